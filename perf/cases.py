"""The work a user of nanoserve_amd has it do, as timed cases through its public entry points
(``Kernels`` and ``Qwen2Runner``): single layers in decode, batched decode and prefill, decode
attention, the calibrated quantizer, and whole decode steps and prompt passes.

A case is a dict of plain values. ``kind`` names the entry point:

  linear  Kernels.w4_linear on the standard W4 format (GEMV for m <= 8, GEMM above)
  mlp     Kernels.w4_linear_swiglu: gate/up projection with the SwiGLU activation
  packed  Kernels.w4_linear_packed on weights repacked once at load time
  attn    Kernels.decode_qkv_attention: one token of one layer over a long KV cache
  gptq    Kernels.w4_gptq: one layer's calibrated quantization
  decode  Qwen2Runner.decode: one token through the model, captured as a graph
  prompt  Qwen2Runner.forward on several tokens, from position 0 or after a cached prefix

Weights are random int4 codes with |N(0, 1)| * 0.02 group scales and activations N(0, 1), as in
this repository's benchmark; whole models are ``Qwen2Runner.random``.
"""
import math

import torch

from nanoserve_amd import gptq
from nanoserve_amd.ops import Kernels
from nanoserve_amd.qwen import Qwen2Runner, Qwen2Shape

BF16 = torch.bfloat16
GROUP = 128
HEAD_DIM = 128

# (hidden, heads, kv heads, intermediate, vocabulary) of the models whose layers the benchmark and
# the tests run: the 7B and 1.5B shapes and a small one.
MODELS = {
    "7b": (3584, 28, 4, 18944, 152064),
    "1.5b": (1536, 12, 2, 8960, 151936),
    "small": (512, 4, 2, 1024, 4096),
}

_kernels = None


def kernels():
    global _kernels
    if _kernels is None:
        _kernels = Kernels()
    return _kernels


def listed():
    return [
        # the smallest call: the 1.5B gate projection for one token, where latency counts
        {"name": "linear decode small", "kind": "linear", "m": 1, "n": 8960, "k": 1536},
        # eight sequences decoding together, the longest rows of the 7B model
        {"name": "linear decode batch 8", "kind": "linear", "m": 8, "n": 3584, "k": 18944},
        # a short, ragged prompt through the 7B q/k/v projection
        {"name": "linear prompt 100", "kind": "linear", "m": 100, "n": 4608, "k": 3584},
        # four sequences decoding together, the 7B gate/up projection and its activation
        {"name": "mlp decode batch 4", "kind": "mlp", "m": 4, "n": 37888, "k": 3584},
        # the largest prompt of the benchmark through the 7B gate/up projection
        {"name": "mlp prompt 2048", "kind": "mlp", "m": 2048, "n": 37888, "k": 3584},
        # sixteen sequences decoding together on weights repacked at load time
        {"name": "packed decode batch 16", "kind": "packed", "m": 16, "n": 37888, "k": 3584},
        # a ragged prompt through the 7B down projection on repacked weights
        {"name": "packed prompt 700", "kind": "packed", "m": 700, "n": 3584, "k": 18944},
        # one layer's attention for one token of a long conversation
        {"name": "attention 16k", "kind": "attn", "heads": 28, "kv": 4, "rows": 16384,
         "pos": 15999},
        # calibrated quantization of the 7B q/k/v projection when a model is loaded
        {"name": "gptq qkv", "kind": "gptq", "n": 4608, "k": 3584},
        # one token at context 1024 through six layers and the head of the 7B model, as a
        # replayed graph (rounding differences grow with depth, so models are cut in depth)
        {"name": "decode step 7b", "kind": "decode", "model": "7b", "layers": 6, "rows": 1024,
         "pos": 1023},
        # a prompt through two layers of the 7B model, its keys and values cached
        {"name": "prompt 1000", "kind": "prompt", "model": "7b", "layers": 2, "t": 1000,
         "pos": 0, "packed": False},
        # the next chunk of a long prompt, attending over what is already cached
        {"name": "prompt chunk 512 at 3000", "kind": "prompt", "model": "7b", "layers": 2,
         "t": 512, "pos": 3000, "packed": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "mlp", "packed", "packed", "attn", "gptq",
                       "decode", "prompt", "prompt"])
    if kind in ("linear", "mlp", "packed"):
        k = 128 * _log_int(rng, 7, 148)
        n = 128 * _log_int(rng, 8, 296)
        if kind == "packed":
            m = _log_int(rng, 2, 2048)
        else:
            m = _log_int(rng, 1, 2048)
        m = min(m, 2048 * 37888 * 3584 // (n * k))  # no more than the largest layer's products
        if kind == "linear" and m <= 8:
            n += rng.randrange(-96, 96)  # decode takes any number of output features
        return {"kind": kind, "m": m, "n": n, "k": k}
    if kind == "attn":
        heads, kv = rng.choice([(28, 4), (12, 2), (32, 8), (16, 16)])
        rows = _log_int(rng, 200, 32768)
        return {"kind": kind, "heads": heads, "kv": kv, "rows": rows,
                "pos": rows - 1 - rng.randrange(0, rows // 4)}
    if kind == "gptq":
        return {"kind": kind, "n": _log_int(rng, 300, 4600), "k": 128 * _log_int(rng, 4, 28)}
    model = rng.choice(["7b", "1.5b", "small"])
    layers = rng.randrange(1, 3)
    if kind == "decode":
        layers *= 2
        rows = _log_int(rng, 64, 8192)
        return {"kind": kind, "model": model, "layers": layers, "rows": rows,
                "pos": rows - 1 - rng.randrange(0, rows // 4)}
    return {"kind": kind, "model": model, "layers": layers, "t": _log_int(rng, 9, 900),
            "pos": rng.choice([0, _log_int(rng, 16, 4096)]), "packed": rng.random() < 0.5}


# ---------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *size, std=1.0):
    return (torch.randn(*size, generator=g, device="cuda") * std).to(BF16)


def _weights(g, n, k):
    """Random int4 codes [n, k / 8] and scales [n, k / 128] of the standard W4 format."""
    wq = torch.randint(-(1 << 31), 1 << 31, (n, k // 8), generator=g, device="cuda",
                       dtype=torch.int64).to(torch.int32)
    s = (torch.randn(n, k // GROUP, generator=g, device="cuda").abs() * 0.02).to(BF16)
    return wq, s


def _shape(case):
    hidden, heads, kv, inter, vocab = MODELS[case["model"]]
    return Qwen2Shape(layers=case["layers"], hidden=hidden, heads=heads, kv_heads=kv,
                      intermediate=inter, vocab=vocab)


def _inputs(case, seed):
    """The tensors of a case, without any plan made from them."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("linear", "mlp", "packed"):
        wq, s = _weights(g, case["n"], case["k"])
        return {"x": _randn(g, case["m"], case["k"]), "wq": wq, "s": s}
    if kind == "attn":
        hq, hk, rows = case["heads"], case["kv"], case["rows"]
        inv = 1.0 / (1e6 ** (torch.arange(0, HEAD_DIM, 2, device="cuda").float() / HEAD_DIM))
        return {"qkv": _randn(g, (hq + 2 * hk) * HEAD_DIM),
                "bias": _randn(g, (hq + 2 * hk) * HEAD_DIM, std=0.02), "inv": inv,
                "kc": _randn(g, hk, rows, HEAD_DIM), "vc": _randn(g, hk, rows, HEAD_DIM),
                "pos": torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")}
    if kind == "gptq":
        w = _randn(g, case["n"], case["k"], std=0.02)
        # activations of a real layer are correlated across features
        mix = torch.randn(64, case["k"], generator=g, device="cuda")
        x = (torch.randn(512, 64, generator=g, device="cuda") @ mix / 8
             + torch.randn(512, case["k"], generator=g, device="cuda"))
        return {"w": w, "u": gptq.hessian_factor(gptq.hessian(x))[0]}
    shape = _shape(case)
    runner = Qwen2Runner.random(shape, seed=seed, kernels=kernels())
    t = case["t"] if kind == "prompt" else 1
    runner.alloc_cache(case["pos"] + t if kind == "prompt" else case["rows"])
    filled = case["pos"]
    for cache in (runner.cache_k, runner.cache_v):
        cache.zero_()
        if filled:
            cache[:, :, :filled] = _randn(g, shape.layers, shape.kv_heads, filled, HEAD_DIM)
    ids = torch.randint(0, shape.vocab, (t,), generator=g, device="cuda")
    return {"runner": runner, "ids": ids}


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"], st["k"] = case, kernels()
    kind = case["kind"]
    if kind == "linear":
        st["work"] = st["k"].w4_linear_workspace(case["m"], case["n"], case["k"])
    elif kind == "packed":
        st["wp"], st["sp"] = st["k"].w4_repack(st["wq"], st["s"])
        del st["wq"], st["s"]
    elif kind == "attn":
        st["work"] = st["k"].decode_attention_workspace(case["heads"], case["kv"], HEAD_DIM,
                                                        case["rows"])
    elif kind == "decode":
        # warm-up and capture write the cache's last row: keep what was there
        r = st["runner"]
        last = [c[:, :, -1].clone() for c in (r.cache_k, r.cache_v)]
        r.capture_decode()
        for c, row in zip((r.cache_k, r.cache_v), last):
            c[:, :, -1] = row
    elif kind == "prompt" and case["packed"]:
        st["runner"].pack_prefill()
    return st


# ---------------------------------------------------------------------------------- one pass
def run(st):
    case, k = st["case"], st["k"]
    kind = case["kind"]
    if kind == "linear":
        return k.w4_linear(st["x"], st["wq"], st["s"], GROUP, work=st["work"])
    if kind == "mlp":
        return k.w4_linear_swiglu(st["x"], st["wq"], st["s"], GROUP)
    if kind == "packed":
        return k.w4_linear_packed(st["x"], st["wp"], st["sp"], case["n"])
    if kind == "attn":
        out = k.decode_qkv_attention(st["qkv"], st["bias"], st["inv"], st["pos"], st["kc"],
                                     st["vc"], case["heads"], case["kv"], HEAD_DIM, st["work"])
        return {"out": out, "k": st["kc"][:, case["pos"]], "v": st["vc"][:, case["pos"]]}
    if kind == "gptq":
        wq, s = k.w4_gptq(st["w"], st["u"])
        return {"wq": wq, "s": s}
    r, p = st["runner"], case["pos"]
    if kind == "decode":
        logits = r.decode(st["ids"], p)
        return {"logits": logits, "k": r.cache_k[:, :, p], "v": r.cache_v[:, :, p]}
    t = case["t"]
    logits = r.forward(st["ids"], p, use_cache=True, last_only=True)
    return {"logits": logits, "k": r.cache_k[:, :, p:p + t], "v": r.cache_v[:, :, p:p + t]}


# ---------------------------------------------------------------------------------- needed work
def _linear_bytes(m, n, k, n_out):
    return n * k // 2 + 2 * n * (k // GROUP) + 2 * m * k + 2 * m * n_out


def work(case):
    kind = case["kind"]
    if kind in ("linear", "mlp", "packed"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _linear_bytes(m, n, k, n // 2 if kind == "mlp" else n),
                "flops": 2 * m * n * k}
    if kind == "attn":
        hq, hk, n = case["heads"], case["kv"], case["pos"] + 1
        return {"bytes": 4 * hk * n * HEAD_DIM + 4 * (hq + hk) * HEAD_DIM * 2,
                "flops": 4 * hq * n * HEAD_DIM}
    if kind == "gptq":
        n, k = case["n"], case["k"]
        return {"bytes": 2 * n * k + 2 * k * k + n * k // 2 + 2 * n * (k // GROUP),
                "flops": n * k * k}
    s = _shape(case)
    t = case["t"] if kind == "prompt" else 1
    p = case["pos"]
    qkv, hd = s.qkv_rows, s.heads * HEAD_DIM
    mats = ((qkv, s.hidden), (s.hidden, hd), (2 * s.intermediate, s.hidden),
            (s.hidden, s.intermediate))
    params = sum(n * k for n, k in mats)
    nbytes = s.layers * (sum(n * k // 2 + 2 * n * (k // GROUP) for n, k in mats)
                         + 4 * s.kv_heads * HEAD_DIM * (p + t))
    nbytes += 2 * s.vocab * s.hidden + 2 * t * s.hidden + 2 * s.vocab
    pairs = t * p + t * (t + 1) // 2  # query-key pairs under the causal mask
    flops = s.layers * (2 * t * params + 4 * s.heads * HEAD_DIM * pairs)
    flops += 2 * s.vocab * s.hidden
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Measured as about four times the error of the outputs against ``exact`` (a bf16 output is
    rounded with a relative error of 1.7e-3 root mean square; GEMMs stage bf16 weights; whole
    models round every activation)."""
    kind = case["kind"]
    if kind == "gptq":
        return "exact"
    if kind in ("linear", "mlp", "packed", "attn"):
        return {"rel": 1e-2, "max": 0.1}
    return {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------------------------- 64 bits
def _deq(wq, s):
    """The weights (q - 8) * s of rows of the standard W4 format, in 64 bits."""
    sh = torch.arange(0, 32, 4, device=wq.device, dtype=torch.int32)
    q = ((wq[:, :, None] >> sh) & 15).reshape(wq.shape[0], -1).double() - 8
    return (q.view(q.shape[0], -1, GROUP) * s.double()[:, :, None]).view(q.shape[0], -1)


def _lin(x, wq, s, rows=4096):
    return torch.cat([x @ _deq(wq[i:i + rows], s[i:i + rows]).t()
                      for i in range(0, wq.shape[0], rows)], dim=1)


def _swiglu(y):
    """silu(gate) * up of columns interleaved in blocks of 8 gate, 8 up."""
    y = y.view(y.shape[0], -1, 2, 8)
    return (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(y.shape[0], -1)


def _norm(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos, inv_freq):
    """x [t, heads, d] rotated at positions pos [t]."""
    a = pos.double()[:, None] * inv_freq.double()
    c, s = a.cos()[:, None], a.sin()[:, None]
    lo, hi = x.chunk(2, dim=-1)
    return torch.cat([lo * c - hi * s, hi * c + lo * s], dim=-1)


def _attend(q, k, v, pos):
    """q [t, hq, d] at positions pos over k, v [hk, n, d], causal; returns [t, hq * d]."""
    t, hq, d = q.shape
    hk, n, _ = k.shape
    out = torch.empty(t, hq, d, dtype=torch.float64, device=q.device)
    mask = torch.arange(n, device=q.device)[None] > pos[:, None]
    for h in range(hq):
        g = h // (hq // hk)
        sc = (q[:, h] @ k[g].t()) / math.sqrt(d)
        out[:, h] = torch.softmax(sc.masked_fill(mask, float("-inf")), -1) @ v[g]
    return out.reshape(t, hq * d)


def _head_rows(w, x, rows=16384):
    return torch.cat([x @ w[i:i + rows].double().t() for i in range(0, w.shape[0], rows)], dim=1)


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "gptq":
        return None  # whole numbers: the codes follow from the order of the updates
    st = _inputs(case, seed)
    if kind in ("linear", "mlp", "packed"):
        y = _lin(st["x"].double(), st["wq"], st["s"])
        return _swiglu(y) if kind == "mlp" else y
    if kind == "attn":
        hq, hk, p = case["heads"], case["kv"], case["pos"]
        qkv = (st["qkv"].double() + st["bias"].double()).view(1, hq + 2 * hk, HEAD_DIM)
        qk, v = qkv[:, :hq + hk], qkv[0, hq + hk:]
        qk = _rope(qk, st["pos"], st["inv"])
        kc, vc = st["kc"][:, :p + 1].double(), st["vc"][:, :p + 1].double()
        kc[:, p], vc[:, p] = qk[0, hq:], v
        return {"out": _attend(qk[:, :hq], kc, vc, st["pos"]), "k": kc[:, p], "v": vc[:, p]}
    r, ids, p = st["runner"], st["ids"], case["pos"]
    s, t = r.shape, ids.shape[0]
    hq, hk = s.heads, s.kv_heads
    pos = torch.arange(p, p + t, device="cuda")
    x = r.embed[ids].double()
    ks, vs = [], []
    for li, layer in enumerate(r.layers):
        qkv = _lin(_norm(x, layer["ln_in"], s.eps), *layer["wqkv"])
        if layer["bqkv"] is not None:
            qkv += layer["bqkv"].double()
        qkv = qkv.view(t, hq + 2 * hk, HEAD_DIM)
        qk, v = _rope(qkv[:, :hq + hk], pos, r.inv_freq), qkv[:, hq + hk:]
        ks.append(qk[:, hq:].transpose(0, 1))
        vs.append(v.transpose(0, 1))
        kc = torch.cat([r.cache_k[li, :, :p].double(), ks[-1]], dim=1)
        vc = torch.cat([r.cache_v[li, :, :p].double(), vs[-1]], dim=1)
        x = x + _lin(_attend(qk[:, :hq], kc, vc, pos), *layer["wo"])
        h = _swiglu(_lin(_norm(x, layer["ln_post"], s.eps), *layer["wgu"]))
        x = x + _lin(h, *layer["wd"])
    logits = _head_rows(r.lm_head, _norm(x[-1:], r.final_norm, s.eps))
    k, v = torch.stack(ks), torch.stack(vs)
    if kind == "decode":
        k, v = k[:, :, 0], v[:, :, 0]
    return {"logits": logits, "k": k, "v": v}
