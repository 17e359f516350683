"""W4A16 Qwen2 decoder on the nanoserve_amd kernels: the caller of the W4 linear layers.

Counterpart of the reference's ``Qwen2Runner`` (python/nanoserve/qwen.py:43-177) with its
options fixed to the fast path (``w4=True``, fused norm / rope / swiglu kernels). Batch 1.

Data flow of one layer, as this runner schedules it: the residual stream enters the q/k/v
projection through a fused add + RMSNorm (the first layer has nothing to add yet); the
attention writes its head outputs, which the o projection consumes; the o output is the addend
that the gate/up projection's fused add + RMSNorm folds into the residual stream; SwiGLU is
applied as the gate/up projection writes its output; the down projection's output is the
addend the next layer's q/k/v projection (or, after the last layer, the final norm in front of
the bf16 lm_head) folds in. Embedding and lm_head stay bf16 as in the reference.

Two differences of layout, not of arithmetic: q/k/v and gate/up are each one W4 projection
(quantization is per row and per 128-column group, so stacking rows before quantizing gives
the same codes and scales as quantizing them one by one), and a one-token decode step runs
on device-resident token id and position (``decode``), so the whole step is captured once as
a HIP graph and replayed for every token (``capture_decode``).

Kernels used per decode step and layer: ns_w4_gemv_decode x3 (the q/k/v and gate/up GEMVs
with the residual add + RMSNorm fused into their activation load, SwiGLU fused into the
gate/up GEMV's output; the down GEMV), ns_decode_qkv_attention (bias + RoPE + KV append +
grouped-query attention over the cache, splits left unmerged) and ns_w4_gemv_decode_attn
(the o GEMV, merging the attention's splits while loading its activation). The gate/up weight
rows are stored interleaved in blocks of 8 (``interleave_gate_up``) so that a gate row and its
up row land in the same 16-row group. The prompt pass (T > 1) uses ns_w4_linear (GEMM for
T > 8) and ns_w4_linear_swiglu, ns_rmsnorm, ns_prompt_qkv (bias + RoPE + KV append) and
ns_prompt_attention (causal attention on matrix cores; PyTorch SDPA for head sizes other than
128); after ``pack_prefill`` prompts of more than 16 tokens run the packed-format GEMMs instead
(ns_w4_linear_packed, ns_w4_linear_packed_swiglu).

No weights are downloaded: ``random`` builds a model of any Qwen2 shape with seeded random
weights (quantized by ns_w4_quantize), ``from_hf`` quantizes a Hugging Face Qwen2 model's
weights.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.nn.functional as F
from torch.nn.attention import SDPBackend, sdpa_kernel

from . import gptq
from .ops import Kernels

# Cache rows per split of the library's decode attention (its workspace grows by one split
# every ATTN_SPLIT_ROWS rows; tests/test_abi.py checks the two agree).
ATTN_SPLIT_ROWS = 128


@dataclass(frozen=True)
class Qwen2Shape:
    """Architecture sizes; defaults are Qwen2.5-7B (hidden 3584, 28 layers, 28 query / 4 kv
    heads of 128, intermediate 18944, vocabulary 152064, rope theta 1e6)."""
    layers: int = 28
    hidden: int = 3584
    heads: int = 28
    kv_heads: int = 4
    head_dim: int = 128
    intermediate: int = 18944
    vocab: int = 152064
    eps: float = 1e-6
    rope_theta: float = 1000000.0
    qkv_bias: bool = True
    group: int = 128

    @property
    def qkv_rows(self) -> int:
        return (self.heads + 2 * self.kv_heads) * self.head_dim

    def w4_bytes_per_layer(self) -> int:
        """Bytes of int4 codes + bf16 scales one layer's four projections read."""
        def lin(n, k):
            return n * k // 2 + n * (k // self.group) * 2
        H, I = self.hidden, self.intermediate
        return (lin(self.qkv_rows, H) + lin(H, self.heads * self.head_dim) + lin(2 * I, H)
                + lin(H, I))

    def decode_bytes(self, context: int) -> int:
        """Bytes one decode step must read at least: every W4 projection, the bf16 lm_head and
        the KV cache rows of ``context`` positions (embedding row, norms and activations are
        negligible and not counted)."""
        kv = 2 * self.layers * self.kv_heads * context * self.head_dim * 2
        return self.layers * self.w4_bytes_per_layer() + self.vocab * self.hidden * 2 + kv


def interleave_gate_up(Wq: torch.Tensor, S: torch.Tensor):
    """Row order of the fused gate/up projection used by the decode GEMV's SwiGLU output: rows
    16b .. 16b+7 are gate rows 8b .. 8b+7 and rows 16b+8 .. 16b+15 the up rows 8b .. 8b+7
    (gate rows 0 .. I-1 then up rows I .. 2I-1 on input). Rows are whole quantized rows, so
    codes and scales move together and nothing is re-quantized."""
    N = Wq.shape[0]
    if N % 16:
        raise ValueError("gate/up interleave needs the intermediate size to be a multiple of 8")

    def perm(t):
        return t.view(2, N // 16, 8, t.shape[1]).transpose(0, 1).reshape(N, t.shape[1]).contiguous()

    return perm(Wq), perm(S)


def _plain_rope_theta(cfg) -> float:
    """RoPE base of a Hugging Face Qwen2 config; only unscaled ("default") RoPE is supported.

    Transformers has kept these settings in three places over its versions: a ``rope_theta``
    attribute, a ``rope_scaling`` dict (whose kind is ``rope_type`` or the older ``type``) and a
    ``rope_parameters`` dict. Every dict present is checked for a scaled kind; the first base
    found in ``rope_parameters``, ``rope_scaling`` or the attribute, in that order, is used, and
    10000 when none is set."""
    specs = [d for d in (getattr(cfg, "rope_parameters", None), getattr(cfg, "rope_scaling", None))
             if isinstance(d, dict)]
    kinds = {d.get("rope_type", d.get("type")) for d in specs} - {None, "default"}
    if kinds:
        raise NotImplementedError(f"scaled RoPE ({', '.join(sorted(map(str, kinds)))}) is not supported")
    bases = [d.get("rope_theta") for d in specs] + [getattr(cfg, "rope_theta", None)]
    return float(next((b for b in bases if b), 10000.0))


def _kernel_operand(t: torch.Tensor, shape) -> bool:
    """Whether the one-launch operators of the prompt pass take this bias or output head: bf16,
    contiguous, 16-byte aligned. PyTorch's operators take the others."""
    return (t.dtype is torch.bfloat16 and t.shape == shape and t.is_contiguous()
            and t.data_ptr() % 16 == 0)


def _calibration_hessians(hf_model, calib_ids: torch.Tensor) -> dict:
    """Run the HF model on calib_ids and return {(layer, stack): H} with H = 2 X^T X / T
    (float64, on the model's device) of the inputs X of each stack of linear layers that share
    an input (wqkv: q/k/v_proj, wo: o_proj, wgu: gate/up_proj, wd: down_proj)."""
    ids = calib_ids if calib_ids.ndim == 2 else calib_ids[None]
    sums: dict = {}
    hooks = []

    def hook(key):
        def fn(_mod, args):
            x = args[0].detach().reshape(-1, args[0].shape[-1]).to(torch.float64)
            s, n = sums.get(key, (0.0, 0))
            sums[key] = (s + x.t() @ x, n + x.shape[0])
        return fn

    for li, layer in enumerate(hf_model.model.layers):
        for name, mod in (("wqkv", layer.self_attn.q_proj), ("wo", layer.self_attn.o_proj),
                          ("wgu", layer.mlp.gate_proj), ("wd", layer.mlp.down_proj)):
            hooks.append(mod.register_forward_pre_hook(hook((li, name))))
    try:
        with torch.no_grad():
            hf_model(ids.to(next(hf_model.parameters()).device))
    finally:
        for h in hooks:
            h.remove()
    return {key: (2.0 / n) * s for key, (s, n) in sums.items()}


class Qwen2Runner:
    """W4A16 Qwen2 runner. Build with ``random`` or ``from_hf``; ``forward`` / ``generate`` have
    the reference's signatures and semantics (qwen.py:137-177)."""

    def __init__(self, shape: Qwen2Shape, embed, final_norm, lm_head, layers,
                 kernels: Kernels | None = None):
        self.shape = shape
        self.k = kernels or Kernels()
        self.embed, self.final_norm, self.lm_head = embed, final_norm, lm_head
        self.layers = layers
        # the RMSNorm weight applied after layer i: layer i + 1's input norm, the final norm last
        self.norm_after = [L["ln_in"] for L in layers[1:]] + [final_norm]
        self.dev = embed.device
        D = shape.head_dim
        if shape.heads % shape.kv_heads:
            raise ValueError("heads must be a multiple of kv_heads")
        # reference qwen.py:64-65: theta^(-2i/D) in fp32 from int64 exponents
        self.inv_freq = 1.0 / (shape.rope_theta ** (
            torch.arange(0, D, 2, dtype=torch.int64, device=self.dev).float() / D))
        self.cache_k = self.cache_v = None
        self.max_len = 0
        self.graph = None
        # one-token decode state: device-resident token id and position, static activations
        H, I = shape.hidden, shape.intermediate
        bf = dict(dtype=torch.bfloat16, device=self.dev)
        self.tok = torch.zeros(1, dtype=torch.int32, device=self.dev)
        self.pos = torch.zeros(1, dtype=torch.int32, device=self.dev)
        # the step's rotation table (cos, sin of pos * inv_freq), written by decode_embed
        self.rot = torch.empty(2, D // 2, dtype=torch.float32, device=self.dev)
        self.x = torch.empty(1, H, **bf)
        self.x2 = torch.empty(1, H, **bf)
        self.h = torch.empty(1, H, **bf)
        self.o = torch.empty(1, H, **bf)
        self.d = torch.empty(1, H, **bf)
        self.qkv = torch.empty(1, shape.qkv_rows, **bf)
        self.attn = torch.empty(1, shape.heads * D, **bf)
        self.act = torch.empty(1, I, **bf)
        self.logits = torch.empty(1, shape.vocab, **bf)
        self.work = None
        self.packed = None  # per layer {name: (Wp, Sp, N)} once pack_prefill has run

    # ------------------------------------------------------------------ construction
    @classmethod
    def random(cls, shape: Qwen2Shape = Qwen2Shape(), device="cuda", seed: int = 0,
               std: float = 0.02, kernels: Kernels | None = None) -> "Qwen2Runner":
        """Seeded random weights: linear and embedding weights N(0, std) in bf16, quantized with
        ns_w4_quantize; biases N(0, std); norm weights 1 + N(0, 0.05)."""
        k = kernels or Kernels()
        g = torch.Generator(device=device)
        g.manual_seed(seed)
        bf = torch.bfloat16

        def randn(*size, scale=std):
            return (torch.randn(*size, generator=g, device=device) * scale).to(bf)

        def norm_w():
            return (1.0 + torch.randn(shape.hidden, generator=g, device=device) * 0.05).to(bf)

        H, I, D = shape.hidden, shape.intermediate, shape.head_dim
        layers = []
        for _ in range(shape.layers):
            L = {"ln_in": norm_w(), "ln_post": norm_w(),
                 "bqkv": randn(shape.qkv_rows) if shape.qkv_bias else None}
            for name, (n, kk) in (("wqkv", (shape.qkv_rows, H)), ("wo", (H, shape.heads * D)),
                                  ("wgu", (2 * I, H)), ("wd", (H, I))):
                W = randn(n, kk)
                L[name] = k.w4_quantize(W, shape.group)
                del W
            L["wgu"] = interleave_gate_up(*L["wgu"])
            layers.append(L)
        embed = randn(shape.vocab, H)
        lm_head = randn(shape.vocab, H)
        return cls(shape, embed, norm_w(), lm_head, layers, k)

    @classmethod
    def from_hf(cls, hf_model, device="cuda", group: int = 128,
                kernels: Kernels | None = None, calib_ids: torch.Tensor | None = None,
                damp: float = 0.01) -> "Qwen2Runner":
        """Quantize a Hugging Face Qwen2ForCausalLM's weights (as the reference's
        Qwen2Runner.__init__ + quantize, qwen.py:43-99; default, unscaled RoPE only).

        Without ``calib_ids`` every linear layer is quantized by round to nearest, as the
        reference does. With ``calib_ids`` (token ids [B, T] or [T]) the HF model is run once on
        them, the inputs of every linear layer are accumulated into that layer's Hessian
        2 X^T X / T (float64), and each layer is quantized by GPTQ (``nanoserve_amd.gptq``) into
        the same format: the calibrated quantizer the reference names as its next step
        (README.md:233-235). The activations come from the unquantized model."""
        cfg = hf_model.config
        k = kernels or Kernels()
        theta = _plain_rope_theta(cfg)
        D = getattr(cfg, "head_dim", None) or cfg.hidden_size // cfg.num_attention_heads
        m = hf_model.model
        at0 = m.layers[0].self_attn
        shape = Qwen2Shape(layers=len(m.layers), hidden=cfg.hidden_size,
                           heads=cfg.num_attention_heads, kv_heads=cfg.num_key_value_heads,
                           head_dim=D, intermediate=cfg.intermediate_size,
                           vocab=m.embed_tokens.weight.shape[0], eps=cfg.rms_norm_eps,
                           rope_theta=float(theta), qkv_bias=at0.q_proj.bias is not None,
                           group=group)

        def bf(t):
            return t.detach().to(device=device, dtype=torch.bfloat16).contiguous()

        hess = _calibration_hessians(hf_model, calib_ids) if calib_ids is not None else None

        def quantize(li, name, ws):
            W = bf(torch.cat([w.detach() for w in ws]))
            if hess is None:
                return k.w4_quantize(W, group)
            return gptq.quantize_layer(k, W, H=hess[(li, name)], group=group, damp=damp)

        layers = []
        for li, layer in enumerate(m.layers):
            at, mlp = layer.self_attn, layer.mlp
            L = {"ln_in": bf(layer.input_layernorm.weight),
                 "ln_post": bf(layer.post_attention_layernorm.weight),
                 "bqkv": (bf(torch.cat([at.q_proj.bias, at.k_proj.bias, at.v_proj.bias]))
                          if shape.qkv_bias else None)}
            stacks = {"wqkv": [at.q_proj.weight, at.k_proj.weight, at.v_proj.weight],
                      "wo": [at.o_proj.weight],
                      "wgu": [mlp.gate_proj.weight, mlp.up_proj.weight],
                      "wd": [mlp.down_proj.weight]}
            for name, ws in stacks.items():
                L[name] = quantize(li, name, ws)
            L["wgu"] = interleave_gate_up(*L["wgu"])
            layers.append(L)
        return cls(shape, bf(m.embed_tokens.weight), bf(m.norm.weight),
                   bf(hf_model.lm_head.weight), layers, k)

    # ------------------------------------------------------------------ cache
    def alloc_cache(self, max_len: int):
        """KV cache [layers, kv_heads, max_len, head_dim] bf16 for K and for V (reference
        qwen.py:114-117), and the decode-attention workspace. Drops a captured graph."""
        s = self.shape
        shape = (s.layers, s.kv_heads, max_len, s.head_dim)
        self.cache_k = torch.empty(shape, dtype=torch.bfloat16, device=self.dev)
        self.cache_v = torch.empty_like(self.cache_k)
        self.max_len = max_len
        self.work = self.k.decode_attention_workspace(s.heads, s.kv_heads, s.head_dim, max_len,
                                                      device=self.dev)
        # Up to 16 cache splits the o projection merges the attention's splits in its own
        # activation load; past that every o workgroup would read every split's partials, and
        # the attention's merge kernel followed by the plain o GEMV is faster (MI355X, 28-layer
        # 7B step at its last position: 1.384 against 1.411 ms at 1024 rows, 1.416 against
        # 1.410 at 2048, 1.552 against 1.416 at 4096, 2.399 against 1.693 at 16384).
        self.merge_in_o = max_len <= 16 * ATTN_SPLIT_ROWS
        self.graph = None

    # ------------------------------------------------------------------ one-token decode step
    def _decode_body(self):
        """One decode step on self.tok / self.pos (device tensors) into self.logits. Launches
        only; no allocation, no host synchronisation, so it can be captured.

        First ns_decode_embed: the token's embedding row, and the position's rotation table,
        which every layer's attention then reads instead of computing the angles itself.
        Per layer five kernels: the q/k/v GEMV with the residual add + input RMSNorm fused
        into its activation load, the attention (bias + RoPE + KV append + attention over
        128-row splits of the cache), the o GEMV, which merges the attention's splits as it
        loads its activation (for caches of more than 16 splits the attention's own merge
        kernel merges them and the o GEMV is the plain one), the gate/up GEMV with the post-attention add + RMSNorm fused in
        and SwiGLU fused into its output, and the down GEMV. The residual stream alternates between two
        buffers (a fused GEMV reads one and one of its workgroups writes the other)."""
        s, k = self.shape, self.k
        D, G, eps = s.head_dim, s.group, s.eps
        k.decode_embed(self.tok, self.pos, self.embed, self.inv_freq, x=self.x, rot=self.rot)
        resid, spare = self.x, self.x2
        pending = None  # the addend not yet in the residual stream (the last down output)
        for li, L in enumerate(self.layers):
            if pending is None:
                k.gemv_decode(*L["wqkv"], G, res=resid, norm_w=L["ln_in"], eps=eps, out=self.qkv)
            else:
                k.gemv_decode(*L["wqkv"], G, res=resid, r=pending, norm_w=L["ln_in"], eps=eps,
                              res_out=spare, out=self.qkv)
                resid, spare = spare, resid
            k.decode_qkv_attention(self.qkv[0], L["bqkv"], self.inv_freq, self.pos,
                                   self.cache_k[li], self.cache_v[li], s.heads, s.kv_heads, D,
                                   self.work, out=self.attn, merge=not self.merge_in_o,
                                   rot=self.rot)
            if self.merge_in_o:
                k.gemv_decode_attn(self.attn, self.work, self.pos, self.max_len, s.heads,
                                   *L["wo"], G, out=self.o)
            else:
                k.gemv_decode(*L["wo"], G, x=self.attn, out=self.o)
            k.gemv_decode(*L["wgu"], G, res=resid, r=self.o, norm_w=L["ln_post"], eps=eps,
                          res_out=spare, swiglu=True, out=self.act)
            resid, spare = spare, resid
            k.gemv_decode(*L["wd"], G, x=self.act, out=self.d)
            pending = self.d
        k.bf16_gemv(self.lm_head, res=resid, r=pending, norm_w=self.final_norm, eps=eps,
                    out=self.logits)

    def _set_step(self, token, pos: int):
        if self.cache_k is None:
            raise RuntimeError("alloc_cache first")
        if not 0 <= pos < self.max_len:
            raise ValueError(f"position {pos} outside the cache (max_len {self.max_len})")
        if isinstance(token, torch.Tensor):
            self.tok.copy_(token.reshape(1))
        else:
            self.tok.fill_(int(token))
        self.pos.fill_(pos)

    def capture_decode(self):
        """Capture one decode step as a HIP graph (replayed by ``decode``). The warm-up runs
        and the capture write cache row max_len - 1, which a step at that position rewrites
        before reading it."""
        if self.cache_k is None:
            raise RuntimeError("alloc_cache first")
        self.pos.fill_(self.max_len - 1)
        side = torch.cuda.Stream(device=self.dev)
        side.wait_stream(torch.cuda.current_stream(self.dev))
        with torch.cuda.stream(side):
            for _ in range(2):
                self._decode_body()
        torch.cuda.current_stream(self.dev).wait_stream(side)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            self._decode_body()
        self.graph = g

    @torch.no_grad()
    def decode(self, token, pos: int) -> torch.Tensor:
        """Logits [1, vocab] of one token at position ``pos``, attending over cache rows
        0 .. pos (the token's own k / v are appended at row pos). Replays the captured graph
        when there is one. Returns the runner's own logits buffer (overwritten by the next
        step)."""
        self._set_step(token, pos)
        if self.graph is not None:
            self.graph.replay()
        else:
            self._decode_body()
        return self.logits

    # ------------------------------------------------------------------ prompt pass
    def pack_prefill(self):
        """Keep a second copy of every layer's W4 weights in the packed tile format
        (ns_w4_repack), so that prompt passes of more than 16 tokens run the packed-format GEMMs
        (w4_linear_packed; w4_linear_packed_swiglu for gate/up): same numerics as the standard
        GEMMs (bf16-staged weights), faster on MI355X. Decode keeps the standard copies, whose
        M = 1 kernels are the faster ones. Costs the W4 bytes once more in device memory (about
        3.4 GB for Qwen2.5-7B). Returns self."""
        if self.shape.group != 128:
            raise ValueError("the packed tile format has group size 128")
        self.packed = []
        for L in self.layers:
            P = {}
            for name in ("wqkv", "wo", "wgu", "wd"):
                Wq, S = L[name]
                P[name] = (*self.k.w4_repack(Wq, S), Wq.shape[0])
            self.packed.append(P)
        return self

    def _prompt_attention_kernel_ok(self, T, pos0, cached):
        """Whether ns_prompt_attention takes this chunk: head size 128, and its limits over the rows
        that hold the keys (the cache's or, without a cache, the projection's)."""
        s = self.shape
        return s.head_dim == 128 and self.k.prompt_attention_fits(
            T, s.heads, s.kv_heads, pos0, s.head_dim if cached else s.qkv_rows)

    def _prompt_attention(self, q, k, v, pos0, li):
        """Causal attention of T query tokens at positions pos0 .. pos0+T-1 over cache / prompt
        keys (PyTorch) where ns_prompt_attention does not apply, returned as bf16 [T, Hq*D]. A
        prompt from position 0 runs the fused SDPA
        kernel (flash or memory-efficient backend: fp32 scores, softmax and sums) on the bf16
        q / k / v with the causal flag; the math backend, whose batched bf16 products are not
        used here, is excluded, and where no fused kernel takes the shape the fp32 path runs.
        A chunk after cached positions (pos0 > 0) attends in fp32 with an explicit mask."""
        s = self.shape
        T, D = q.shape[0], s.head_dim
        rep = s.heads // s.kv_heads
        if pos0 == 0:
            qb = q.reshape(T, s.heads, D).transpose(0, 1).contiguous()
            kb = k.reshape(T, s.kv_heads, D).transpose(0, 1).repeat_interleave(rep, dim=0).contiguous()
            vb = v.reshape(T, s.kv_heads, D).transpose(0, 1).repeat_interleave(rep, dim=0).contiguous()
            try:
                with sdpa_kernel([SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION]):
                    o = F.scaled_dot_product_attention(qb[None], kb[None], vb[None], is_causal=True)
                return o[0].transpose(0, 1).reshape(T, s.heads * D)
            except RuntimeError as e:
                if "No available kernel" not in str(e):
                    raise
                # no fused kernel for this shape: the fp32 path below
        qh = q.reshape(T, s.heads, D).transpose(0, 1).float().contiguous()
        if pos0 == 0:
            kh = k.reshape(T, s.kv_heads, D).transpose(0, 1).float()
            vh = v.reshape(T, s.kv_heads, D).transpose(0, 1).float()
        else:
            kh = self.cache_k[li, :, :pos0 + T].float()
            vh = self.cache_v[li, :, :pos0 + T].float()
        kh = kh.repeat_interleave(rep, dim=0).contiguous()
        vh = vh.repeat_interleave(rep, dim=0).contiguous()
        n = kh.shape[1]
        qpos = torch.arange(pos0, pos0 + T, device=q.device)[:, None]
        mask = torch.arange(n, device=q.device)[None, :] <= qpos
        o = F.scaled_dot_product_attention(qh[None], kh[None], vh[None], attn_mask=mask)
        return o[0].transpose(0, 1).reshape(T, s.heads * D).to(torch.bfloat16)

    @torch.no_grad()
    def forward(self, ids, pos0: int = 0, use_cache: bool = False, last_only: bool = False):
        """ids: [T] token ids at positions pos0 .. pos0+T-1; returns logits [T, vocab] (or
        [1, vocab] with ``last_only``). Reference qwen.py:137-164. A one-token call with
        pos0 > 0 is a decode step (cache required, its k / v row is always stored); other
        calls attend causally over the prompt (and, for pos0 > 0, the cache)."""
        s, k = self.shape, self.k
        T = ids.shape[0]
        if T == 1 and pos0 > 0:
            logits = self.decode(ids.reshape(1), pos0)
            return logits.clone()
        if (use_cache or pos0 > 0) and (self.cache_k is None or pos0 + T > self.max_len):
            raise RuntimeError("cache too small: alloc_cache(max_len) first")
        if T == 0:
            return self.embed.new_empty((0, s.vocab))
        D, G = s.head_dim, s.group
        qn, kn = s.heads * D, s.kv_heads * D
        x = self.embed.index_select(0, ids.to(self.dev)).contiguous()
        h = k.rmsnorm(x, None, self.layers[0]["ln_in"], s.eps)
        packed = self.packed is not None and T > 16

        def lin(a, li, name):
            if packed:
                return k.w4_linear_packed(a, *self.packed[li][name])
            return k.w4_linear(a, *self.layers[li][name], G)

        def gate_up_swiglu(a, li):  # gate/up rows interleaved by 8
            if packed:
                return k.w4_linear_packed_swiglu(a, *self.packed[li]["wgu"])
            return k.w4_linear_swiglu(a, *self.layers[li]["wgu"], G)

        cached = use_cache or pos0 > 0
        in_kernel = self._prompt_attention_kernel_ok(T, pos0, cached)
        # one workspace for the pass: the layers' launches follow each other on one stream
        work = (k.prompt_attention_workspace(T, s.heads, s.kv_heads, pos0, device=self.dev)
                if in_kernel else None)

        def attention(qkv, bias, li):
            """Bias, RoPE, KV append and attention of the fused projection's output."""
            caches = (self.cache_k[li], self.cache_v[li]) if cached else (None, None)
            if bias is not None and not _kernel_operand(bias, (s.qkv_rows,)):
                qkv += bias
                bias = None
            k.prompt_qkv(qkv, bias, self.inv_freq, s.heads, s.kv_heads, D, pos0, *caches)
            q, kk, v = qkv[:, :qn], qkv[:, qn:qn + kn], qkv[:, qn + kn:]
            if not in_kernel:
                if cached and pos0 == 0:  # the rotated heads of this chunk are in the cache
                    kk, v = (c[:, :T].transpose(0, 1).reshape(T, kn) for c in caches)
                return self._prompt_attention(q, kk, v, pos0, li)
            if not cached:
                caches = (x.unflatten(1, (s.kv_heads, D)).transpose(0, 1) for x in (kk, v))
            return k.prompt_attention(q, *caches, s.heads, pos0, work=work)

        for li, L in enumerate(self.layers):
            a = attention(lin(h, li, "wqkv"), L["bqkv"], li)
            h = k.rmsnorm(x, lin(a, li, "wo"), L["ln_post"], s.eps)
            act = gate_up_swiglu(h, li)
            # the down output joins the residual stream under the norm that follows this layer
            h = k.rmsnorm(x, lin(act, li, "wd"), self.norm_after[li], s.eps)
        if last_only:
            h = h[-1:]
        if (h.shape[0] == 1 and s.hidden % 8 == 0 and s.hidden <= 8192
                and _kernel_operand(self.lm_head, (self.lm_head.shape[0], s.hidden))):
            return k.bf16_gemv(self.lm_head, x=h)  # 1.09 GB at 6.4 TB/s, against 4.6 for F.linear
        return F.linear(h, self.lm_head)

    @torch.no_grad()
    def generate(self, prompt_ids, n_new: int, use_graph: bool = True):
        """Greedy decoding (reference qwen.py:166-177): returns the ``n_new`` generated ids. The
        decode steps replay one captured graph when ``use_graph``."""
        T = prompt_ids.shape[0]
        self.alloc_cache(T + n_new)
        if use_graph and n_new > 1:
            self.capture_decode()
        # generated ids stay on the device until the end: no host synchronisation per token
        ids = torch.empty(n_new, dtype=torch.int64, device=self.dev)
        ids[0] = self.forward(prompt_ids, 0, use_cache=True, last_only=True)[-1].argmax()
        for n in range(1, n_new):
            ids[n] = self.decode(ids[n - 1], T + n - 1)[-1].argmax()
        return ids.tolist()
