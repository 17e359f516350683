"""The prompt pass's attention operators against a float64 reference: ns_prompt_qkv (bias + RoPE +
KV append) and ns_prompt_attention (causal grouped-query attention with a position offset)."""
import math

import pytest
import torch

BF16 = torch.bfloat16


def _ref(q, k, v, pos0):
    """q [T, Hq, 128], k / v [Hk, n, 128] float64 -> [T, Hq * 128]."""
    T, Hq, D = q.shape
    rep = Hq // k.shape[0]
    kk, vv = k.repeat_interleave(rep, 0), v.repeat_interleave(rep, 0)
    s = q.transpose(0, 1) @ kk.transpose(1, 2).contiguous() / math.sqrt(D)
    qp = torch.arange(pos0, pos0 + T, device=q.device)[:, None]
    s = s.masked_fill(torch.arange(k.shape[1], device=q.device)[None] > qp, float("-inf"))
    return (torch.softmax(s, -1) @ vv).transpose(0, 1).reshape(T, Hq * D)


# rows = T * Hq / Hk around the wave (32) and tile (128) sizes, keys around the 64-key block,
# with one split and several, one and many kv heads
@pytest.mark.gpu
@pytest.mark.parametrize("T,pos0,Hq,Hk", [
    (2, 0, 1, 1), (31, 0, 2, 2), (33, 31, 4, 4), (64, 0, 7, 1), (65, 63, 7, 1), (18, 1, 28, 4),
    (19, 4077, 28, 4), (128, 128, 2, 1), (129, 383, 12, 2), (300, 0, 28, 4), (9, 5000, 16, 16),
    (520, 1000, 32, 8), (1100, 0, 40, 8)])
@pytest.mark.parametrize("cached", [True, False])
def test_prompt_attention(kernels, T, pos0, Hq, Hk, cached):
    n = pos0 + T
    g = torch.Generator(device="cuda").manual_seed(T * 7 + pos0)
    rows = torch.randn(n, (Hq + 2 * Hk) * 128, generator=g, device="cuda").to(BF16)
    rows[:, :Hq * 128] *= 3  # peaked rows as well as flat ones
    q = rows[pos0:, :Hq * 128]
    k, v = (rows[:, a * 128:(a + Hk) * 128].unflatten(1, (Hk, 128)).transpose(0, 1)
            for a in (Hq, Hq + Hk))
    want = _ref(q.double().reshape(T, Hq, 128), k.double(), v.double(), pos0)
    if cached:  # rows past the last key are never read into a result
        kc, vc = (torch.full((Hk, n + 70, 128), float("nan"), dtype=BF16, device="cuda")
                  for _ in range(2))
        kc[:, :n], vc[:, :n] = k, v
        k, v = kc, vc
    work = kernels.prompt_attention_workspace(T, Hq, Hk, pos0)
    got = kernels.prompt_attention(q, k, v, Hq, pos0, work=work)
    again = kernels.prompt_attention(q, k, v, Hq, pos0, work=work)
    assert torch.equal(got, again)
    # half a bf16 ulp of the result (at most 2^-8 of it), the probabilities' split from position 0
    # (2^-16 of the values' magnitude) and fp32 sums
    err = (got.double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + 2.0 ** -14 * v[:, :n].double().abs().amax()
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.gpu
def test_prompt_attention_keeps_fp32_probabilities(kernels):
    """Behind cached positions the second product holds the whole fp32 probability: three keys whose
    values cancel to about 2^-18 of them, so that an error of a probability is the result's error."""
    Hk, T, pos0 = 16, 2, 3
    g = torch.Generator(device="cuda").manual_seed(8)
    # scores 0, about -0.5 and about -5 nats; the chunk's own keys score below -1000 (probability 0)
    b = torch.tensor([0.0, -0.5, -5.0], device="cuda") * (1 + 0.3 * torch.rand(Hk, 3, generator=g, device="cuda"))
    kk, v = (torch.zeros(Hk, pos0 + T, 128, dtype=BF16, device="cuda") for _ in range(2))
    kk[:, :3, 0], kk[:, 3:, 0] = b.to(BF16), -1024.0
    q = torch.zeros(T, Hk, 128, dtype=BF16, device="cuda")
    q[..., 0] = 11.3125
    p = torch.exp(kk[:, :3, :1].double() * 11.3125 / math.sqrt(128))
    v[:, 1] = torch.randn(Hk, 128, generator=g, device="cuda").to(BF16)
    v[:, 0] = -(p[:, 1] * v[:, 1].double()).to(BF16)
    v[:, 2] = -((p[:, 1] * v[:, 1].double() + v[:, 0].double()) / p[:, 2]).to(BF16)
    want = (p * v[:, :3].double()).sum(1) / p.sum(1)
    work = kernels.prompt_attention_workspace(T, Hk, Hk, pos0)
    got = kernels.prompt_attention(q.view(T, -1), kk, v, Hk, pos0, work=work).view(T, Hk, 128).double()
    # exp2 and its argument to 2^-22 of the probability, a handful of fp32 sums, the result's bf16
    # rounding; a probability of 16 bits is up to 2^-18 off
    bound = 2.0 ** -20 * (p[:, 1] * v[:, 1].double()).abs() + 2.0 ** -8 * want.abs() + 1e-9
    assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() / bound).max())


@pytest.mark.gpu
def test_prompt_attention_special_values(kernels):
    """A NaN value reaches every query that attends to it and no other kv head (a masked key of the
    same block contributes 0 * NaN, as in a plain masked product); scores of +-1e4 do not overflow."""
    T, Hq, Hk = 200, 4, 2
    g = torch.Generator(device="cuda").manual_seed(3)
    q = (torch.randn(T, Hq * 128, generator=g, device="cuda") * 30).to(BF16)
    k = (torch.randn(Hk, T, 128, generator=g, device="cuda") * 30).to(BF16)
    v = torch.randn(Hk, T, 128, generator=g, device="cuda").to(BF16)
    work = kernels.prompt_attention_workspace(T, Hq, Hk, 0)
    got = kernels.prompt_attention(q, k, v, Hq, 0, work=work).double()
    want = _ref(q.double().reshape(T, Hq, 128), k.double(), v.double(), 0)
    # fp32 scores of magnitude 1e4 carry 1e4 * 2^-22 in the exponent
    assert float((got - want).norm() / want.norm()) < 1e-2
    v[1, 77, 5] = float("nan")
    got = kernels.prompt_attention(q, k, v, Hq, 0, work=work).view(T, Hq, 128)
    bad = torch.isnan(got)
    assert not bad[:, :2].any() and not bad[..., :5].any() and bool(bad[77:, 2:, 5].all())


@pytest.mark.gpu
@pytest.mark.parametrize("T,Hq,Hk,D,pos0,cached,bias", [
    (1, 1, 1, 128, 5, True, True), (3, 28, 4, 128, 0, True, True), (257, 12, 2, 128, 300, True, False),
    (40, 7, 1, 64, 11, False, True), (5, 3, 3, 16, 0, False, False), (9, 2, 1, 256, 7, True, True)])
def test_prompt_qkv(kernels, T, Hq, Hk, D, pos0, cached, bias):
    """Against the float64 bias + RoPE; cache rows outside the chunk stay as they are."""
    g = torch.Generator(device="cuda").manual_seed(T + Hq)
    H = Hq + 2 * Hk
    qkv = torch.randn(T, H * D, generator=g, device="cuda").to(BF16)
    b = torch.randn(H * D, generator=g, device="cuda").to(BF16) if bias else None
    inv = (1.0 / 1e6 ** (torch.arange(0, D, 2).float() / D)).cuda()
    x = (qkv + b if bias else qkv).double().view(T, H, D)
    ang = (torch.arange(pos0, pos0 + T, device="cuda").float()[:, None] * inv).double()[:, None]
    lo, hi = x[:, :Hq + Hk].chunk(2, -1)
    want = torch.cat([torch.cat([lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin()], -1),
                      x[:, Hq + Hk:]], 1)
    caches = [None, None]
    if cached:
        caches = [torch.full((Hk, pos0 + T + 3, D), 9.0, dtype=BF16, device="cuda") for _ in range(2)]
    got = qkv.clone()
    kernels.prompt_qkv(got, b, inv, Hq, Hk, D, pos0, *caches)
    out = got.view(T, H, D).clone()
    if cached:
        assert torch.equal(out[:, Hq:], qkv.view(T, H, D)[:, Hq:])
        for i, c in enumerate(caches):
            assert bool((c[:, :pos0] == 9).all()) and bool((c[:, pos0 + T:] == 9).all())
            out[:, Hq + i * Hk:Hq + (i + 1) * Hk] = c[:, pos0:pos0 + T].transpose(0, 1)
    assert torch.equal(out[:, Hq + Hk:].double(), want[:, Hq + Hk:])
    err = (out.double() - want).abs()
    mag = x.abs().view(T, H, 2, D // 2).amax(2).repeat(1, 1, 2)
    assert bool((err <= want.abs() * 2.0 ** -8 + mag * 1e-5).all())


def test_prompt_ops_reject_bad_arguments():
    from nanoserve_amd import Kernels

    lib, P = Kernels().lib, 0x10000
    ok = dict(q=P, qs=512, k=P, v=P, ks=128, hs=1 << 20, out=P, T=4, Hq=4, Hk=2, pos0=0)

    def attn(**kw):
        a = {**ok, **kw}
        return lib.ns_prompt_attention(a["q"], a["qs"], a["k"], a["v"], a["ks"], a["hs"], a["out"], None,
                                       0, a["T"], a["Hq"], a["Hk"], a["pos0"], None)

    for bad in (dict(q=None), dict(k=P + 8), dict(v=None), dict(out=P + 2), dict(qs=508), dict(qs=256),
                dict(ks=64), dict(hs=-8), dict(T=0), dict(Hq=5), dict(Hk=0), dict(pos0=-1),
                dict(pos0=1 << 29), dict(pos0=9000000)):
        assert attn(**bad) == -2, bad
    assert attn(T=300, pos0=3000) == -2  # needs a workspace
    assert lib.ns_prompt_attention_workspace(4, 4, 2, 0) == 0
    qkv = lib.ns_prompt_qkv
    assert qkv(None, None, P, None, None, 4, 4, 2, 128, 0, 0, None) == -2
    assert qkv(P, None, P, P, None, 4, 4, 2, 128, 0, 16, None) == -2
    assert qkv(P, None, P, P, P, 4, 4, 2, 128, 13, 16, None) == -2
    assert qkv(P, None, P, P, P, 4, 4, 2, 72, 0, 16, None) == -2
    assert qkv(P, P + 2, P, P, P, 4, 4, 2, 128, 0, 16, None) == -2


# past the position where the projection's row stride would end the 32-bit offsets, and the last one a
# cache's rows reach: keys planted at the start, the middle and the end decide the result
@pytest.mark.gpu
@pytest.mark.parametrize("T,pos0", [(70, 300000), (40, (1 << 23) - 169)])
def test_prompt_attention_far_positions(kernels, T, pos0):
    n, Hq = pos0 + T, 2
    assert kernels.prompt_attention_fits(T, Hq, 1, pos0, 128)
    assert T > 40 or not kernels.prompt_attention_fits(T, Hq, 1, pos0 + 1, 128)
    g = torch.Generator(device="cuda").manual_seed(T)
    k, v = (torch.randn(1, n, 128, generator=g, device="cuda", dtype=BF16) for _ in range(2))
    k *= 0.05
    q = torch.randn(T, Hq * 128, generator=g, device="cuda").to(BF16)
    q[:, ::128] = 16.0
    for j in (5, n // 2, n - T - 1, n - 2):
        k[0, j, 0] = 18.0
    work = kernels.prompt_attention_workspace(T, Hq, 1, pos0)
    got = kernels.prompt_attention(q, k, v, Hq, pos0, work=work).double().view(T, Hq, 128)
    for h in range(Hq):
        want = _ref(q.double().view(T, Hq, 128)[:, h:h + 1], k.double(), v.double(), pos0)
        err = (got[:, h] - want).abs()
        assert bool((err <= want.abs() * 2.0 ** -8 + 2.0 ** -14 * v.double().abs().amax()).all())


def test_prompt_attention_limits_follow_the_key_rows():
    """The runner's choice of the kernel is the kernel's own rule: 32-bit offsets over the rows the keys
    lie in (128 values in a cache, the projection's width without one) and 65535 row tiles."""
    from nanoserve_amd import Kernels
    from nanoserve_amd.qwen import Qwen2Runner, Qwen2Shape

    r = Qwen2Runner.__new__(Qwen2Runner)
    r.k, r.shape = Kernels(), Qwen2Shape(layers=1, hidden=3584, heads=28, kv_heads=4)
    P = 0x10000

    def ok(T, pos0, cached):
        fits = r._prompt_attention_kernel_ok(T, pos0, cached)
        stride = 128 if cached else r.shape.qkv_rows
        if not fits:  # refused before any launch
            assert r.k.lib.ns_prompt_attention(P, r.shape.qkv_rows, P, P, stride, 128, P, P, 1 << 62, T,
                                               28, 4, pos0, None) == -2
        return fits

    assert ok(512, 3000, True) and ok(512, 0, False)
    assert ok(512, 300000, True) and ok(512, (1 << 23) - 641, True)
    assert not ok(512, (1 << 23) - 640, True)
    assert ok(232000, 0, False) and not ok(233000, 0, False)
    # 7 heads per kv head: 65535 * 128 / 7 = 1198354.3 tokens
    assert ok(1198354, 0, True) and not ok(1198355, 0, True) and not ok(1198372, 0, True)
    assert not ok(0, 0, True) and not ok(1 << 30, 0, True)
    r.shape = Qwen2Shape(layers=1, hidden=1024, heads=16, kv_heads=16, head_dim=64)
    assert not r._prompt_attention_kernel_ok(512, 0, True)


# Caches past the streaming line (128-row pieces of all kv heads > CUs): positions at the edges of a
# 16-row block, a 128-row piece and a workgroup's range, one range and many, empty waves and ranges
@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hk,max_len", [(28, 4, 9000), (8, 8, 4200), (16, 16, 2200), (3, 1, 33000)])
def test_decode_attention_streamed(kernels, Hq, Hk, max_len):
    g = torch.Generator(device="cuda").manual_seed(Hq + max_len)
    kc, vc = (torch.randn(Hk, max_len, 128, generator=g, device="cuda").to(BF16) for _ in range(2))
    qkv = torch.randn((Hq + 2 * Hk) * 128, generator=g, device="cuda").to(BF16)
    qkv[:Hq * 128] *= 3
    b = torch.randn((Hq + 2 * Hk) * 128, generator=g, device="cuda").to(BF16)
    inv = (1.0 / 1e6 ** (torch.arange(0, 128, 2).float() / 128)).cuda()
    work = kernels.decode_attention_workspace(Hq, Hk, 128, max_len)
    for pos in (0, 15, 16, 127, 128, 255, 1000, 2047, 2200 - 1, max_len // 2 + 1, max_len - 1, max_len + 5):
        p = torch.tensor([pos], dtype=torch.int32, device="cuda")
        k2, v2 = kc.clone(), vc.clone()
        if pos + 1 < max_len:  # rows past the position must not matter
            k2[:, pos + 1:] = float("nan")
            v2[:, pos + 1:] = float("nan")
        if pos < max_len:
            k2[:, pos] = v2[:, pos] = float("nan")  # the token's own row is written by the call
        got = kernels.decode_qkv_attention(qkv, b, inv, p, k2, v2, Hq, Hk, 128, work)
        rot = torch.stack([torch.cos(pos * inv), torch.sin(pos * inv)])
        ref = (qkv + b).clone()
        kernels.decode_qkv(ref, None, inv, p, kc.clone(), vc.clone(), Hq, Hk, 128)
        ref = ref.double().view(Hq + 2 * Hk, 1, 128)
        n = min(pos + 1, max_len)
        kk, vv = kc[:, :n].double(), vc[:, :n].double()
        if pos < max_len:
            kk[:, pos], vv[:, pos] = ref[Hq:Hq + Hk, 0], ref[Hq + Hk:, 0]
            assert torch.equal(k2[:, pos].double(), kk[:, pos]) and torch.equal(v2[:, pos].double(), vv[:, pos])
        q = ref[:Hq].transpose(0, 1).contiguous()
        want = _ref(q, kk, vv, n - 1)
        # half a bf16 ulp, the probabilities' two-term split and fp32 sums
        bound = want.abs() * 2.0 ** -8 + 2.0 ** -14 * vv.abs().amax()
        assert bool(((got.double() - want).abs() <= bound).all()), pos
        plain = kernels.decode_attention(q.to(BF16).reshape(-1), k2, v2, p, Hq, Hk, 128, work)
        assert torch.equal(plain, got), pos
        if pos < max_len:  # an angle table gives the same angles' outputs
            with_rot = kernels.decode_qkv_attention(qkv, b, inv, p, k2, v2, Hq, Hk, 128, work, rot=rot)
            assert bool(((with_rot.double() - want).abs() <= 4 * bound + 1e-2).all()), pos
