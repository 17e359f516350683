"""W4 layers on row counts that are no multiple of 128: the GEMM on ragged M (every small-tile plan,
tile and K remainders, the register-staged fallback), and SwiGLU behind M = 2..8 and ragged M."""
import pytest
import torch

BF16 = torch.bfloat16


def _weights(N, K, G, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    wq = torch.randint(-(1 << 31), 1 << 31, (N, K // 8), generator=g, device="cuda",
                       dtype=torch.int64).to(torch.int32)
    s = (torch.randn(N, K // G, generator=g, device="cuda").abs() * 0.02).to(BF16)
    return wq, s


def _x(M, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(M, K, generator=g, device="cuda").to(BF16)


def _deq(wq, s, G):
    sh = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((wq[:, :, None] >> sh) & 15).reshape(wq.shape[0], -1).double() - 8
    w = q.view(q.shape[0], -1, G) * s.double()[:, :, None]
    return w.view(q.shape[0], -1)


# (M, N, K, G): every tile plan with ragged M (32 to 192 rows, 32 to 128 columns, one round of the CUs
# and several), at one row, at tile edges and past them, K whose blocks do not divide among the K
# groups, and the register-staged kernel (G = 96, K % 64 == 32)
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,G", [
    (9, 128, 64, 64), (32, 256, 192, 64), (33, 1024, 704, 64), (65, 896, 1152, 128),
    (63, 4608, 3584, 128), (100, 3584, 1280, 128), (129, 3584, 640, 128),
    (200, 1536, 8960, 128), (250, 1024, 2048, 32), (17, 16384, 576, 64), (31, 9216, 1536, 128),
    (64, 17920, 1536, 128), (57, 16512, 448, 64), (100, 4608, 3584, 128), (129, 4608, 512, 128),
    (300, 3328, 1024, 128), (700, 1792, 896, 128), (1000, 8960, 256, 128), (2047, 18944, 128, 128),
    (20, 17920, 448, 64), (40, 33024, 128, 128), (700, 3584, 384, 128), (1000, 4608, 192, 64),
    (1200, 4608, 192, 32), (300, 12800, 128, 128), (1700, 3584, 8192, 128), (390, 3584, 8192, 128),
    (500, 3584, 320, 64), (2000, 18944, 64, 64), (333, 8960, 320, 64), (1790, 3584, 8256, 64),
    (10, 128, 96, 96), (77, 256, 288, 96), (130, 384, 160, 32)])
def test_linear_ragged_rows(kernels, M, N, K, G):
    wq, s = _weights(N, K, G, M + N)
    x = _x(M, K, K)
    y = kernels.w4_linear(x, wq, s, G)
    assert y.shape == (M, N)
    # the GEMM's numerics: weights staged as bf16, fp32 accumulation, half a bf16 ulp of rounding
    ref = x.double() @ _deq(wq, s, G).to(BF16).double().t()
    err = (y.double() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + 2e-5 * ref.abs().max()).all())
    assert torch.equal(y, kernels.w4_linear(x, wq, s, G))


@pytest.mark.gpu
def test_linear_ragged_rows_views(kernels):
    """A row slice at an address that is not 16-byte aligned, and rows that are not contiguous."""
    wq, s = _weights(256, 256, 128, 1)
    flat = _x(1, 40 * 256 + 8, 2).view(-1)
    for x in (flat[1:1 + 20 * 256].view(20, 256), flat[:40 * 256].view(20, 512)[:, 256:]):
        assert torch.equal(kernels.w4_linear(x, wq, s), kernels.w4_linear(x.clone(), wq, s))
        assert torch.equal(kernels.w4_linear_swiglu(x, wq, s),
                           kernels.w4_linear_swiglu(x.clone(), wq, s))


def _two_step(kernels, x, wq, s, G):
    M, N = x.shape[0], wq.shape[0]
    gu = kernels.w4_linear(x, wq, s, G).view(M, N // 16, 2, 8)
    return kernels.swiglu(*(gu[:, :, i].reshape(M, N // 2).contiguous() for i in (0, 1)))


# M = 2..8: SwiGLU in the GEMV (one to five pairs per wave, both group heights, N tails inside a
# group) and through the interleaved activation kernel (odd group counts, other group sizes)
@pytest.mark.gpu
@pytest.mark.parametrize("N,K,G", [(16, 256, 128), (48, 512, 128), (1040, 3584, 128), (37888, 3584, 128),
                                   (17920, 1536, 128), (4112, 5120, 128), (528, 9216, 128),
                                   (272, 13312, 128), (160, 18944, 128), (2064, 896, 128),
                                   (96, 4224, 128), (64, 192, 96), (32, 256, 64)])
@pytest.mark.parametrize("M", [2, 5, 8])
def test_mlp_small_batch(kernels, M, N, K, G):
    wq, s = _weights(N, K, G, N + K)
    x = _x(M, K, M)
    out = torch.empty(M, N // 2, dtype=BF16, device="cuda")
    got = kernels.w4_linear_swiglu(x, wq, s, G, out=out)
    assert got is out and torch.equal(got, _two_step(kernels, x, wq, s, G))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,G", [(9, 256, 256, 128), (40, 4608, 512, 128), (33, 17920, 256, 64),
                                     (100, 3584, 640, 32), (61, 18944, 128, 128), (200, 1536, 1920, 128),
                                     (333, 8960, 256, 128), (900, 18944, 128, 128),
                                     (20, 17920, 128, 128), (40, 33024, 128, 128), (300, 3328, 256, 128),
                                     (700, 3584, 256, 128), (1000, 4608, 256, 128),
                                     (1200, 4608, 256, 128), (500, 3584, 256, 128),
                                     (390, 3584, 8192, 128), (1790, 3584, 8192, 128),
                                     (1040, 18944, 64, 64)])
def test_mlp_ragged_rows(kernels, M, N, K, G):
    wq, s = _weights(N, K, G, N + K)
    x = _x(M, K, M)
    assert torch.equal(kernels.w4_linear_swiglu(x, wq, s, G), _two_step(kernels, x, wq, s, G))


# the packed GEMM's tile plans, ragged in M and N
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (17, 128, 128), (100, 896, 1024), (77, 200, 128), (260, 4096, 128), (410, 3584, 2048), (400, 3584, 128),
    (500, 4608, 256), (700, 3504, 384), (333, 8960, 256), (1000, 4608, 2048), (1210, 4608, 2176),
    (1900, 4608, 128), (350, 18944, 128), (700, 1800, 256), (1153, 3584, 2048), (548, 9984, 256),
    (155, 7536, 384), (806, 1536, 1920)])
def test_packed_ragged(kernels, M, N, K):
    wq, s = _weights(N, K, 128, M + N)
    wp, sp = kernels.w4_repack(wq, s)
    x = _x(M, K, K)
    y = kernels.w4_linear_packed(x, wp, sp, N)
    ref = x.double() @ _deq(wq, s, 128).to(BF16).double().t()
    err = (y.double() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + 2e-5 * ref.abs().max()).all())
    if N % 16 == 0:
        gu = y.view(M, N // 16, 2, 8)
        two = kernels.swiglu(*(gu[:, :, i].reshape(M, N // 2).contiguous() for i in (0, 1)))
        assert torch.equal(kernels.w4_linear_packed_swiglu(x, wp, sp, N), two)


# rows that are no whole 16-byte segments (N % 8 != 0, or an output at another address), in each of the
# packed GEMM's plans and at full and ragged tiles; the elements around the output stay as they are
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (64, 201, 128), (100, 897, 1024), (128, 8201, 1024), (77, 203, 256), (260, 4097, 128), (410, 3583, 2048),
    (500, 4606, 256), (700, 3501, 384), (333, 8962, 256), (1000, 4610, 2048), (1210, 4607, 2176),
    (1900, 4609, 128), (1153, 3585, 2048), (548, 9986, 256), (128, 4609, 256), (700, 4608, 384),
    (1000, 4608, 2048), (1210, 4608, 2176), (260, 4096, 128)])
def test_packed_rows_without_segments(kernels, M, N, K):
    wq, s = _weights(N, K, 128, M + N)
    wp, sp = kernels.w4_repack(wq, s)
    x = _x(M, K, K)

    def at(cols, off):
        flat = torch.full((M * cols + 64,), 7.0, dtype=BF16, device="cuda")
        return flat, flat[32 + off:32 + off + M * cols].view(M, cols)

    flat, y = at(N, 1 if N % 8 == 0 else 0)
    assert kernels.w4_linear_packed(x, wp, sp, N, out=y) is y
    lo = (y.data_ptr() - flat.data_ptr()) // 2
    assert bool((flat[:lo] == 7).all()) and bool((flat[lo + M * N:] == 7).all())
    ref = x.double() @ _deq(wq, s, 128).to(BF16).double().t()
    err = (y.double() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + 2e-5 * ref.abs().max()).all())
    if N % 16 == 0:
        flat, y = at(N // 2, 1)
        kernels.w4_linear_packed_swiglu(x, wp, sp, N, out=y)
        assert torch.equal(y, kernels.w4_linear_packed_swiglu(x, wp, sp, N))
        assert bool((flat[:33] == 7).all()) and bool((flat[33 + M * N // 2:] == 7).all())


def test_rows_entry_points_reject():
    from nanoserve_amd import Kernels

    lib, P = Kernels().lib, 0x10000
    lin, mlp = lib.ns_w4_linear_rows, lib.ns_w4_linear_swiglu_rows
    assert lin(P, P, P, P, 9, 100, 128, 128, None) == -2      # N % 128
    assert lin(P, P, P, P, 9, 128, 100, 128, None) == -2
    assert lin(P + 8, P, P, P, 9, 128, 128, 128, None) == -2
    assert lin(P, P, P, P, 0, 128, 128, 128, None) == -2
    assert lib.ns_w4_linear_swiglu_rows_workspace(4, 512, 896, 128) == 4 * 512 * 2
    assert lib.ns_w4_linear_swiglu_rows_workspace(4, 512, 1024, 128) == 0
    assert lib.ns_w4_linear_swiglu_rows_workspace(9, 512, 896, 128) == 0
    assert mlp(P, P, P, P, None, 0, 4, 512, 896, 128, None) == -2   # needs tmp
    assert mlp(P, P, P, P, P, 4095, 4, 512, 896, 128, None) == -2
    assert mlp(P, P, P, P + 2, None, 0, 4, 512, 1024, 128, None) == -2
    assert mlp(P, P, P, P, None, 0, 9, 48, 1024, 128, None) == -2   # N % 128 above 8 rows
    assert mlp(P, P, P, P, None, 0, 4, 24, 1024, 128, None) == -2   # N % 16
    assert mlp(P, P, P, P, None, 0, 20, 128, 96, 96, None) == -2    # no SwiGLU epilogue there
