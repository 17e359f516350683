"""What the Kernels wrappers hand to the library for strided and overlapping arguments: a contiguous
copy must live until the launch has been issued (an address read from a copy that is already gone can
belong to the next copy), and a launch must not write where it still reads."""
import weakref

import pytest
import torch

from nanoserve_amd import Kernels, ops

BF16 = torch.bfloat16


class _Lib:
    """Stands in for the library: every launch notes whether the copies made for it still exist."""

    def __init__(self, copies):
        self.copies, self.launches = copies, []

    def __getattr__(self, name):
        def call(*args):
            if not name.endswith("_workspace"):
                self.launches.append((name, len(self.copies), all(c() is not None for c in self.copies)))
                self.args = args
            return 0

        return call


def _strided(*size, dtype=BF16):
    return torch.ones(size[0], 2 * size[1], dtype=dtype)[:, ::2]


@pytest.fixture
def stub(monkeypatch):
    copies, contiguous = [], torch.Tensor.contiguous

    def spy(t, *args, **kw):
        c = contiguous(t, *args, **kw)
        if c is not t:
            copies.append(weakref.ref(c))
        return c

    monkeypatch.setattr(ops, "_require_gpu_tensor", lambda *a: None)
    monkeypatch.setattr(torch.Tensor, "contiguous", spy)
    k = Kernels.__new__(Kernels)
    k.lib = _Lib(copies)
    monkeypatch.setattr(Kernels, "_stream", staticmethod(lambda: 0))
    return k



@pytest.mark.parametrize("call,copies", [
    (lambda k, wq, s: k.w4_linear(_strided(4, 256), wq, s), 3),
    (lambda k, wq, s: k.w4_linear_swiglu(_strided(1, 256), wq, s), 3),
    (lambda k, wq, s: k.w4_linear_swiglu(_strided(4, 256), wq, s), 3),
    (lambda k, wq, s: k.w4_linear_swiglu(_strided(128, 256), wq, s), 3),
    (lambda k, wq, s: k.w4_repack(wq, s), 2),
    (lambda k, wq, s: k.w4_quantize(_strided(32, 256)), 1),
    (lambda k, wq, s: k.w4_linear_packed(_strided(4, 256), torch.ones(2, 2, 256, dtype=torch.int32),
                                         torch.ones(2, 2, 16, dtype=BF16), 32), 1),
    (lambda k, wq, s: k.w4_linear_packed_swiglu(_strided(32, 256), torch.ones(2, 2, 256, dtype=torch.int32),
                                                torch.ones(2, 2, 16, dtype=BF16), 32), 1),
    (lambda k, wq, s: k.rmsnorm(torch.ones(2, 16, dtype=BF16), _strided(2, 16), _strided(16, 1)[:, 0], 1e-6), 2),
    (lambda k, wq, s: k.rope(torch.ones(2, 128, dtype=BF16), torch.ones(2, 128, dtype=BF16),
                             _strided(64, 1)[:, 0], 1, 1, 128, 0), 1)])
def test_copies_outlive_the_launch(stub, call, copies):
    call(stub, _strided(32, 32, dtype=torch.int32), _strided(32, 2))
    assert [(n, alive) for _, n, alive in stub.lib.launches] == [(copies, True)]


# rows for which the activation was padded or the activation function ran as a launch of its own
@pytest.mark.parametrize("M", [2, 5, 8, 9, 100, 130])
@pytest.mark.parametrize("shift", [0, 128, -128])
def test_swiglu_over_its_input(stub, M, shift):
    wq, s = torch.ones(512, 32, dtype=torch.int32), torch.ones(512, 2, dtype=BF16)
    buf = torch.ones(M * 256 + 256, dtype=BF16)
    x, out = (buf[o:o + M * 256].view(M, 256) for o in (128, 128 + shift))
    got = stub.w4_linear_swiglu(x, wq, s, out=out)
    y = stub.lib.args[3]
    assert got is out and (y + out.nbytes <= x.data_ptr() or y >= x.data_ptr() + x.nbytes)


@pytest.mark.parametrize("M", [1, 4, 100, 128])
def test_swiglu_writes_out_in_place(stub, M):
    wq, s = torch.ones(512, 32, dtype=torch.int32), torch.ones(512, 2, dtype=BF16)
    out = torch.ones(M, 256, dtype=BF16)
    assert stub.w4_linear_swiglu(torch.ones(M, 256, dtype=BF16), wq, s, out=out) is out
    assert stub.lib.args[3] == out.data_ptr()


# scales above 1 MiB, so that the allocator serves them from the blocks it serves the codes from
@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 4, 8, 20, 128])
def test_strided_weights(kernels, M):
    N, K = 18944, 3584
    g = torch.Generator(device="cuda").manual_seed(M)
    wq = torch.randint(-(1 << 31), 1 << 31, (N, K // 4), generator=g, device="cuda",
                       dtype=torch.int64).to(torch.int32)[:, K // 8:]
    s = (torch.randn(N, K // 64, generator=g, device="cuda").abs() * 0.02).to(BF16)[:, K // 128:]
    x = torch.randn(M, K, generator=g, device="cuda").to(BF16)
    wc, sc = wq.contiguous(), s.contiguous()
    assert not wq.is_contiguous() and not s.is_contiguous()
    assert torch.equal(kernels.w4_linear(x, wq, s), kernels.w4_linear(x, wc, sc))
    assert torch.equal(kernels.w4_linear_swiglu(x, wq, s), kernels.w4_linear_swiglu(x, wc, sc))
    y = kernels.w4_linear_swiglu(x, wc[:2 * K], sc[:2 * K])
    if M not in (1, 128):  # out over the input
        z = x.clone()
        assert torch.equal(kernels.w4_linear_swiglu(z, wc[:2 * K], sc[:2 * K], out=z), y)
    for a, b in zip(kernels.w4_repack(wq, s), kernels.w4_repack(wc, sc)):
        assert torch.equal(a, b)
