"""Prompt passes on hand-built runners: biases and output heads that the one-launch operators do not
take (other types, strides, addresses) give what their contiguous bf16 forms give."""
import pytest
import torch

from nanoserve_amd.qwen import Qwen2Runner, Qwen2Shape

BF16 = torch.bfloat16
SHAPE = Qwen2Shape(layers=2, hidden=512, heads=4, kv_heads=2, intermediate=1024, vocab=1003)


def _off_by_one(t):
    """The same values at an address that is 2 bytes past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view_as(t)
    return flat.copy_(t)


def _every_other(t):
    wide = torch.empty(*t.shape[:-1], 2 * t.shape[-1], dtype=t.dtype, device=t.device)
    wide[..., ::2] = t
    return wide[..., ::2]


@pytest.mark.gpu
@pytest.mark.parametrize("form", [torch.Tensor.float, _off_by_one, _every_other])
def test_forward_takes_any_bias(kernels, form):
    r = Qwen2Runner.random(SHAPE, seed=3, kernels=kernels)
    ids = torch.arange(37, device="cuda") * 7
    r.alloc_cache(64)
    want = r.forward(ids, 0, use_cache=True)
    kc, vc = r.cache_k[:, :, :37].clone(), r.cache_v[:, :, :37].clone()
    for layer in r.layers:
        layer["bqkv"] = form(layer["bqkv"])
    assert torch.equal(r.forward(ids, 0, use_cache=True), want)
    assert torch.equal(r.cache_k[:, :, :37], kc) and torch.equal(r.cache_v[:, :, :37], vc)
    assert torch.equal(r.forward(ids), want)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [_off_by_one, _every_other])
def test_forward_takes_any_head(kernels, form):
    r = Qwen2Runner.random(SHAPE, seed=4, kernels=kernels)
    ids = torch.arange(21, device="cuda") * 5
    want = r.forward(ids, last_only=True).double()
    r.lm_head = form(r.lm_head)
    got = r.forward(ids, last_only=True).double()
    assert got.shape == (1, SHAPE.vocab)
    # fp32 sums in another order, half a bf16 ulp each
    assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 1e-4 * want.abs().max()).all())
