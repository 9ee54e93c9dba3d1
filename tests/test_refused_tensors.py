"""Tensors that a call must refuse before anything reaches the native library (no GPU needed: the library is a recorder that
fails the test when it is called)."""
import pytest
import torch

from opentail.stingray_amd import SamplerContext, SamplingParams


class _NoCalls:
    def __getattr__(self, name):
        raise RuntimeError(f"{name} was called")


@pytest.fixture()
def ctx():
    c = SamplerContext.__new__(SamplerContext)
    c.L, c.h, c._batches = _NoCalls(), None, set()
    return c


@pytest.mark.parametrize("rows", [0, 2])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sample_batch_refuses_logits_in_host_memory(ctx, rows, dtype):
    """(a host address given to a kernel would fault the GPU; such logits were always refused, with no rows as well)"""
    with pytest.raises(AssertionError):
        ctx.sample_batch(torch.zeros((rows, 64), dtype=dtype), [SamplingParams()] * rows, [0.5] * rows)
