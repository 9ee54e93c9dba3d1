"""Row argmax where a workgroup's tiles, chunks and vectors end: the first index of the largest element (a zero of either
sign), the first NaN before everything, the original bits as the value; fp32 and bf16, rows at every address."""
import numpy as np
import pytest

from opentail.stingray_amd import SamplerContext, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = SamplerContext(0)
    yield c
    c.close()


def _want(row):
    nan = np.isnan(row)
    if nan.any():
        return int(np.argmax(nan))
    return int(np.argmax(row == row.max()))


# a vector, a tile of a workgroup (256 threads x 4 vectors) and two of them, one element less and more; several chunks a row
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("vocab", [1, 3, 8, 9, 1023, 4095, 4096, 4097, 8191, 8192, 8193, 16_385, 33_001, 100_003])
def test_first_of_the_largest(ctx, vocab, bf16):
    import torch

    rng = np.random.default_rng(vocab)
    rows = 40
    x = rng.normal(0, 1, (rows, vocab)).astype(np.float32)
    for r in range(rows):
        a, b = (int(v) for v in np.sort(rng.integers(0, vocab, 2)))
        kind = r % 8
        if kind == 0:
            x[r, a] = x[r, b] = 9.0
        elif kind == 1:
            x[r, -1] = 9.0
        elif kind == 2:
            x[r] = -np.abs(x[r]) - 1
            x[r, a], x[r, b] = (np.float32(-0.0), np.float32(0.0)) if r % 16 == 2 else (np.float32(0.0), np.float32(-0.0))
        elif kind == 3:
            x[r, b] = np.inf
            x[r, a] = -np.nan if r % 16 == 3 else np.nan
        elif kind == 4:
            x[r] = -np.inf
        elif kind == 5:
            x[r] = -np.inf
            x[r, b] = np.nan
            x[r, a] = -np.nan
        elif kind == 6:
            x[r] = -np.abs(x[r]) - 3
        else:
            x[r] = np.round(x[r])
    bits = x.view(np.uint32)
    if bf16:
        half = np.where(np.isnan(x), (bits >> 16) | 0x40, synthetic.to_bf16_bits(x)).astype(np.uint16)
        x = (half.astype(np.uint32) << 16).view(np.float32)
    want = [_want(row) for row in x]
    for off, pad in [(0, -vocab % 8), (1, 0), (3, 5)]:
        stride = vocab + pad
        if bf16:
            flat = torch.zeros(off + rows * stride, dtype=torch.int16, device="cuda")
            view = flat[off:].view(rows, stride)[:, :vocab]
            view.copy_(torch.from_numpy(half.view(np.int16)).cuda())
            dev = flat.view(torch.bfloat16)[off:].view(rows, stride)[:, :vocab]
        else:
            flat = torch.zeros(off + rows * stride, device="cuda")
            dev = flat[off:].view(rows, stride)[:, :vocab]
            dev.copy_(torch.from_numpy(x).cuda())
        idx, val = ctx.argmax_rows(dev)
        assert list(idx) == want, (vocab, bf16, off, pad)
        assert np.array_equal(np.asarray(val).view(np.uint32), x[np.arange(rows), want].view(np.uint32)), (vocab, bf16, off, pad)
