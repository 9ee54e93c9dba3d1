"""Results that kernels leave in pinned host memory, and uniforms that they read there: the row argmax with device and host
results, sample_batch, and steps whose uniforms change while earlier launches still read theirs (the pinned ring goes
round, the context changes streams in between)."""
import numpy as np
import pytest

from opentail.stingray_amd import SamplerContext, SamplingParams
from oracle import binding as orc
from tests.helpers import oracle_tokens

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ctx():
    c = SamplerContext(0)
    yield c
    c.close()


@pytest.mark.parametrize("rows,vocab", [(1, 1), (1, 70_001), (3, 2048), (130, 40_000), (1500, 513)])
def test_argmax_host_and_device_results_agree(ctx, rows, vocab):
    import torch

    m = np.random.default_rng(rows).normal(0, 2, (rows, vocab)).astype(np.float32)
    dev = torch.from_numpy(m).cuda()
    out = (torch.full((rows,), -3, dtype=torch.int32, device="cuda"), torch.full((rows,), 9.0, device="cuda"))
    want = np.array([orc.greedy(r) for r in m])
    for _ in range(3):
        i0, v0 = ctx.argmax_rows(dev, out=out)
        i1, v1 = ctx.argmax_rows(dev)
        assert np.array_equal(i0, want) and np.array_equal(i1, want)
        assert np.array_equal(v0, m[np.arange(rows), want]) and np.array_equal(v1, v0)
        assert np.array_equal(out[0].cpu().numpy(), want) and np.array_equal(out[1].cpu().numpy(), v0)


@pytest.mark.parametrize("own_stream", [False, True])
@pytest.mark.parametrize("rows,vocab", [(1, 40_000), (33, 151_936), (257, 2048), (1500, 513)])
def test_argmax_device_results_are_there_for_other_streams(rows, vocab, own_stream):
    """The device arrays are read on a stream that is not ordered behind the context's, and given away at once: what the
    allocator hands out next keeps what is put there."""
    import torch

    torch.cuda.synchronize()
    c = SamplerContext(0, use_torch_stream=not own_stream)
    rng = np.random.default_rng(rows)
    m = rng.normal(0, 2, (4, rows, vocab)).astype(np.float32)
    dev = [torch.from_numpy(x).cuda() for x in m]
    want = m.argmax(axis=2)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    for i in range(24):
        k = i % 4
        with torch.cuda.stream(other):
            out = (torch.full((rows,), -3, dtype=torch.int32, device="cuda"), torch.full((rows,), 9.0, device="cuda"))
            other.synchronize()
            idx, val = c.argmax_rows(dev[k], out=out)
            got = (out[0].clone(), out[1].clone())
            del out
            new = [torch.full((rows,), 77, dtype=torch.int32, device="cuda") for _ in range(2)]
        other.synchronize()
        assert np.array_equal(idx, want[k]) and np.array_equal(val, m[k][np.arange(rows), want[k]])
        assert np.array_equal(got[0].cpu().numpy(), idx) and np.array_equal(got[1].cpu().numpy(), val), i
        assert all(bool((t == 77).all()) for t in new), i
    c.close()


@pytest.mark.parametrize("topk", [0, 40])
def test_uniforms_of_launches_in_flight_are_not_overwritten(ctx, topk):
    """400 steps of new uniforms without a wait (the ring of a batch of 40 rows goes round several times), the context on
    another stream every 50 steps; every step's tokens against the oracle."""
    import torch

    rng = np.random.default_rng(5)
    rows, vocab, steps = 40, 5_003, 400
    x = rng.normal(0, 2, (rows, vocab)).astype(np.float32)
    params = [SamplingParams(Temperature=0.9, TopK=topk, TopP=0.97) for _ in range(rows)]
    u = rng.random((steps, rows))
    dev = torch.from_numpy(x).cuda()
    out = torch.zeros((steps, rows), dtype=torch.int32, device="cuda")
    batch = ctx.new_batch().upload(params, vocab, u[0])
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for i in range(steps):
        if i % 50 == 0:
            ctx.set_stream(streams[(i // 50) % 2].cuda_stream)
        if i:
            if i % 3:
                batch.set_uniforms(u[i])
            else:
                batch.append_tokens(np.full(rows, -1), u[i])
        ctx.sample_launch(batch, dev, out[i])
    ctx.synchronize()
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for i in range(0, steps, 7):
        assert np.array_equal(got[i], oracle_tokens(x, params, u[i])), i
    batch.close()
    ctx.set_stream(None)
