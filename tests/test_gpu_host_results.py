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
