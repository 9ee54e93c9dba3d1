"""The ways in which the selection kernel's workers take the rows of a launch, at the sizes where one way ends and the next
begins, against the CPU oracle.  Token ids are the same."""
import numpy as np
import pytest

from opentail.stingray_amd import SamplerContext, SamplingParams, pack_allow_mask, synthetic
from tests.helpers import oracle_tokens

pytestmark = pytest.mark.gpu
CHUNK = 512 * 19 * 4  # elements of fp32 logits that a worker's registers hold (bf16: 512 * 10 * 8)


@pytest.fixture(scope="module")
def ctx():
    c = SamplerContext(0)
    yield c
    c.close()


def _batch(rng, rows, vocab, longest):
    logits = synthetic.zipf_head_logits(rng, rows, vocab)
    logits[rows // 2] = np.round(logits[rows // 2])  # ties, and hundreds of entries at the bound
    logits[rows // 3, :] = -3.0
    params, allowed = [], np.ones((rows, vocab), dtype=bool)
    for r in range(rows):
        p = SamplingParams(Temperature=0.0 if r % 9 == 4 else float(rng.uniform(0.3, 1.6)), TopK=int(rng.integers(1, min(longest, vocab - 1) + 1)),
                           TopP=float(rng.choice([1.0, 0.95, 0.6])), MinP=float(rng.choice([0.0, 0.02])))
        if r % 3 == 1:
            p.PreviousTokens = rng.integers(0, vocab, 50).tolist() + np.argsort(-logits[r])[:10].tolist()
            p.RepetitionPenalty, p.FrequencyPenalty = 1.2, 0.1
        if r % 5 == 2:
            allowed[r] = rng.random(vocab) < 0.3
            allowed[r, 0] = True
        params.append(p)
    return logits, params, pack_allow_mask(allowed), np.array([r % 5 == 2 for r in range(rows)], dtype=np.uint8)


def _check(ctx, rng, rows, vocab, longest, bf16):
    import torch

    logits, params, mask, active = _batch(rng, rows, vocab, longest)
    u = rng.random(rows)
    if bf16:
        bits = synthetic.to_bf16_bits(logits)
        logits = synthetic.bf16_bits_to_f32(bits)
        dev = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
    else:
        dev = torch.from_numpy(logits).cuda()
    got = ctx.sample_batch(dev, params, u, mask, active)
    want = oracle_tokens(logits, params, u, mask, active)
    assert np.array_equal(got, want), (rows, vocab, longest, bf16, np.nonzero(got != want)[0][:10])


# Two workers to a compute unit that keep their rows' results: one row more than the device has compute units, the rows of a
# second turn, and chunks that end with a chunk's last vector and one element behind it.
@pytest.mark.parametrize("rows,vocab,longest,bf16", [
    (257, 1000, 900, False), (257, CHUNK, 40, False), (257, CHUNK + 1, 1000, False), (300, 2 * CHUNK - 3, 1000, False), (257, 2 * CHUNK + 1, 1000, False),
    (257, 3 * CHUNK + 1, 1000, False), (520, 9_001, 64, False), (513, 4 * CHUNK - 4, 300, False), (257, 4 * CHUNK + 1, 1000, False),
    (600, 33_333, 1000, True), (257, 512 * 10 * 8 + 1, 1000, True), (300, 100_003, 200, True), (257, 131_072, 1000, True)])
def test_more_rows_than_compute_units(ctx, rows, vocab, longest, bf16):
    _check(ctx, np.random.default_rng(rows * 7 + vocab), rows, vocab, longest, bf16)


# Where rows get a worker of their own, and what the others' chunks are: rows of one chunk in any number, and both sides of the lines
# for two, three and four chunks, short and long lists.
@pytest.mark.parametrize("rows,vocab,longest,bf16", [
    (1, CHUNK, 40, False), (5, CHUNK, 1000, False), (1, CHUNK + 1, 40, False), (64, 49_152, 1000, False), (64, 49_152, 1000, True), (24, 24_001, 64, True),
    (128, 2 * CHUNK - 3, 40, False), (129, 2 * CHUNK - 3, 40, False), (97, 100_003, 40, False), (96, 100_003, 40, False), (118, 100_003, 1000, False),
    (117, 100_003, 1000, False), (81, 4 * CHUNK - 4, 64, False), (121, 131_072, 1000, False), (113, 131_072, 40, True), (193, 60_000, 1000, True), (192, 60_000, 1000, True)])
def test_rows_with_and_without_a_worker_of_their_own(ctx, rows, vocab, longest, bf16):
    _check(ctx, np.random.default_rng(rows * 5 + vocab), rows, vocab, longest, bf16)


# Rows of five to eight chunks, whose second four join the groups of the first, and of nine: the chunks' edges, with the largest
# entries in both chunks of a pair and ties across them, dealt out, a worker to a row, and two to a compute unit.
@pytest.mark.parametrize("rows", [1, 7, 90, 140, 258])
@pytest.mark.parametrize("vocab,longest,bf16", [(4 * CHUNK + 1, 1000, False), (6 * CHUNK + 5, 64, False), (8 * CHUNK - 3, 1000, False), (8 * CHUNK + 3, 300, False),
                                                (7 * 512 * 10 * 8 - 1, 1000, True)])
def test_rows_of_more_than_four_chunks(ctx, rows, vocab, longest, bf16):
    if rows > 100 and vocab > 7 * CHUNK:
        vocab = 5 * CHUNK + 7
    _check(ctx, np.random.default_rng(rows * 3 + vocab), rows, vocab, longest, bf16)


def test_ties_across_chunks_that_share_their_groups(ctx):
    import torch

    rng = np.random.default_rng(5)
    vocab, rows = 6 * CHUNK, 9
    for n in (rows, 150):
        logits = rng.normal(0, 1, (n, vocab)).astype(np.float32)
        at = 4 * (512 * 4 * 3 + 200) + 1  # an element of a group, and the ones at its place in the chunk that joins it
        logits[:, at] = logits[:, at + 4 * CHUNK] = 9.0
        logits[::2, at + CHUNK] = logits[::2, at + 5 * CHUNK] = 9.0
        logits[1::3, at + 4 * CHUNK] = 9.5
        params = [SamplingParams(Temperature=0.0 if r % 3 == 0 else 0.7, TopK=[1, 2, 3, 50][r % 4], RepetitionPenalty=1.0) for r in range(n)]
        u = rng.random(n)
        got = ctx.sample_batch(torch.from_numpy(logits).cuda(), params, u)
        assert np.array_equal(got, oracle_tokens(logits, params, u)), n


# Launches of more than two turns of workers, whose second ones start late: the same tokens at every step, alone and between passes of two
# other streams over 64 MB each, which are queued with the steps and last longer than these do
@pytest.mark.parametrize("rows,vocab,bf16", [(513, 20_011, False), (1030, 40_000, True)])
def test_launches_of_several_turns_beside_other_work(ctx, rows, vocab, bf16):
    import torch

    rng = np.random.default_rng(rows)
    logits, params, mask, active = _batch(rng, rows, vocab, 1000)
    u = rng.random(rows)
    dev = torch.from_numpy(logits).cuda()
    if bf16:
        bits = synthetic.to_bf16_bits(logits)
        logits = synthetic.bf16_bits_to_f32(bits)
        dev = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
    want = oracle_tokens(logits, params, u, mask, active)
    steps = 8
    tokens = torch.full((2 * steps, rows), -7, dtype=torch.int32, device="cuda")
    noise = [torch.randn(4096, 4096, device="cuda") for _ in range(2)]
    sides = [torch.cuda.Stream() for _ in noise]
    batch = ctx.new_batch().upload(params, vocab, u, mask, active)
    for t in range(steps):
        ctx.sample_launch(batch, dev, tokens[t])
    for side in sides:
        side.wait_stream(torch.cuda.current_stream())
    for t in range(steps, 2 * steps):
        for x, side in zip(noise, sides):
            with torch.cuda.stream(side):
                for _ in range(10):
                    x.mul_(0.5).add_(1.0)
        ctx.sample_launch(batch, dev, tokens[t])
    ctx.synchronize()
    torch.cuda.synchronize()
    batch.close()
    for t, got in enumerate(tokens.cpu().numpy()):
        assert np.array_equal(got, want), (t, np.nonzero(got != want)[0][:10])


# Short lists over many waves: each gives its two largest, of which the bound comes also where one a wave would do (lists of up to as
# many entries as waves); waves with one entry and with none among them
@pytest.mark.parametrize("vocab,bf16", [(4 * CHUNK - 1, False), (5 * CHUNK, False), (8 * CHUNK - 3, False), (8 * CHUNK + 1, False), (327_000, True)])
def test_short_lists_of_rows_that_many_waves_stream(ctx, vocab, bf16):
    import torch

    rng = np.random.default_rng(vocab)
    rows = 12
    logits = rng.normal(0, 1.5, (rows, vocab)).astype(np.float32)
    allowed = np.ones((rows, vocab), dtype=bool)
    allowed[1] = False
    allowed[1, rng.integers(0, vocab, 9)] = True           # most waves have nothing, the others one
    allowed[2, : vocab // 2] = False                       # half the waves have nothing
    logits[3, : 3000] += 20.0                              # a few waves have everything
    logits[4] = np.round(logits[4] * 2) / 2                # ties at the bound
    bits = synthetic.to_bf16_bits(logits)
    if bf16:
        logits = synthetic.bf16_bits_to_f32(bits)
    dev = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16) if bf16 else torch.from_numpy(logits).cuda()
    active = np.isin(np.arange(rows), (1, 2)).astype(np.uint8)
    for k in (1, 2, 31, 32, 33, 40, 63, 64):
        params = [SamplingParams(Temperature=0.8, TopK=k, TopP=0.95, RepetitionPenalty=1.1 if r % 2 else 1.0,
                                 PreviousTokens=rng.integers(0, vocab, 60).tolist() if r % 2 else []) for r in range(rows)]
        mask, u = pack_allow_mask(allowed), rng.random(rows)
        got = ctx.sample_batch(dev, params, u, mask, active)
        assert np.array_equal(got, oracle_tokens(logits, params, u, mask, active)), (vocab, bf16, k)
