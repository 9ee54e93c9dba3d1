"""Nuclei cut from lists of thousands of candidates, which are not put in order but for the entries that need it: list lengths around
the sizes at which the tables change, cuts early, late and nowhere, on smooth values, on coarse grids and on plateaus."""
import numpy as np
import pytest

from opentail.stingray_amd import SamplerContext, SamplingParams, pack_allow_mask, synthetic
from tests.helpers import oracle_tokens, to_oracle
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = SamplerContext(0)
    yield c
    c.close()


def _rows(rng, rows, vocab, allowed_counts, bf16):
    logits = rng.normal(0, 1.5, (rows, vocab)).astype(np.float32)
    allowed = np.zeros((rows, vocab), dtype=bool)
    params = []
    for r in range(rows):
        allowed[r, rng.choice(vocab, allowed_counts[r % len(allowed_counts)], replace=False)] = True
        shape = (r // len(allowed_counts)) % 5
        if shape == 1:
            logits[r] = np.round(logits[r] * 64) / 64
        elif shape == 2:
            logits[r] = np.round(logits[r] * 4) / 4           # hundreds of entries of one value
        elif shape == 3:
            logits[r, rng.random(vocab) < 0.5] = 0.5            # a plateau of half of the row
        elif shape == 4:
            logits[r] = rng.uniform(-0.01, 0.01, vocab)       # all but flat
        p = SamplingParams(Temperature=float(rng.choice([0.6, 1.0, 1.7])), TopP=float(rng.choice([0.05, 0.5, 0.95, 0.999, 0.9999999])))
        if r % 4 == 3:
            p.MinP = float(rng.choice([1e-4, 1e-3, 0.02]))
        params.append(p)
    if bf16:
        logits = synthetic.bf16_bits_to_f32(synthetic.to_bf16_bits(logits))
    return logits, params, allowed


@pytest.mark.parametrize("rows,vocab,counts,bf16", [
    (30, 40_000, (1023, 1024, 1025, 1100, 2047, 2049), False), (30, 40_000, (4095, 4096, 4097, 6000, 8191, 8200), False),
    (15, 60_000, (16_383, 16_384, 16_385), False), (20, 60_000, (3000, 9000, 14_000, 20_000), True), (270, 8_192, (1500, 4096, 4097), False)])
def test_nuclei_of_long_lists(ctx, rows, vocab, counts, bf16):
    import torch

    rng = np.random.default_rng(rows + vocab + counts[0])
    logits, params, allowed = _rows(rng, rows, vocab, counts, bf16)
    mask, active, u = pack_allow_mask(allowed), np.ones(rows, dtype=np.uint8), rng.random(rows)
    dev = torch.from_numpy(logits).cuda()
    if bf16:
        dev = dev.to(torch.bfloat16)
    got = ctx.sample_batch(dev, params, u, mask, active)
    want = oracle_tokens(logits, params, u, mask, active)
    assert np.array_equal(got, want), np.nonzero(got != want)[0][:10]


# ... and the whole distribution, which names every member of the nucleus
@pytest.mark.parametrize("count", [1025, 3000, 4097, 12_000])
def test_distributions_of_long_lists(ctx, count):
    import torch

    rows, vocab = 10, 30_000
    rng = np.random.default_rng(count)
    logits, params, allowed = _rows(rng, rows, vocab, (count, count + 7), False)
    logits = np.where(allowed, logits, -np.inf).astype(np.float32)
    got = ctx.build_distribution(torch.from_numpy(logits).cuda(), params).cpu().numpy()
    for r in range(rows):
        want = orc.build_filtered_distribution(logits[r], to_oracle(params[r]))
        assert np.array_equal(got[r], want), (r, np.count_nonzero(got[r]), np.count_nonzero(want))
