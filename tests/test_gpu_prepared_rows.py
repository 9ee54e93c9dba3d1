"""Rows of the full-vocabulary path whose cut comes from a list of candidates and whose normalisation and draw are left to
the whole device: the sizes at which segments, half blocks and blocks end, coarse logits (runs of equal probabilities across
the cut), lists that are empty, short, longer than they may be, and launches with too many rows for that way."""
import numpy as np
import pytest
import torch

from opentail.stingray_amd import SamplerContext, SamplingParams, pack_allow_mask
from oracle import binding as orc
from tests.helpers import oracle_tokens, to_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = SamplerContext(0)
    yield c
    c.close()


PARAMS = [SamplingParams(), SamplingParams(Temperature=0.7, TopP=0.9), SamplingParams(Temperature=1.3, TopP=0.999),
          SamplingParams(TopP=1e-6), SamplingParams(Temperature=0.8, MinP=1e-4), SamplingParams(MinP=1e-3, TopP=0.95),
          SamplingParams(Temperature=2.0, TopP=0.5), SamplingParams(MinP=1e-34, TopP=0.9),
          SamplingParams(Temperature=0.9, TopP=0.97, FrequencyPenalty=0.3, PreviousTokens=[5, 4000, 5, 17])]


def _check(ctx, logits, dev, params, rng):
    for r, u in enumerate([rng.random(len(params)), np.zeros(len(params)), np.full(len(params), 1.0 - 2.0 ** -53)]):
        got = ctx.sample_batch(dev, params, u)
        assert np.array_equal(got, oracle_tokens(logits, params, u)), (logits.shape, r)
    tokens, probs = ctx.sample_with_distribution(dev, params, u)
    probs = probs.cpu().numpy()
    assert np.array_equal(tokens, got), logits.shape
    for r, p in enumerate(params):
        want = orc.build_filtered_distribution(logits[r], to_oracle(p))
        assert np.array_equal(probs[r].view(np.uint32), want.view(np.uint32)), (logits.shape, r)


@pytest.mark.parametrize("vocab", [4096, 4097, 8191, 16385, 31_745, 32_768, 33_791, 36_865, 40_967, 65_537, 151_936])
@pytest.mark.parametrize("kind", ["f32", "bf16", "coarse"])
def test_rows_prepared_by_the_whole_device(ctx, vocab, kind):
    rng = np.random.default_rng(vocab)
    x = torch.from_numpy(rng.normal(0, 1.5, (len(PARAMS), vocab)).astype(np.float32))
    if kind == "bf16":
        x = x.to(torch.bfloat16)
    elif kind == "coarse":
        x = torch.round(x * 2) / 2
    _check(ctx, x.float().numpy(), x.cuda(), PARAMS, rng)


def test_rows_with_a_sharp_head_and_rows_with_equal_logits(ctx):
    rng = np.random.default_rng(3)
    logits = rng.normal(0, 1.5, (len(PARAMS), 20_011)).astype(np.float32)
    logits[:, 4_321] = 40.0                        # lists of a single entry
    _check(ctx, logits, torch.from_numpy(logits).cuda(), PARAMS, rng)
    logits[:] = 0.25                               # every entry in the first bucket
    _check(ctx, logits, torch.from_numpy(logits).cuda(), PARAMS, rng)
    logits[:, 9:] = float("-inf")
    _check(ctx, logits, torch.from_numpy(logits).cuda(), PARAMS, rng)


def test_launches_of_more_rows_than_the_whole_device_takes(ctx):
    rng = np.random.default_rng(4)
    base = rng.normal(0, 1.5, (len(PARAMS), 66_000)).astype(np.float32)
    rows = 520                                     # 65 segments each: beyond the limits of tokens and distributions
    params = [PARAMS[i % len(PARAMS)] for i in range(rows)]
    u = np.repeat(rng.random(rows // len(PARAMS) + 1), len(PARAMS))[:rows]
    dev = torch.from_numpy(base).cuda()[torch.arange(rows, device="cuda") % len(PARAMS)].contiguous()
    got = ctx.sample_batch(dev, params, u)
    want = oracle_tokens(base[np.arange(18) % len(PARAMS)], params[:18], u[:18])
    assert np.array_equal(got[:18], want)
    few = ctx.sample_batch(dev[:90], params[:90], u[:90])
    assert np.array_equal(got[:90], few)


@pytest.mark.parametrize("vocab", [8_191, 40_003])
@pytest.mark.parametrize("spread", [0.0, 0.02, 6.0, 60.0])
def test_rows_whose_mass_lies_anywhere_between_one_size_and_many(ctx, vocab, spread):
    """What a row's workgroups add up by size decides how much of the row is listed: mass in one bucket (to its full count of a
    workgroup, 8,192 equal entries), around a boundary of two, over every doubling that there is, in zeros and denormals."""
    rng = np.random.default_rng(int(10 * spread))
    logits = (-spread * rng.random((len(PARAMS), vocab))).astype(np.float32)
    logits[:, vocab // 2] = 0.0
    if spread == 60.0:
        logits[:, ::3] -= 60.0                     # e down to 1e-52: denormals, zeros
    _check(ctx, logits, torch.from_numpy(logits).cuda(), PARAMS, rng)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows,candidates", [(9, 16_383), (9, 16_384), (9, 16_385), (9, 18_700), (9, 40_003), (300, 4_096), (300, 4_097), (300, 4_800)])
def test_lists_around_the_longest_that_a_row_takes(ctx, rows, candidates, dtype):
    """`candidates` entries near the maximum, the rest far below: lists that just fit, that do not but cannot be told from the
    sums by size, and that are not made; rows at odd addresses, with a compute unit each and without."""
    vocab = 40_003
    rng = np.random.default_rng(candidates)
    base = rng.normal(-30.0, 0.5, (9, vocab)).astype(np.float32)
    for r in range(9):
        at = rng.permutation(vocab)[:candidates]
        base[r, at] = 3.0 + 0.25 * rng.random(candidates).astype(np.float32) * (r % 3)
    x = torch.from_numpy(base).to(torch.bfloat16 if dtype == "bf16" else torch.float32)
    base = x.float().numpy()
    some = [SamplingParams(TopP=0.9999), SamplingParams(MinP=0.3), SamplingParams(MinP=0.3, TopP=0.9), SamplingParams(TopP=0.6),
            SamplingParams(MinP=0.02, TopP=0.999), SamplingParams(MinP=0.9), SamplingParams(TopP=0.9999, FrequencyPenalty=0.1, PreviousTokens=[1, 2, 2]),
            SamplingParams(MinP=0.3, TopP=0.2), SamplingParams(Temperature=2.0, TopP=0.9)]
    params, u = [some[i % 9] for i in range(rows)], np.repeat(rng.random(rows // 9 + 1), 9)[:rows]
    dev = x.cuda()[torch.arange(rows, device="cuda") % 9].contiguous()
    few = rows if rows < 20 else 18
    logits = base[np.arange(few) % 9]
    got = ctx.sample_batch(dev, params, u)
    assert np.array_equal(got[:few], oracle_tokens(logits, params[:few], u[:few]))
    tokens, probs = ctx.sample_with_distribution(dev, params, u)
    assert np.array_equal(tokens, got)
    for r in range(9):
        want = orc.build_filtered_distribution(logits[r], to_oracle(params[r]))
        assert np.array_equal(probs[r].cpu().numpy().view(np.uint32), want.view(np.uint32)), r


@pytest.mark.parametrize("vocab", [8, 900, 4_095, 1_048_577])
def test_rows_that_their_own_workgroup_adds(ctx, vocab):
    """Too short or too long for the whole device, cut by min-p: nothing but the maximum left, a few entries, as many as the
    survivors' list holds and more, a threshold too small to bound anything."""
    rng = np.random.default_rng(vocab)
    some = [SamplingParams(MinP=0.3), SamplingParams(MinP=0.05, TopP=0.9), SamplingParams(Temperature=2.0, MinP=0.002), SamplingParams(MinP=1e-33),
            SamplingParams(MinP=1.0), SamplingParams(Temperature=0.5, MinP=0.01, PresencePenalty=0.5, PreviousTokens=[3, 3, 5])]
    some = some[:3] if vocab > 1_000_000 else some
    logits = rng.normal(0, 1.5, (len(some), vocab)).astype(np.float32)
    _check(ctx, logits, torch.from_numpy(logits).cuda(), some, rng)
    at = rng.permutation(vocab)
    for close in (vocab, 4_097, 4_096):            # equal entries at the top: as many as the list holds, one more, all
        logits[:] = -9.0
        logits[:, at[:close]] = 1.0
        _check(ctx, logits, torch.from_numpy(logits).cuda(), some, rng)
        if close >= vocab and vocab < 4_096:
            break


@pytest.mark.parametrize("vocab", [16_385, 40_000, 98_305, 131_072])
@pytest.mark.parametrize("rows", [1, 17, 40])
def test_launches_that_min_p_alone_cuts(ctx, vocab, rows):
    """On both sides of the lines between the whole device and the row's workgroup: distributions of few long rows, of more and of
    shorter ones, with a handful, hundreds and most of the entries left."""
    rng = np.random.default_rng(vocab + rows)
    some = [SamplingParams(MinP=0.05), SamplingParams(Temperature=2.0, MinP=0.002, TopP=0.9), SamplingParams(Temperature=30.0, MinP=0.6)]
    base = rng.normal(0, 1.5, (3, vocab)).astype(np.float32)
    base[0, :20] += 12.0 * np.arange(1, 21, dtype=np.float32) ** -1.1
    params, u = [some[i % 3] for i in range(rows)], rng.random(rows)
    x = torch.from_numpy(base).cuda()[torch.arange(rows, device="cuda") % 3].contiguous()
    tokens, probs = ctx.sample_with_distribution(x, params, u)
    few = min(rows, 6)
    logits = base[np.arange(few) % 3]
    want = oracle_tokens(logits, params[:few], u[:few])
    assert np.array_equal(tokens[:few], want)
    assert np.array_equal(ctx.sample_batch(x, params, u), tokens)
    for r in range(rows):
        assert torch.equal(probs[r], probs[r % 3])
    for r in range(min(rows, 3)):
        want = orc.build_filtered_distribution(logits[r], to_oracle(params[r]))
        assert np.array_equal(probs[r].cpu().numpy().view(np.uint32), want.view(np.uint32)), r


def test_masked_biased_and_penalised_rows(ctx):
    """Allow-masks from three tokens to nearly all, logit bias (on ids that are masked, outside the vocabulary, enough to change the
    maximum) and long histories, on every way that a prepared row takes; distributions built alone as well."""
    rng = np.random.default_rng(8)
    vocab = 50_021
    some = [SamplingParams(), SamplingParams(TopP=0.9), SamplingParams(Temperature=1.5, TopP=0.98), SamplingParams(MinP=0.02),
            SamplingParams(Temperature=0.7, MinP=0.001, TopP=0.95)]
    rows = 3 * len(some)
    logits = rng.normal(0, 1.5, (rows, vocab)).astype(np.float32)
    allowed = np.ones((rows, vocab), dtype=bool)
    params = []
    for r in range(rows):
        p = some[r % len(some)]
        if r < 5:
            allowed[r] = rng.random(vocab) < (0.5, 0.01, 0.9, 0.3, 0.05)[r]
            allowed[r, [3, 4_000, vocab - 1]] = True
        elif r < 10:
            ids = [int(i) for i in rng.integers(0, vocab, 40)] + [0, vocab - 1]
            p = SamplingParams(Temperature=p.Temperature, TopP=p.TopP, MinP=p.MinP, LogitBias={**{i: float(b) for i, b in zip(ids, rng.normal(0, 4, len(ids)))}, 7: 9.5, vocab + 3: 50.0})
        else:
            p = SamplingParams(Temperature=p.Temperature, TopP=p.TopP, MinP=p.MinP, RepetitionPenalty=1.3, FrequencyPenalty=0.2,
                               RepeatLastN=300, PreviousTokens=[int(i) for i in rng.integers(0, vocab, 700)])
        params.append(p)
    allowed[12, ::2] = False                       # a mask beside penalties
    allowed[6, 7] = False                          # ... and in front of a bias
    mask = pack_allow_mask(allowed)
    u = rng.random(rows)
    got = ctx.sample_batch(torch.from_numpy(logits).cuda(), params, u, mask)
    assert np.array_equal(got, oracle_tokens(logits, params, u, mask))
    masked = np.where(allowed, logits, -np.inf).astype(np.float32)
    with_masks = ctx.build_distribution(torch.from_numpy(logits).cuda(), params, allow_mask=mask).cpu().numpy()
    tokens, drawn_from = ctx.sample_with_distribution(torch.from_numpy(masked).cuda(), params, u)
    for r, p in enumerate(params):
        want = orc.build_filtered_distribution(masked[r], to_oracle(p))
        assert np.array_equal(with_masks[r].view(np.uint32), want.view(np.uint32)), r
        assert np.array_equal(drawn_from[r].cpu().numpy().view(np.uint32), want.view(np.uint32)), r
    assert np.array_equal(tokens, got)
