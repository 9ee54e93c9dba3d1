"""Rows whose largest entry decides the token: around the lines where it just does and just does not, in every shape of the
launch that asks.  Tokens are the oracle's, and tokens and flags those of the way that never asks (forced from the host: a poll limit
of zero for the kernels' bounded waits)."""

import numpy as np
import pytest
from opentail.stingray_amd import SamplerContext, SamplingParams, pack_allow_mask, synthetic
from tests.helpers import hooks_lib, oracle_tokens

pytestmark = pytest.mark.gpu
CHUNK = 512 * 19 * 4  # elements of a worker's chunk of fp32 logits


@pytest.fixture()
def ctx():
    c = SamplerContext(0)
    yield c
    c.close()


def _rows(rng, rows, vocab, top_k, bf16):
    """Rows with one entry well above the rest: `gap` nats above all others that count together.  top-p, min-p and the uniform lie on both
    sides of what that entry covers, some within a few roundings of it."""
    logits = rng.normal(0, 1, (rows, vocab)).astype(np.float32)
    params, u = [], rng.random(rows)
    for r in range(rows):
        k = int(rng.integers(2, top_k + 1)) if top_k else 0
        t = float(np.float32(rng.uniform(0.4, 1.3)))
        x = np.sort(logits[r].astype(np.float64))[::-1][: k - 1 if k else None] / t
        rest = x[0] + np.log(np.exp(x - x[0]).sum())
        gap = rng.uniform(-1.0, 7.0)
        at = int(rng.choice([0, vocab - 1, int(rng.integers(vocab))]))
        raised = 0.0
        p = SamplingParams(Temperature=t, TopK=k)
        if r % 3 == 1:  # the entry is in the history, and what the penalty takes away was added
            p.PresencePenalty, p.FrequencyPenalty = 0.25, 0.125
            p.PreviousTokens = rng.integers(0, vocab, 40).tolist() + ([at] * 3 if r % 2 else [])
            raised = 0.25 + 0.125 * p.PreviousTokens.count(at) if at in p.PreviousTokens else 0.0
        logits[r, at] = np.float32((rest + gap) * t + raised)
        covers = 1.0 / (1.0 + np.exp(-gap))
        near = covers * (1.0 + float(rng.choice([-1e-2, -1e-3, -2e-4, -1e-6, 0.0, 1e-6, 1e-3])))
        kind = r % 4
        if kind == 0:
            p.TopP = float(np.float32(min(near, 0.9999)))
        elif kind == 1:
            p.MinP = float(np.float32(np.exp(x[0] - rest - gap) * rng.choice([0.5, 1.0, 1.001, 2.0, 50.0])))
            p.TopP = float(rng.choice([1.0, 0.9]))
        elif kind == 2:
            u[r] = min(near, 0.9999999)
        if r % 7 == 3:
            u[r] = rng.choice([0.0, 1e-7, 1e-6, 0.9999995, 0.99999997])
        if r % 11 == 5:
            logits[r, (at + vocab // 2) % vocab] = logits[r, at]  # not the only one
        params.append(p)
    if bf16:
        logits = synthetic.bf16_bits_to_f32(synthetic.to_bf16_bits(logits))
    return logits, params, u


def _check(ctx, rng, rows, vocab, top_k, bf16, rounds, make=_rows):
    import torch

    h = hooks_lib()
    for _ in range(rounds):
        logits, params, u, *masks = make(rng, rows, vocab, top_k, bf16)
        dev = torch.from_numpy(logits).cuda()
        if bf16:
            dev = dev.to(torch.bfloat16)
        got, flags = ctx.sample_batch(dev, params, u, *masks, return_flags=True)
        want = oracle_tokens(logits, params, u, *masks)
        assert np.array_equal(got, want), np.nonzero(got != want)[0][:10]
        h.sr_debug_set_spin_limit(ctx.h, 0)
        h.sr_debug_set_row_wait_limit(ctx.h, 0)
        other, other_flags = ctx.sample_batch(dev, params, u, *masks, return_flags=True)
        h.sr_debug_set_spin_limit(ctx.h, 1 << 22)
        h.sr_debug_set_row_wait_limit(ctx.h, 1 << 15)
        assert np.array_equal(got, other)
        assert np.array_equal(flags, other_flags), np.nonzero(flags != other_flags)[0][:10]


# Dealt rows of one and of several chunks, short and long lists; chunks that join in pairs; a row to a worker; two workers to a
# compute unit; more of them than that.
@pytest.mark.parametrize("rows,vocab,top_k,bf16", [
    (1, 49_152, 40, False), (9, 4 * CHUNK - 1, 64, False), (24, 100_003, 300, True), (7, 6 * CHUNK + 3, 500, False), (5, 5 * CHUNK, 64, False),
    (20, 12_345, 50, False), (270, 9_001, 900, False), (300, 20_011, 60, True), (530, 16_384, 200, False), (260, 4 * CHUNK + 9, 100, False)])
def test_rows_that_their_largest_entry_decides(ctx, rows, vocab, top_k, bf16):
    _check(ctx, np.random.default_rng(rows + vocab), rows, vocab, top_k, bf16, 12 if rows < 10 else 3 if rows < 100 else 1)


def _scaled(x, t):
    """fl(x / T) as the sampler takes it: times a rounded 1 / T."""
    return np.asarray(x, dtype=np.float32) * (np.float32(1.0) / np.float32(t))


def _cold_rows(rng, rows, vocab, top_k, bf16, most):
    """Two entries a few of their last places apart, far above the rest, at temperatures at which the roundings of x / T are as large as what
    lies between them: what the larger one covers by the values as they stand and by the scaled, rounded ones differs, and the uniform or top-p
    lies in between, or near it.  |x| / T up to about `most`; beyond 1e9 some rows' scaled maximum is no finite number."""
    logits = rng.normal(-5, 1, (rows, vocab)).astype(np.float32)
    params, u = [], rng.random(rows)
    for r in range(rows):
        size = float(rng.choice([0.7, 20.0, 28.0, 300.0, 1e4])) * rng.uniform(0.7, 1.3)
        t = np.float32(max(10.0 ** rng.uniform(-5.2, -2), size / most))
        if r % 5 == 2:
            size = -size
            logits[r] = np.float32(4 * size - 1.0) + logits[r]
        at, other = (int(i) for i in rng.choice(vocab, 2, replace=False))
        p = SamplingParams(Temperature=float(t), TopK=int(rng.integers(2, top_k + 1)))
        x0 = np.float32(size)
        if bf16:
            x0 = synthetic.bf16_bits_to_f32(synthetic.to_bf16_bits(np.array([x0])))[0]
        if r % 3 == 1:  # one of them, or both, through the history
            p.PresencePenalty, p.FrequencyPenalty = 0.25, 0.125
            p.PreviousTokens = rng.integers(0, vocab, 30).tolist() + [at] * 3 + ([other] if r % 2 else [])
        gap = float(rng.choice([0.3, 1.0, 2.0, 4.0])) * float(t)  # ... of each other, or the next value below if that is more
        x1 = np.float32(float(x0) - gap)
        if bf16:
            x1 = synthetic.bf16_bits_to_f32(synthetic.to_bf16_bits(np.array([x1])))[0]
        if x1 == x0:
            x1 = np.nextafter(x0, np.float32(-np.inf)) if not bf16 else x0
        logits[r, at], logits[r, other] = x0, x1
        # what they have behind the penalties, and what the larger one covers, by differences as they stand and by scaled values
        adj = {}
        for i in (at, other):
            v, c = logits[r, i], (p.PreviousTokens or []).count(i)
            adj[i] = v - (np.float32(0.25) + np.float32(0.125) * np.float32(c)) if c else v
        hi, lo = max(adj.values()), min(adj.values())
        with np.errstate(over="ignore", invalid="ignore"):
            stands = 1.0 / (1.0 + np.exp(-(float(hi) - float(lo)) / float(t)))
            scaled = 1.0 / (1.0 + np.exp(-float(_scaled(hi, t) - _scaled(lo, t))))
        line = float(rng.choice([stands, scaled, 0.5 * (stands + scaled)])) * (1.0 + float(rng.choice([-1e-2, -6e-4, -1e-5, 0.0, 1e-5])))
        line = min(max(line, 0.0), 0.9999999)
        if r % 2:
            p.TopP = float(np.float32(min(max(line, 1e-3), 0.9999)))
            u[r] = rng.choice([0.3, 0.8, 0.999])
        else:
            u[r] = line
        if r % 4 == 3:
            p.MinP = float(np.float32(rng.choice([0.02, 0.4, 0.9])))
        if most > 1e9 and r % 13 == 6:
            p.Temperature = float(np.float32(rng.choice([1e-35, 1e-38])))
        params.append(p)
    if bf16:
        logits = synthetic.bf16_bits_to_f32(synthetic.to_bf16_bits(logits))
    return logits, params, u


# (from |x| / T of some 1e7 on, entries tens of T below the largest may have its scaled value)
@pytest.mark.parametrize("most", [8e6, 4e9])
@pytest.mark.parametrize("rows,vocab,top_k,bf16", [
    (1, 49_152, 40, False), (20, 12_345, 50, False), (24, 100_003, 300, False), (24, 30_001, 300, True), (7, 6 * CHUNK + 3, 500, False), (300, 20_011, 60, False),
    (200, 40_000, 900, False), (530, 16_384, 200, False), (530, 9_001, 50, True)])
def test_rows_at_temperatures_at_which_scaled_values_round_apart(ctx, rows, vocab, top_k, bf16, most):
    _check(ctx, np.random.default_rng(rows + vocab), rows, vocab, top_k, bf16, 24 if rows == 1 else 6 if rows < 100 else 1,
           lambda *how: _cold_rows(*how, most))


def test_a_row_at_a_thousandth_whose_draw_lies_between_the_two(ctx):
    import torch

    logits = np.full((1, 49_152), -5.0, dtype=np.float32)
    logits[0, 100], logits[0, 200] = 28.457004547, 28.456491470
    params, u = [SamplingParams(Temperature=1e-3, TopK=40)], np.array([0.6252147])
    assert oracle_tokens(logits, params, u)[0] == 200
    assert ctx.sample_batch(torch.from_numpy(logits).cuda(), params, u)[0] == 200


# The full-vocabulary path: one, two and four segments a wave, rows that end inside a segment, rows of odd addresses, several turns of workgroups.
@pytest.mark.parametrize("rows,vocab,bf16", [(1, 4_096, False), (3, 5_001, False), (30, 100_003, True), (33, 100_003, False), (6, 262_144, False),
                                             (66, 200_064, False), (40, 50_257, True), (280, 16_385, False)])
def test_rows_of_the_whole_vocabulary_that_their_largest_entry_decides(ctx, rows, vocab, bf16):
    _check(ctx, np.random.default_rng(rows + vocab), rows, vocab, 0, bf16, 8 if rows < 10 else 2 if rows < 50 else 1)


def _odd_rows(rng, rows, vocab, top_k, bf16):
    """Every second entry is masked away, far above all others; the largest of the rest carries a bias where no top-k is asked for.  Some
    rows hold a NaN, a +inf, one or two finite entries, or values a thousand times as large at as many times the temperature."""
    half, params, u = _rows(rng, rows, vocab // 2, top_k, False)
    logits = np.full((rows, vocab), 60.0, dtype=np.float32)
    allowed = np.zeros((rows, vocab), dtype=bool)
    allowed[:, 1:2 * (vocab // 2):2] = True
    for r in range(rows):
        at, p = int(np.argmax(half[r])), params[r]
        if p.PreviousTokens:
            p.PreviousTokens = [2 * t + 1 for t in p.PreviousTokens]
        if not top_k and r % 2:
            half[r, at] -= np.float32(2.0)
            p.LogitBias = {2 * at + 1: 2.0, 2 * int(rng.integers(vocab // 2)): -1.0}
        odd = r % 9
        if odd == 1:
            half[r, rng.integers(vocab // 2)] = np.nan
        elif odd == 2:
            half[r, rng.integers(vocab // 2)] = np.inf
        elif odd in (3, 4):
            keep = rng.choice(vocab // 2, odd - 2, replace=False)
            half[r] = np.where(np.isin(np.arange(vocab // 2), keep), half[r], -np.inf)
        elif odd in (5, 6) and not p.PreviousTokens and not p.LogitBias:
            half[r] *= np.float32(1000.0)
            p.Temperature *= 1000.0
        logits[r, 1:2 * (vocab // 2):2] = half[r]
    if bf16:
        logits = synthetic.bf16_bits_to_f32(synthetic.to_bf16_bits(logits))
    return logits, params, u, pack_allow_mask(allowed), np.ones(rows, dtype=np.uint8)


@pytest.mark.parametrize("rows,vocab,top_k,bf16", [(9, 40_000, 50, False), (20, 100_003, 300, True), (540, 16_385, 60, False), (9, 50_001, 0, False),
                                                   (40, 100_003, 0, True), (70, 151_936, 0, False)])
def test_masked_and_biased_rows_and_odd_values_of_which_the_largest_may_decide(ctx, rows, vocab, top_k, bf16):
    _check(ctx, np.random.default_rng(rows + vocab + top_k), rows, vocab, top_k, bf16, 8 if rows < 10 else 2 if rows < 50 else 1, _odd_rows)


# A row whose largest entry decides is written by the pass, once: not again by the launch behind it, although some workgroup of the row has
# stopped waiting.  A row that nothing decided gets its token there.
@pytest.mark.parametrize("rows,vocab,bf16", [(1, 49_152, False), (40, 100_003, True), (30, 151_936, False)])
def test_a_decided_row_that_a_workgroup_has_marked_late_is_not_written_again(ctx, rows, vocab, bf16):
    import torch

    h, none = hooks_lib(), -77
    rng = np.random.default_rng(rows)
    seen = set()
    for _ in range(24 if rows == 1 else 2):
        logits, params, u = _rows(rng, rows, vocab, 0, bf16)
        dev = torch.from_numpy(logits).cuda()
        if bf16:
            dev = dev.to(torch.bfloat16)
        batch = ctx.new_batch().upload(params, vocab, u)
        tok, flags = (torch.zeros(rows, dtype=torch.int32, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        ctx._check(h.sr_selftest_late_rows(ctx.h, batch.h, dev.data_ptr(), int(bf16), vocab, none, tok.data_ptr(), flags.data_ptr()))
        got, want, left = tok.cpu().numpy(), oracle_tokens(logits, params, u), flags.cpu().numpy() == none
        assert np.array_equal(got == none, left)
        assert np.array_equal(got[~left], want[~left])
        seen |= set(left.tolist())
        for polls in (1, 2, 3, 6):  # (few enough that some workgroups leave and others decide; results in pinned memory, call after call)
            h.sr_debug_set_row_wait_limit(ctx.h, polls)
            assert np.array_equal(ctx.sample_batch(dev, params, u), want), polls
        h.sr_debug_set_row_wait_limit(ctx.h, 1 << 15)
        batch.close()
    assert seen == {False, True}


# ... and where the distribution is handed out beside the token, that is written whole, by two launches (many rows) and by one: rows that nothing
# cuts, nuclei and min-p cuts of a few entries.
@pytest.mark.parametrize("rows,vocab,bf16", [(3, 20_001, False), (12, 100_003, True), (20, 65_536, False), (90, 65_537, False)])
def test_distributions_of_rows_that_their_largest_entry_decides(ctx, rows, vocab, bf16):
    import torch
    from oracle import binding as orc
    from tests.helpers import to_oracle

    rng = np.random.default_rng(rows * vocab)
    for _ in range(2):
        logits, params, u = _rows(rng, rows, vocab, 0, bf16)
        dev = torch.from_numpy(logits).cuda()
        if bf16:
            dev = dev.to(torch.bfloat16)
        toks, probs = ctx.sample_with_distribution(dev, params, u)
        alone = ctx.build_distribution(dev, params).cpu().numpy()
        probs = probs.cpu().numpy()
        assert np.array_equal(toks, oracle_tokens(logits, params, u)), np.nonzero(toks != oracle_tokens(logits, params, u))[0][:10]
        for r in range(rows):
            want = orc.build_filtered_distribution(logits[r], to_oracle(params[r]))
            assert np.array_equal(probs[r], want) and np.array_equal(alone[r], want), r

# Verifications: sequences whose drafts are all accepted for certain, where the bonus row's largest entry is its token or is not, beside some that
# reject a draft and some with up to three tests too close to tell from about the sums.  A row and a half of blocks, one entry in a unit of its own, a
# block's last entry; short rows, many positions (of which several are worked out side by side).
@pytest.mark.parametrize("rows,drafts,vocab", [(16, 2, 50_001), (9, 8, 65_537), (3, 4, 262_144), (40, 7, 8_193), (300, 1, 4_096), (2, 3, 16_385), (16, 8, 20_011)])
def test_bonus_rows_that_their_largest_entry_decides(ctx, rows, drafts, vocab):
    import torch
    from oracle import binding as orc
    from tests.helpers import to_oracle

    rng = np.random.default_rng(rows + vocab)
    rejected = close = 0
    for turn in range(3 if rows < 100 else 1):
        t = rng.normal(0, 1, (rows, drafts + 1, vocab)).astype(np.float32)
        u = rng.uniform(0.05, 0.5, (rows, drafts + 1))
        temps = [float(np.float32(rng.choice([1.0, rng.uniform(0.5, 1.3)]))) for _ in range(rows)]
        k = rng.integers(0, vocab, (rows, drafts))
        q = np.full((rows, drafts, vocab), 1e-9, dtype=np.float32)
        for r in range(rows):
            for i in range(drafts):
                t[r, i, k[r, i]] = 30.0  # accepted for certain
                q[r, i, k[r, i]] = 0.9
            x = t[r, drafts].astype(np.float64) / temps[r]
            rest = x.max() + np.log(np.exp(x - x.max()).sum())
            gap = rng.uniform(-1.0, 7.0)
            at = int(rng.choice([0, vocab - 1, 8_191 % vocab, 2_048 % vocab, int(rng.integers(vocab))]))
            t[r, drafts, at] = np.float32((rest + gap) * temps[r])
            # the sum in front of the entry and behind it, of all
            x = t[r, drafts].astype(np.float64) / temps[r]
            p = np.exp(x - x.max())
            line = p[: at + int(rng.integers(2))].sum() / p.sum()
            u[r, drafts] = np.clip(line + rng.choice([-0.3, -3e-2, -1e-3, -1e-5, 0.0, 1e-5, 1e-3, 3e-2, 0.3]), 0.0, 0.99999999)
            if r % 9 == 4:
                u[r, drafts] = rng.choice([0.0, 1e-7, 0.9999999])
            if r % 9 == 5:
                t[r, drafts, (at + vocab // 2) % vocab] = t[r, drafts, at]  # not the only one
            kind = (r + turn) % 4
            if kind in (1, 2):  # a rejected draft, or up to three whose test is close: p about half of q, u above p / q or at it
                for i in rng.choice(drafts, 1 if kind == 1 else min(3, drafts), replace=False):
                    x = t[r, i].astype(np.float64) / temps[r]
                    x[k[r, i]] = -np.inf
                    t[r, i, k[r, i]] = np.float32((x.max() + np.log(np.exp(x - x.max()).sum()) + rng.uniform(-0.5, 0.2)) * temps[r])
                    x = t[r, i].astype(np.float64) / temps[r]
                    p = np.exp(x - x.max())
                    u[r, i] = 0.95 if kind == 1 else p[k[r, i]] / p.sum() / 0.9 * (1.0 + rng.choice([-2e-7, -1e-8, 0.0, 1e-8, 2e-7]))
                close += kind == 2
        params = [SamplingParams(Temperature=T) for T in temps]
        dev = [torch.from_numpy(v).cuda() for v in (t, q, k.astype(np.int32))]
        acc, tok = ctx.spec_verify(dev[0], dev[1], dev[2], params, u)
        for r in range(rows):
            wa, wt = orc.spec_verify_row(t[r], q[r], k[r], to_oracle(params[r]), orc.Rng(replay=u[r]))
            assert acc[r] == wa and np.array_equal(tok[r][: len(wt)], wt), (r, acc[r], wa, tok[r], wt)
            rejected += wa < drafts
    assert rejected > 0 and close > 0
