"""SR_OUT_AMBIGUOUS: the row's token is still the one the documented conventions give, but it rests on something the
managed runtime leaves open -- the draw or a cut lies within a few ulp of a boundary of the running sum (the lane
order of TensorPrimitives.Sum, Sampler.cs:555, and the last bit of MathF.Exp can move such a sum by an ulp or two), or
a top-p cut splits a run of equal probabilities (the unstable sort of Sampler.cs:533).  A managed caller re-runs such a
row on the CPU.  Tested here: draws placed exactly on a boundary are flagged (the boundary is found by bisecting the
oracle's own answer in u), draws in the middle of a token's interval are not, cuts inside runs of equal
probabilities are, and a random batch flags few rows."""
import numpy as np
import pytest

from opentail.stingray_amd import SR_OUT_AMBIGUOUS, SamplerContext, SamplingParams, synthetic
from oracle import binding as orc
from tests.helpers import oracle_tokens, to_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = SamplerContext(0)
    yield c
    c.close()


def _cuda(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _boundaries(row, p, n_want, rng):
    """Pairs (u_lo, u_hi) of adjacent doubles between which the oracle's token changes, and mid-interval u's."""
    op = to_oracle(p)
    on, mid = [], []
    for _ in range(200):
        a, b = sorted(rng.random(2))
        ta, tb = orc.sample_u(row, op, a), orc.sample_u(row, op, b)
        if ta == tb:
            continue
        for _ in range(80):                       # bisect down to neighbouring doubles
            m = 0.5 * (a + b)
            if m == a or m == b:
                break
            if orc.sample_u(row, op, m) == ta:
                a = m
            else:
                b, tb = m, orc.sample_u(row, op, m)
        on.extend([a, b])
        if len(on) >= n_want:
            break
    # a u whose token's interval in u is wide, taken at the interval's middle
    for _ in range(400):
        u = rng.random()
        t = orc.sample_u(row, op, u)
        d = 1e-4
        if orc.sample_u(row, op, max(u - d, 0.0)) == t and orc.sample_u(row, op, min(u + d, 1.0 - 1e-12)) == t:
            mid.append(u)
        if len(mid) >= n_want:
            break
    return on, mid


@pytest.mark.parametrize("kind", ["topk", "full_top_p", "full_min_p", "full_plain"])
def test_draws_on_a_boundary_are_flagged_and_draws_inside_an_interval_are_not(ctx, kind):
    rng = np.random.default_rng({"topk": 1, "full_top_p": 2, "full_min_p": 3, "full_plain": 4}[kind])
    V = 3_000
    row = rng.normal(0, 1.5, V).astype(np.float32)
    row[rng.integers(0, V, 8)] += np.linspace(6, 2, 8).astype(np.float32)
    p = {"topk": SamplingParams(Temperature=0.9, TopK=50, TopP=0.97),
         "full_top_p": SamplingParams(Temperature=0.8, TopP=0.9),
         "full_min_p": SamplingParams(Temperature=1.1, MinP=0.01),
         "full_plain": SamplingParams(Temperature=1.3)}[kind]
    on, mid = _boundaries(row, p, 12, rng)
    assert len(on) >= 8 and len(mid) >= 8
    us = np.array(on + mid)
    logits = np.tile(row, (len(us), 1))
    got, flags = ctx.sample_batch(_cuda(logits), [p] * len(us), us, return_flags=True)
    assert np.array_equal(got, oracle_tokens(logits, [p] * len(us), us))
    amb = (flags & SR_OUT_AMBIGUOUS) != 0
    assert amb[: len(on)].all(), (kind, np.nonzero(~amb[: len(on)])[0])
    assert not amb[len(on):].any(), (kind, np.nonzero(amb[len(on):])[0])


def test_a_top_p_cut_inside_a_run_of_equal_probabilities_is_flagged(ctx):
    V = 4_096
    rng = np.random.default_rng(9)
    flat = np.full(V, -4.0, dtype=np.float32)
    flat[:64] = 1.0                                   # 64 equal logits carry nearly all the mass; top-p cuts among them
    sharp = rng.normal(0, 1.0, V).astype(np.float32)
    sharp[7] = 9.0                                    # one token far above: the cut is nowhere near a tie
    params = [SamplingParams(Temperature=1.0, TopP=0.5), SamplingParams(Temperature=1.0, TopP=0.5)]
    logits = np.stack([flat, sharp])
    u = np.array([0.3, 0.3])
    got, flags = ctx.sample_batch(_cuda(logits), params, u, return_flags=True)
    assert np.array_equal(got, oracle_tokens(logits, params, u))
    assert flags[0] & SR_OUT_AMBIGUOUS and not flags[1] & SR_OUT_AMBIGUOUS


def test_a_random_batch_flags_few_rows(ctx):
    w = synthetic.config3(rows=256, bf16=False, full_chain=True)
    got, flags = ctx.sample_batch(_cuda(w.logits), w.params, w.uniforms, return_flags=True)
    assert np.array_equal(got, oracle_tokens(w.logits, w.params, w.uniforms))
    assert int(((flags & SR_OUT_AMBIGUOUS) != 0).sum()) <= 2
    w2 = synthetic.config2()
    got, flags = ctx.sample_batch(_cuda(w2.logits), w2.params, w2.uniforms, return_flags=True)
    assert int(((flags & SR_OUT_AMBIGUOUS) != 0).sum()) <= 1


# ---- rows that the whole device prepares (4,096 entries and more; normalised and drawn by it from 32,768 on) ---------------

LONG = {"short_list": SamplingParams(Temperature=0.35, TopP=0.9),  # a nucleus of a handful: one wave cuts and draws
        "list": SamplingParams(Temperature=0.8, TopP=0.5),          # hundreds: the row's workgroup
        "long_nucleus": SamplingParams(TopP=0.9),                   # thousands: the whole device
        "min_p": SamplingParams(Temperature=0.9, MinP=0.02),
        "min_p_top_p": SamplingParams(Temperature=0.9, MinP=0.1, TopP=0.9),
        "plain": SamplingParams(Temperature=1.2)}
# (how many members each has, which is what decides the way that the row takes)
LONG_MEMBERS = {"short_list": (4, 30), "list": (100, 1_000), "long_nucleus": (1_100, 16_000), "min_p": (100, 1_000),
                "min_p_top_p": (65, 1_000), "plain": (33_000, 33_000)}


def _long_row(rng):
    row = rng.normal(0, 1.5, 33_000).astype(np.float32)
    row[rng.integers(0, len(row), 12)] += np.linspace(6, 2, 12).astype(np.float32)
    return row


@pytest.mark.parametrize("kind", list(LONG))
def test_draws_of_long_rows_on_and_off_a_boundary(ctx, kind):
    rng = np.random.default_rng(list(LONG).index(kind) + 20)
    row, p = _long_row(rng), LONG[kind]
    lo, hi = LONG_MEMBERS[kind]
    assert lo <= int((orc.build_filtered_distribution(row, to_oracle(p)) > 0).sum()) <= hi
    on, mid = _boundaries(row, p, 8, rng)
    assert len(on) >= 6 and len(mid) >= 6
    us = np.array(on + mid)
    logits = np.tile(row, (len(us), 1))
    got, flags = ctx.sample_batch(_cuda(logits), [p] * len(us), us, return_flags=True)
    assert np.array_equal(got, oracle_tokens(logits, [p] * len(us), us))
    amb = (flags & SR_OUT_AMBIGUOUS) != 0
    assert amb[: len(on)].all(), (kind, np.nonzero(~amb[: len(on)])[0])
    assert not amb[len(on):].any(), (kind, np.nonzero(amb[len(on):])[0])


def test_cuts_of_long_rows_on_and_off_a_boundary(ctx):
    """top-p set to the running sum behind the k-th probability and min-p to the ratio of the k-th to the first: the cut is flagged
    wherever it is made, and not when it lies between two far apart."""
    rng = np.random.default_rng(31)
    row = _long_row(rng)
    e = np.exp(row - row.max())
    y = np.sort(e * np.float32(1.0 / np.cumsum(e, dtype=np.float32)[-1]))[::-1]
    run = np.cumsum(y, dtype=np.float32)
    params, want = [], []
    for k in (1, 9, 40, 300, 900, 1_500, 7_000):
        params += [SamplingParams(TopP=float(run[k])), SamplingParams(MinP=float(y[k] / y[0])), SamplingParams(MinP=1e-4, TopP=float(run[k]))]
        want += [True, True, True]
    for k in (1, 3, 6):                                # halfway between sums, between probabilities
        params += [SamplingParams(TopP=float(run[k] + y[k + 1] / 2)), SamplingParams(MinP=float((y[k] + y[k + 1]) / 2 / y[0]))]
        want += [False, False]
    u = np.full(len(params), 0.0)                      # (the first member: far from any boundary of the draw)
    first = int(np.argmax(row))
    row[[0, first]] = row[[first, 0]]                  # ... the row's largest entry, so that u = 0.2 of it draws it
    u[:] = 0.2 * float(y[0])
    logits = np.tile(row, (len(params), 1))
    got, flags = ctx.sample_batch(_cuda(logits), params, u, return_flags=True)
    assert np.array_equal(got, oracle_tokens(logits, params, u))
    amb = (flags & SR_OUT_AMBIGUOUS) != 0
    assert np.array_equal(amb, np.array(want)), [(i, params[i]) for i in np.nonzero(amb != np.array(want))[0]]


@pytest.mark.parametrize("run_length", [30, 500, 6_000])
def test_cuts_of_long_rows_inside_a_run_of_equal_probabilities_are_flagged(ctx, run_length):
    rng = np.random.default_rng(run_length)
    row = rng.normal(-12.0, 0.5, 33_000).astype(np.float32)
    row[rng.permutation(len(row))[:run_length]] = 2.0
    params = [SamplingParams(TopP=0.5), SamplingParams(MinP=0.5, TopP=0.5), SamplingParams(MinP=0.5)]  # (min-p keeps the whole run)
    logits = np.tile(row, (3, 1))
    u = np.full(3, 0.3)
    got, flags = ctx.sample_batch(_cuda(logits), params, u, return_flags=True)
    assert np.array_equal(got, oracle_tokens(logits, params, u))
    assert ((flags & SR_OUT_AMBIGUOUS) != 0).tolist()[:2] == [True, True]
