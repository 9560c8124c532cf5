"""BetaE, the one-call backward with Adam that finishes rows of one pair in the stream of the query gradient: full batches of
64 pairs, several of them, and every number of such rows in one, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.util import REL_F32, assert_close, seed

pytestmark = pytest.mark.gpu


# Pairs that are a segment of their own, per wavefront of eight and per batch of 64: none, all, all but one, odd and even counts.
# K = 512: full batches; 520: 64 + 1; 1,024: two full batches; 300: 38 each, the last one 34.  Features on both sides of 256: two
# rows requested at a time and one.
@pytest.mark.parametrize("k", [300, 512, 520, 1024])
@pytest.mark.parametrize("dim", [64, 128, 256, 260, 400])
def test_rows_in_the_stream_in_every_batch(dim, k):
    rng = np.random.default_rng(seed("beta rows in the stream", dim, k))
    b, per_wave = 4, -(-k // 8)
    hot = 24                               # ids that occur again and again
    idx, fresh = np.empty((b, k), dtype=np.int64), hot
    counts = iter(rng.permutation([0, 1, 2, 31, 32, 33, 62, 63, 64] * 16))
    for q in range(b):
        idx[q] = np.arange(k) % hot
        for first in range(0, k, per_wave):
            for at in range(first, min(first + per_wave, k), 64):
                cnt = min(64, first + per_wave - at, k - at)
                n = min(int(next(counts)), cnt)
                idx[q, at + np.sort(rng.permutation(cnt)[:n])] = fresh + np.arange(n)
                fresh += n
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    place = rng.permutation(fresh + 50)
    raw = f32(rng.standard_normal((fresh + 50, 2 * dim)) * 0.5)
    qa, qb = (f32(np.clip(1 + 0.5 * rng.standard_normal((b, dim)), 0.05, 1e9)) for _ in range(2))
    one_step(raw, qa, qb, place[idx], f32(rng.standard_normal((b, k))))


def one_step(raw, qa, qb, idx, gs):
    """Scores, query gradients and the one-call backward with Adam, against the oracle."""
    from smore_amd import fused
    n, dim, (b, k) = raw.shape[0], qa.shape[1], idx.shape
    rows = orc.gather(orc.regularizer(raw), idx).reshape(b, k, -1)
    want = orc.score_forward("beta_kl", rows, qa[:, None], qb[:, None], 60.0)
    g_rows, g_a, g_b = orc.score_backward("beta_kl", gs, rows, qa[:, None], qb[:, None])
    uniq, inverse, _, _ = orc.merge_indices(idx)
    merged = orc.merge_grads(g_rows.reshape(b * k, -1), inverse, uniq.size)
    terms = orc.merge_grads(np.abs(g_rows).reshape(b * k, -1), inverse, uniq.size)
    merged *= raw[uniq] + 1 >= 0.05

    dev = lambda x: torch.tensor(x, dtype=torch.float32, device="cuda")
    table, q1, q2, g, ids = dev(raw), dev(qa), dev(qb), dev(gs), torch.tensor(idx, device="cuda")
    params = fused.score_params(60.0, 0.0, regularizer=(1.0, 0.05, 1e9))
    score = fused.score_forward("beta_kl", table, ids, q1, q2, params)
    assert_close(score.cpu().numpy(), want, REL_F32, "score")
    gq = fused.score_backward_query("beta_kl", table, ids, q1, q2, score, g, params)
    plan = fused.build_plan(ids, n)
    assert (plan.pair_seg < 0).any() and (plan.pair_seg >= 0).any()
    m, v = torch.zeros_like(table), torch.zeros_like(table)
    one = fused.score_backward_fused("beta_kl", plan, table, ids, q1, q2, score, g, params, m=m, v=v, adam=fused.adam_params(1e-3, 1))
    for got, ref in ((gq[0], g_a), (gq[1], g_b), (one[0], g_a), (one[1], g_b)):
        # a sum over k terms of either sign: one ulp of their magnitudes is the floor of any order
        assert_close(got.cpu().numpy(), ref[:, 0], REL_F32, "query gradient", sum_abs=np.abs(gs).sum(1)[:, None] * np.ones(dim))
    assert_close(m.cpu().numpy()[uniq], 0.1 * merged, REL_F32, "first moments", sum_abs=0.1 * terms)
    assert_close(v.cpu().numpy()[uniq], 1e-3 * merged ** 2, 2 * REL_F32, "second moments", sum_abs=2e-3 * np.abs(merged) * terms)
    untouched = np.setdiff1d(np.arange(n), uniq)
    assert not m[untouched].any() and torch.equal(table[untouched], dev(raw)[untouched])
    w = raw.copy()
    orc.adam_rows(w, np.zeros_like(raw), np.zeros_like(raw), uniq, m.cpu().numpy()[uniq].astype(np.float64) / np.float32(0.1), 1e-3, 1)
    # a first step moves a weight by at most the learning rate, known to a few ulps from the moments the device holds
    assert np.all(np.abs(table.cpu().numpy()[uniq] - w[uniq]) <= 1e-3 * 1e-4 + 2.0 ** -22 * np.abs(w[uniq]))


# queries of more than 4 MiB: rows of one pair are finished by the query-gradient kernel whatever the optimizer
@pytest.mark.parametrize("kind", ["merged", "squeeze", "adam and merged"])
@pytest.mark.parametrize("dim,b", [(64, 8300), (260, 2100), (516, 1100), (33, 16000)])
def test_rows_finished_outside_the_stream(dim, b, kind):
    """The one call against its two halves: query gradients, and the entity pass's rows."""
    from smore_amd import fused
    rng = np.random.default_rng(seed("outside the stream", dim, kind))
    k = 70
    n = b * k // 2
    table = torch.tensor(rng.standard_normal((n, 2 * dim)) * 0.5, dtype=torch.float32, device="cuda")
    q1, q2 = (torch.tensor(np.clip(1 + 0.5 * rng.standard_normal((b, dim)), 0.05, None), dtype=torch.float32, device="cuda") for _ in range(2))
    ids = torch.tensor(rng.integers(0, n, (b, k)), device="cuda")
    g = torch.tensor(rng.standard_normal((b, k)), dtype=torch.float32, device="cuda")
    params = fused.score_params(60.0, 0.0, regularizer=(1.0, 0.05, 1e9))
    score = fused.score_forward("beta_kl", table, ids, q1, q2, params)
    plan = fused.build_plan(ids, n)
    want_q = fused.score_backward_query("beta_kl", table, ids, q1, q2, score, g, params)
    want = torch.empty(plan.uniq.numel(), 2 * dim, device="cuda")
    fused.score_backward_entity("beta_kl", plan, table, q1, q2, score, g, params, merged=want)
    merged = None if kind == "squeeze" else torch.empty_like(want)
    state = {}
    if kind != "merged":
        squeeze = kind == "squeeze"
        state = dict(m=torch.zeros_like(table), v=torch.zeros(n, 1, device="cuda") if squeeze else torch.zeros_like(table),
                     adam=fused.adam_params(1e-3, 1, squeeze=squeeze))
    got_q = fused.score_backward_fused("beta_kl", plan, table, ids, q1, q2, score, g, params, merged=merged, **state)
    uniq = plan.uniq[:int(plan.n_uniq)]
    want = want[:uniq.numel()]
    for a, w in zip(got_q, want_q):
        # the wavefronts' sums may be of other lengths: an ulp of the terms' magnitudes
        assert_close(a.cpu().numpy(), w.cpu().numpy(), REL_F32, "query gradient", sum_abs=g.abs().sum(1, keepdim=True).cpu().numpy() * np.ones(dim))
    if merged is not None:
        assert_close(merged[:uniq.numel()].cpu().numpy(), want.cpu().numpy(), REL_F32, "merged rows")
    if state:
        assert_close(state["m"][uniq].cpu().numpy(), 0.1 * want.cpu().numpy(), REL_F32, "first moments")
