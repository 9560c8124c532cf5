"""BetaE rows of every number of floats per lane, with features inside and outside the interval of the fast forms, against
the oracle: scores, query gradients, and the one-call backward with Adam that finishes rows of one pair in its stream."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.util import REL_F32, assert_close, seed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [4, 64, 68, 128, 132, 192, 196, 256, 260, 320, 324, 384, 388, 448, 452, 512])
@pytest.mark.parametrize("clamped", [True, False])
def test_row_lengths(dim, clamped):
    from smore_amd import fused
    rng = np.random.default_rng(seed("beta rows", dim, clamped))
    n, b, k = 300, 5, 67                  # 335 pairs: a third of the touched rows occur once; 67: a remainder per wavefront
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    raw = f32(rng.standard_normal((n, 2 * dim)) * 0.5)
    if not clamped:
        raw = f32(np.clip(raw + 1.0, 0.05, None))
        raw[7, :] = f32(np.full(2 * dim, 0.004))      # below the interval
        raw[8, dim - 1] = 0.011
    raw[9, 0] = 1200.0                                # beyond it
    qa, qb = (f32(np.clip(1 + 0.5 * rng.standard_normal((b, dim)), 0.05, 1e9)) for _ in range(2))
    idx = rng.integers(0, n, (b, k))
    idx[0, :3] = (7, 8, 9)
    gs = f32(rng.standard_normal((b, k)))
    reg = orc.regularizer(raw) if clamped else raw
    rows = orc.gather(reg, idx).reshape(b, k, -1)
    want = orc.score_forward("beta_kl", rows, qa[:, None], qb[:, None], 60.0)
    g_rows, g_a, g_b = orc.score_backward("beta_kl", gs, rows, qa[:, None], qb[:, None])
    uniq, inverse, _, _ = orc.merge_indices(idx)
    merged = orc.merge_grads(g_rows.reshape(b * k, -1), inverse, uniq.size)
    terms = orc.merge_grads(np.abs(g_rows).reshape(b * k, -1), inverse, uniq.size)
    if clamped:
        merged *= raw[uniq] + 1 >= 0.05

    dev = lambda x: torch.tensor(x, dtype=torch.float32, device="cuda")
    table, q1, q2, g, ids = dev(raw), dev(qa), dev(qb), dev(gs), torch.tensor(idx, device="cuda")
    params = fused.score_params(60.0, 0.0, regularizer=(1.0, 0.05, 1e9) if clamped else None)
    score = fused.score_forward("beta_kl", table, ids, q1, q2, params)
    # entity 9: lgamma and (x - q) psi(x) of 1,201 are 7,313 and 8,500, and four terms of that size cancel: an ulp of each
    assert_close(score.cpu().numpy(), want, REL_F32, "score", sum_abs=4 * 8500.0 * (idx == 9))
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
    assert np.abs(table.cpu().numpy()[uniq] - w[uniq]).max() <= 1e-3 * 1e-4 + 2.0 ** -23 * np.abs(w[uniq]).max()
