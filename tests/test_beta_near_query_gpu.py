"""BetaE where the terms of row and query cancel: rows that equal their query or lie near it, rows at the ends of the interval of
the fast forms, and the error against 64 bits beside that of the distance operators, which take the general forms for every
feature."""
import numpy as np
import pytest
import torch
from scipy.special import gammaln, polygamma, psi

from tests.util import seed

pytestmark = pytest.mark.gpu


def _dev(x):
    return torch.tensor(x, dtype=torch.float32, device="cuda")


def _rms(x):
    return float(np.sqrt(np.mean(np.square(x))))


def _kl(ea, eb, qa, qb):
    log_beta = lambda a, b: gammaln(a) + gammaln(b) - gammaln(a + b)
    return log_beta(qa, qb) - log_beta(ea, eb) + (ea - qa) * psi(ea) + (eb - qb) * psi(eb) + (qa + qb - ea - eb) * psi(ea + eb)


def _draw(rng, low, high, shape):
    """low None: a normal around 1, clamped at 0.05, as the regularizer leaves rows."""
    x = np.clip(1 + 0.5 * rng.standard_normal(shape), 0.05, None) if low is None else np.exp(rng.uniform(np.log(low), np.log(high), shape))
    return x.astype(np.float32).astype(np.float64)


def test_shared_list_constants_of_row_and_query_are_of_one_form():
    """A list of the queries' own rows.  A pair's three sums (the row's constant, the query's, the product's 800 terms of one
    sign, about 1 each) are rounded 800 times at most, half the sum high on average: sqrt(800 / 12) * 2^-24 * 800 = 3.9e-4 rms a pair,
    0.17e-4 in the mean of 512 that are independent; six times that.  What hardware logarithms and reciprocals are off by is
    the same in both constants, unless their forms differ."""
    from smore_amd import fused
    rng = np.random.default_rng(seed("one form"))
    n, dim = 512, 400
    qa, qb = (_draw(rng, None, None, (n, dim)) for _ in range(2))
    table = _dev(np.concatenate([qa, qb], 1))
    score = fused.score_forward_shared("beta_kl", table, torch.arange(n, device="cuda"), _dev(qa), _dev(qb), fused.score_params(0.0))
    assert abs(score.diagonal().double().mean().item()) <= 1.0e-4


def _mixed(rng, shape):
    """Features in the interval of the fast forms, below it, beyond it and at its ends, the sum of a pair included."""
    x = _draw(rng, 0.05, 60.0, shape)
    x[..., ::7] = _draw(rng, 0.001, 0.019, x[..., ::7].shape)
    x[..., 3::11] = _draw(rng, 1001.0, 5000.0, x[..., 3::11].shape)
    x[0, 0], x[1, 1], x[2, 2], x[3, 3] = np.float32(0.02), 1000.0, 999.5, np.float32(0.0199)
    return x


# every number of floats per lane, in columns of one and of four, and rows that are not
WIDTHS = [4, 33, 64, 200, 256, 260, 400, 452, 512, 516, 1000]


@pytest.mark.parametrize("inside", [True, False])
@pytest.mark.parametrize("dim", WIDTHS)
def test_a_row_is_at_no_distance_from_itself(dim, inside):
    from smore_amd import fused
    from smore_amd.evaluation import candidate_ranks
    rng = np.random.default_rng(seed("itself", dim, inside))
    n, k = 40, 140
    qa, qb = (_draw(rng, 0.05, 60.0, (n, dim)) if inside else _mixed(rng, (n, dim)) for _ in range(2))
    table, q1, q2 = _dev(np.concatenate([qa, qb], 1)), _dev(qa), _dev(qb)
    idx = torch.tensor(rng.integers(0, n, (n, k)), device="cuda")
    own = torch.tensor(rng.integers(0, k, n), device="cuda")
    at = torch.arange(n, device="cuda")
    idx[at, own] = at
    params = fused.score_params(60.0)
    score = fused.score_forward("beta_kl", table, idx, q1, q2, params)
    logit = candidate_ranks("beta_kl", table, q1, q2, params, idx, [1] * n)[0]
    assert (score[at, own] == 60.0).all() and (logit[at, own] == 60.0).all()
    assert torch.isfinite(score).all()


# widths with one and two columns of four a lane, in single columns, unaligned
@pytest.mark.parametrize("low,high", [(None, None), (0.05, 5.0), (1.0, 5.0), (1.0, 20.0), (20.0, 60.0), (60.0, 480.0)])
@pytest.mark.parametrize("near", [0.01, 0.1])
@pytest.mark.parametrize("dim", [36, 250, 400, 512])
def test_scores_near_the_query_round_no_worse_than_the_general_forms(dim, near, low, high):
    """The operators sum a row's features in another order: a tenth for that and for the spread of two samples of 2,048."""
    from smore_amd import fused
    from smore_amd.torchext import ext_ops
    rng = np.random.default_rng(seed("near", dim, near, low))
    b, k = 256, 8
    qa, qb = (_draw(rng, low, high, (b, dim)) for _ in range(2))
    ea, eb = ((np.repeat(q, k, 0) * rng.uniform(1 - near, 1 + near, (b * k, dim))).astype(np.float32).astype(np.float64) for q in (qa, qb))
    want = _kl(ea, eb, np.repeat(qa, k, 0), np.repeat(qb, k, 0)).sum(1).reshape(b, k)
    rows, q1, q2 = _dev(np.concatenate([ea, eb], 1)), _dev(qa), _dev(qb)
    idx = torch.arange(b * k, device="cuda").reshape(b, k)
    got = -fused.score_forward("beta_kl", rows, idx, q1, q2, fused.score_params(0.0)).cpu().numpy().astype(np.float64)
    with torch.no_grad():
        general = ext_ops.beta_kl(rows.view(b, k, -1), ext_ops.BetaDist(q1[:, None], q2[:, None])).cpu().numpy().astype(np.float64)
    assert _rms(got - want) <= 1.1 * _rms(general - want)


@pytest.mark.parametrize("inside", [True, False])
@pytest.mark.parametrize("dim", WIDTHS)
def test_a_row_does_not_pull_at_a_query_that_equals_it(dim, inside):
    """One pair a query: the query gradient is that pair's, and the row's own is 0 in every form of the backward."""
    from smore_amd import fused
    rng = np.random.default_rng(seed("pull", dim, inside))
    n = 40
    qa, qb = (_draw(rng, 0.05, 60.0, (n, dim)) if inside else _mixed(rng, (n, dim)) for _ in range(2))
    table, q1, q2 = _dev(np.concatenate([qa, qb], 1)), _dev(qa), _dev(qb)
    idx = torch.arange(n, device="cuda").reshape(n, 1)
    gs, params = _dev(rng.standard_normal((n, 1))), fused.score_params(60.0)
    score = fused.score_forward("beta_kl", table, idx, q1, q2, params)
    for g in fused.score_backward_query("beta_kl", table, idx, q1, q2, score, gs, params):
        assert not g.any()
    plan = fused.build_plan(idx, n)
    m, v, before = torch.zeros_like(table), torch.zeros_like(table), table.clone()
    for g in fused.score_backward_fused("beta_kl", plan, table, idx, q1, q2, score, gs, params, m=m, v=v, adam=fused.adam_params(1e-3, 1)):
        assert not g.any()
    assert not m.any() and not v.any() and torch.equal(table, before)


@pytest.mark.parametrize("outside", [0.004, 1500.0])
@pytest.mark.parametrize("dim", WIDTHS)
def test_a_feature_outside_the_interval_changes_no_other(dim, outside):
    """The form is chosen by the feature, whatever path its row takes."""
    from smore_amd import fused
    rng = np.random.default_rng(seed("outside", dim, outside))
    n = 40
    qa, qb = (_draw(rng, 0.05, 60.0, (n, dim)) for _ in range(2))
    rows = np.concatenate([_draw(rng, None, None, (n, dim)), _draw(rng, 1.0, 60.0, (n, dim))], 1)
    idx = torch.arange(n, device="cuda").reshape(n, 1)
    q1, q2, gs, params = _dev(qa), _dev(qb), _dev(rng.standard_normal((n, 1))), fused.score_params(60.0)
    score = torch.zeros_like(gs)
    at = rng.integers(0, dim, n)
    moved = rows.copy()
    moved[np.arange(n), at] = outside
    plain, other = (fused.score_backward_query("beta_kl", _dev(t), idx, q1, q2, score, gs, params) for t in (rows, moved))
    same = torch.ones(n, dim, dtype=torch.bool, device="cuda")
    same[torch.arange(n), torch.tensor(at)] = False
    for a, b in zip(plain, other):
        assert torch.equal(a[same], b[same]) and not torch.equal(a, b)


@pytest.mark.parametrize("low,high", [(None, None), (0.05, 5.0), (1.0, 20.0), (20.0, 60.0), (60.0, 480.0)])
def test_gradients_of_rows_round_no_worse_than_the_general_forms(low, high):
    """Relative errors of single pairs' gradients, out of trigammas alone: 51,200 features."""
    from smore_amd import fused
    from smore_amd.torchext import ext_ops
    rng = np.random.default_rng(seed("rows' gradients", low))
    n, dim = 128, 400
    ea, eb = (_draw(rng, low, high, (n, dim)) for _ in range(2))
    ea = np.round(ea * 2 ** 14) / 2 ** 14                 # (ea + 1/4 and their difference are exact)
    qa, qb = ea + 0.25, eb
    table, q1, q2 = _dev(np.concatenate([ea, eb], 1)), _dev(qa), _dev(qb)
    idx = torch.arange(n, device="cuda").reshape(n, 1)
    gs, params = torch.ones(n, 1, device="cuda"), fused.score_params(0.0)
    plan = fused.build_plan(idx, n)
    merged = torch.empty_like(table)
    fused.score_backward_entity("beta_kl", plan, table, q1, q2, torch.zeros_like(gs), gs, params, merged=merged)
    rows = table.view(n, 1, -1).clone().requires_grad_(True)
    ext_ops.beta_kl(rows, ext_ops.BetaDist(q1[:, None], q2[:, None])).backward(-gs)
    want = 0.25 * (polygamma(1, ea) - polygamma(1, ea + eb))
    error = lambda g: _rms((g.detach().cpu().numpy().astype(np.float64).reshape(n, -1)[:, :dim] / want - 1))
    assert error(merged) <= error(rows.grad)


def test_ranking_knows_the_digamma_to_an_ulp():
    """Features of 1/31 to 1/17, where psi(x) - psi(x + 1) = -1/x is 17 to 31 and an ulp 2^-19: 1/x and the sum are off by 0.58 and 0.29
    of one, the difference by 0.29 more, the logit's own roundings by 0.2 each.  The logit is that difference times about
    -40, plus parts in 64 bits."""
    from smore_amd import fused
    from tests.test_rank_numerics_gpu import _all_ids, _keys
    rng = np.random.default_rng(seed("digamma"))
    n, dim = 2000, 4
    ea, eb = np.full((n, dim), 1.0), np.full((n, dim), 1.0)
    ea[:, 0] = _draw(rng, 1 / 31, 1 / 17, n)
    qa, qb = np.ones((1, dim)), np.ones((1, dim))
    qa[0, 0] = 40.0
    want = -_kl(ea, eb, qa, qb).sum(1)
    got = _keys("beta_kl", _dev(np.concatenate([ea, eb], 1)), _dev(qa), _dev(qb), fused.score_params(0.0), _all_ids(1, n))[0]
    error = (got.cpu().numpy().astype(np.float64)[0] - want) / (ea[:, 0] - 40.0)
    assert _rms(error) <= 2.0 ** -19


@pytest.mark.parametrize("outside", [0.004, 1500.0])
@pytest.mark.parametrize("dim", WIDTHS)
def test_a_feature_outside_the_interval_changes_no_other_gradient_of_its_row(dim, outside):
    """One pair a query and Adam: rows finished in the stream up to 512 floats a half, by the entity pass beyond."""
    from smore_amd import fused
    rng = np.random.default_rng(seed("outside, rows", dim, outside))
    n = 40
    qa, qb = (_draw(rng, 0.05, 60.0, (n, dim)) for _ in range(2))
    rows = np.concatenate([_draw(rng, None, None, (n, dim)), _draw(rng, 1.0, 60.0, (n, dim))], 1)
    idx = torch.arange(n, device="cuda").reshape(n, 1)
    q1, q2, gs, params = _dev(qa), _dev(qb), _dev(rng.standard_normal((n, 1))), fused.score_params(60.0)
    score, plan = torch.zeros_like(gs), fused.build_plan(idx, n)
    at = rng.integers(0, dim, n)
    moved = rows.copy()
    moved[np.arange(n), at] = outside
    moments = []
    for t in (rows, moved):
        table = _dev(t)
        m, v = torch.zeros_like(table), torch.zeros_like(table)
        fused.score_backward_fused("beta_kl", plan, table, idx, q1, q2, score, gs, params, m=m, v=v, adam=fused.adam_params(1e-3, 1))
        moments.append(m)
    same = torch.ones(n, 2 * dim, dtype=torch.bool, device="cuda")
    for half in (0, dim):
        same[torch.arange(n), torch.tensor(at + half)] = False
    assert torch.equal(moments[0][same], moments[1][same]) and not torch.equal(moments[0], moments[1])
