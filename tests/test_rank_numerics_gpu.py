"""All-entity ranking: values that are not finite, keys from elsewhere, rows that occur twice, and the rounding error of the
scores against that of the scoring kernels (a row per wavefront, summed as a tree)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

GAMMA = {"l1": 24.0, "l2": 12.0, "box": 24.0, "rotate": 9.0, "beta_kl": 60.0, "complex": 0.0, "distmult": 0.0}
TWO_HALVES = ("rotate", "beta_kl", "complex")
ONE_QUERY = ("l1", "l2", "distmult")


def _ptr(t):
    return None if t is None else t.data_ptr()


def _row(model, dim):
    return dim * (2 if model in TWO_HALVES else 1)


def _keys(model, table, q1, q2, params, ids, branches=1):
    """smx_rank_answer_keys_union on the device ids [B, A]: scores and keys (as signed 64-bit)."""
    from smore_amd import _lib
    from smore_amd.fused import MODELS
    b, a = ids.shape
    counts = torch.full((b,), a, dtype=torch.int32, device="cuda")
    keys, scores = torch.empty((b, a), dtype=torch.int64, device="cuda"), torch.empty((b, a), device="cuda")
    _lib.call("smx_rank_answer_keys_union", MODELS[model], None, _ptr(table), table.shape[0], _ptr(q1), _ptr(q2), b, branches,
              q1.shape[-1], ctypes.byref(params), _ptr(ids), _ptr(counts), a, _ptr(scores), _ptr(keys))
    return scores, keys


def _scan(model, table, q1, q2, params, ids, keys, branches=1):
    """smx_rank_scan_union with the keys given, in the slots of `ids`."""
    from smore_amd import _lib
    from smore_amd.fused import MODELS
    b, a = ids.shape
    counts = torch.full((b,), a, dtype=torch.int32, device="cuda")
    order = torch.argsort(keys ^ -(1 << 63), dim=1, descending=True, stable=True)
    ids_s, keys_s = torch.gather(ids, 1, order).contiguous(), torch.gather(keys, 1, order).contiguous()
    ranks = torch.empty((b, a), dtype=torch.int64, device="cuda")
    ws = torch.empty(_lib.load().smx_rank_workspace_bytes(b, a), dtype=torch.uint8, device="cuda")
    _lib.call("smx_rank_scan_union", MODELS[model], None, _ptr(table), table.shape[0], _ptr(q1), _ptr(q2), b, branches,
              q1.shape[-1], ctypes.byref(params), _ptr(ids_s), _ptr(keys_s), _ptr(counts), a, _ptr(ranks), _ptr(ws), ws.numel())
    return torch.empty_like(ranks).scatter_(1, order, ranks)


def _all_ids(b, n):
    return torch.arange(n, device="cuda").expand(b, n).contiguous()


@pytest.mark.parametrize("model", ["l1", "l2", "box", "rotate", "complex", "distmult"])
@pytest.mark.parametrize("b,dim", [(1, 100), (5, 36), (5, 33)])
def test_rows_that_are_not_finite_rank_where_the_scoring_kernels_put_them(model, b, dim):
    """A diverged row (an infinite feature, sums or squares beyond fp32) scores -inf or +inf, not NaN: it must not move the
    ranks of the others.  Integer coordinates elsewhere: every finite sum is exact."""
    from smore_amd import fused
    from smore_amd.evaluation import filtered_ranks
    rng = np.random.default_rng(dim)
    n = 300
    table = rng.integers(-3, 4, (n, _row(model, dim))).astype(np.float32)
    q1 = rng.integers(1, 4, (b, dim)).astype(np.float32)
    q2 = None if model in ONE_QUERY else rng.integers(1, 4, (b, dim)).astype(np.float32)
    table[3, 5], table[130, dim - 1], table[131, 0] = np.inf, -np.inf, 1e38
    if model in ("l1", "l2", "box", "rotate"):
        table[7], table[299] = 3e38, -1e30
    t, a, c = (None if x is None else torch.tensor(x, device="cuda") for x in (table, q1, q2))
    params = fused.score_params(GAMMA[model], 0.5 if model == "box" else 0.0)
    want = fused.score_forward(model, t, _all_ids(b, n), a, c, params)
    got, _ = _keys(model, t, a, c, params, _all_ids(b, n))
    assert not want.isnan().any() and int(want.isinf().sum()) >= b
    assert torch.equal(got.isinf(), want.isinf()) and not got.isnan().any()
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    answers = [rng.choice(n, size=9, replace=False).tolist() + [3] for _ in range(b)]
    answers = [list(dict.fromkeys(x)) for x in answers]
    ranks = filtered_ranks(model, t, a, c, params, [x[:4] for x in answers], [x[4:] for x in answers])
    # (rotate: irrational sums, the order of two rows within rounding is either kernel's own)
    scores = (got if model == "rotate" else want).cpu().numpy().astype(np.float64)
    for i in range(b):
        want_h, want_e = orc.filtered_ranks(scores[i], answers[i][:4], answers[i][4:])
        assert ranks[i][0].tolist() == want_h.tolist() and ranks[i][1].tolist() == want_e.tolist()


def _rms(x):
    return float(np.sqrt(np.mean(np.square(x))))


@pytest.mark.parametrize("dim", [100, 400])
def test_box_scores_keep_their_digits_where_distances_are_near_the_offsets(dim):
    """Outside distances near zero: |d| - offset is exact there, and what a form that scales it by 1 / cen rounds away is
    1 / cen times larger.  Bound: up to 64 additions one after another round by sqrt(64 / 3) x 2^-24 / sqrt(3) of the sum,
    2.7 x 2^-24."""
    from smore_amd import fused
    rng = np.random.default_rng(dim)
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    n, b, cen = 1500, 3, float(np.float32(0.02))
    table = f32(rng.choice([-1.0, 1.0], (n, dim)) * 0.05 * (1 + 0.01 * rng.random((n, dim))))
    q1, q2 = np.zeros((b, dim)), f32(0.05 * (1 + 0.001 * rng.random((b, dim))))
    want = orc.score_forward("box", np.broadcast_to(table[None], (b, n, dim)), q1[:, None], q2[:, None], 0.0, cen)
    t, a, c = (torch.tensor(x, dtype=torch.float32, device="cuda") for x in (table, q1, q2))
    got, _ = _keys("box", t, a, c, fused.score_params(0.0, cen), _all_ids(b, n))
    assert _rms(got.cpu().numpy() - want) <= 4 * 2.0 ** -24 * _rms(want)


def test_box_scores_with_a_weight_too_small_to_invert():
    from smore_amd import fused
    rng = np.random.default_rng(0)
    n, b, dim = 200, 2, 40
    table, q1 = rng.integers(-3, 4, (n, dim)).astype(np.float32), rng.integers(-3, 4, (b, dim)).astype(np.float32)
    q2 = rng.integers(0, 3, (b, dim)).astype(np.float32)
    want = -np.maximum(np.abs(table[None] - q1[:, None]) - q2[:, None], 0).sum(axis=-1)
    t, a, c = (torch.tensor(x, device="cuda") for x in (table, q1, q2))
    got, _ = _keys("box", t, a, c, fused.score_params(0.0, 1e-40), _all_ids(b, n))
    assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("model", ["l1", "l2", "box", "rotate", "complex", "distmult", "complex_norm", "distmult_norm"])
@pytest.mark.parametrize("dim", [12, 33, 100, 255, 400])
def test_scores_round_no_worse_than_those_of_the_scoring_kernels(model, dim):
    """The scan sums a row feature by feature in one lane, the scoring kernels as a tree over a wavefront: error against
    float64, a tenth for the spread of two samples of a few thousand logits."""
    from smore_amd import fused
    rng = np.random.default_rng(dim)
    model, norm = model.removesuffix("_norm"), model.endswith("_norm")
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    n, b, cen = 1500, 4, float(np.float32(0.02))
    r = 26.0 / dim
    table, q1 = f32(rng.uniform(-r, r, (n, _row(model, dim)))), f32(rng.uniform(-r, r, (b, dim)))
    q2 = None if model in ONE_QUERY else f32(rng.uniform(0 if model == "box" else -r, r, (b, dim)))
    want = orc.score_forward(model, np.broadcast_to(table[None], (b,) + table.shape), q1[:, None],
                             None if q2 is None else q2[:, None], 0.0, cen, norm=norm)
    t, a, c = (None if x is None else torch.tensor(x, dtype=torch.float32, device="cuda") for x in (table, q1, q2))
    params = fused.score_params(0.0, cen if model == "box" else 0.0, norm=norm)
    scan, _ = _keys(model, t, a, c, params, _all_ids(b, n))
    tree = fused.score_forward(model, t, _all_ids(b, n), a, c, params)
    assert _rms(scan.cpu().numpy() - want) <= 1.1 * _rms(tree.cpu().numpy() - want)


@pytest.mark.parametrize("low,high", [(0.05, 3.0), (1.0, 20.0), (20.0, 100.0)])
@pytest.mark.parametrize("dim", [30, 100, 404])
def test_divergences_round_no_worse_than_those_of_the_scoring_kernels(low, high, dim):
    """BetaE: the log-Beta terms of row and query, thousands of times the divergence's last digits, cancel.  Whole error, and
    the part that can reorder entities (without each query's mean); a tenth for the spread of two samples."""
    from smore_amd import fused
    rng = np.random.default_rng(dim)
    f32 = lambda x: x.astype(np.float32).astype(np.float64)
    n, b = 600, 3
    table, q1, q2 = (f32(rng.uniform(low, high, s)) for s in ((n, 2 * dim), (b, dim), (b, dim)))
    want = orc.score_forward("beta_kl", np.broadcast_to(table[None], (b,) + table.shape), q1[:, None], q2[:, None], 0.0, 0.0)
    t, a, c = (torch.tensor(x, dtype=torch.float32, device="cuda") for x in (table, q1, q2))
    params = fused.score_params(0.0)
    scan = _keys("beta_kl", t, a, c, params, _all_ids(b, n))[0].cpu().numpy() - want
    tree = fused.score_forward("beta_kl", t, _all_ids(b, n), a, c, params).cpu().numpy() - want
    assert _rms(scan) <= 1.1 * _rms(tree)
    assert _rms(scan - scan.mean(axis=1, keepdims=True)) <= 1.1 * _rms(tree - tree.mean(axis=1, keepdims=True))


@pytest.mark.parametrize("model", ["l1", "box", "rotate", "beta_kl", "complex_norm", "l2"])
@pytest.mark.parametrize("b,branches,dim", [(1, 1, 100), (6, 1, 37), (3, 2, 36)])
def test_answers_are_known_by_their_ids_not_by_their_scores(model, b, branches, dim):
    """Every entity is an answer, one of them listed twice: nothing ranks before any of them, whatever the keys' scores --
    those of smx_rank_answer_keys, the same an ulp off, or scores of the scoring kernels."""
    from smore_amd import fused
    from smore_amd.evaluation import filtered_ranks
    rng = np.random.default_rng(dim)
    model, norm = model.removesuffix("_norm"), model.endswith("_norm")
    n = 333
    low, high = (0.1, 4.0) if model == "beta_kl" else (-0.2, 0.2)
    t = torch.tensor(rng.uniform(low, high, (n, _row(model, dim))), dtype=torch.float32, device="cuda")
    q = [torch.tensor(np.abs(rng.uniform(low, high, (b, branches, dim))), dtype=torch.float32, device="cuda") for _ in range(2)]
    q1, q2 = q[0], None if model in ONE_QUERY else q[1]
    params = fused.score_params(GAMMA[model], 0.02 if model == "box" else 0.0, norm=norm)
    ids = torch.cat([_all_ids(b, n), torch.full((b, 1), 7, device="cuda")], dim=1).contiguous()
    _, keys = _keys(model, t, q1, q2, params, ids, branches)
    ulp = torch.tensor(rng.integers(-1, 2, tuple(keys.shape)), device="cuda") << 32
    elsewhere = (torch.tensor(rng.integers(0, 2 ** 31, tuple(keys.shape)), device="cuda") << 32) | (keys & 0xFFFFFFFF)
    for k in (keys, keys + ulp, elsewhere):
        assert (_scan(model, t, q1, q2, params, ids, k, branches) == 1).all()
    ranks = filtered_ranks(model, t, q1, q2, params, [list(range(0, n, 2))] * b, [list(range(1, n, 2))] * b, branches)
    assert all((x == 1).all() for pair in ranks for x in pair)


@pytest.mark.parametrize("model", ["complex", "distmult"])
@pytest.mark.parametrize("b,dim", [(1, 100), (5, 33)])
def test_unit_length_rows_beyond_fp32_score_as_among_candidates(model, b, dim):
    """A row whose squared length leaves fp32 is scaled to zeros (its logit is gamma), to a NaN where a feature is infinite,
    also where its product with the query is infinite: the candidate call scales first."""
    from smore_amd import fused
    from smore_amd.evaluation import candidate_ranks
    rng = np.random.default_rng(dim)
    n = 200
    table = rng.uniform(-1, 1, (n, _row(model, dim))).astype(np.float32)
    table[3], table[77, :5], table[130, dim - 1], table[199, 0] = 3e38, -2e38, np.inf, 1e30
    q = [torch.tensor(rng.uniform(1, 3, (b, dim)), dtype=torch.float32, device="cuda") for _ in range(2)]
    t, q2 = torch.tensor(table, device="cuda"), None if model in ONE_QUERY else q[1]
    params = fused.score_params(0.0, norm=True)
    want, _, _ = candidate_ranks(model, t, q[0], q2, params, _all_ids(b, n), [1] * b)
    got, keys = _keys(model, t, q[0], q2, params, _all_ids(b, n))
    assert torch.equal(got.isnan(), want.isnan()) and want.isnan().sum() == b and (got[:, [3, 77, 199]] - want[:, [3, 77, 199]]).abs().max() < 1e-5
    ids = torch.tensor([[3, 77, 8, 199]], device="cuda").expand(b, 4).contiguous()
    _, some = _keys(model, t, q[0], q2, params, ids)
    ranks = _scan(model, t, q[0], q2, params, ids, some)
    others = np.setdiff1d(np.arange(n), [3, 77, 8, 199])
    order = keys ^ -(1 << 63)
    for i in range(b):
        beats = (order[i, others][:, None] > order[i, ids[i]][None]).sum(dim=0)
        assert (ranks[i] == beats + 1).all()
