"""The evaluation kernels at the sizes where their work split can go wrong: groups of 128 rows, steps of 32 (16, 8)
features with tails, one to four query rows per wavefront, histograms in LDS and in memory, tiles of 64 candidates.
Integer-valued inputs: every fp32 sum is exact, scores tie in large numbers, and the ranks must be the oracle's."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def dev(a, dtype=torch.float32):
    return None if a is None else torch.tensor(a, dtype=dtype, device="cuda")


def _integers(model, n, b, dim, rng, offsets=(0, 5)):
    mul = 2 if model == "complex" else 1
    table = rng.integers(-3, 4, (n, dim * mul)).astype(np.float64)
    q1 = rng.integers(-3, 4, (b, dim)).astype(np.float64)
    q2 = rng.integers(*offsets, (b, dim)).astype(np.float64) if model in ("box", "complex") else None
    return table, q1, q2


def _answers(n, b, most, rng):
    lists = [rng.choice(n, size=min(n, int(rng.integers(1, most + 1))), replace=False).tolist() for _ in range(b)]
    return [x[: len(x) // 2] for x in lists], [x[len(x) // 2:] for x in lists]


def _scan_by_parts(model, table, q1, q2, params, lists):
    """smx_rank_answer_keys, a sort on the host, smx_rank_scan: the two-call form of the same ranks."""
    from smore_amd import _lib
    from smore_amd.fused import MODELS
    lib, b, dim, n = _lib.load(), q1.shape[0], q1.shape[1], table.shape[0]
    a = max(len(x) for x in lists)
    ids = torch.tensor([x + [0] * (a - len(x)) for x in lists], device="cuda")
    counts = torch.tensor([len(x) for x in lists], dtype=torch.int32, device="cuda")
    keys, scores = torch.empty((b, a), dtype=torch.int64, device="cuda"), torch.empty((b, a), device="cuda")
    p = lambda t: None if t is None else t.data_ptr()
    _lib.call("smx_rank_answer_keys", MODELS[model], None, p(table), n, p(q1), p(q2), b, dim, ctypes.byref(params), p(ids),
              p(counts), a, p(scores), p(keys))
    order = torch.argsort(keys ^ -(1 << 63), dim=1, descending=True, stable=True)
    ids_s, keys_s = torch.gather(ids, 1, order).contiguous(), torch.gather(keys, 1, order).contiguous()
    ranks = torch.empty((b, a), dtype=torch.int64, device="cuda")
    ws = torch.empty(lib.smx_rank_workspace_bytes(b, a), dtype=torch.uint8, device="cuda")
    _lib.call("smx_rank_scan", MODELS[model], None, p(table), n, p(q1), p(q2), b, dim, ctypes.byref(params), p(ids_s),
              p(keys_s), p(counts), a, p(ranks), p(ws), ws.numel())
    return torch.empty_like(ranks).scatter_(1, order, ranks).cpu().numpy()


@pytest.mark.parametrize("model,n,b,dim,most,cen", [
    ("l1", 127, 1, 32, 5, 0.0), ("l1", 128, 4, 33, 9, 0.0), ("l1", 129, 5, 3, 70, 0.0), ("l1", 1000, 17, 70, 12, 0.0),
    ("box", 300, 9, 36, 20, 0.5), ("box", 257, 8, 31, 4, 0.5), ("box", 300, 3, 44, 20, 2.0), ("box", 200, 3, 8, 6, 0.0),
    ("complex", 385, 6, 19, 7, 0.0), ("complex", 130, 2, 16, 7, 0.0), ("distmult", 260, 16, 65, 30, 0.0),
    ("distmult", 700, 9, 12, 600, 0.0),        # histograms of up to 600 answers: counted in memory
])
def test_ranks_over_the_edges_of_the_scan(model, n, b, dim, most, cen):
    from smore_amd import fused
    from smore_amd.evaluation import filtered_ranks
    rng = np.random.default_rng(n + b)
    # (box: some offsets are negative, the reference's inside distance is then |offset|)
    table, q1, q2 = _integers(model, n, b, dim, rng, offsets=(-2, 5) if model == "box" else (-3, 4))
    easy, hard = _answers(n, b, most, rng)
    params = fused.score_params(0.0, cen)
    rows = np.broadcast_to(table[None], (b,) + table.shape)
    scores = orc.score_forward(model, rows, q1[:, None], None if q2 is None else q2[:, None], 0.0, cen)
    t, a, c = dev(table), dev(q1), dev(q2)
    got = filtered_ranks(model, t, a, c, params, easy, hard)
    parts = _scan_by_parts(model, t, a, c, params, [e + h for e, h in zip(easy, hard)])
    for i in range(b):
        want_h, want_e = orc.filtered_ranks(scores[i], easy[i], hard[i])
        assert got[i][0].tolist() == want_h.tolist() and got[i][1].tolist() == want_e.tolist()
        assert parts[i, : len(easy[i]) + len(hard[i])].tolist() == want_e.tolist() + want_h.tolist()


@pytest.mark.parametrize("model,b,u,dim,most", [
    ("l1", 1, 1, 96, 64), ("l1", 1, 1, 33, 40), ("l1", 1, 1, 96, 65), ("box", 2, 1, 100, 64), ("box", 1, 2, 100, 30),
    ("complex", 1, 1, 50, 9), ("complex", 1, 2, 21, 64), ("complex", 2, 1, 129, 20), ("distmult", 1, 1, 260, 3),
])
def test_ranks_of_one_and_two_queries_over_a_long_table(model, b, u, dim, most):
    """The streaming form: from 20 MB of table, up to two query rows and 64 answers (one case just past each limit)."""
    from smore_amd import fused
    from smore_amd.evaluation import filtered_ranks
    rng = np.random.default_rng(dim)
    width = dim * (2 if model == "complex" else 1)
    n = (20 << 20) // (4 * width) + (1 if dim != 50 else -1)
    table, q1, q2 = _integers(model, n, b * u, dim, rng, offsets=(-2, 5) if model == "box" else (-3, 4))
    lists = [rng.choice(n, size=most, replace=False).tolist() for _ in range(b)]
    scores = np.concatenate([orc.score_forward(model, table[None, i:i + 16384].repeat(b * u, 0), q1[:, None],
                                               None if q2 is None else q2[:, None], 0.0, 0.5) for i in range(0, n, 16384)], axis=1)
    scores = scores.reshape(b, u, n).max(axis=1)
    shape = (b, u, dim) if u > 1 else (b, dim)
    q1, q2 = q1.reshape(shape), None if q2 is None else q2.reshape(shape)
    got = filtered_ranks(model, dev(table), dev(q1), dev(q2), fused.score_params(0.0, 0.5), [x[::2] for x in lists],
                         [x[1::2] for x in lists], branches=u)
    for i in range(b):
        want_h, want_e = orc.filtered_ranks(scores[i], lists[i][::2], lists[i][1::2])
        assert got[i][0].tolist() == want_h.tolist() and got[i][1].tolist() == want_e.tolist()


@pytest.mark.parametrize("b,u", [(3, 2), (9, 2), (5, 3), (5, 4)])
def test_union_ranks_with_several_queries_per_pass(b, u):
    from smore_amd import fused
    from smore_amd.evaluation import filtered_ranks
    rng = np.random.default_rng(b * u)
    n, dim = 400, 40
    table, q1, _ = _integers("l1", n, b * u, dim, rng)
    easy, hard = _answers(n, b, 15, rng)
    rows = np.broadcast_to(table[None], (b * u,) + table.shape)
    scores = orc.score_forward("l1", rows, q1[:, None], None, 0.0, 0.0).reshape(b, u, n).max(axis=1)
    got = filtered_ranks("l1", dev(table), dev(q1.reshape(b, u, dim)), None, fused.score_params(0.0), easy, hard, branches=u)
    for i in range(b):
        want_h, want_e = orc.filtered_ranks(scores[i], easy[i], hard[i])
        assert got[i][0].tolist() == want_h.tolist() and got[i][1].tolist() == want_e.tolist()


@pytest.mark.parametrize("b,c,h", [(1, 1, 1), (2, 63, 63), (3, 64, 2), (2, 65, 65), (5, 257, 70), (1, 4096, 130)])
def test_candidate_ranks_over_the_edges_of_the_tiles(b, c, h):
    """With and without the logits as an output (the ranking's slots then hold the scores in between)."""
    from smore_amd import _lib, fused
    from smore_amd.fused import MODELS
    rng = np.random.default_rng(c)
    n, dim = 300, 20
    table, q1, _ = _integers("l1", n, b, dim, rng)
    neg = rng.integers(0, n, (b, c))
    neg[:, c - c // 5:] = -1
    n_hard = rng.integers(0, h + 1, b).astype(np.int32)
    n_hard[0] = h
    rows = table[np.where(neg == -1, 0, neg)]
    logits = orc.score_forward("l1", rows, q1[:, None], None, 24.0, 0.0)
    t, q, cand, counts = dev(table), dev(q1), dev(neg, torch.int64), dev(n_hard, torch.int32)
    params = fused.score_params(24.0)
    for with_logits in (True, False):
        logit = torch.empty((b, c), device="cuda") if with_logits else None
        ranking, hard = torch.empty((b, c), dtype=torch.int64, device="cuda"), torch.empty((b, h), dtype=torch.int64, device="cuda")
        _lib.call("smx_rank_candidates", MODELS["l1"], None, t.data_ptr(), n, q.data_ptr(), None, b, dim, ctypes.byref(params),
                  cand.data_ptr(), c, counts.data_ptr(), h, logit.data_ptr() if with_logits else None, ranking.data_ptr(),
                  hard.data_ptr(), None)
        for i in range(b):
            biased, rk, filt = orc.candidate_ranks(logits[i].astype(np.float32), neg[i], int(n_hard[i]))
            assert np.array_equal(ranking[i].cpu().numpy(), rk)
            assert hard[i].tolist() == filt.tolist() + [0] * (h - len(filt))
            assert logit is None or np.array_equal(logit[i].cpu().numpy(), biased)


@pytest.mark.parametrize("model,b,u,dim", [("l2", 1, 1, 200), ("rotate", 2, 1, 130), ("rotate", 1, 2, 75), ("complex_norm", 2, 1, 100),
                                           ("complex_norm", 1, 1, 61), ("distmult_norm", 1, 1, 260), ("box", 2, 1, 500)])
def test_streamed_ranks_lie_where_fp32_allows_and_equal_rows_tie(model, b, u, dim):
    """Random floats; a copy of each answer's row ranks before it from a lower id and does not from a higher one."""
    from smore_amd import fused
    from smore_amd.evaluation import filtered_ranks
    rng = np.random.default_rng(dim)
    model, norm = model.removesuffix("_norm"), model.endswith("_norm")
    width = dim * (2 if model in ("rotate", "complex") else 1)
    n = (20 << 20) // (4 * width) + 5
    t = dev(rng.uniform(-0.2, 0.2, (n, width)))
    q1 = dev(rng.uniform(-0.2, 0.2, (b, u, dim)))
    q2 = None if model in ("l2", "distmult") else dev(rng.uniform(0, 0.2, (b, u, dim)))
    answers = rng.choice(np.arange(1, n - 1), size=(b, 12), replace=False)
    t[0], t[n - 1] = t[answers[0, 0]], t[answers[0, 1]]
    params = fused.score_params(0.0, 0.02 if model == "box" else 0.0, norm=norm)
    got = filtered_ranks(model, t, q1, q2, params, [[]] * b, answers.tolist(), branches=u)
    table, a, c = t.cpu().numpy().astype(np.float64), q1.cpu().numpy().reshape(b * u, 1, dim).astype(np.float64), None
    if q2 is not None:
        c = q2.cpu().numpy().reshape(b * u, 1, dim).astype(np.float64)
    scores = np.concatenate([orc.score_forward(model, np.broadcast_to(table[None, i:i + 8192], (b * u,) + table[i:i + 8192].shape), a, c,
                                               0.0, 0.02, norm=norm) for i in range(0, n, 8192)], axis=1).reshape(b, u, n).max(axis=1)
    for i in range(b):
        others = np.sort(np.delete(scores[i], answers[i]))
        tol = 2e-5 * max(1.0, np.abs(scores[i]).max())
        ranks = got[i][0].cpu().numpy()
        for x, r in zip(answers[i], ranks):
            assert 1 + np.sum(others > scores[i, x] + tol) <= r <= 1 + np.sum(others > scores[i, x] - tol)
    # without the copies (rows behind every other): one rank less after the lower id, the same before the higher one
    far = q1[0, 0] if q2 is None or model == "box" else torch.cat([q1[0, 0], q2[0, 0]])
    t[0] = t[n - 1] = -far if model in ("complex", "distmult") else far + 100.0
    again = filtered_ranks(model, t, q1, q2, params, [[]] * b, answers.tolist(), branches=u)
    s0, s1 = scores[0, answers[0, 0]], scores[0, answers[0, 1]]
    assert abs(s0 - s1) > 1e-5
    assert got[0][0][0].item() == again[0][0][0].item() + 1 + int(s1 > s0)
    assert got[0][0][1].item() == again[0][0][1].item() + int(s0 > s1)


@pytest.mark.parametrize("model", ["l1", "l2", "box", "rotate", "beta_kl", "complex", "complex_norm", "distmult_norm"])
@pytest.mark.parametrize("b,c,dim", [(1, 1, 40), (3, 33, 37), (5, 64, 520)])
def test_short_candidate_lists_are_those_of_long_ones(model, b, c, dim):
    """Up to 64 candidates one launch scores and ranks them: the same bits as a list padded beyond that."""
    from smore_amd import fused
    from smore_amd.evaluation import candidate_ranks
    if dim == 520 and model != "l1":
        dim = 264
    rng = np.random.default_rng(c)
    model, norm = model.removesuffix("_norm"), model.endswith("_norm")
    n = 300
    t = dev(rng.uniform(0.1, 2.0, (n, dim * (2 if model in ("rotate", "complex", "beta_kl") else 1))))
    q1 = dev(rng.uniform(0.1, 2.0, (b, dim)))
    q2 = None if model in ("l1", "l2", "distmult") else dev(rng.uniform(0.1, 2.0, (b, dim)))
    params = fused.score_params(24.0, 0.02 if model == "box" else 0.0, norm=norm)
    neg = rng.integers(0, n, (b, c))
    neg[:, c // 2: c // 2 + 3] = -1
    n_hard = [min(3, c)] * b
    short = candidate_ranks(model, t, q1, q2, params, dev(neg, torch.int64), n_hard)
    long = candidate_ranks(model, t, q1, q2, params, dev(np.concatenate([neg, np.full((b, 70), -1)], axis=1), torch.int64), n_hard)
    assert torch.equal(short[0], long[0][:, :c])
    for i in range(b):
        _, rank, filtered = orc.candidate_ranks(short[0][i].cpu().numpy() - np.where(neg[i] == -1, np.float32(-1e6), 0), neg[i], n_hard[i])
        real = neg[i] != -1
        assert np.array_equal(short[1][i].cpu().numpy()[real], rank[real]) and short[2][i].tolist() == filtered.tolist()
        assert torch.equal(short[1][i][dev(real, torch.bool)], long[1][i, :c][dev(real, torch.bool)])
