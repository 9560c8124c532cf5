"""Rows of a table that no cache holds are loaded past the caches in tiles of different ids: the scores and the sign codes are
those of a table of the same rows that is small enough to be read in the ordinary way."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.util import REL_F32, assert_close, seed

pytestmark = pytest.mark.gpu


# tables of 1.6 GiB where sign codes are kept and of 4.1 GiB where not; halves of 132 floats (a last column of one lane) and of
# 260 (two columns per lane); tiles of 256 pairs with a last one of 44, and of 200; a fifth to a half of them hold no id twice
@pytest.mark.parametrize("model,dim,n,b,k", [("box", 132, 3_300_000, 4100, 300), ("l1", 260, 1_700_000, 4100, 300),
                                             ("rotate", 132, 4_200_000, 8200, 200), ("l2", 260, 4_300_000, 8200, 200),
                                             ("complex", 260, 2_150_000, 8200, 200), ("distmult", 132, 8_400_000, 16400, 200)])
def test_same_bits_as_a_small_table(model, dim, n, b, k):
    from smore_amd import fused
    rng = np.random.default_rng(seed("rows read once", model, dim))
    width = dim * (2 if model in ("rotate", "complex") else 1)
    pool = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, 20_000)]))
    pick = rng.integers(0, pool.size, (b, k))
    pick[0, :2] = (0, pool.size - 1)
    small = torch.tensor(rng.standard_normal((pool.size, width)) * 0.5, dtype=torch.float32, device="cuda")
    rows = torch.tensor(pool, device="cuda")
    large = torch.empty(n, width, dtype=torch.float32, device="cuda")
    large[rows] = small
    local = torch.tensor(pick, device="cuda")
    q1 = torch.tensor(rng.standard_normal((b, dim)) * 0.5, dtype=torch.float32, device="cuda")
    q2 = None if model in ("l1", "l2", "distmult") else torch.tensor(rng.random((b, dim)), dtype=torch.float32, device="cuda")
    params = fused.score_params(24.0, 0.02)
    codes = [fused.new_codes(model, t, local, q1) for t in (large, small)]
    got = fused.score_forward(model, large, rows[local], q1, q2, params, codes=codes[0])
    ref = fused.score_forward(model, small, local, q1, q2, params, codes=codes[1])
    assert torch.equal(got, ref)
    if codes[0] is not None:
        assert torch.equal(codes[0], codes[1])
    for i in (0, b - 1):
        f64 = lambda t: t.cpu().numpy().astype(np.float64)
        want = orc.score_forward(model, f64(small[local[i]])[None], f64(q1[i])[None, None], None if q2 is None else f64(q2[i])[None, None],
                                 24.0, *([0.02] if model == "box" else []))
        # the terms of a row: at most some 2 each
        assert_close(got[i].cpu().numpy(), want[0], REL_F32, "score", sum_abs=24.0 + 2.0 * dim)


# 1.27 GiB a half, lists of 128 MiB; the last wavefront of a list takes nine candidates of its sixteen
@pytest.mark.parametrize("model,dim,n", [("box", 260, 1_320_000), ("l1", 132, 2_600_000), ("rotate", 132, 2_600_000), ("complex", 260, 1_320_000)])
def test_candidates_as_from_a_small_table(model, dim, n):
    from smore_amd import fused
    from smore_amd.evaluation import candidate_ranks
    rng = np.random.default_rng(seed("candidates read once", model, dim))
    width = dim * (2 if model in ("rotate", "complex") else 1)
    b, c = -(-(1 << 27) // (width * 4 * 1001)), 1001
    pool = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, 5000)]))
    pick = rng.integers(0, pool.size, (b, c))
    pick[0, :2] = (0, pool.size - 1)
    small = torch.tensor(rng.standard_normal((pool.size, width)) * 0.5, dtype=torch.float32, device="cuda")
    rows = torch.tensor(pool, device="cuda")
    large = torch.empty(n, width, dtype=torch.float32, device="cuda")
    large[rows] = small
    local = torch.tensor(pick, device="cuda")
    ids = rows[local]
    local[:, -30:], ids[:, -30:] = -1, -1                 # padding reads entity 0, the same row in both
    q1 = torch.tensor(rng.standard_normal((b, dim)) * 0.5, dtype=torch.float32, device="cuda")
    q2 = None if model == "l1" else torch.tensor(rng.random((b, dim)), dtype=torch.float32, device="cuda")
    params = fused.score_params(24.0, 0.02)
    n_hard = rng.integers(1, 11, b).tolist()
    for got, ref in zip(candidate_ranks(model, large, q1, q2, params, ids, n_hard), candidate_ranks(model, small, q1, q2, params, local, n_hard)):
        assert torch.equal(got, ref)
