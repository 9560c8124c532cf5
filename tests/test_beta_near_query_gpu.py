"""BetaE where the terms of row and query cancel: rows that equal their query or lie near it, rows at the ends of the interval of
the fast forms, and the error against 64 bits beside that of the distance operators, which take the general forms for every
feature."""
import numpy as np
import pytest
import torch

from tests.util import seed

pytestmark = pytest.mark.gpu


def _dev(x):
    return torch.tensor(x, dtype=torch.float32, device="cuda")


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
