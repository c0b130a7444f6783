"""The training step's gradient (k_guide_train) at the edges of its split.

A block takes 256 rows per iteration, a wave 32 of them in two groups of 16, and
a launch at most one block per CU.  Rows with no contribution add nothing, and a
batch 2^k times as long scales every delta by 2^-k exactly, so the gradient of n
rows spread over n 2^k (the others without contribution) times 2^k must be the
gradient of the n rows up to the order of the float32 sums: chains of at most
about 300 additions, 300 x 2^-24 = 1.8e-5 of the sum of magnitudes; 1e-4 of the
gradient's norm allows for cancellation by a factor of 5.
"""
import numpy as np
import pytest

import test_gpu_guide as base

pytestmark = pytest.mark.gpu
guide = base.guide  # the fixture


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 63, 255, 256, 257, 511, 1025])
@pytest.mark.parametrize("k", [1, 3, 7])
def test_spread_rows_give_the_same_gradient(guide, device, n, k):
    guide.set_params(base.make_params())
    rows = base.G.random_rows(n, seed=n)
    g0, l0 = guide.gradient(base.to_dev(rows, device))
    wide = base.G.random_rows(n << k, seed=n + 1)
    wide[:, 12] = 0.0
    wide[np.arange(n) * (1 << k) + (5 * n) % (1 << k)] = rows
    g1, l1 = guide.gradient(base.to_dev(wide, device))
    a, b = g0.cpu().numpy().astype(np.float64), g1.cpu().numpy().astype(np.float64) * (1 << k)
    assert np.linalg.norm(a) > 0
    for name, (lo, hi) in base.BLOCKS.items():
        assert np.linalg.norm(a[lo:hi] - b[lo:hi]) <= 1e-4 * np.linalg.norm(a[lo:hi]), name
    assert abs(l0 - l1 * (1 << k)) <= 1e-4 * abs(l0)


@pytest.mark.parametrize("n", [33, 70001])
def test_gradient_repeats_and_takes_any_base(guide, device, n):
    """Sums in a fixed order: the same bits again, and from rows that start 4
    bytes past a 16-byte boundary."""
    import torch

    guide.set_params(base.make_params())
    rows = base.to_dev(base.G.random_rows(n, seed=n), device)
    shifted = torch.empty(n * 16 + 1, dtype=torch.float32, device=device)[1:].view(n, 16)
    shifted.copy_(rows)
    g0, l0 = guide.gradient(rows)
    for r in (rows, shifted):
        g1, l1 = guide.gradient(r)
        assert torch.equal(g0, g1) and l0 == l1


def test_training_wraps_around_the_rows(guide, device):
    """Batches that start late in the rows take the rest from their beginning."""
    import torch

    rows = base.G.random_rows(1000, seed=9)
    p = base.make_params()
    guide.set_params(p)
    guide.train(base.to_dev(rows, device), n_batch=700, iters=2, lr=1e-3)
    a = guide.get_params()
    # the second step of the same run, its batch laid out without wrapping
    guide.set_params(p)
    guide.train(base.to_dev(np.concatenate([rows[:700], rows[700:], rows[:400]]), device), n_batch=700, iters=2, lr=1e-3)
    assert np.array_equal(a, guide.get_params())
    assert torch.isfinite(torch.as_tensor(a)).all()
