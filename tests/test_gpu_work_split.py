"""The kernels' splits of the work at the sizes where they can go wrong (one
unit, a partly filled last unit, many units), against NumPy in 64 bits."""
import sys

import numpy as np
import pytest

import cutc_amd as ct

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    return ct.Context(0)


def coo(dims, nnz, seed):
    rng = np.random.default_rng(seed)
    flat = rng.choice(int(np.prod(dims)), size=nnz, replace=False)
    ind = [a.astype(np.uint32) for a in np.unravel_index(flat, dims)]
    vals = rng.uniform(1.0, 5.0, nnz)
    return ct.Coo.from_arrays(ind, vals, dims), ind, vals


def predict(ind, F):
    h = np.ones((len(ind[0]), F[0].shape[1]))
    for i, f in zip(ind, F):
        h *= f.astype(np.float64)[i]
    return h.sum(1)


@pytest.mark.parametrize("dims", [(60, 50, 40), (20, 15, 12, 10)], ids=["3way", "4way"])
def test_batch_rmse_of_segments(ctx, dims):
    """Per-problem RMSE with problems of one nonzero, about a workgroup's
    walkers and many times a segment's blocks, at every rank.  An FP32 prediction
    of R products of at most 1 is off by at most R 2^-24 = 4e-6."""
    sizes, ranks = [1, 7, 31, 129, 4097, 20011], (8, 16, 32, 64)
    probs, tests, rk, want = [], [], [], []
    rng = np.random.default_rng(5)
    for k, (n, R) in enumerate((n, R) for R in ranks for n in sizes):
        say(f"[batch rmse] n={n} R={R} dims={dims}")
        t, ind, vals = coo(dims, n, 100 + k)
        e, eind, evals = coo(dims, max(1, n // 9), 300 + k)
        F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
        probs.append(t), tests.append(e), rk.append(R)
        want.append((F, np.sqrt(np.mean((vals - predict(ind, F)) ** 2)),
                     np.sqrt(np.mean((evals - predict(eind, F)) ** 2))))
    b = ct.Batch(ctx, probs, tests, rk)
    for p, (F, _, _) in enumerate(want):
        for m, f in enumerate(F):
            b.set_factor(p, m, f)
    tr, te = b.rmse()
    np.testing.assert_allclose(tr, [w[1] for w in want], rtol=1e-6, atol=4e-6)
    np.testing.assert_allclose(te, [w[2] for w in want], rtol=1e-6, atol=4e-6)
