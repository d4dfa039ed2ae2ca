"""Calls at the limits of what the entry points take: the widest ranks, work
space that holds anything, files that contradict themselves, outputs that share
memory, tensors without nonzeros.

Tolerances: CP-ALS fits within 1e-4 of the float64 ALS and float32 sums within
1e-5 relative (Frobenius) of float64, as in test_gpu_cpd.py and
test_gpu_paths.py; refusals by their error."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_builder import random_tensor

pytestmark = pytest.mark.gpu


def rel(a, b):
    b = np.asarray(b, dtype=np.float64)
    n = np.linalg.norm(b)
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / (n if n > 0 else 1.0))


# ---- CP-ALS past 128 columns ---------------------------------------------------------

def dirty_scratch(cuda):
    """Leaves large floats of both signs over the first 4.4 MB of the
    allocation-free call's work space: a rank-4 fit whose last mode, of 280000
    rows, keeps its MTTKRP output there."""
    import torch
    import mmcsf
    rng = np.random.default_rng(1)
    dims = [40, 30, 280_000]
    inds = [rng.integers(0, 40, dims[2]), rng.integers(0, 30, dims[2]), np.arange(dims[2])]
    vals = (-1e9 * (rng.random(dims[2]) + 0.5)).astype(np.float32)
    f = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 12)
    U = [torch.from_numpy(rng.random((d, 4)).astype(np.float32)).to(cuda) for d in dims]
    mmcsf.cpd_als(f, U, iters=1, tol=0.0, no_alloc=True)


@pytest.mark.parametrize("R", [128, 129, 132, 256])
@pytest.mark.parametrize("dims", [[500, 400, 300], [400, 300, 290, 280]])
def test_cpd_norms_at_wide_ranks(cuda, dims, R):
    """The column norms of every update start from zero at any rank, whatever the
    work space held."""
    import torch
    import mmcsf
    from oracle import dense as D
    rng = np.random.default_rng(R + len(dims))
    inds, vals = random_tensor(rng, dims, 20_000)
    U0 = [rng.standard_normal((d, R)).astype(np.float32) for d in dims]
    fits, _, lam64 = D.cpd_als(inds, vals, dims, [u.astype(np.float64) for u in U0], 2, tol=0.0)
    f = mmcsf.Format(mmcsf.Tensor.from_numpy(dims, inds, vals), 12, fbr_threshold=128)
    for no_alloc in (True, True, False):
        dirty_scratch(cuda)
        U = [torch.from_numpy(u.copy()).to(cuda) for u in U0]
        lam, st = mmcsf.cpd_als(f, U, iters=2, tol=0.0, no_alloc=no_alloc)
        np.testing.assert_allclose(st["fit_history"], fits, atol=1e-4, rtol=0)
        assert np.isfinite(lam).all() and all(bool(torch.isfinite(u).all()) for u in U)
