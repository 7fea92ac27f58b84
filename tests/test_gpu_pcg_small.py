"""The one-workgroup PCG of small systems: row counts either side of a slice of
64 rows and of a row per thread, uneven row lengths, rows without a diagonal
entry, systems whose rows do not fit its slots (the launch-per-step iteration
takes over, from the same x), a start that is not zero; repeated solves are
bitwise equal."""
import numpy as np
import pytest

import anifem_amd as af

pytestmark = pytest.mark.gpu


def spd(n, extra, seed, hubs=0):
    """Symmetric diagonally dominant CSR arrays and the dense matrix."""
    rng = np.random.default_rng(seed)
    A = np.zeros((n, n))
    if n > 1:
        i, j = rng.integers(0, n, extra * n), rng.integers(0, n, extra * n)
        v = rng.uniform(-1, 1, extra * n)
        A[i, j] = v
        for h in range(0, n, max(1, n // hubs)) if hubs else ():
            A[h, rng.choice(n, min(n - 1, 300), replace=False)] = 0.01
    A = np.triu(A, 1)
    A += A.T
    A[np.arange(n), np.arange(n)] = np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n)
    mask = A != 0
    rp = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int64)
    return rp, np.nonzero(mask)[1].astype(np.int32), A[mask], A


@pytest.mark.parametrize("n,extra,hubs", [(1, 0, 0), (63, 2, 0), (64, 3, 0), (65, 1, 0), (1023, 2, 0), (1025, 2, 0),
                                          (2049, 3, 0), (5120, 1, 0), (5121, 1, 0), (2000, 1, 32)])
def test_small_pcg_matches_direct_solve(n, extra, hubs):
    import torch
    rp, ci, v, A = spd(n, extra, n + extra, hubs)
    rng = np.random.default_rng(n)
    b, x0 = rng.normal(size=n), rng.normal(size=n)
    d = [torch.from_numpy(a).cuda() for a in (rp, ci, v, b)]
    xs = []
    for _ in range(2):
        x = torch.from_numpy(x0.copy()).cuda()
        res, ok = af.pcg_jacobi(n, *d, x, rtol=1e-12)
        assert ok and res.true_relres < 1e-11
        xs.append(x.cpu().numpy())
    assert np.array_equal(xs[0], xs[1])
    ref = np.linalg.solve(A, b)
    # ||x - ref|| <= ||A^-1|| ||b - A x||, and the rows are dominant by at least 0.5
    assert np.linalg.norm(xs[0] - ref) <= 2 * 1e-11 * np.linalg.norm(b) + 1e-12 * np.linalg.norm(ref)
    x = torch.from_numpy(x0.copy()).cuda()
    res, ok = af.pcg_jacobi(n, *d, x, rtol=1e-14, maxit=0)
    assert not ok and res.iterations == 0 and np.array_equal(x.cpu().numpy(), x0)
