"""Jacobi-PCG that breaks down (a NaN in the data): not converged, every iteration
counted, a NaN solution, as one launch after another gives them, and without the
one-workgroup solver running its iterations to the end."""
import time

import numpy as np
import pytest

import anifem_amd as af

pytestmark = pytest.mark.gpu


def tridiagonal(n):
    rp = np.concatenate([[0], np.cumsum([2] + [3] * (n - 2) + [2])]).astype(np.int64)
    i = np.arange(n)
    ci = np.stack([i - 1, i, i + 1], 1).ravel()
    v = np.tile([-1.0, 2.5, -1.0], n)
    keep = (ci >= 0) & (ci < n)
    return rp, ci[keep].astype(np.int32), v[keep]


@pytest.mark.parametrize("where", ["b", "x", "matrix"])
def test_breakdown_ends_the_one_workgroup_solve(where):
    import torch
    n, maxit = 700, 2_000_000
    rp, ci, v = tridiagonal(n)
    b, x0 = np.ones(n), np.zeros(n)
    {"b": b, "x": x0, "matrix": v}[where][n // 2] = np.nan
    d = [torch.from_numpy(a).cuda() for a in (rp, ci, v, b)]
    x = torch.from_numpy(x0).cuda()
    torch.cuda.synchronize()
    t = time.perf_counter()
    res, ok = af.pcg_jacobi(n, *d, x, maxit=maxit)
    assert time.perf_counter() - t < 2.0
    assert not ok and res.iterations == maxit and np.isnan(res.relres) and bool(torch.isnan(x).all())


@pytest.mark.parametrize("where", ["b", "matrix"])
@pytest.mark.parametrize("maxit", [0, 1, 2, 3, 5])
def test_breakdown_agrees_with_the_launches(where, maxit):
    """The same system padded with unconnected rows to a size that the launches
    solve: iterations, status and which entries are NaN agree."""
    import torch
    out = []
    for pad in (0, 6000):
        n = 300
        rp, ci, v = tridiagonal(n)
        b = np.ones(n + pad)
        if where == "b":
            b[7] = np.nan
        else:
            v[7] = np.nan
        rp = np.concatenate([rp, rp[-1] + 1 + np.arange(pad)]).astype(np.int64)
        ci = np.concatenate([ci, n + np.arange(pad)]).astype(np.int32)
        v = np.concatenate([v, np.ones(pad)])
        x = torch.zeros(n + pad, dtype=torch.float64, device="cuda")
        res, ok = af.pcg_jacobi(n + pad, *[torch.from_numpy(a).cuda() for a in (rp, ci, v, b)], x, maxit=maxit)
        out.append((res.iterations, ok, np.isnan(res.relres), torch.isnan(x[:n]).cpu().numpy().tolist()))
    assert out[0] == out[1]
