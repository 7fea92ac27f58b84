"""Which form solves a system: the one-workgroup solver takes it up to 5,120 rows,
49,152 entries and 192 load groups of its padded layout, the launches per
iteration otherwise.  Three uncoupled copies of the system with a right-hand side
on the first always go to the launches, with the same lanes per row, and their
sums gain zeros only: the first copy's solution is that of the system alone, bit
for bit, if the launches solved it too, and differs in its last digits if the
other form did, whose sums run in another order."""
import numpy as np
import pytest

import anifem_amd as af
from test_gpu_pcg_small import spd

pytestmark = pytest.mark.gpu


def banded(n, half):
    """Symmetric, diagonally dominant, about 2 half + 1 entries per row."""
    i = np.arange(n)[:, None] + np.arange(-half, half + 1)[None, :]
    ok = (i >= 0) & (i < n)
    v = np.where(np.arange(-half, half + 1) == 0, 2.0 * half + 0.1, -1.0)[None, :] * np.ones((n, 1))
    rp = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int64)
    return rp, i[ok].astype(np.int32), v[ok]


def solve(rp, ci, v, b):
    import torch
    x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
    res, ok = af.pcg_jacobi(len(b), *[torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (rp, ci, v, b)], x,
                            rtol=1e-11)
    assert ok
    return x.cpu().numpy(), res.iterations


SYSTEMS = {
    "most rows": (lambda: banded(5120, 1), True), "one row more": (lambda: banded(5121, 1), False),
    "most entries": (lambda: banded(3280, 7), True), "entries above": (lambda: banded(3281, 7), False),
    "one slice": (lambda: banded(64, 31), True), "uneven rows": (lambda: spd(2000, 1, 3, 5)[:3], True),
    "too many long rows": (lambda: spd(2000, 1, 2001, 32)[:3], False)}


@pytest.mark.parametrize("name", list(SYSTEMS))
def test_form_by_size(name):
    make, one_workgroup = SYSTEMS[name]
    rp, ci, v = make()
    n = len(rp) - 1
    b = np.random.default_rng(n).normal(size=n)
    x, it = solve(rp, ci, v, b)
    k = max(3, -(-5121 // n))
    xs, its = solve(np.concatenate([[0]] + [rp[1:] + rp[-1] * c for c in range(k)]),
                    np.concatenate([ci + n * c for c in range(k)]).astype(np.int32), np.tile(v, k),
                    np.concatenate([b, np.zeros((k - 1) * n)]))
    assert not xs[n:].any()
    assert np.linalg.norm(xs[:n] - x) <= 1e-9 * np.linalg.norm(x)
    assert np.array_equal(xs[:n], x) != one_workgroup
    if not one_workgroup:
        assert it == its
