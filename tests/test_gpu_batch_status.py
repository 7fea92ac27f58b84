"""The counts of a batched pass: non-finite entries and flat cells of this pass
alone, over several geometry workgroups and from threads that come and go, as
the single contexts report them."""
import threading

import numpy as np
import pytest

import anifem_amd as af

pytestmark = pytest.mark.gpu


def test_batch_counts_match_single_contexts_and_reset():
    import torch
    specs, flat = [(2, af.FEM_P1), (5, af.FEM_P2)], 1
    meshes = []
    for n, fem in specs:
        c, t = af.kuhn_cube(n, 0.2, n)
        extra = np.concatenate([c, np.array([[2.0, 0, 0], [3.0, 0, 0], [2.0, 1, 0], [3.0, 1, 0]])])  # one plane
        more = np.tile(np.arange(len(c), len(c) + 4, dtype=t.dtype), (flat, 1))
        meshes.append((extra, np.concatenate([t, more]), fem))
    f = torch.ones(1, dtype=torch.float64, device="cuda")
    B = af.Batch(meshes, dirichlet=af.DIRICHLET_NONE, autotune=False)
    good = torch.ones(B.n_tets, dtype=torch.float64, device="cuda")
    expect = [0, 0]
    for c, t, fem in meshes:
        A = af.Assembler(c, t, af.Op(af.GRAD, fem), order=2, tensor_type=af.TENSOR_SCALAR,
                         tensor_storage=af.COEF_PER_TET, rhs_order=2, rhs_tensor_type=af.TENSOR_SCALAR,
                         rhs_tensor_storage=af.COEF_CONST, dirichlet=af.DIRICHLET_NONE)
        k = torch.ones((1, len(t)), dtype=torch.float64, device="cuda")
        _, _, st = A.assemble(D=k, F=f)
        expect[0] += st.n_nonfinite
        expect[1] += st.n_degenerate
    got = []

    def run():
        for _ in range(2):
            _, _, st = B.run(good, f)
            got.append((st.n_nonfinite, st.n_degenerate))

    run()
    for _ in range(3):  # each thread takes the words of the one before
        t = threading.Thread(target=run)
        t.start()
        t.join()
    assert got == [tuple(expect)] * 8
    bad = good.clone()
    bad[7] = float("nan")
    _, _, st = B.run(bad, f)
    assert st.code == af.ERR_NONFINITE and st.n_nonfinite > expect[0] and st.n_degenerate == expect[1]
    _, _, st = B.run(good, f)
    assert (st.n_nonfinite, st.n_degenerate) == tuple(expect)
