"""Meshes with nodes that no cell uses: their rows have no (row, cell) pair, only
the diagonal.  A row block holds no more rows than a workgroup has lanes for, and
every pass stores zeros there and the oracle's values elsewhere."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T


def mesh(extra):
    coords, tets = T.shuffled_mesh(*af.kuhn_cube(2, 0.2, 1), 4)
    coords = np.concatenate([coords, 2.0 + np.random.default_rng(2).random((extra, 3))])
    return coords, tets


@pytest.mark.parametrize("fem,nc,tt,budget", [(af.FEM_P1, 1, af.TENSOR_SCALAR, 256), (af.FEM_P3, 1, af.TENSOR_SCALAR, 128),
                                              (af.FEM_P2, 3, af.TENSOR_LAME, 128)])
def test_blocks_hold_a_row_per_lane(fem, nc, tt, budget):
    A = af.Assembler(*mesh(1500), af.Op(af.GRAD, fem, nc), tensor_type=tt, tensor_storage=af.COEF_PER_TET,
                     host_only=True)
    B = A.blocks()
    assert np.diff(B["blk_row0"]).max() <= budget
    assert np.diff(B["blk_row0"]).max() <= B["layout"].max_block_pairs <= budget


@pytest.mark.gpu
@pytest.mark.parametrize("fem,nc,tt", [(af.FEM_P1, 1, af.TENSOR_SCALAR), (af.FEM_P2, 1, af.TENSOR_SCALAR),
                                       (af.FEM_P3, 1, af.TENSOR_SCALAR), (af.FEM_P1, 3, af.TENSOR_LAME),
                                       (af.FEM_P2, 3, af.TENSOR_LAME), (af.FEM_ND0, 1, af.TENSOR_SCALAR),
                                       (af.FEM_CR1, 1, af.TENSOR_SCALAR)])
def test_passes_over_unused_nodes_match_oracle(fem, nc, tt):
    import torch
    coords, tets = mesh(1500)
    n = len(tets)
    rng = np.random.default_rng(fem + nc)
    op = af.CURL if fem == af.FEM_ND0 else af.GRAD
    load = 3 if nc == 3 or fem == af.FEM_ND0 else 1
    A = af.Assembler(coords, tets, af.Op(op, fem, nc), order=4, tensor_type=tt, tensor_storage=af.COEF_PER_TET,
                     rhs_order=4, rhs_tensor_type=af.TENSOR_GENERAL if load == 3 else af.TENSOR_SCALAR,
                     rhs_tensor_storage=af.COEF_PER_TET, dirichlet=af.DIRICHLET_NONE)
    s, nf, sg = A.setup(), A.nf, A.signs().astype(np.float64)
    xyz = coords[A.tets()].reshape(n, 12)
    D, f = rng.uniform(0.5, 2.0, (n, 2 if tt == af.TENSOR_LAME else 1)), rng.uniform(0.5, 2.0, (n, load))
    ttor, Dor = tt, D
    if tt == af.TENSOR_LAME:  # the 9 x 9 tensor it stands for
        I = np.eye(3)
        C1, C2 = np.einsum("ij,kl->jilk", I, I), np.einsum("ik,jl->jilk", I, I) + np.einsum("il,jk->jilk", I, I)
        ttor, Dor = af.TENSOR_GENERAL, D[:, :1] * C1.reshape(1, 81) + D[:, 1:] * C2.reshape(1, 81)
    Ae = T.orc_elem(op, fem, nc, op, fem, nc, ttor, 1, 4, xyz, Dor)
    Fe = T.orc_elem(af.IDEN, af.FEM_P0, 1, af.IDEN, fem, nc,
                    af.TENSOR_GENERAL if load == 3 else af.TENSOR_SCALAR, 1, 4, xyz, f)
    loc = torch.from_numpy(Ae.reshape(n, nf, nf)).cuda(), torch.from_numpy(Fe).cuda()
    Ae = (Ae.reshape(n, nf, nf) * sg[:, None, :] * sg[:, :, None]).reshape(n, -1)
    rc, v_or, r_or = T.oracle_scatter(n, nf, s["dofs"], s["slot"], Ae, Fe * sg, A.nnz, A.ndof)
    assert rc == 0
    unused = np.setdiff1d(np.arange(A.ndof), s["dofs"])
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a.T)).cuda()
    for persistent in (True, False):
        A.set_persistent(persistent)
        for val, rhs, st in (A.assemble(to(D), to(f)), A.assemble_elements(*loc), (None, *A.assemble_rhs(loc[1]))):
            assert st.code == 0
            if val is not None:
                assert np.abs(val.cpu().numpy() - v_or).max() <= 1e-12 * np.abs(v_or).max()
            assert np.abs(rhs.cpu().numpy() - r_or).max() <= 1e-12 * np.abs(r_or).max()
            assert not rhs.cpu().numpy()[unused].any()
