"""Evaluation where the points of a cell range are dealt out to several
workgroups (few cells, many points) and where the passes are longer (many of
both): runs of points that do not divide evenly, one cell, the last lane of a
workgroup, cells that fill the chip by themselves.  <= 1e-12 of the largest value
against the oracle, and every copy of a cell gets the same values."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T

pytestmark = pytest.mark.gpu

BASE = 61  # distinct cells; larger batches repeat them


@pytest.mark.parametrize("op,fem,nc,q,n", [
    (af.GRAD, af.FEM_P3, 3, 96, 1), (af.GRAD, af.FEM_P2, 3, 95, 255), (af.GRAD, af.FEM_ND0, 1, 31, 257),
    (af.GRAD, af.FEM_RT0, 1, 96, 513), (af.IDEN, af.FEM_P3, 2, 29, 300), (af.IDEN, af.FEM_P1, 1, 96, 256),
    (af.GRAD, af.FEM_P2, 1, 47, 3001), (af.IDEN, af.FEM_P2, 3, 96, 8191), (af.GRAD, af.FEM_P1, 3, 14, 20001),
    (af.IDEN, af.FEM_P1, 1, 17, 1023 * 256 + 1)])
def test_split_points_match_oracle(op, fem, nc, q, n):
    import torch
    rng = np.random.default_rng(q * 1000 + n % 997)
    o = af.Op(op, fem, nc)
    m = min(n, BASE)
    xyz, dofs = rng.uniform(-1, 1, (m, 12)), rng.normal(size=(m, o.nfa))
    xyl = rng.dirichlet(np.ones(4), q)
    ref = T.orc_apply(op, fem, nc, xyl, xyz, dofs)
    cell = np.arange(n) % m
    out = af.fem3dapply_batch(o, xyl, torch.from_numpy(T.soa_xyz(xyz[cell])).cuda(),
                              torch.from_numpy(np.ascontiguousarray(dofs[cell])).cuda())
    torch.cuda.synchronize()
    got = out[:m].cpu().numpy()
    scale = np.abs(ref).max(axis=(1, 2), keepdims=True)
    assert (np.abs(got - ref) <= 1e-12 * scale).all()
    assert torch.equal(out, out[:m][torch.from_numpy(cell).cuda()])


@pytest.mark.parametrize("fem", [af.FEM_P0, af.FEM_P1, af.FEM_P2, af.FEM_P3, af.FEM_CR1, af.FEM_B2, af.FEM_B4,
                                 af.FEM_RT0, af.FEM_ND0])
def test_points_of_each_cell_match_oracle(fem):
    """Every space and operator at each cell's own physical points
    (anifem_fem3dapplyx_batch): the cells of a mesh, whose barycentric coordinates
    lose no digits; <= 1e-12 of the largest value."""
    import torch
    vector = fem in (af.FEM_RT0, af.FEM_ND0)
    coords, tets = af.kuhn_cube(3, 0.2, 11)
    n, q = 129, 3
    xyz = coords[tets[:n]].reshape(n, 12)
    rng = np.random.default_rng(fem)
    X = T.points_physical(xyz, rng.dirichlet(np.ones(4), q))
    for op, nc in [(af.IDEN, 1), (af.GRAD, 1)] + ([(af.DIV, 1), (af.CURL, 1)] if vector else
                                                  [(af.IDEN, 2), (af.IDEN, 3), (af.GRAD, 2), (af.GRAD, 3)]):
        o = af.Op(op, fem, nc)
        dofs = rng.normal(size=(n, o.nfa))
        got = af.fem3dapplyx_batch(o, torch.from_numpy(X).cuda(), torch.from_numpy(T.soa_xyz(xyz)).cuda(),
                                   torch.from_numpy(dofs).cuda()).cpu().numpy()
        if fem == af.FEM_P0 and op == af.GRAD:  # zero; the oracle has values of P0 only
            ref = np.zeros((n, q, o.dim))
        else:
            ref = T.orc_applyx(op, fem, nc, X, xyz, dofs)
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max(), (op, nc)
