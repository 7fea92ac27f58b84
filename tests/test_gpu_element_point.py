"""Element matrices with a coefficient at the quadrature points, at the edges of
the per-point kernel's launch shapes: one cell, cells either side of a
workgroup's tile, the wide shapes of large batches, entries of one to 25 tiles,
an output that is not 16-byte aligned.  FP64 <= 1e-12, FP32 <= 5e-6 relative
Frobenius per element against the oracle, as for the other element kernels."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T

pytestmark = pytest.mark.gpu

BASE = 97  # distinct cells; larger batches repeat them


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


@pytest.mark.parametrize("op,fem,nc,tt,order,n", [
    (af.GRAD, af.FEM_P1, 1, af.TENSOR_SCALAR, 2, 1), (af.GRAD, af.FEM_P1, 1, af.TENSOR_GENERAL, 2, 65),
    (af.GRAD, af.FEM_P2, 1, af.TENSOR_SCALAR, 4, 17), (af.GRAD, af.FEM_P2, 1, af.TENSOR_SYMMETRIC, 4, 512 * 64 + 5),
    (af.GRAD, af.FEM_P2, 1, af.TENSOR_GENERAL, 6, 512 * 64 + 63), (af.GRAD, af.FEM_P3, 1, af.TENSOR_SCALAR, 6, 97),
    (af.GRAD, af.FEM_P3, 1, af.TENSOR_SCALAR, 6, 512 * 64 + 1), (af.GRAD, af.FEM_P3, 1, af.TENSOR_GENERAL, 4, 512 * 32 + 31),
    (af.GRAD, af.FEM_P3, 1, af.TENSOR_GENERAL, 6, 33), (af.IDEN, af.FEM_P3, 1, af.TENSOR_SCALAR, 6, 512 * 32 + 33),
    (af.GRAD, af.FEM_P2, 3, af.TENSOR_LAME, 4, 70), (af.IDEN, af.FEM_ND0, 1, af.TENSOR_SCALAR, 2, 129),
    (af.CURL, af.FEM_ND0, 1, af.TENSOR_SYMMETRIC, 2, 64), (af.IDEN, af.FEM_RT0, 1, af.TENSOR_GENERAL, 4, 63),
    (af.IDEN, af.FEM_B4, 1, af.TENSOR_SCALAR, 6, 66)])
def test_point_kernel_shapes_match_oracle(op, fem, nc, tt, order, n):
    import torch
    rng = np.random.default_rng(order * 1000 + n % 1000 + fem)
    o = af.Op(op, fem, nc)
    m = min(n, BASE)
    xyz = rng.uniform(-1, 1, (m, 12))
    perm = T.point_permutation(order)
    q = len(perm)
    dd = {af.TENSOR_SCALAR: 1, af.TENSOR_LAME: 2}.get(tt, o.dim * o.dim)
    D = rng.uniform(0.5, 2.0, (m, q, dd))
    Dprod = Dor = D
    ttor = tt
    if tt == af.TENSOR_SYMMETRIC:
        M = D.reshape(m * q, o.dim, o.dim)
        Dor = (M + M.transpose(0, 2, 1)).reshape(m, q, -1)
        Dprod = T.pack_sym(Dor.reshape(m * q, -1), o.dim).reshape(m, q, -1)
    elif tt == af.TENSOR_LAME:  # the 9 x 9 tensor it stands for
        ttor = af.TENSOR_GENERAL
        I = np.eye(3)
        C1, C2 = np.einsum("ij,kl->jilk", I, I), np.einsum("ik,jl->jilk", I, I) + np.einsum("il,jk->jilk", I, I)
        Dor = (D[:, :, :1] * C1.reshape(1, 1, 81) + D[:, :, 1:] * C2.reshape(1, 1, 81)).reshape(m, q, 81)
    ref = T.orc_elem(op, fem, nc, op, fem, nc, ttor, af.COEF_PER_POINT, order, xyz, Dor.reshape(m, -1))
    cell = np.arange(n) % m
    xd = dev(T.soa_xyz(xyz[cell]))
    Dd = dev(Dprod[:, perm, :][cell].transpose(2, 1, 0))
    for prec, dt, tol in [(af.PREC_FP64, torch.float64, 1e-12), (af.PREC_FP32, torch.float32, 5e-6)]:
        for shift in (0, 1):  # the second output starts one value past a 16-byte boundary
            buf = torch.full((n * o.nfa * o.nfa + 2,), -7.0, dtype=dt, device="cuda")
            out = buf[shift:shift + n * o.nfa * o.nfa].view(n, o.nfa, o.nfa)
            af.fem3dtet_batch(o, o, tt, af.COEF_PER_POINT, Dd, order, xd, precision=prec, out=out)
            A = out.cpu().numpy().reshape(n, -1).astype(np.float64)
            assert (buf[shift + n * o.nfa * o.nfa:] == -7.0).all() and (buf[:shift] == -7.0).all()
            assert T.rel_frob(A[:m], ref) <= tol
            assert np.array_equal(A, A[cell])  # a cell's matrix does not depend on its place


def test_point_kernel_keeps_nonfinite_values_in_their_cell():
    rng = np.random.default_rng(3)
    n, q = 40, len(T.point_permutation(4))
    xyz, D = rng.uniform(-1, 1, (n, 12)), rng.uniform(0.5, 2.0, (1, q, n))
    D[0, 3, 17] = np.nan
    o = af.Op(af.GRAD, af.FEM_P2)
    A = af.fem3dtet_batch(o, o, af.TENSOR_SCALAR, af.COEF_PER_POINT, dev(D), 4, dev(T.soa_xyz(xyz))).cpu().numpy()
    bad = np.isnan(A).reshape(n, -1).any(axis=1)
    assert bad[17] and bad.sum() == 1
