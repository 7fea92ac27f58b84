"""Element matrices with a constant tensor per cell at the edges of the kernel's
launch shapes: one cell, batches either side of a change of the cells per
workgroup, an output aligned to one value only (single rows instead of row
pairs), spaces with an odd number of rows, columns that do not fill the lane
groups.  FP64 <= 1e-12, FP32 <= 5e-6 relative Frobenius per element against the
oracle, as for the other element kernels."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T

pytestmark = pytest.mark.gpu

BASE = 61  # distinct cells; larger batches repeat them


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


@pytest.mark.parametrize("pair,tt,n", [
    ((2, 2, 1, 2, 2, 1), af.TENSOR_SCALAR, 1), ((2, 2, 1, 2, 2, 1), af.TENSOR_GENERAL, 512 * 32 + 1),
    ((2, 3, 1, 2, 3, 1), af.TENSOR_SYMMETRIC, 512 * 32 - 1), ((2, 3, 1, 2, 3, 1), af.TENSOR_GENERAL, 512 * 256 + 3),
    ((2, 4, 1, 2, 4, 1), af.TENSOR_SCALAR, 257), ((1, 4, 1, 1, 4, 1), af.TENSOR_SCALAR, 19),
    ((2, 2, 3, 2, 2, 3), af.TENSOR_LAME, 23), ((2, 3, 3, 2, 3, 3), af.TENSOR_LAME, 512 * 64 + 7),
    ((2, 4, 3, 2, 4, 3), af.TENSOR_LAME, 33), ((2, 3, 3, 2, 3, 3), af.TENSOR_SCALAR, 40),
    ((2, 4, 1, 2, 2, 3), af.TENSOR_GENERAL, 50), ((1, 1, 1, 1, 3, 3), af.TENSOR_SCALAR, 35),
    ((1, 1004, 1, 1, 1004, 1), af.TENSOR_SCALAR, 70), ((1, 2, 1, 1, 1004, 1), af.TENSOR_SCALAR, 31),
    ((1, 25, 1, 1, 25, 1), af.TENSOR_SYMMETRIC, 129), ((4, 25, 1, 4, 25, 1), af.TENSOR_GENERAL, 15),
    ((1, 21, 1, 1, 21, 1), af.TENSOR_SCALAR, 64), ((4, 25, 1, 1, 21, 1), af.TENSOR_GENERAL, 17)])
def test_const_kernel_shapes_match_oracle(pair, tt, n):
    import torch
    oa, fa, ca, ob, fb, cb = pair
    opA, opB = af.Op(oa, fa, ca), af.Op(ob, fb, cb)
    dA, dB = opA.dim, opB.dim
    rng = np.random.default_rng(fa * 7 + fb + n % 1000)
    m = min(n, BASE)
    xyz = rng.uniform(-1, 1, (m, 12))
    dd = {af.TENSOR_SCALAR: 1, af.TENSOR_LAME: 2}.get(tt, dA * dB)
    D = rng.uniform(0.5, 2.0, (m, dd))
    Dprod, Dor, ttor = D, D, tt
    if tt == af.TENSOR_SYMMETRIC:
        M = D.reshape(m, dB, dB)
        Dor = (M + M.transpose(0, 2, 1)).reshape(m, -1)
        Dprod = T.pack_sym(Dor, dB)
    elif tt == af.TENSOR_LAME:  # the 9 x 9 tensor it stands for
        ttor, I = af.TENSOR_GENERAL, np.eye(3)
        C1, C2 = np.einsum("ij,kl->jilk", I, I), np.einsum("ik,jl->jilk", I, I) + np.einsum("il,jk->jilk", I, I)
        Dor = D[:, :1] * C1.reshape(1, 81) + D[:, 1:] * C2.reshape(1, 81)
    ref = T.orc_elem(oa, fa, ca, ob, fb, cb, ttor, af.COEF_PER_TET, 4, xyz, Dor)
    cell = np.arange(n) % m
    xd, Dd = dev(T.soa_xyz(xyz[cell])), dev(Dprod[cell].T)
    E = opA.nfa * opB.nfa
    for prec, dt, tol in [(af.PREC_FP64, torch.float64, 1e-12), (af.PREC_FP32, torch.float32, 5e-6)]:
        for shift in (0, 1):
            buf = torch.full((n * E + 2,), -7.0, dtype=dt, device="cuda")
            out = buf[shift:shift + n * E].view(n, opA.nfa, opB.nfa)
            af.fem3dtet_batch(opA, opB, tt, af.COEF_PER_TET, Dd, 4, xd, precision=prec, out=out)
            A = out.cpu().numpy().reshape(n, -1).astype(np.float64)
            assert (buf[shift + n * E:] == -7.0).all() and (buf[:shift] == -7.0).all()
            assert T.rel_frob(A[:m], ref) <= tol
            assert np.array_equal(A, A[cell])  # a cell's matrix does not depend on its place


@pytest.mark.parametrize("pair,tt,n", [
    ((2, 4, 3, 2, 4, 3), af.TENSOR_GENERAL, 1), ((1, 4, 3, 1, 4, 3), af.TENSOR_SCALAR, 37),
    ((2, 4, 3, 2, 4, 3), af.TENSOR_SYMMETRIC, 512 * 32 + 1), ((1, 4, 1, 2, 4, 3), af.TENSOR_GENERAL, 51),
    ((2, 4, 3, 1, 4, 1), af.TENSOR_GENERAL, 49), ((2, 3, 1, 2, 4, 3), af.TENSOR_GENERAL, 18),
    ((2, 3, 3, 2, 4, 3), af.TENSOR_GENERAL, 41), ((2, 4, 3, 2, 3, 3), af.TENSOR_GENERAL, 41),
    ((1, 3, 3, 1, 4, 3), af.TENSOR_SCALAR, 1)])
def test_matrices_of_several_passes_match_oracle(pair, tt, n):
    """More items than lanes: whole columns per pass, the last pass's cells dealt
    out to groups of lanes."""
    test_const_kernel_shapes_match_oracle(pair, tt, n)


@pytest.mark.parametrize("pair,tt", [((1, 21, 1, 1, 21, 1), af.TENSOR_GENERAL), ((2, 25, 1, 2, 25, 1), af.TENSOR_SYMMETRIC),
                                     ((4, 25, 1, 4, 25, 1), af.TENSOR_GENERAL), ((1, 4, 3, 1, 21, 1), af.TENSOR_GENERAL)])
@pytest.mark.parametrize("n", [384 * 32 - 1, 384 * 32, 384 * 128 + 5, 384 * 256 - 1, 384 * 256 + 1])
def test_face_and_edge_spaces_either_side_of_a_change_of_cells_per_workgroup(pair, tt, n):
    test_const_kernel_shapes_match_oracle(pair, tt, n)
