"""Element matrices and face integrals of the operators that select part of a
gradient (DUDX, DUDY, DUDZ on both sides; DIV and CURL of three components; the
normal form) for every form of the coefficient, and above all for coefficients
that vary over the points of a cell.  Cell counts are odd.  FP64 <= 1e-12, FP32
<= 5e-6 relative Frobenius per element against the oracle, as for the other
element kernels."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T

pytestmark = pytest.mark.gpu

N = 35
PRECISIONS = [(af.PREC_FP64, 1e-12), (af.PREC_FP32, 5e-6)]
# degree of the basis functions' derivatives
DERIVATIVE_DEGREE = {af.FEM_P1: 0, af.FEM_P2: 1, af.FEM_P3: 2, af.FEM_CR1: 0, af.FEM_B2: 1, af.FEM_B4: 3}


def dev(a):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def host(t):
    return t.cpu().numpy().reshape(t.shape[0], -1).astype(np.float64)


def cells(seed):
    return np.random.default_rng(seed).uniform(-1, 1, (N, 12))


def coefficients(tt, storage, nv, q, rng):
    """nv values per cell and point, constant as `storage` says: (N, q, nv)."""
    shape = {af.COEF_CONST: (1, 1, nv), af.COEF_PER_TET: (N, 1, nv), af.COEF_PER_POINT: (N, q, nv)}[storage]
    return np.broadcast_to(rng.uniform(0.5, 2.0, shape), (N, q, nv))


def stored(values, tt, storage):
    """The product's array of coefficients (N, q, nv)."""
    if tt == af.TENSOR_NULL:
        return None
    if storage == af.COEF_CONST:
        return dev(values[0, 0])
    v = values[:, :1] if storage == af.COEF_PER_TET else values
    return dev(v.transpose(2, 1, 0))


@pytest.mark.parametrize("fem", list(DERIVATIVE_DEGREE))
@pytest.mark.parametrize("op", [af.DUDX, af.DUDY, af.DUDZ])
def test_derivative_pairs_match_oracle(op, fem):
    o = af.Op(op, fem)
    rng = np.random.default_rng(100 * op + fem)
    xyz = cells(op + fem)
    xd = dev(T.soa_xyz(xyz))
    deg = 2 * DERIVATIVE_DEGREE[fem] + 2  # of an integrand with a quadratic coefficient
    for tt in (af.TENSOR_NULL, af.TENSOR_SCALAR, af.TENSOR_SYMMETRIC):
        for storage in (af.COEF_CONST, af.COEF_PER_TET, af.COEF_PER_POINT):
            for order in (2, 5):
                perm = T.point_permutation(order)
                c = coefficients(tt, storage, 1, len(perm), rng)
                ref = T.orc_elem(op, fem, 1, op, fem, 1, tt, af.COEF_PER_POINT, order, xyz, c.reshape(N, -1))
                D = stored(c[:, perm], tt, storage)
                for prec, tol in PRECISIONS:
                    A = host(af.fem3dtet_batch(o, o, tt, storage, D, order, xd, precision=prec))
                    assert T.rel_frob(A, ref) <= tol, ("volume", tt, storage, order, prec)
            for face in (0, 3):
                p, po = af.face_quadrature(deg, face)[0], T.orc_face_quadrature(face)[0]
                c = coefficients(tt, storage, 1, 1, rng)[:, 0, :]
                m, mo = (T.xdep_field(T.points_physical(xyz, x)) if storage == af.COEF_PER_POINT
                         else np.ones((N, len(x))) for x in (p, po))
                ref = T.orc_face(op, fem, 1, op, fem, 1, tt, af.COEF_PER_POINT, face, 0, xyz, c * mo)
                D = stored((c * m)[:, :, None], tt, storage)
                for prec, tol in PRECISIONS:
                    A = host(af.fem3dface_batch(o, o, tt, storage, D, deg, face, xd, precision=prec))
                    assert T.rel_frob(A, ref) <= tol, ("face", face, tt, storage, prec)


@pytest.mark.parametrize("opA,ncA,opB,ncB,fem,tt,rows,cols", [
    (af.DIV, 3, af.DIV, 3, af.FEM_P2, af.TENSOR_SCALAR, 1, 1), (af.DIV, 3, af.DIV, 3, af.FEM_P1, af.TENSOR_GENERAL, 1, 1),
    (af.CURL, 3, af.CURL, 3, af.FEM_P2, af.TENSOR_SCALAR, 3, 3), (af.CURL, 3, af.CURL, 3, af.FEM_P1, af.TENSOR_GENERAL, 3, 3),
    (af.CURL, 3, af.IDEN, 3, af.FEM_P2, af.TENSOR_GENERAL, 3, 3), (af.DUDX, 1, af.DUDY, 1, af.FEM_P2, af.TENSOR_SCALAR, 1, 1),
    (af.DUDZ, 3, af.DUDZ, 3, af.FEM_P1, af.TENSOR_SCALAR, 3, 3)])
def test_selecting_operators_with_point_coefficients_match_oracle(opA, ncA, opB, ncB, fem, tt, rows, cols):
    order = 4
    oa, ob = af.Op(opA, fem, ncA), af.Op(opB, fem, ncB)
    rng = np.random.default_rng(opA * 10 + opB)
    xyz = cells(opA * 7 + fem)
    perm = T.point_permutation(order)
    nv = 1 if tt == af.TENSOR_SCALAR else rows * cols
    c = coefficients(tt, af.COEF_PER_POINT, nv, len(perm), rng)
    ref = T.orc_elem(opA, fem, ncA, opB, fem, ncB, tt, af.COEF_PER_POINT, order, xyz, c.reshape(N, -1))
    D = stored(c[:, perm], tt, af.COEF_PER_POINT)
    for prec, tol in PRECISIONS:
        A = host(af.fem3dtet_batch(oa, ob, tt, af.COEF_PER_POINT, D, order, dev(T.soa_xyz(xyz)), precision=prec))
        assert T.rel_frob(A, ref) <= tol, prec


@pytest.mark.parametrize("opA,ncA,fem,cols,face", [(af.GRAD, 1, af.FEM_P2, 3, 1), (af.GRAD, 1, af.FEM_P1, 3, 2),
                                                   (af.DUDY, 1, af.FEM_P2, 1, 0), (af.DIV, 3, af.FEM_P1, 1, 3)])
def test_normal_form_with_point_coefficients_matches_oracle(opA, ncA, fem, cols, face):
    """((D OpA(u)) . n) v: D has the three rows of the normal's components."""
    order = 6  # derivative 1, coefficient 2, value 2
    oa, ob = af.Op(opA, fem, ncA), af.Op(af.IDEN, fem)
    xyz = cells(fem + face)
    c = np.random.default_rng(opA + face).normal(size=(N, 3 * cols))
    p, po = af.face_quadrature(order, face)[0], T.orc_face_quadrature(face)[0]
    m, mo = (T.xdep_field(T.points_physical(xyz, x))[:, :, None] for x in (p, po))
    ref = T.orc_face(opA, fem, ncA, af.IDEN, fem, 1, af.TENSOR_GENERAL, af.COEF_PER_POINT, face, 1, xyz,
                     (mo * c[:, None, :]).reshape(N, -1))
    D = stored(m * c[:, None, :], af.TENSOR_GENERAL, af.COEF_PER_POINT)
    for prec, tol in PRECISIONS:
        A = host(af.fem3dface_batch(oa, ob, af.TENSOR_GENERAL, af.COEF_PER_POINT, D, order, face, dev(T.soa_xyz(xyz)),
                                    dot_normal=True, precision=prec))
        assert T.rel_frob(A, ref) <= tol, prec
