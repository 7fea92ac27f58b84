"""The fused RT0 / ND0 assembly against the oracle for every tensor form it
takes (packed symmetric, general, constant over the mesh), in FP32, without a
load vector, and its non-finite count.  FP64 within 1e-12 and FP32 within 2e-5 of
the row maximum, as for the other assembled matrices."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T
from test_gpu_assembly import dev

pytestmark = pytest.mark.gpu

RT0, ND0, P0 = af.FEM_RT0, af.FEM_ND0, af.FEM_P0


@pytest.mark.parametrize("op,fem,tt,storage,n", [
    (af.IDEN, ND0, af.TENSOR_SYMMETRIC, af.COEF_PER_TET, 4), (af.CURL, ND0, af.TENSOR_GENERAL, af.COEF_PER_TET, 4),
    (af.IDEN, RT0, af.TENSOR_GENERAL, af.COEF_CONST, 3), (af.IDEN, RT0, af.TENSOR_SYMMETRIC, af.COEF_PER_TET, 5),
    (af.DIV, RT0, af.TENSOR_SCALAR, af.COEF_CONST, 1), (af.GRAD, ND0, af.TENSOR_GENERAL, af.COEF_PER_TET, 2)])
def test_fused_tensor_forms_match_oracle(op, fem, tt, storage, n):
    import torch
    coords, tets = T.shuffled_mesh(*af.kuhn_cube(n, 0.2, 5), 6)
    m = len(tets)
    rng = np.random.default_rng(op * 10 + n)
    d = af.Op(op, fem).dim
    k = 1 if storage == af.COEF_CONST else m
    D = rng.uniform(-1, 1, (k, 1 if tt == af.TENSOR_SCALAR else d * d))
    Dprod = Dor = D
    if tt == af.TENSOR_SYMMETRIC:
        M = D.reshape(k, d, d)
        Dor = (M + M.transpose(0, 2, 1)).reshape(k, -1)
        Dprod = T.pack_sym(Dor, d)
    Asm = af.Assembler(coords, tets, af.Op(op, fem), order=2, tensor_type=tt, tensor_storage=storage, rhs_order=2,
                       rhs_tensor_type=af.TENSOR_GENERAL, rhs_tensor_storage=af.COEF_PER_TET,
                       dirichlet=af.DIRICHLET_BOUNDARY)
    f = rng.uniform(-1, 1, (m, 3))
    s, rt, sg, nf = Asm.setup(), Asm.tets(), Asm.signs().astype(np.float64), Asm.nf
    xyz = coords[rt].reshape(m, 12)
    A = T.orc_elem(op, fem, 1, op, fem, 1, tt, storage, 2, xyz, Dor)
    F = T.orc_elem(af.IDEN, P0, 1, af.IDEN, fem, 1, af.TENSOR_GENERAL, 1, 2, xyz, f) * sg
    A = (A.reshape(m, nf, nf) * sg[:, None, :] * sg[:, :, None]).reshape(m, -1)
    A, F = T.apply_dir_elementwise(A, F, s["dofs"], s["dirichlet"])
    rc, v_or, r_or = T.oracle_scatter(m, nf, s["dofs"], s["slot"], A, F, Asm.nnz, Asm.ndof)
    assert rc == 0
    rowmax = np.repeat(np.maximum.reduceat(np.abs(v_or), s["row_ptr"][:-1]), np.diff(s["row_ptr"]))
    Dd = dev(Dprod.ravel() if k == 1 else Dprod.T.copy())
    for prec, tol in [(af.PREC_FP64, 1e-12), (af.PREC_FP32, 2e-5)]:
        val, rhs, st = Asm.assemble(D=Dd, F=dev(f.T.copy()), precision=prec)
        assert st.code == 0
        assert np.abs((val.cpu().numpy() - v_or) / rowmax).max() <= tol
        assert np.abs(rhs.cpu().numpy() - r_or).max() <= tol * max(np.abs(r_or).max(), 1e-300)
    v2 = torch.empty_like(val)
    r2 = torch.full_like(rhs, 7.0)  # no load vector: the values alone, a zero right-hand side
    Asm.assemble(D=Dd, val=v2, rhs=r2)
    assert np.abs((v2.cpu().numpy() - v_or) / rowmax).max() <= 1e-12 and (r2 == 0).all()


def test_fused_nonfinite_count_and_reset():
    coords, tets = af.kuhn_cube(2, 0.2, 1)
    kappa = np.ones((1, len(tets)))
    kappa[0, 7] = np.nan
    Asm = af.Assembler(coords, tets, af.Op(af.IDEN, ND0), order=2, tensor_type=af.TENSOR_SCALAR,
                       tensor_storage=af.COEF_PER_TET, dirichlet=af.DIRICHLET_NONE)
    _, _, st = Asm.assemble(D=dev(kappa))
    assert st.code == af.ERR_NONFINITE and st.n_nonfinite == 36  # every entry of one 6 x 6 matrix
    _, _, st = Asm.assemble(D=dev(np.ones((1, len(tets)))))
    assert st.code == 0 and st.n_nonfinite == 0
