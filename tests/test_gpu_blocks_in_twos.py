"""Elasticity contexts on three components of P2 have blocks of at most 128 pairs;
general element matrices and load vectors take them in twos.  Values and
right-hand sides equal those of one workgroup per block bit for bit, and the
oracle's sequential scatter: one block, an odd number, blocks that stay alone (a
node of many cells), Dirichlet rows, rows without a cell."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T

pytestmark = pytest.mark.gpu


def meshes(name):
    if name == "fan":
        return T.fan_mesh(30)
    coords, tets = T.shuffled_mesh(*af.kuhn_cube({"one": 1, "small": 2, "cube": 4, "unused": 2}[name], 0.2, 3), 5)
    if name == "unused":
        coords = np.concatenate([coords, np.random.default_rng(1).random((300, 3)) + 2.0])
    return coords, tets


@pytest.mark.parametrize("dirichlet", [af.DIRICHLET_NONE, af.DIRICHLET_BOUNDARY])
@pytest.mark.parametrize("name", ["one", "small", "cube", "fan", "unused"])
def test_general_matrices_and_load_vectors(name, dirichlet):
    import torch
    coords, tets = meshes(name)
    A = af.Assembler(coords, tets, af.Op(af.GRAD, af.FEM_P2, 3), tensor_type=af.TENSOR_LAME,
                     tensor_storage=af.COEF_PER_TET, dirichlet=dirichlet)
    assert A.block_layout().max_block_pairs <= 128
    n, nf, s = len(tets), A.nf, A.setup()
    rng = np.random.default_rng(n)
    Ae, Fe = rng.normal(size=(n, nf * nf)), rng.normal(size=(n, nf))
    Ao, Fo = T.apply_dir_elementwise(Ae, Fe, s["dofs"], s["dirichlet"])
    for dt in (torch.float64, torch.float32):
        E, F = torch.from_numpy(Ae.reshape(n, nf, nf)).to(dt).cuda(), torch.from_numpy(Fe).to(dt).cuda()
        got = []
        for persistent in (True, False):
            A.set_persistent(persistent)
            val, rhs, st = A.assemble_elements(E, F)
            assert st.code == 0
            got.append((val, rhs))
        rhs2, st = A.assemble_rhs(F)
        assert st.code == 0
        assert torch.equal(got[0][0], got[1][0])
        assert torch.equal(got[0][1], got[1][1]) and torch.equal(rhs2, got[1][1])
        if dt == torch.float64:
            rc, v_or, r_or = T.oracle_scatter(n, nf, s["dofs"], s["slot"], Ao, Fo, A.nnz, A.ndof)
            assert rc == 0
            assert np.abs(got[0][0].cpu().numpy() - v_or).max() <= 1e-14 * np.abs(v_or).max()
            assert np.abs(rhs2.cpu().numpy() - r_or).max() <= 1e-14 * np.abs(r_or).max()
    # counts of entries that are not finite, over both blocks of a record
    E = torch.from_numpy(Ae.reshape(n, nf, nf)).cuda()
    E[n // 2, 3, :] = np.nan
    A.set_persistent(True)
    c1 = A.assemble_elements(E)[2]
    A.set_persistent(False)
    c0 = A.assemble_elements(E)[2]
    assert c1.code == c0.code and c1.n_nonfinite == c0.n_nonfinite
