"""Two lanes per pair in the P2^3 elasticity pass (blocks of at most 128 pairs):
bitwise the values of the one-lane pass over blocks of 256 pairs and of the
per-block kernel, FP64 and FP32, with and without Dirichlet rows and load
vector; a mesh one of whose nodes exceeds the blocks takes the wider ones."""
import numpy as np
import pytest

import anifem_amd as af
import anifem_testlib as T
from test_gpu_assembly import dev

pytestmark = pytest.mark.gpu


def _context(coords, tets, dirichlet, budget=None):
    return af.Assembler(coords, tets, af.Op(af.GRAD, af.FEM_P2, 3), order=2, tensor_type=af.TENSOR_LAME,
                        tensor_storage=af.COEF_PER_TET, rhs_order=2, rhs_tensor_type=af.TENSOR_GENERAL,
                        rhs_tensor_storage=af.COEF_CONST, dirichlet=dirichlet, budget=budget)


@pytest.mark.parametrize("n,dirichlet", [(1, af.DIRICHLET_NONE), (4, af.DIRICHLET_BOUNDARY), (5, af.DIRICHLET_NONE)])
def test_two_lanes_match_one_lane_and_per_block(n, dirichlet):
    coords, tets = T.shuffled_mesh(*af.kuhn_cube(n, 0.2, 3), 2)
    rng = np.random.default_rng(n)
    D, F = dev(rng.uniform(0.5, 2.0, (2, len(tets)))), dev(rng.uniform(-1, 1, 3))
    A, W = _context(coords, tets, dirichlet), _context(coords, tets, dirichlet, (4096, 8192, 256))
    assert A.block_layout().max_block_pairs <= 128
    for prec in (af.PREC_FP64, af.PREC_FP32):
        for load in (F, None):
            got = []
            for ctx, mode in ((A, 1), (A, 0), (W, 1), (W, 0)):
                ctx.set_persistent(mode)
                val, rhs, st = ctx.assemble(D=D, F=load, precision=prec)
                assert st.code == 0
                got.append((val.cpu().numpy(), None if rhs is None else rhs.cpu().numpy()))
            for v, r in got[1:]:
                assert np.array_equal(v, got[0][0])
                assert r is None or np.array_equal(r, got[0][1])


def test_node_beyond_the_split_blocks():
    coords, tets = T.fan_mesh(80)  # a node of 160 cells
    A = _context(coords, tets, af.DIRICHLET_NONE)
    assert A.block_layout().max_block_pairs > 128
    D = dev(np.ones((2, len(tets))))
    val, rhs, st = A.assemble(D=D, F=dev(np.array([0.0, 0.0, -1.0])))
    A.set_persistent(0)
    v0, r0, _ = A.assemble(D=D, F=dev(np.array([0.0, 0.0, -1.0])))
    assert st.code == 0 and np.array_equal(val.cpu().numpy(), v0.cpu().numpy())
    assert np.array_equal(rhs.cpu().numpy(), r0.cpu().numpy())
