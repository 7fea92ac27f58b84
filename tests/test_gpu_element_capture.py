"""Element matrices with coefficients at the points under stream capture: once the
table of an operator pair, rule and storage is there, from a call with another
tensor or from an assembly, a call allocates nothing and can be captured; every
replay equals the eager call."""
import numpy as np
import pytest

import anifem_amd as af

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fem,order,first", [(af.FEM_B2, 3, "general"), (af.FEM_CR1, 3, "assembly"),
                                             (af.FEM_B2, 7, "symmetric")])
def test_capture_after_another_tensor(fem, order, first):
    import torch
    rng = np.random.default_rng(order)
    coords, tets = af.kuhn_cube(2, 0.2, 1)
    n, q = len(tets), len(af.quadrature(order)[1])
    op = af.Op(af.GRAD, fem)
    xyz = torch.from_numpy(np.ascontiguousarray(coords[tets].reshape(n, 12).T)).cuda()
    D = {t: torch.from_numpy(rng.uniform(0.5, 2.0, (k, q, n))).cuda()
         for t, k in ((af.TENSOR_SCALAR, 1), (af.TENSOR_SYMMETRIC, 6), (af.TENSOR_GENERAL, 9))}
    if first == "assembly":
        asm = af.Assembler(coords, tets, op, order=order, tensor_type=af.TENSOR_SCALAR,
                           tensor_storage=af.COEF_PER_POINT, dirichlet=af.DIRICHLET_NONE)
        asm.assemble(D[af.TENSOR_SCALAR])
    else:
        tt = {"general": af.TENSOR_GENERAL, "symmetric": af.TENSOR_SYMMETRIC}[first]
        af.fem3dtet_batch(op, op, tt, af.COEF_PER_POINT, D[tt], order, xyz)
    out = {t: torch.empty((n, op.nfa, op.nfa), dtype=torch.float64, device="cuda") for t in D}
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for t in D:
            af.fem3dtet_batch(op, op, t, af.COEF_PER_POINT, D[t], order, xyz, out=out[t])
    for k in range(4):
        for t in D:
            out[t].fill_(np.nan)
            D[t].mul_(1.25)
        g.replay()
        for t in D:
            eager = af.fem3dtet_batch(op, op, t, af.COEF_PER_POINT, D[t], order, xyz)
            assert torch.equal(out[t], eager), (k, t)
