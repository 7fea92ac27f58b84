"""Evaluation on several streams: the tables that a context uploads on the first
use are there for a call that follows on another stream, also when the first
stream is busy."""
import numpy as np
import pytest

import anifem_amd as af

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", ["evaluate", "coloured"])
def test_first_use_of_the_dof_map_is_complete_for_other_streams(first):
    import torch
    coords, tets = af.kuhn_cube(6, 0.2, 3)
    xyl = np.random.default_rng(4).dirichlet(np.ones(4), 5)
    make = lambda: af.Assembler(coords, tets, af.Op(af.GRAD, af.FEM_P2), dirichlet=af.DIRICHLET_NONE)
    ref = make()
    u = torch.from_numpy(np.random.default_rng(5).normal(size=ref.ndof)).cuda()
    expected = ref.evaluate(u, xyl)
    torch.cuda.synchronize()
    asm = make()
    outs = [torch.full_like(expected, np.nan) for _ in range(2)]
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(20_000_000)
    if first == "evaluate":
        asm.evaluate(u, xyl, out=outs[0], stream=busy)
    else:
        asm.set_scatter(af.SCATTER_COLOURED)
        asm.evaluate(u, xyl, out=outs[0], stream=busy)
    asm.evaluate(u, xyl, out=outs[1], stream=other)
    busy.synchronize()
    other.synchronize()
    for o in outs:
        assert torch.equal(o, expected)
