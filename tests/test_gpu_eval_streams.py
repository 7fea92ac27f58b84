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


@pytest.mark.parametrize("handle", [False, True])
@pytest.mark.parametrize("call", ["evaluate", "apply"])
def test_result_of_another_stream_is_read_in_order(call, handle):
    """The current stream follows the stream that was given to the call: reading
    the result at once gives the values, with the given stream still busy."""
    import torch
    coords, tets = af.kuhn_cube(5, 0.2, 7)
    xyl = np.random.default_rng(8).dirichlet(np.ones(4), 3)
    op = af.Op(af.GRAD, af.FEM_P2)
    asm = af.Assembler(coords, tets, op, dirichlet=af.DIRICHLET_BOUNDARY)
    u = torch.from_numpy(np.random.default_rng(9).normal(size=asm.ndof)).cuda()
    dofs = torch.from_numpy(np.random.default_rng(9).normal(size=(len(tets), op.nfa))).cuda()
    xyz = torch.from_numpy(np.ascontiguousarray(coords[tets].reshape(len(tets), 12).T)).cuda()
    run = {"evaluate": lambda **k: asm.evaluate(u, xyl, **k),
           "apply": lambda **k: af.fem3dapply_batch(op, xyl, xyz, dofs, **k)}[call]
    expected = run().cpu()
    out = torch.full(expected.shape, np.nan, dtype=torch.float64, device="cuda")
    busy = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(20_000_000)
    got = run(out=out, stream=busy.cuda_stream if handle else busy).cpu()
    assert torch.equal(got, expected)
