"""Performance cases of the element-matrix and assembly library.

A case is a dict of plain values; `kind` names the part of the library that a
program calls:

  element    element matrices of a batch of cells (fem3dtet_batch)
  assemble   matrix and load vector of a mesh (Assembler.assemble)
  evaluate   a global solution vector at points of every cell (Assembler.evaluate)
  batch      many meshes of different sizes and orders at once (Batch.run)
  pcg        Jacobi-preconditioned CG on an assembled system (pcg_jacobi)

Meshes are boxes of nx x ny x nz sub-cubes of six Kuhn tetrahedra with jittered
interior nodes, made here so that the float64 references need none of the
library's code.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "inmost-fem_amd"))
import anifem_amd as af  # noqa: E402

DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")
F64 = torch.float64

# ---- cases -------------------------------------------------------------------
FEM = {"P0": af.FEM_P0, "P1": af.FEM_P1, "P2": af.FEM_P2, "P3": af.FEM_P3, "ND0": af.FEM_ND0, "RT0": af.FEM_RT0}
OP = {"iden": af.IDEN, "grad": af.GRAD, "div": af.DIV, "curl": af.CURL}
TENSOR = {"scalar": af.TENSOR_SCALAR, "symmetric": af.TENSOR_SYMMETRIC, "general": af.TENSOR_GENERAL,
          "lame": af.TENSOR_LAME}
STORAGE = {"const": af.COEF_CONST, "tet": af.COEF_PER_TET, "point": af.COEF_PER_POINT}
PREC = {"fp64": af.PREC_FP64, "fp32": af.PREC_FP32, "fp16x3": af.PREC_FP16X3}
DEGREE = {"P0": 0, "P1": 1, "P2": 2, "P3": 3, "ND0": 1, "RT0": 1}
NFA = {"P0": 1, "P1": 4, "P2": 10, "P3": 20, "ND0": 6, "RT0": 4}
# stored couplings per sub-cube of an unbounded Kuhn lattice: ordered pairs of
# DOFs that share a cell (1 node, 7 edges, 12 faces, 6 cells per sub-cube)
COUPLINGS = {"P1": 15, "P2": 230, "P3": 1311, "ND0": 115, "RT0": 84}
DOFS = {"P1": 1, "P2": 8, "P3": 27, "ND0": 7, "RT0": 12}


def element(name, fem, op, tensor, storage, order, n, nc=1, prec="fp64"):
    return dict(name=name, kind="element", fem=fem, op=op, tensor=tensor, storage=storage, order=order, n=n, nc=nc,
                prec=prec)


def assemble(name, fem, op, tensor, nx, ny, nz, nc=1, prec="fp64", status=False):
    return dict(name=name, kind="assemble", fem=fem, op=op, tensor=tensor, nx=nx, ny=ny, nz=nz, nc=nc, prec=prec,
                status=status)


def listed():
    return [
        # a handful of cells, e.g. one refinement patch: the latency of a call
        element("element_p1_small", "P1", "grad", "scalar", "tet", 1, 384),
        # anisotropic diffusion element matrices for a user's own scatter (the benchmark's size)
        element("element_p2_aniso", "P2", "grad", "symmetric", "tet", 2, 1572864),
        # coefficient that varies inside the cells, given at the rule's points
        element("element_p3_pointwise", "P3", "grad", "scalar", "point", 6, 93701),
        # 30 x 30 elasticity matrices in single precision
        element("element_p2vec_fp32", "P2", "grad", "lame", "tet", 2, 663552, 3, "fp32"),
        # a small Poisson problem, status checked as a program does by default
        assemble("assemble_p1_small", "P1", "grad", "scalar", 16, 16, 16, status=True),
        # the headline workload: P2 anisotropic diffusion at 64^3
        assemble("assemble_p2_aniso", "P2", "grad", "symmetric", 64, 64, 64),
        # linear elasticity, P2^3, per-cell Lame parameters: the largest system
        assemble("assemble_p2vec", "P2", "grad", "lame", 48, 48, 48, 3),
        # curl-curl matrix of edge elements (Maxwell)
        assemble("assemble_nd0_curl", "ND0", "curl", "scalar", 33, 31, 32),
        # post-processing: the gradient of a P2 solution at four points of every cell
        dict(name="evaluate_p2_grad", kind="evaluate", fem="P2", op="grad", nc=1, q=4, nx=48, ny=48, nz=48),
        # many meshes of uneven size and order in one call
        dict(name="batch_mixed", kind="batch", meshes=32, lo=4, hi=24),
        # a small solve: 16^3 P1 Poisson to 1e-10
        dict(name="pcg_p1_small", kind="pcg", fem="P1", nx=16, ny=16, nz=16, rtol=1e-10),
        # a solve whose matrix outweighs the caches of one chiplet
        dict(name="pcg_p2", kind="pcg", fem="P2", nx=40, ny=40, nz=40, rtol=1e-8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """Side lengths around one log-uniform size, not all equal."""
    s = _log(rng, lo, hi)
    return [max(2, min(hi, s + rng.randint(-2, 2))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["element"] * 4 + ["assemble"] * 4 + ["evaluate"] * 2 + ["batch", "pcg"])
    if kind == "element":
        fem, op, nc, top = rng.choice([("P1", "grad", 1, 1500000), ("P2", "grad", 1, 1200000), ("P3", "grad", 1, 90000),
                                       ("P1", "iden", 1, 1500000), ("P2", "iden", 1, 1200000),
                                       ("P1", "grad", 3, 600000), ("P2", "grad", 3, 400000), ("ND0", "iden", 1, 600000),
                                       ("ND0", "curl", 1, 600000), ("RT0", "iden", 1, 600000),
                                       ("RT0", "div", 1, 600000)])
        vector = fem in ("ND0", "RT0")
        if nc == 3:
            tensor, storage = "lame", rng.choice(["tet", "tet", "const"])
        elif op == "div" or (op == "iden" and not vector):
            tensor, storage = "scalar", rng.choice(["tet", "const"])
        else:
            tensor = rng.choice(["scalar", "symmetric", "general"])
            storage = rng.choice(["tet", "tet", "const", "point"]) if tensor == "scalar" else "tet"
        deg = DEGREE[fem]
        if op == "iden":
            order = 2 * deg
        else:
            order = 1 if vector else max(1, 2 * (deg - 1))
        if storage == "point":
            order = {1: 2, 2: 4, 3: 4, 4: rng.choice([5, 6])}[order]
        prec = rng.choice(["fp64", "fp64", "fp32"] + ([] if vector or storage == "point" else ["fp16x3"]))
        if storage == "point":
            top = min(top, 400000)
        c = element("", fem, op, tensor, storage, order, _log(rng, 384, top), nc, prec)
    elif kind == "assemble":
        fem, op, nc, tensor, hi = rng.choice([("P1", "grad", 1, "scalar", 60), ("P1", "grad", 1, "symmetric", 60),
                                              ("P2", "grad", 1, "scalar", 52), ("P2", "grad", 1, "general", 48),
                                              ("P3", "grad", 1, "scalar", 24), ("P1", "grad", 3, "lame", 40),
                                              ("P2", "grad", 3, "lame", 30), ("ND0", "curl", 1, "scalar", 30),
                                              ("ND0", "iden", 1, "symmetric", 30), ("RT0", "iden", 1, "symmetric", 30),
                                              ("RT0", "div", 1, "scalar", 30)])
        c = assemble("", fem, op, tensor, *_box(rng, 4, hi), nc, rng.choice(["fp64", "fp64", "fp32"]),
                     rng.random() < 0.3)
    elif kind == "evaluate":
        fem, nc = rng.choice([("P1", 1), ("P2", 1), ("P3", 1), ("P2", 3), ("ND0", 1), ("RT0", 1)])
        op = rng.choice(["iden", {"ND0": "curl", "RT0": "div"}.get(fem, "grad")])
        nx, ny, nz = _box(rng, 4, {"P1": 50, "P2": 44}.get(fem, 30) if nc == 1 else 30)
        c = dict(kind=kind, fem=fem, op=op, nc=nc, q=rng.choice([1, 3, 4, 5, 8, 14]), nx=nx, ny=ny, nz=nz)
    elif kind == "batch":
        c = dict(kind=kind, meshes=rng.randint(8, 40), lo=rng.randint(3, 5), hi=_log(rng, 8, 22))
    else:
        fem = rng.choice(["P1", "P2"])
        nx, ny, nz = _box(rng, 6, 40 if fem == "P1" else 30)
        c = dict(kind=kind, fem=fem, nx=nx, ny=ny, nz=nz, rtol=rng.choice([1e-6, 1e-8, 1e-10]))
    c.pop("name", None)
    return c


# ---- inputs --------------------------------------------------------------------
PERMS = [(0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)]


def box_mesh(nx, ny, nz, seed):
    """(coords (N, 3) float64, tets (6 nx ny nz, 4) int32): Kuhn cells, interior
    nodes moved by up to a fifth of the spacing."""
    h = 1.0 / max(nx, ny, nz)
    dims = np.array([nx, ny, nz])
    idx = np.stack(np.meshgrid(*[np.arange(d + 1) for d in dims], indexing="ij"), axis=-1).reshape(-1, 3)
    inner = ((idx > 0) & (idx < dims)).all(axis=1)
    coords = idx * h
    move = np.random.default_rng(seed).uniform(-0.2 * h, 0.2 * h, coords.shape)
    coords[inner] += move[inner]
    stride = np.array([(ny + 1) * (nz + 1), nz + 1, 1])
    cell = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), axis=-1).reshape(-1, 3)
    base = cell @ stride
    tets = np.empty((len(base), 6, 4), dtype=np.int32)
    for p, perm in enumerate(PERMS):
        v = base.copy()
        tets[:, p, 0] = v
        for s, axis in enumerate(perm):
            v = v + stride[axis]
            tets[:, p, s + 1] = v
    return coords, tets.reshape(-1, 4)


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 + seed)
    return g


def _uniform(g, lo, hi, *shape):
    return torch.empty(shape, dtype=F64, device=DEV).uniform_(lo, hi, generator=g)


def coefficient(tensor, n, g, dim=3):
    """The tensor of n cells: (values in the library's per-cell layout, full tensor (n, dim, dim) or None)."""
    if tensor == "scalar":
        k = 10.0 ** _uniform(g, -1, 1, n)
        return k[None], None
    if tensor == "lame":  # Young's modulus over three decades
        e, nu = 10.0 ** _uniform(g, 0, 3, n), _uniform(g, 0.2, 0.45, n)
        return torch.stack([e * nu / ((1 + nu) * (1 - 2 * nu)), e / (2 * (1 + nu))]), None
    # R diag(1, 10^a, 10^b) R^T with random rotations (unit quaternions)
    w, x, y, z = torch.nn.functional.normalize(
        torch.empty((4, n), dtype=F64, device=DEV).normal_(generator=g), dim=0)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], dim=1).view(n, 3, 3)
    lam = torch.cat([torch.ones((n, 1), dtype=F64, device=DEV), 10.0 ** _uniform(g, -2, 2, n, 2)], dim=1)
    D = (R * lam[:, None, :]) @ R.transpose(1, 2).contiguous()
    if tensor == "general":  # with a rotational part, as a magnetised medium has
        s = _uniform(g, -0.3, 0.3, n)
        D[:, 0, 1] += s
        D[:, 1, 0] -= s
        return torch.stack([D[:, k, j] for j in range(3) for k in range(3)]).contiguous(), D
    D = 0.5 * (D + D.transpose(1, 2))
    return torch.stack([D[:, i, j] for j in range(3) for i in range(j + 1)]).contiguous(), D


def affine(g):
    """Coefficients of a positive affine function on the unit box: c0 + c . x."""
    return torch.cat([_uniform(g, 1.0, 2.0, 1), _uniform(g, -0.3, 0.3, 3)])


def load_of(case):
    """Constant load: f of scalar spaces, a vector for vector-valued ones."""
    return torch.tensor([0.3, -0.2, -1.0] if case["nc"] == 3 or case["fem"] in ("ND0", "RT0") else [1.0], dtype=F64,
                        device=DEV)


def batch_meshes(case, seed):
    # sizes and orders belong to the case: the same for every seed
    rng = np.random.default_rng(case["meshes"] * 1009 + case["lo"] * 31 + case["hi"])
    sides = np.round(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), case["meshes"]))).astype(int)
    fems = rng.integers(1, 4, case["meshes"])
    return [box_mesh(int(s), int(s), int(s), seed * 977 + i) + ("P%d" % f,) for i, (s, f) in enumerate(zip(sides, fems))]


def element_inputs(case, seed):
    n = case["n"]
    side = 1
    while 6 * side ** 3 < n:
        side += 1
    coords, tets = box_mesh(side, side, side, seed)
    c = torch.from_numpy(coords).to(DEV)
    P = c[torch.from_numpy(tets[:n]).to(DEV).long()]  # (n, 4, 3)
    g = _generator(seed)
    D, full = coefficient(case["tensor"], 1 if case["storage"] == "const" else n, g)
    return P, D, full, affine(g)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "element":
        P, D, _, aff = element_inputs(case, seed)
        n = case["n"]
        xyz = P.reshape(n, 12).t().contiguous()
        if case["storage"] == "point":
            X = af.quadrature_points_batch(case["order"], xyz)
            D = (D[0] * (aff[0] + aff[1] * X[0] + aff[2] * X[1] + aff[3] * X[2])).contiguous()
        elif case["storage"] == "const":
            D = D[:, 0].contiguous()
        op = af.Operator(OP[case["op"]], FEM[case["fem"]], case["nc"])
        nf = NFA[case["fem"]] * case["nc"]
        out = torch.empty((n, nf, nf), dtype=F64 if case["prec"] == "fp64" else torch.float32, device=DEV)
        return dict(case=case, op=op, xyz=xyz, D=D, out=out)
    if kind == "batch":
        meshes = batch_meshes(case, seed)
        B = af.Batch([(c, t, FEM[f]) for c, t, f in meshes])
        kappa = 10.0 ** _uniform(_generator(seed), -1, 1, B.n_tets)
        return dict(case=case, B=B, kappa=kappa, f=torch.ones(1, dtype=F64, device=DEV),
                    val=torch.empty(B.nnz, dtype=F64, device=DEV), rhs=torch.empty(B.ndof, dtype=F64, device=DEV))
    coords, tets = box_mesh(case["nx"], case["ny"], case["nz"], seed)
    g = _generator(seed)
    if kind == "assemble":
        D, _ = coefficient(case["tensor"], len(tets), g)
        F = load_of(case)
        vector = len(F) == 3
        A = af.Assembler(coords, tets, af.Op(OP[case["op"]], FEM[case["fem"]], case["nc"]), order=assembly_order(case),
                         tensor_type=TENSOR[case["tensor"]], tensor_storage=af.COEF_PER_TET, rhs_order=DEGREE[case["fem"]],
                         rhs_tensor_type=af.TENSOR_GENERAL if vector else af.TENSOR_SCALAR,
                         rhs_tensor_storage=af.COEF_CONST, dirichlet=af.DIRICHLET_BOUNDARY)
        return dict(case=case, A=A, D=D, F=F, val=torch.empty(A.nnz, dtype=F64, device=DEV),
                    rhs=torch.empty(A.ndof, dtype=F64, device=DEV))
    if kind == "evaluate":
        A = af.Assembler(coords, tets, af.Op(af.IDEN, FEM[case["fem"]], case["nc"]), order=1,
                         tensor_type=af.TENSOR_NULL, dirichlet=af.DIRICHLET_NONE)
        dim = eval_dim(case)
        return dict(case=case, A=A, u=_uniform(g, -1, 1, A.ndof), xyl=eval_points(case, seed),
                    out=torch.empty((len(tets), case["q"], dim), dtype=F64, device=DEV))
    A = af.Assembler(coords, tets, af.Op(af.GRAD, FEM[case["fem"]]), order=2, dirichlet=af.DIRICHLET_BOUNDARY)
    val, rhs, _ = A.assemble(F=torch.ones(1, dtype=F64, device=DEV))
    rp, ci = A.csr()
    return dict(case=case, A=A, rp=rp, ci=ci, val=val, rhs=rhs, x=torch.zeros(A.ndof, dtype=F64, device=DEV))


def assembly_order(case):
    deg = DEGREE[case["fem"]]
    if case["op"] == "iden":
        return 2 * deg
    return 1 if case["fem"] in ("ND0", "RT0") else max(1, 2 * (deg - 1))


def eval_dim(case):
    if case["fem"] in ("ND0", "RT0"):
        return 1 if case["op"] == "div" else 3
    return case["nc"] * (3 if case["op"] == "grad" else 1)


def eval_points(case, seed):
    return np.random.default_rng(seed + 17).dirichlet(np.ones(4), case["q"])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "element":
        return af.fem3dtet_batch(state["op"], state["op"], TENSOR[case["tensor"]], STORAGE[case["storage"]], state["D"],
                                 case["order"], state["xyz"], PREC[case["prec"]], out=state["out"])
    if kind == "assemble":
        val, rhs, _ = state["A"].assemble(D=state["D"], F=state["F"], precision=PREC[case["prec"]], val=state["val"],
                                          rhs=state["rhs"], status=case["status"])
        return val, rhs
    if kind == "evaluate":
        return state["A"].evaluate(state["u"], state["xyl"], op=OP[case["op"]], out=state["out"])
    if kind == "batch":
        val, rhs, _ = state["B"].run(state["kappa"], state["f"], state["val"], state["rhs"], status=False)
        return val, rhs
    state["x"].zero_()
    af.pcg_jacobi(state["A"].ndof, state["rp"], state["ci"], state["val"], state["rhs"], state["x"], rtol=case["rtol"])
    return state["x"]


# ---- work ----------------------------------------------------------------------
def work(case):
    """Each input read once, each output written once; the products of the
    factored element contraction (six distinct geometry values where symmetric)."""
    kind = case["kind"]
    coef = {"scalar": 1, "symmetric": 6, "general": 9, "lame": 2}
    if kind == "element":
        n, nf, nc = case["n"], NFA[case["fem"]], case["nc"]
        q = {1: 1, 2: 4, 3: 8, 4: 14, 5: 14, 6: 24}[case["order"]] if case["storage"] == "point" else 1
        D = 0 if case["storage"] == "const" else 8 * coef[case["tensor"]] * q
        E = nf * nf * nc * nc
        size = 8 if case["prec"] == "fp64" else 4
        kk = 1 if case["op"] == "div" or (case["op"] == "iden" and case["fem"][0] == "P") else \
            (9 if case["tensor"] == "general" or nc == 3 else 6)
        pairs = E if case["tensor"] == "general" else E // 2 + nf * nc // 2
        return {"bytes": n * (96 + D + E * size), "flops": n * (2 * kk * q * pairs + 120)}
    if kind == "batch":
        b = f = 0
        for c, t, fem in batch_meshes(case, 1):
            n, nf, cells = len(t), NFA[fem], len(t) // 6
            b += 24 * len(c) + n * (16 + 8) + 8 * cells * (COUPLINGS[fem] + DOFS[fem])
            f += n * (6 * nf * (nf + 1) + 120)
        return {"bytes": b, "flops": f}
    cells = case["nx"] * case["ny"] * case["nz"]
    n = 6 * cells
    nc = case.get("nc", 1)
    ndof, nnz = DOFS[case["fem"]] * cells * nc, COUPLINGS[case["fem"]] * cells * nc * nc
    nf = NFA[case["fem"]] * nc
    if kind == "assemble":
        kk = 1 if case["op"] == "div" else (9 if case["tensor"] in ("general", "lame") else 6)
        return {"bytes": 24 * cells + n * (16 + 8 * coef[case["tensor"]]) + 8 * (nnz + ndof),
                "flops": n * (kk * nf * (nf + 1) + 120)}
    if kind == "evaluate":
        d = eval_dim(case)
        return {"bytes": 24 * cells + n * (16 + 4 * nf) + 8 * ndof + 8 * n * case["q"] * d,
                "flops": n * case["q"] * 2 * nf * d}
    its = 5 * max(case["nx"], case["ny"], case["nz"]) * DEGREE[case["fem"]]  # about the iterations of such a solve
    return {"bytes": 12 * nnz + 24 * ndof, "flops": its * (2 * nnz + 12 * ndof)}


# ---- float64 references ---------------------------------------------------------
EDGES = [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)]
FACES = [(0, 1, 2), (1, 2, 3), (2, 3, 0), (3, 0, 1)]


def _t(a):
    return torch.as_tensor(a, dtype=F64, device=DEV)


def gauss_tet(m):
    """Collapsed Gauss-Legendre rule, exact to degree 2m - 3: barycentric points
    (m^3, 4) and weights that sum to 1."""
    x, w = np.polynomial.legendre.leggauss(m)
    x, w = (x + 1) / 2, w / 2
    u, v, s = np.meshgrid(x, x, x, indexing="ij")
    W = w[:, None, None] * w[None, :, None] * w[None, None, :] * (1 - u) ** 2 * (1 - v) * 6
    a, b, c = u, (1 - u) * v, (1 - u) * (1 - v) * s
    L = np.stack([1 - a - b - c, a, b, c], axis=-1).reshape(-1, 4)
    return L, W.ravel()


def reference_basis(fem, op, L):
    """Reference values (points, nf, d): basis values, gradients, or the reference fields of ND0 / RT0."""
    g = np.array([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    q = len(L)
    l = [L[:, i] for i in range(4)]
    if fem == "ND0":
        if op == "iden":
            return np.stack([l[a][:, None] * g[b] - l[b][:, None] * g[a] for a, b in EDGES], axis=1)
        return np.broadcast_to(np.stack([2 * np.cross(g[a], g[b]) for a, b in EDGES]), (q, 6, 3)).copy()
    if fem == "RT0":
        if op == "iden":
            v = np.array([[0.0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
            return np.stack([L[:, 1:] - v[(i + 3) % 4] for i in range(4)], axis=1)
        return np.full((q, 4, 1), 3.0)
    # Lagrange spaces: value and derivatives by the barycentric coordinates
    val, dl = [], []

    def add(f, d):
        val.append(f)
        dl.append(np.stack([d.get(k, np.zeros(q)) for k in range(4)], axis=-1))

    one = np.ones(q)
    if fem == "P0":
        add(one, {})
    elif fem == "P1":
        for i in range(4):
            add(l[i], {i: one})
    elif fem == "P2":
        for i in range(4):
            add(l[i] * (2 * l[i] - 1), {i: 4 * l[i] - 1})
        for a, b in EDGES:
            add(4 * l[a] * l[b], {a: 4 * l[b], b: 4 * l[a]})
    else:
        for i in range(4):
            add(0.5 * l[i] * (3 * l[i] - 1) * (3 * l[i] - 2), {i: 0.5 * (27 * l[i] ** 2 - 18 * l[i] + 2)})
        for a, b in EDGES:
            add(4.5 * l[a] * l[b] * (3 * l[a] - 1), {a: 4.5 * l[b] * (6 * l[a] - 1), b: 4.5 * l[a] * (3 * l[a] - 1)})
            add(4.5 * l[a] * l[b] * (3 * l[b] - 1), {b: 4.5 * l[a] * (6 * l[b] - 1), a: 4.5 * l[b] * (3 * l[b] - 1)})
        for a, b, c in FACES:
            add(27 * l[a] * l[b] * l[c], {a: 27 * l[b] * l[c], b: 27 * l[a] * l[c], c: 27 * l[a] * l[b]})
    if op == "iden":
        return np.stack(val, axis=1)[:, :, None]
    return np.einsum("qik,ka->qia", np.stack(dl, axis=1), g)


def geometry(P):
    """J (n, 3, 3), its inverse and determinant."""
    J = (P[:, 1:] - P[:, :1]).transpose(1, 2).contiguous()
    a, b, c = J[:, :, 0], J[:, :, 1], J[:, :, 2]
    bc, ca, ab = torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)
    det = (a * bc).sum(1)
    return J, torch.stack([bc, ca, ab], dim=1) / det[:, None, None], det


def maps(fem, op, P):
    """The map T (n, dim, d) from reference to physical components (None: 1) and
    the factor per basis function (n, nf) (None: 1)."""
    J, Ji, det = geometry(P)
    T = s = None
    if fem == "ND0":
        length = torch.stack([(P[:, b] - P[:, a]).norm(dim=1) for a, b in EDGES], dim=1)
        T, s = (Ji.transpose(1, 2), length) if op == "iden" else (J, length / det[:, None])
    elif fem == "RT0":
        area = torch.stack([0.5 * torch.linalg.cross(P[:, b] - P[:, a], P[:, c] - P[:, a]).norm(dim=1)
                            for a, b, c in FACES], dim=1)
        T, s = (J if op == "iden" else None), area / (0.5 * det.abs()[:, None])
    elif op == "grad":
        T = Ji.transpose(1, 2)
    return T, s, det.abs() / 6


def element_matrices(case, P, D, full, aff=None):
    """(n, nf_test, nf_trial) of the case's form."""
    fem, op, nc, n = case["fem"], case["op"], case["nc"], len(P)
    T, s, vol = maps(fem, op, P)
    L, w = gauss_tet(DEGREE[fem] + 3)
    B = _t(reference_basis(fem, op, L))
    L, w = _t(L), _t(w)
    nf, d = B.shape[1], B.shape[2]
    if nc == 3:  # isotropic elasticity, component blocks
        R = torch.einsum("q,qib,qja->baij", w, B, B).reshape(9, nf * nf)
        lam, mu = [vol * v for v in D]
        A = torch.empty((n, 3, nf, 3, nf), dtype=F64, device=P.device)
        G = T.transpose(1, 2) @ T.contiguous()
        for cb in range(3):
            for ca in range(3):
                K = lam[:, None, None] * T[:, cb, :, None] * T[:, ca, None, :] \
                    + mu[:, None, None] * T[:, ca, :, None] * T[:, cb, None, :]
                if cb == ca:
                    K = K + mu[:, None, None] * G
                A[:, cb, :, ca, :] = (K.reshape(n, 9) @ R).view(n, nf, nf)
        return A.view(n, 3 * nf, 3 * nf)
    if full is not None:
        K = T.transpose(1, 2) @ full @ T.contiguous()
    elif T is not None:
        K = T.transpose(1, 2) @ T.contiguous() * D[0][:, None, None]
    else:
        K = D[0][:, None, None] * torch.ones((len(P), 1, 1), dtype=F64, device=P.device)
    K = K * vol[:, None, None]
    if aff is None:
        A = K.reshape(n, d * d) @ torch.einsum("q,qib,qja->baij", w, B, B).reshape(d * d, nf * nf)
    else:
        X = torch.einsum("qv,nvc->nqc", L, P)
        k = (aff[0] + X @ aff[1:]) * w
        A = torch.zeros((n, nf * nf), dtype=F64, device=P.device)
        for i in range(len(w)):
            Ri = torch.einsum("ib,ja->baij", B[i], B[i]).reshape(d * d, nf * nf)
            A.addmm_(K.reshape(n, d * d) * k[:, i, None], Ri)
    A = A.view(n, nf, nf)
    return A if s is None else A * s[:, :, None] * s[:, None, :]


def load_vectors(case, P, f):
    fem, nc = case["fem"], case["nc"]
    T, s, vol = maps(fem, "iden", P)
    L, w = gauss_tet(DEGREE[fem] + 2)
    m = torch.einsum("q,qid->id", _t(w), _t(reference_basis(fem, "iden", L)))  # mean of the reference fields
    if T is not None:
        return torch.einsum("nkd,id,k,n->ni", T, m, f, vol) * s
    return (vol[:, None, None] * f[None, :, None] * m[None, None, :, 0]).reshape(len(P), -1)


def first_appearance(key):
    """Ids of the distinct keys in the order in which they first appear, and their counts."""
    u, inv, cnt = torch.unique(key, return_inverse=True, return_counts=True)
    first = torch.full((len(u),), len(key), dtype=torch.int64, device=key.device)
    first.scatter_reduce_(0, inv, torch.arange(len(key), device=key.device), "amin")
    order = torch.argsort(first)
    rank = torch.empty_like(order)
    rank[order] = torch.arange(len(order), device=key.device)
    return rank[inv], cnt[order], len(u)


def numbering(fem, nc, coords, tets):
    """Cells with positive orientation, DOF ids (n, nf), orientation signs, Dirichlet flags, DOF count:
    nodes, edges, faces, each by first appearance, component after component."""
    c, t = torch.from_numpy(coords).to(DEV), torch.from_numpy(tets).to(DEV).long()
    P = c[t]
    m = P[:, :3] - P[:, 3:]
    flip = (m[:, 0] * torch.linalg.cross(m[:, 1], m[:, 2])).sum(1) < 0
    t = torch.where(flip[:, None], t[:, [0, 1, 3, 2]], t)
    n, nn = len(t), len(c)
    e = torch.stack([t[:, [a, b]] for a, b in EDGES], dim=1)
    ek = (e.min(2).values * nn + e.max(2).values).reshape(-1)
    f = torch.stack([t[:, list(v)] for v in FACES], dim=1).sort(dim=2).values
    fk = ((f[:, :, 0] * nn + f[:, :, 1]) * nn + f[:, :, 2]).reshape(-1)
    eid, _, ne = first_appearance(ek)
    fid, fcount, nfaces = first_appearance(fk)
    eid, fid = eid.view(n, 6), fid.view(n, 4)
    outer = fcount[fid] == 1  # boundary faces: their closure is Dirichlet
    node = torch.zeros(nn, dtype=torch.bool, device=DEV)
    edge = torch.zeros(ne, dtype=torch.bool, device=DEV)
    face = fcount == 1
    for k, v in enumerate(FACES):
        for i in v:
            node[t[outer[:, k], i]] = True
        for j, (a, b) in enumerate(EDGES):
            if a in v and b in v:
                edge[eid[outer[:, k], j]] = True
    up = e[:, :, 0] < e[:, :, 1]
    sign = None
    if fem == "P1":
        dofs, dirichlet = t, node
    elif fem == "P2":
        dofs, dirichlet = torch.cat([t, nn + eid], dim=1), torch.cat([node, edge])
    elif fem == "P3":
        near, far = nn + 2 * eid + (~up).long(), nn + 2 * eid + up.long()
        dofs = torch.cat([t, torch.stack([near, far], dim=2).view(n, 12), nn + 2 * ne + fid], dim=1)
        dirichlet = torch.cat([node, edge.repeat_interleave(2), face])
    elif fem == "ND0":
        dofs, dirichlet, sign = eid, edge, torch.where(up, 1.0, -1.0).to(F64)
    else:
        v = torch.stack([t[:, list(i)] for i in FACES], dim=1)
        odd = (v[:, :, 0] > v[:, :, 1]).long() + (v[:, :, 0] > v[:, :, 2]).long() + (v[:, :, 1] > v[:, :, 2]).long()
        odd = (odd + torch.arange(4, device=DEV)) % 2
        dofs, dirichlet, sign = fid, face, 1.0 - 2.0 * odd.to(F64)
    ns = len(dirichlet)
    return P, c[t], torch.cat([dofs + k * ns for k in range(nc)], dim=1), sign, dirichlet.repeat(nc), ns * nc


def scatter(A, F, dofs, sign, dirichlet, ndof):
    """CSR values (rows, then columns, ascending) and right-hand side with homogeneous Dirichlet rows and columns."""
    if sign is not None:
        A = A * sign[:, :, None] * sign[:, None, :]
        F = F * sign
    row, col = dofs[:, :, None].expand_as(A), dofs[:, None, :].expand_as(A)
    fixed = dirichlet[dofs]
    drop = fixed[:, :, None] | fixed[:, None, :]
    diag = row == col
    A = torch.where(drop, diag.to(F64), A)
    keep = (diag | ~drop).reshape(-1)
    key = (row * ndof + col).reshape(-1)[keep]
    a = A.reshape(-1)[keep]
    del row, col, drop, diag, A, keep
    key, at = key.sort()
    a = a[at]
    del at
    _, inv = torch.unique_consecutive(key, return_inverse=True)
    val = torch.zeros(int(inv[-1]) + 1, dtype=F64, device=a.device).index_add_(0, inv, a)
    F = torch.where(fixed, torch.zeros_like(F), F)
    return val, torch.zeros(ndof, dtype=F64, device=a.device).index_add_(0, dofs.reshape(-1), F.reshape(-1))


def system(fem, nc, form, coords, tets, D, full, f):
    """Assembled (values, right-hand side) of a form on a mesh."""
    P, Pr, dofs, sign, dirichlet, ndof = numbering(fem, nc, coords, tets)
    A = element_matrices(form, Pr, D, full)
    return scatter(A, load_vectors(form, Pr, f), dofs, sign, dirichlet, ndof) + (dofs, dirichlet, ndof)


def exact(case, seed):
    kind = case["kind"]
    if kind == "element":
        P, D, full, aff = element_inputs(case, seed)
        aff = aff if case["storage"] == "point" else None
        out = []
        for i in range(0, case["n"], 1 << 17):
            Dc = D if case["storage"] == "const" else D[:, i:i + (1 << 17)]
            fc = full if full is None or case["storage"] == "const" else full[i:i + (1 << 17)]
            # trial DOFs outermost: the column-major matrices of the library
            out.append(element_matrices(case, P[i:i + (1 << 17)], Dc, fc, aff).transpose(1, 2).contiguous())
        return torch.cat(out)
    if kind == "batch":
        kappa, at, vals, rhss = None, 0, [], []
        meshes = batch_meshes(case, seed)
        kappa = 10.0 ** _uniform(_generator(seed), -1, 1, sum(len(t) for _, t, _ in meshes))
        for c, t, fem in meshes:
            form = dict(fem=fem, op="grad", nc=1)
            v, r = system(fem, 1, form, c, t, kappa[None, at:at + len(t)], None, _t([1.0]))[:2]
            at += len(t)
            vals.append(v)
            rhss.append(r)
        return torch.cat(vals), torch.cat(rhss)
    coords, tets = box_mesh(case["nx"], case["ny"], case["nz"], seed)
    g = _generator(seed)
    if kind == "assemble":
        D, full = coefficient(case["tensor"], len(tets), g)
        return system(case["fem"], case["nc"], case, coords, tets, D, full, load_of(case))[:2]
    if kind == "evaluate":
        _, P, dofs, sign, _, ndof = numbering(case["fem"], case["nc"], coords, tets)
        u = _uniform(g, -1, 1, ndof)[dofs]
        u = u if sign is None else u * sign
        T, s, _ = maps(case["fem"], case["op"], P)
        u = u if s is None else u * s
        B = _t(reference_basis(case["fem"], case["op"], eval_points(case, seed)))
        v = torch.einsum("qid,nci->nqcd", B, u.view(len(P), case["nc"], -1))
        v = v if T is None else torch.einsum("nkd,nqcd->nqck", T, v)
        return v.reshape(len(P), case["q"], -1)
    if (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1) * DEGREE[case["fem"]] ** 3 > 8000:
        return None  # the dense solve would take too long
    form = dict(fem=case["fem"], op="grad", nc=1)
    one = torch.ones((1, len(tets)), dtype=F64, device=DEV)
    P, Pr, dofs, _, dirichlet, ndof = numbering(case["fem"], 1, coords, tets)
    A = element_matrices(form, Pr, one, None)
    f = load_vectors(form, Pr, _t([1.0]))
    M = torch.zeros(ndof * ndof, dtype=F64, device=DEV)
    M.index_add_(0, (dofs[:, :, None] * ndof + dofs[:, None, :]).reshape(-1), A.reshape(-1))
    b = torch.zeros(ndof, dtype=F64, device=DEV).index_add_(0, dofs.reshape(-1), f.reshape(-1))
    inner = torch.nonzero(~dirichlet)[:, 0]
    x = torch.zeros(ndof, dtype=F64, device=DEV)
    x[inner] = torch.linalg.solve(M.view(ndof, ndof)[inner][:, inner], b[inner])
    return x
