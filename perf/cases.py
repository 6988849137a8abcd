"""The work a program has this library do, as cases that can be timed and compared.

Kinds of case (``case["kind"]``):

  product   one operator-vector product on device vectors, the call every iteration of a solver makes:
            FP64, real or complex kernels
  products  several right-hand sides at once, host arrays in and out
  solve     one GMRES solve A x = b from x0 = 1: plain FP64, or FP32 inner solves inside FP64 refinement
  batch     independent systems of different sizes solved together, several right-hand sides each
  assemble  a new point set: tree, skeletons, operators, and the first product

An assembled operator is what a program keeps between its products and solves, so ``prepare`` assembles
an operator once per geometry and makes new vectors for every seed.  An ``assemble`` case has new points
for every seed and builds its operator inside ``run``.
"""
import collections
import math

import numpy as np
import torch

import h2weak_amd as h2w

IE, RBF, HELMHOLTZ, HANKEL = h2w.CHOICE_IE, h2w.CHOICE_RBF, h2w.CHOICE_HELMHOLTZ, h2w.CHOICE_HANKEL
GMRES_TOL = {"fp64": 1e-12, "refined": 1e-10}


def listed():
    return [
        # a small 1D system on a grid: the whole product is a chain of small launches
        dict(name="product_1d_small", kind="product", dim=1, N=2048, n_max=64, tol=12, choice=RBF, variant=h2w.NESTED,
             points="grid"),
        # the 1D integral equation on 250000 random points: a deep tree of low ranks
        dict(name="product_1d", kind="product", dim=1, N=250000, n_max=100, tol=12, choice=IE, variant=h2w.NESTED,
             points="uniform"),
        # the 2D integral equation on the 400 x 400 grid, semi-nested: per-pair column factors
        dict(name="product_2d_semi", kind="product", dim=2, N=160000, n_max=64, tol=10, choice=IE,
             variant=h2w.SEMI_NESTED, points="grid"),
        # scattered 3D points: leaves of every size between a few and over a hundred points
        dict(name="product_3d", kind="product", dim=3, N=20011, n_max=64, tol=8, choice=RBF, variant=h2w.NESTED,
             points="uniform"),
        # the 3D grid 64^3: tens of gigabytes of operator blocks streamed per product
        dict(name="product_3d_large", kind="product", dim=3, N=262144, n_max=64, tol=8, choice=RBF, variant=h2w.NESTED,
             points="grid"),
        # the 3D Helmholtz kernel: complex blocks and vectors
        dict(name="product_helmholtz", kind="product", dim=3, N=32768, n_max=64, tol=8, choice=HELMHOLTZ,
             variant=h2w.NESTED, points="grid"),
        # 16 right-hand sides against one operator
        dict(name="products_16", kind="products", dim=3, N=32768, n_max=64, tol=10, choice=RBF, variant=h2w.NESTED,
             points="grid", nrhs=16),
        # the 2D run of the published transcripts: FP64 GMRES on the 300 x 300 grid
        dict(name="solve_2d", kind="solve", dim=2, N=90000, n_max=100, tol=12, choice=RBF, variant=h2w.NESTED,
             points="grid", mode="fp64", deflation=0),
        # the refined solve of 3D systems with its deflation space
        dict(name="solve_3d_refined", kind="solve", dim=3, N=32768, n_max=64, tol=10, choice=RBF, variant=h2w.NESTED,
             points="grid", mode="refined", deflation=48),
        # six systems of 4096 to 16384 scattered points, 16 right-hand sides each
        dict(name="batch_solve", kind="batch", systems=6, N_min=4096, N_max=16384, n_max=64, tol=8, nrhs=16),
        # setting up a 2D system on new points
        dict(name="assemble_2d", kind="assemble", dim=2, N=40000, n_max=64, tol=10, choice=IE, variant=h2w.NESTED),
        # setting up a 3D system on new points
        dict(name="assemble_3d", kind="assemble", dim=3, N=20011, n_max=64, tol=8, choice=RBF, variant=h2w.NESTED),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _on_grid(dim, N):
    return N if dim == 1 else max(2, int(round(N ** (1.0 / dim)))) ** dim


def _geometry(rng, largest):
    """A system: dimension, size (up to largest[dim]), leaf size, kernel, format, points."""
    dim = rng.choice([1, 2, 3, 3])
    N = _log_int(rng, {1: 1000, 2: 1000, 3: 2000}[dim], largest[dim])
    points = rng.choice(["grid", "uniform"])
    if points == "grid":
        N = _on_grid(dim, N)
    tol = rng.choice({1: [10, 12], 2: [8, 10, 12], 3: [6, 8, 10]}[dim])
    if dim == 3 and N > 35000:
        tol = min(tol, 8)
    variant = rng.choice([h2w.NESTED, h2w.NESTED, h2w.SEMI_NESTED])
    if dim == 3 and N > 35000:
        variant = h2w.NESTED
    n_max = {1: rng.randint(40, 128), 2: rng.randint(30, 100), 3: rng.randint(40, 125)}[dim]
    return dict(dim=dim, N=N, n_max=n_max, tol=tol, choice=rng.choice([IE, RBF]), variant=variant, points=points)


def draw(rng):
    kind = rng.choice(["product", "product", "product", "complex", "products", "solve", "solve", "batch", "assemble"])
    if kind == "product":
        return dict(kind="product", **_geometry(rng, {1: 250000, 2: 160000, 3: 200000}))
    if kind == "complex":
        choice = rng.choice([HELMHOLTZ, HANKEL])
        dim = 3 if choice == HELMHOLTZ else 2
        points = rng.choice(["grid", "uniform"])
        N = _log_int(rng, 2500, 32768 if dim == 3 else 65536)
        if points == "grid":
            N = _on_grid(dim, N)
        return dict(kind="product", dim=dim, N=N, n_max=rng.randint(40, 100), tol=rng.choice([6, 8]), choice=choice,
                    variant=h2w.NESTED, points=points)
    if kind == "products":
        return dict(kind="products", nrhs=rng.randint(2, 24), **_geometry(rng, {1: 60000, 2: 60000, 3: 32768}))
    if kind == "solve":
        c = _geometry(rng, {1: 60000, 2: 90000, 3: 60000})
        if c["dim"] == 1:
            c["choice"] = IE  # (the 1D RBF matrix is near-singular: its solutions are not determined to 1e-8)
        mode = rng.choice(["fp64", "refined"]) if c["dim"] == 3 else "fp64"
        if mode == "refined":
            c["tol"] = max(c["tol"], 8)  # (the inner operator is truncated to 1e-6)
        return dict(kind="solve", mode=mode, deflation=rng.choice([0, 48]) if mode == "refined" else 0, **c)
    if kind == "batch":
        lo = _log_int(rng, 2000, 6000)
        return dict(kind="batch", systems=rng.randint(2, 6), N_min=lo, N_max=_log_int(rng, lo, 16384),
                    n_max=rng.randint(40, 100), tol=rng.choice([6, 8]), nrhs=rng.randint(2, 16))
    c = _geometry(rng, {1: 100000, 2: 40000, 3: 25000})
    if c["dim"] == 3 and c["N"] > 10000:
        c["tol"] = min(c["tol"], 8)
    del c["points"]
    return dict(kind="assemble", **c)


# ---------------------------------------------------------------- geometry and operators

def _points(c, seed):
    """dim x N coordinates of a scattered point set, or of the reference's grid, on the host."""
    dim, N = c["dim"], c["N"]
    if c.get("points") == "grid":
        n = int(round(N ** (1.0 / dim)))
        nd = -1.0 + 2.0 * (np.arange(n) + 1.0) / (n + 1.0)
        if dim == 1:
            return nd[None, :]
        if dim == 2:
            return np.stack([np.tile(nd, n), np.repeat(nd, n)])
        J, K, I = np.meshgrid(nd, nd, nd, indexing="ij")
        return np.stack([K.ravel(), J.ravel(), I.ravel()])
    return np.random.default_rng(seed).uniform(-1.0, 1.0, (dim, N))


def _initialisation(c, seed):
    P = None if c.get("points") == "grid" else _points(c, seed)
    return h2w.Initialisation(c["dim"], c["N"], c["n_max"], 1.0, c["tol"], c["choice"], c["variant"], points=P)


def _systems(c):
    """The systems of a batch: sizes spread over [N_min, N_max] by their logarithm."""
    S = c["systems"]
    for q in range(S):
        N = int(round(c["N_min"] * (c["N_max"] / c["N_min"]) ** (q / max(1, S - 1))))
        yield dict(dim=3, N=N, n_max=c["n_max"], tol=c["tol"], choice=RBF, variant=h2w.NESTED, points="uniform")


_kept = collections.OrderedDict()  # assembled operators by geometry, the least recently used first


def _operator(c):
    """The assembled operator (or batch of them) of a case; the oldest ones go when the card fills up."""
    key = tuple(sorted((k, v) for k, v in c.items() if k not in ("name", "kind", "nrhs", "mode")))
    if key in _kept:
        _kept.move_to_end(key)
        return _kept[key]
    if torch.cuda.is_available():
        while _kept:
            free, total = torch.cuda.mem_get_info()
            if free > 0.5 * total:
                break
            _kept.popitem(last=False)
    if "systems" in c:
        gs = [_initialisation(s, 100 + q) for q, s in enumerate(_systems(c))]
        h2w.assemble_many(gs, 4)
        op = h2w.Batch(gs)
    else:
        op = _initialisation(c, 1)
        op.tree_initialisation()
        if c.get("deflation"):
            op.set_deflation(128, c["deflation"])
    _kept[key] = op
    return op


# ---------------------------------------------------------------- inputs and passes

def _uniform(seed, *shape, cplx=False):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    x = torch.rand(*shape, 2 if cplx else 1, generator=g, dtype=torch.float64, device="cuda") * 2.0 - 1.0
    return torch.view_as_complex(x) if cplx else x[..., 0].contiguous()


def _rhs(c, P, seed, n=1):
    """n vectors x of a seed and the dense products A x, both (n, N)."""
    X = _uniform(seed, n, c["N"])
    return X, _dense(c, P, X)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "assemble":
        P = np.random.default_rng(seed).uniform(-1.0, 1.0, (case["dim"], case["N"]))
        return dict(case=case, points=P, x=np.random.default_rng(seed + 1).uniform(-1.0, 1.0, case["N"]))
    op = _operator(case)
    if kind == "product":
        x = _uniform(seed, case["N"], cplx=op.cplx)
        return dict(case=case, op=op, x=x, y=torch.empty_like(x))
    if kind == "products":
        return dict(case=case, op=op, X=_uniform(seed, case["nrhs"], case["N"]).cpu().numpy())
    if kind == "solve":
        return dict(case=case, op=op, b=_rhs(case, _points(case, 1), seed)[1][0].cpu().numpy())
    B = [_rhs(s, _points(s, 100 + q), seed + 1000 * q, case["nrhs"])[1].cpu().numpy()
         for q, s in enumerate(_systems(case))]
    return dict(case=case, op=op, B=B)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "product":
        return state["op"].mat_vec_prod(state["x"], state["y"])
    if kind == "products":
        return state["op"].matvec_multi(state["X"])
    if kind == "solve":
        mode = h2w.GMRES_FP64 if case["mode"] == "fp64" else h2w.GMRES_FP32_INNER_IR
        return state["op"].gmres(state["b"], None, 500, GMRES_TOL[case["mode"]], mode)[0]
    if kind == "batch":
        return state["op"].gmres(state["B"], None, 300, 10.0 ** -case["tol"], h2w.GMRES_FP64)[0]
    A = h2w.Initialisation(case["dim"], case["N"], case["n_max"], 1.0, case["tol"], case["choice"], case["variant"],
                           points=state["points"])
    A.tree_initialisation()
    return A.mat_vec_prod(state["x"])


# ---------------------------------------------------------------- what a pass cannot do without

def _products_of(case, op):
    """FP64 and FP32 products of a solve's columns (one set of columns for a batch's lockstep)."""
    if case["kind"] == "solve":
        mode = h2w.GMRES_FP64 if case["mode"] == "fp64" else h2w.GMRES_FP32_INNER_IR
        st = op.gmres(prepare(case, 0)["b"], None, 500, GMRES_TOL[case["mode"]], mode)[1]
        return st["matvecs_fp64"], st["matvecs_fp32"]
    st = op.gmres(prepare(case, 0)["B"], None, 300, 10.0 ** -case["tol"], h2w.GMRES_FP64)[1]
    return max(c["matvecs_fp64"] for row in st for c in row), 0


def work(case):
    """The kernels are symmetric: of the operator elements that the reference's storage formula counts
    (both directions of every block), half have to be read, or written by an assembly, and a multiplication
    and an addition per counted element and right-hand side made.  Vectors are read and written once.  Kernel
    entries of an assembly are taken as 12 operations."""
    if case["kind"] == "assemble":
        A = _initialisation(case, 1)
        A.tree_initialisation()
        half = 0.5 * A.memory
        return {"bytes": 8 * half + 8 * (case["dim"] + 2) * case["N"], "flops": 12 * half}
    op = _operator(case)
    elems = sum(s.memory for s in op.systems) if case["kind"] == "batch" else op.memory
    N = sum(s.N for s in op.systems) if case["kind"] == "batch" else case["N"]
    if case["kind"] in ("product", "products"):
        n = case.get("nrhs", 1)
        if op.cplx:
            return {"bytes": 16 * 0.5 * elems + 32 * N, "flops": 8 * elems}
        return {"bytes": 8 * 0.5 * elems + 16 * n * N, "flops": 2 * elems * n}
    n64, n32 = _products_of(case, op)
    n = case.get("nrhs", 1)
    return {"bytes": (8 * n64 + 4 * n32) * 0.5 * elems + 16 * n * N, "flops": 2 * elems * n * (n64 + n32)}


# ---------------------------------------------------------------- the same in plain 64-bit torch

def _diagonal(c):
    """The matrix's diagonal value (one value for all points)."""
    dim, choice, N = c["dim"], c["choice"], c["N"]
    if choice == RBF:
        return {1: math.sqrt(2.0 * N), 2: 1.0, 3: math.sqrt(N)}[dim]
    if choice == HELMHOLTZ:
        return 500.0 * math.sqrt(N)
    # 1 + the integral of the kernel over the cell of size h around the point, 16-point Gauss-Legendre
    # on one orthant, over h^dim
    t, w = np.polynomial.legendre.leggauss(16)
    h = N ** (-1.0 / dim)
    t, w = 0.25 * h * (t + 1.0), 0.25 * h * w
    T = np.meshgrid(*[t] * dim, indexing="ij")
    W = np.ones_like(T[0])
    for q in range(dim):
        W = W * w.reshape([-1 if q == a else 1 for a in range(dim)])
    R2 = torch.from_numpy(sum(v * v for v in T))
    K = (torch.from_numpy(W) * _kernel(dim, choice, R2)).sum().item() * 2.0 ** dim
    return ((1.0 + 15.0 * math.log(N) if choice == HANKEL else 1.0) + K) / h ** dim


def _kernel(dim, choice, R2):
    """Entries of the matrix off its diagonal, from the squared distances (R2 is overwritten)."""
    a = 1e-4
    if choice == HELMHOLTZ:
        R = R2.sqrt_()
        return torch.complex(R.cos(), R.sin()).div_(4.0 * math.pi)
    if choice == HANKEL:
        R = R2.sqrt_()
        return torch.complex(torch.special.bessel_y0(R).div_(-4.0), torch.special.bessel_j0(R).div_(4.0))
    if choice == IE:
        if dim == 1:
            return R2.log_().mul_(0.5)
        if dim == 2:
            return R2.log_().mul_(-0.25 / math.pi)
        return R2.rsqrt_().div_(4.0 * math.pi)
    if dim < 3:
        R = R2.sqrt_()
        return torch.where(R < a, R / a, a / R)
    near = R2 < a * a
    few = bool(near.any())
    R = R2[near].sqrt() if few else None
    K = R2.log_().mul_(0.5 / math.log(a))
    if few:
        K[near] = (R * R.log() - 1.0) / (a * math.log(a) - 1.0)
    return K


def _dense(c, P, X):
    """A X^T of the dense matrix, row block by row block: X (n, N) on the GPU, the result (n, N)."""
    N = c["N"]
    P = torch.from_numpy(np.ascontiguousarray(P)).cuda()
    d = _diagonal(c)
    Y = torch.empty_like(X)
    step = max(1, (1 << 26) // N)
    for i in range(0, N, step):
        j = min(N, i + step)
        R2 = (P[0, i:j, None] - P[0][None, :]).square_()
        for q in range(1, P.shape[0]):
            R2 += (P[q, i:j, None] - P[q][None, :]).square_()
        R2[torch.arange(j - i), torch.arange(i, j)] = 1.0
        K = _kernel(c["dim"], c["choice"], R2)
        K[torch.arange(j - i), torch.arange(i, j)] = d
        Y[:, i:j] = (K @ X.T.contiguous()).T
    return Y


def exact(case, seed):
    kind = case["kind"]
    if kind == "assemble":
        s = prepare(case, seed)
        return _dense(case, s["points"], torch.from_numpy(s["x"]).cuda()[None, :])[0]
    if kind == "product":
        x = _uniform(seed, case["N"], cplx=case["choice"] in (HELMHOLTZ, HANKEL))
        return _dense(case, _points(case, 1), x[None, :])[0]
    if kind == "products":
        return _dense(case, _points(case, 1), _uniform(seed, case["nrhs"], case["N"]))
    if kind == "solve":
        return _uniform(seed, 1, case["N"])[0]
    return [_uniform(seed + 1000 * q, case["nrhs"], s["N"]) for q, s in enumerate(_systems(case))]
