"""The work that users of this package have it do, as timed cases.

Every case goes through the public entry points (LdltSymbolic / LdltSolver /
MixedLdltSolver, the Krylov consumers, LuSymbolic / LuSolver). The analysis is
done once per pattern and is in hand before a pass, as in a program that
factors many value sets of one pattern (Newton and time steps, frequency
sweeps, interior-point iterations). The kinds of pass:

* step    new values and right-hand sides in device memory: refactor, then the
          refinement ladder to the case's backward error
* host    the same from host buffers, as the reference's API hands them over
* solve   one more solve with a factor in hand (time stepping, adjoints)
* batch   many independent small systems under one plan, refactor and refine
* krylov  block GMRES preconditioned by a factor of a nearby matrix
* lu      the unsymmetric LU: refactor and solve_refined, host buffers
"""
from functools import lru_cache

import numpy as np
import torch

import rslab_amd as R
from rslab_amd import matgen

PRECISION = {"f64": R.Precision.FP64, "fp32": R.Precision.FP32_SCHUR, "bf16": R.Precision.BF16_SCHUR}
ORDERING = {"amd": R.OrderingMethod.Amd, "nd": R.OrderingMethod.MetisND}


def _c(kind, matrix, nx, ny, nz, nrhs, shift=-1.5, field="real", precision="f64", ordering="nd", target=1e-14):
    return dict(kind=kind, matrix=matrix, nx=nx, ny=ny, nz=nz, nrhs=nrhs, shift=shift, field=field,
                precision=precision, ordering=ordering, target=target)


def listed():
    return [
        # a small 2D indefinite system from host memory: one interior-point or
        # Newton step of a small model, where launches and copies count
        dict(_c("host", "grid", 33, 31, 1, 1, shift=-2.0, ordering="amd"), name="small_2d_host"),
        # an ensemble of independent 2D systems of uneven sizes under one plan
        dict(_c("batch", "grid", 16, 96, 1, 1), count=96, name="batch_2d"),
        # an ordinary ragged 3D grid, few right-hand sides
        dict(_c("step", "grid", 37, 29, 23, 3), name="ragged_3d"),
        # the headline: 216,000 unknowns, refactor and refine to 1e-14
        dict(_c("step", "grid", 60, 60, 60, 8), name="cube60"),
        # the reduced-precision factor of a mid-size grid under the same ladder
        dict(_c("step", "grid", 44, 44, 44, 8, precision="fp32"), name="cube44_fp32"),
        # one more right-hand side with the factor in hand (a time step)
        dict(_c("solve", "grid", 48, 48, 48, 1), name="solve_1rhs"),
        # a block of right-hand sides with the factor in hand (sources, modes)
        dict(_c("solve", "grid", 36, 36, 36, 32), name="solve_32rhs"),
        # complex symmetric Helmholtz with an absorbing layer, 16 sources
        dict(_c("step", "helmholtz", 40, 40, 40, 16, shift=-1.2, field="complex"), name="helmholtz40"),
        # 3 unknowns per node, 27-point coupling: one frequency of a sweep
        dict(_c("step", "vector27", 20, 20, 20, 32, shift=0.2, precision="fp32", target=1e-12), name="vector27_sweep"),
        # block GMRES on a matrix whose neighbour was factored in bf16 products
        dict(_c("krylov", "grid", 33, 33, 33, 4, shift=0.2, precision="bf16", target=1e-12), name="gmres_bf16"),
        # unsymmetric convection-diffusion, real and complex
        dict(_c("lu", "convection", 40, 40, 40, 8), name="lu_real"),
        dict(_c("lu", "convection", 26, 26, 26, 5, field="complex"), name="lu_complex"),
    ]


def _side(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step2d", "step3d", "step3d", "step3d", "host", "solve", "solve", "batch", "helmholtz", "helmholtz", "vector27",
                       "krylov", "lu", "lu"])
    if kind == "step2d":
        return _c("step", "grid", _side(rng, 24, 300), _side(rng, 24, 300), 1, _side(rng, 1, 16),
                  shift=-0.5 - 2 * rng.random(), ordering=rng.choice(["amd", "nd"]))
    if kind == "step3d":
        return _c("step", "grid", _side(rng, 10, 46), _side(rng, 10, 46), _side(rng, 10, 46), _side(rng, 1, 16),
                  shift=-0.5 - 2 * rng.random(), precision=rng.choice(["f64", "f64", "fp32"]))
    if kind == "host":
        return _c("host", "grid", _side(rng, 20, 160), _side(rng, 20, 160), 1, _side(rng, 1, 8),
                  shift=-0.5 - 2 * rng.random(), ordering=rng.choice(["amd", "nd"]))
    if kind == "solve":
        return _c("solve", "grid", _side(rng, 10, 46), _side(rng, 10, 46), _side(rng, 10, 46), _side(rng, 1, 48),
                  shift=-0.5 - 2 * rng.random())
    if kind == "batch":
        lo = _side(rng, 8, 32)
        return dict(_c("batch", "grid", lo, _side(rng, lo + 1, 96), 1, _side(rng, 1, 4)), count=_side(rng, 16, 96))
    if kind == "helmholtz":
        return _c("step", "helmholtz", _side(rng, 9, 36), _side(rng, 9, 36), _side(rng, 9, 36), _side(rng, 1, 16),
                  shift=-0.6 - rng.random(), field="complex")
    if kind == "vector27":
        m = _side(rng, 6, 19)
        return _c("step", "vector27", m, m, m, _side(rng, 1, 32), shift=0.05 + 0.45 * rng.random(),
                  precision=rng.choice(["f64", "fp32"]), target=1e-12)
    if kind == "krylov":
        return _c("krylov", "grid", _side(rng, 10, 33), _side(rng, 10, 33), _side(rng, 10, 33), _side(rng, 1, 8),
                  shift=0.1 + 0.4 * rng.random(), precision=rng.choice(["f64", "fp32", "bf16"]), target=1e-12)
    return _c("lu", "convection", _side(rng, 9, 36), _side(rng, 9, 36), _side(rng, 9, 36), _side(rng, 1, 16),
              shift=-0.5 - 1.5 * rng.random(), field=rng.choice(["real", "complex"]))


# ------------------------------------------------------------------ inputs
def _dims(case):
    return tuple(case[k] for k in ("nx", "ny", "nz") if case[k] > 1)


def _absorbing(dims, layer=4, peak=0.5):
    """Damping that grows over the outer `layer` nodes towards every face."""
    dist = None
    for ax, d in enumerate(dims):
        g = np.minimum(np.arange(d), d - 1 - np.arange(d)).reshape([-1 if k == ax else 1 for k in range(len(dims))])
        dist = np.broadcast_to(g, dims) if dist is None else np.minimum(dist, g)
    dist = dist.transpose().reshape(-1)  # the first dimension runs fastest
    return np.where(dist < layer, peak * ((layer - dist) / layer) ** 2, 0.0)


def _uniform(rng, shape, cplx):
    v = rng.uniform(-1.0, 1.0, shape)
    return v + 1j * rng.uniform(-1.0, 1.0, shape) if cplx else v


@lru_cache(maxsize=1)
def _vector27(m):
    return matgen.vector_stencil27(m=m, omega2=0.0)


def _sides(case):
    """The batch's grids: fixed by the case, so that its plan is too."""
    rng = np.random.default_rng(case["count"] * 1000 + case["nx"] + case["ny"])
    return rng.integers(case["nx"], case["ny"] + 1, case["count"])


def _inputs(case, seed):
    """(matrix, or the list of a batch's, and right-hand sides) of a seed."""
    rng = np.random.default_rng(seed)
    cplx = case["field"] == "complex"
    if case["kind"] == "batch":
        mats = [matgen.grid_laplacian((int(s), int(s)), shift=-rng.uniform(0.5, 3.5), diag_real=rng.uniform(-0.01, 0.01, s * s))
                for s in _sides(case)]
        return mats, _uniform(rng, (sum(m.n for m in mats), case["nrhs"]), False)
    dims = _dims(case)
    n = int(np.prod(dims))
    delta = rng.uniform(-0.01, 0.01, n)
    if case["matrix"] == "grid":
        a = matgen.grid_laplacian(dims, shift=case["shift"], diag_real=delta)
    elif case["matrix"] == "helmholtz":
        a = matgen.grid_laplacian(dims, shift=case["shift"], diag_real=delta, diag_imag=_absorbing(dims))
    elif case["matrix"] == "vector27":
        base = _vector27(case["nx"])
        on_diag = base.row_idx == np.repeat(np.arange(base.n), np.diff(base.col_ptr))
        a = base.with_values(base.values + np.where(on_diag, -case["shift"] + 0.01 * rng.uniform(-1, 1, base.nnz), 0.0))
    else:
        a = matgen.convection_diffusion(dims, shift=case["shift"], delta=delta, eta=np.full(n, 0.1) if cplx else None)
    return a, _uniform(rng, (a.n, case["nrhs"]), cplx)


def _settings(case):
    return R.SolverSettings().with_ordering(ORDERING[case["ordering"]]).with_precision(PRECISION[case["precision"]])


def _analyze(case, a, st):
    if case["kind"] == "lu":
        return R.LuSymbolic.analyze_with(a, st)
    if case["kind"] == "batch":
        return R.LdltSymbolic.analyze_batch(a, st)
    return R.LdltSymbolic.analyze_with(a, st)


def prepare(case, seed):
    a, b = _inputs(case, seed)
    st = _settings(case)
    sym = _analyze(case, a, st)
    if case["kind"] == "batch":
        a = R.CscMatrix.block_diag(a)
    first = a
    if case["kind"] == "krylov":  # the preconditioner: a neighbour's factor
        rng = np.random.default_rng(seed + 1)
        on_diag = a.row_idx == np.repeat(np.arange(a.n), np.diff(a.col_ptr))
        first = a.with_values(a.values + np.where(on_diag, rng.uniform(0.0, 0.1, a.nnz), 0.0))
    s = dict(case=case, a=a, b=b, f=sym.factor(first, st))
    if case["kind"] in ("step", "host", "batch"):
        s["mixed"] = R.MixedLdltSolver(s["f"], a)
    if case["kind"] in ("step", "solve", "batch"):
        s["values"] = torch.from_numpy(a.values).cuda()
        s["db"] = torch.from_numpy(b).cuda()
        s["dx"] = torch.empty_like(s["db"])
    return s


def run(s):
    case, f = s["case"], s["f"]
    k = case["nrhs"]
    if case["kind"] == "solve":
        f.solve_device(s["db"].data_ptr(), k, s["dx"].data_ptr())
        return s["dx"]
    if case["kind"] == "krylov":
        return R.gmres_block(s["a"], s["b"], k, f, case["target"], 100, 30).x
    if case["kind"] == "lu":
        f.refactor(s["a"])
        return f.solve_refined(s["a"], s["b"], 2)
    if case["kind"] == "host":
        f.refactor(s["a"])
        x, _ = s["mixed"].solve_to(s["a"], s["b"], case["target"])
        return x, np.array(f.inertia().as_tuple())
    f.refactor_device(s["values"].data_ptr())
    s["mixed"].solve_to_device(s["values"].data_ptr(), s["db"].data_ptr(), k, s["dx"].data_ptr(), case["target"])
    if case["kind"] == "batch":
        return s["dx"], np.array([i.as_tuple() for i in f.inertia_batch(case["count"])])
    if case["field"] == "complex" or case["precision"] != "f64":
        return s["dx"]  # their inertia is decided by rounding, or has no meaning
    return s["dx"], np.array(f.inertia().as_tuple())


# -------------------------------------------------------- work and tolerance
@lru_cache(maxsize=32)
def _plan_size(key):
    """(matrix entries, factor entries, factor operations, n) of a pattern."""
    case = dict(key)
    a, _ = _inputs(case, 0)
    inf = _analyze(case, a, _settings(case)).info()
    nnz = sum(m.nnz for m in a) if case["kind"] == "batch" else a.nnz
    n = sum(m.n for m in a) if case["kind"] == "batch" else a.n
    entries = inf["l_entries"] + inf["u_entries"] if case["kind"] == "lu" else inf["nnzl_padded"]
    return nnz, entries, inf["factor_flops"], n


def work(case):
    """A factor's operations are counted once and its entries written once; a
    solve is one forward and one backward substitution that read the factor
    once. Refinement's further solves are not counted."""
    nnz, entries, flops, n = _plan_size(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    cplx = case["field"] == "complex"
    size, mul = (16, 4) if cplx else (8, 1)
    k = case["nrhs"]
    solve = mul * (2 if case["kind"] == "lu" else 4) * entries * k
    moved = size * (entries + 2 * n * k)
    if case["kind"] == "solve":
        return {"bytes": moved, "flops": solve}
    if case["kind"] == "krylov":
        return {"bytes": moved + size * nnz, "flops": solve}
    return {"bytes": moved + size * (nnz + entries), "flops": mul * flops + solve}


def tolerance(case):
    """Against a 64-bit block elimination with refinement, over the listed
    cases and forty drawn ones, refined solutions were off by up to 8e-13, the
    plain solve by up to 8e-12, the sweep that stops at a backward error of
    1e-12 by 3e-9, and GMRES stopped at a residual of 1e-12 by 4e-12. What a
    backward error leaves grows with the condition number, so nearly singular
    shifts may show more than the largest seen."""
    if case["matrix"] == "vector27":
        return {"rel": 1.3e-8}
    if case["kind"] == "solve":
        return {"rel": 5e-11}
    if case["kind"] == "krylov":
        return {"rel": 2e-11}
    return {"rel": 1e-11}


# ------------------------------------------------------------------- exact
def _apply(rows, cols, vals, x):
    return torch.zeros_like(x).index_add_(0, rows, vals[:, None] * x[cols])


def _block_solve(n, bs, rows, cols, vals, b):
    """x of A x = b for a matrix that couples only neighbouring blocks of `bs`
    rows: block elimination in 64 bits, then refinement against A. `b` may
    hold several systems' blocks side by side in leading dimensions."""
    count = n // bs
    r, c = rows // bs, cols // bs

    def block(i, j):
        m = (r == i) & (c == j)
        d = torch.zeros(bs, bs, dtype=vals.dtype, device=vals.device)
        d.index_put_((rows[m] - i * bs, cols[m] - j * bs), vals[m], accumulate=True)
        return d

    lus, ups, los = [], [], []
    s = block(0, 0)
    for p in range(count):
        lus.append(torch.linalg.lu_factor(s))
        if p + 1 < count:
            ups.append(torch.linalg.lu_solve(*lus[p], block(p, p + 1)))
            los.append(block(p + 1, p))
            s = block(p + 1, p + 1) - los[p] @ ups[p]

    def solve(v):
        v = v.reshape(count, bs, -1).clone()
        for p in range(count):
            if p:
                v[p] -= los[p - 1] @ v[p - 1]
            v[p] = torch.linalg.lu_solve(*lus[p], v[p].contiguous())
        for p in range(count - 2, -1, -1):
            v[p] -= ups[p] @ v[p + 1]
        return v.reshape(n, -1)

    x = solve(b)
    for _ in range(5):
        x = x + solve(b - _apply(rows, cols, vals, x))
    return x


def _triplets(a):
    cols = np.repeat(np.arange(a.n), np.diff(a.col_ptr))
    rows, vals = a.row_idx, a.values
    if isinstance(a, R.CscMatrix):  # the lower triangle only
        off = rows != cols
        rows, cols, vals = np.r_[rows, cols[off]], np.r_[cols, rows[off]], np.r_[vals, vals[off]]
    return [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (rows, cols, vals)]


def exact(case, seed):
    a, b = _inputs(case, seed)
    if case["kind"] == "batch":
        out, at = [], 0
        for m in a:
            dense = torch.zeros(m.n, m.n, dtype=torch.float64, device="cuda")
            rows, cols, vals = _triplets(m)
            dense.index_put_((rows, cols), vals)
            lu = torch.linalg.lu_factor(dense)
            rhs = torch.from_numpy(b[at:at + m.n]).cuda()
            x = torch.linalg.lu_solve(*lu, rhs)
            out.append(x + torch.linalg.lu_solve(*lu, rhs - dense @ x))
            at += m.n
        return torch.cat(out), None
    dims = _dims(case)
    bs = a.n // dims[-1]
    x = _block_solve(a.n, bs, *_triplets(a), torch.from_numpy(b).cuda())
    if case["kind"] in ("krylov", "lu"):
        return x.cpu().numpy()
    if case["kind"] == "host":
        return x.cpu().numpy(), None
    if case["kind"] == "solve" or case["field"] == "complex" or case["precision"] != "f64":
        return x
    return x, None
