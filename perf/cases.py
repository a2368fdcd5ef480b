"""The solves that a user of this framework has it do, as measurable cases.

A case is a dict of plain values.  Its "kind" names the entry point that the
work goes through:

  solve      SolverMesh.solve: a steady solve of one hex box (the cantilever
             and the jittered cube of the benchmark, plain FP64 or mixed
             precision, diagonal or multigrid preconditioner)
  model      solid_model_new(...).evolve(): the reference's solidModel
             interface, a cube on zero-shear rollers under tension
  two_laws   evolve() and write_fields() of a case with two linearElastic laws
             on cellZones (sub-meshes)
  tets       SolverMesh.solve on tetrahedra with E per cell (spherical
             inclusions), full-delta least squares
  step       one Euler time step with body force, from given old-time fields
  batch      Batch.solve of uneven boxes packed together
  serve      Server: a burst of requests submitted, polled and collected
  ldu        LduSolver.solve: the lduMatrix::solver seam, one component

Converging cases run to outer tolerances of 1e-12, where the converged field
no longer depends on the path of the inner solver (rounding, preconditioner
and reduction order move it by less than 1e-9); the plain cantilever stops
after its configuration's fixed number of outer iterations, in FP64
throughout.  The mesh's jitter, the material values and the loads come from
the seed; sizes and the Poisson's ratios (which set the iteration counts) from
the case.
"""
import math

import numpy as np

import solids4foam_amd as s4f
from solids4foam_amd import _abi, cases
from solids4foam_amd.batch import Batch
from solids4foam_amd.serve import Server
from solids4foam_amd.solid import LduSolver, PolyMesh, SolverMesh, solid_model_new

DIAGONAL, GAMG, GAMG_SMOOTHED = _abi.PRECOND_DIAGONAL, _abi.PRECOND_GAMG, _abi.PRECOND_GAMG_SMOOTHED
FP64, MIXED = _abi.PRECISION_FP64, _abi.PRECISION_MIXED
TOL = 1e-12


def listed():
    return [
        # the small case of the framework: the 5,000-cell cantilever on the plain path, solver settings of its
        # configuration (PCG 1e-9, relTol 0.1), a fixed count of outer iterations: launches and latency
        dict(name="cantilever_5k_fp64", kind="solve", nx=50, ny=10, nz=10, lx=1.0, ly=0.2, lz=0.2, jitter=0.0, nu=0.3,
             load="cantilever", precision=FP64, precond=DIAGONAL, rel_tol=0.1, outer=100, relax=0.0),
        # the smallest box of the sweep and serving generators, alone: the latency of a tiny solve
        dict(name="box_8_mixed", kind="solve", nx=8, ny=8, nz=8, lx=0.08, ly=0.08, lz=0.08, jitter=0.1, nu=0.3,
             load="cantilever", precision=MIXED, precond=GAMG, rel_tol=0.9, outer=0, relax=0.0),
        # a model built through the solidModel table: zero-shear rollers, full-delta gradient, exact field known
        dict(name="rollers_25_mixed", kind="model", n=25, nu=0.3, precision=MIXED, precond=GAMG),
        # the jittered cube of the benchmark at an ordinary size, mixed precision
        dict(name="cube_64_mixed", kind="solve", nx=64, ny=64, nz=64, lx=1.0, ly=1.0, lz=1.0, jitter=0.15, nu=0.3,
             load="tension", precision=MIXED, precond=GAMG_SMOOTHED, rel_tol=0.9, outer=0, relax=0.0),
        # an odd, uneven box on the plain FP64 path with the multigrid preconditioner
        dict(name="box_91x75x83_fp64", kind="solve", nx=91, ny=75, nz=83, lx=0.91, ly=0.75, lz=0.83, jitter=0.15,
             nu=0.3, load="tension", precision=FP64, precond=GAMG_SMOOTHED, rel_tol=0.9, outer=0, relax=0.0),
        # the largest: the jittered cube with 2.1 million cells, mixed precision
        dict(name="cube_128_mixed", kind="solve", nx=128, ny=128, nz=128, lx=1.0, ly=1.0, lz=1.0, jitter=0.15, nu=0.3,
             load="tension", precision=MIXED, precond=GAMG_SMOOTHED, rel_tol=0.9, outer=0, relax=0.0),
        # heterogeneous tetrahedra: inclusions as E per cell, shear load
        dict(name="tets_15_mixed", kind="tets", n=15, nu=0.3, precision=MIXED, precond=GAMG),
        # two laws on sub-meshes (matrix and a soft core) and the fields written after the loop
        dict(name="two_laws_18_fp64", kind="two_laws", n=18, nu=0.3, precision=FP64, precond=GAMG),
        # a dynamic case's time step: Euler d2dt2, gravity, old-time fields in
        dict(name="step_47_mixed", kind="step", nx=47, ny=40, nz=45, nu=0.3, precision=MIXED, precond=GAMG),
        # the batched sweep's kind of work: uneven boxes in one packed structure, field relaxation
        dict(name="batch_24", kind="batch", count=24, nmin=8, nmax=32, nu=0.3, shapes=5, precision=MIXED,
             precond=GAMG_SMOOTHED),
        # the serving stream's kind of work: a burst of requests on resident meshes, loads new each time
        dict(name="serve_12", kind="serve", count=12, nmin=8, nmax=48, nu=0.3, shapes=7, precision=MIXED,
             precond=GAMG),
        # one component of a momentum matrix handed over by an lduMatrix host program
        dict(name="ldu_60x64x71", kind="ldu", nx=60, ny=64, nz=71),
    ]


def _log(rng, a, b):
    """An integer of [a, b], spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def _box(rng, a, b):
    """Three sizes of at most a factor 1.6 from one another (slender boxes take many more outer iterations)."""
    n = _log(rng, a, b)
    return [min(b, max(a, int(round(n * rng.uniform(0.79, 1.26))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "cantilever", "model", "tets", "two_laws", "step", "step",
                       "batch", "serve", "ldu", "ldu"])
    mg = rng.choice([GAMG, GAMG_SMOOTHED])
    precision = rng.choice([FP64, MIXED, MIXED])
    nu = round(rng.uniform(0.2, 0.3), 3)
    if kind == "cantilever":
        n = rng.randint(8, 14)
        return dict(kind="solve", nx=5 * n + rng.randint(-3, 3), ny=n, nz=rng.randint(8, 14), lx=1.0, ly=0.2, lz=0.2,
                    jitter=0.0, nu=nu, load="cantilever", precision=FP64, precond=DIAGONAL, rel_tol=0.1,
                    outer=rng.randint(50, 100), relax=0.0)
    if kind == "solve":
        nx, ny, nz = _box(rng, 8, 88)
        return dict(kind="solve", nx=nx, ny=ny, nz=nz, lx=nx * 0.01, ly=ny * 0.01, lz=nz * 0.01,
                    jitter=rng.choice([0.1, 0.15]), nu=nu, load="tension", precision=precision, precond=mg,
                    rel_tol=0.9, outer=0, relax=rng.choice([0.0, 0.0, 0.9]))
    if kind == "model":
        return dict(kind="model", n=_log(rng, 8, 40), nu=nu, precision=precision, precond=mg)
    if kind == "tets":
        return dict(kind="tets", n=rng.randint(8, 15), nu=0.3, precision=MIXED, precond=mg)
    if kind == "two_laws":
        return dict(kind="two_laws", n=_log(rng, 8, 18), nu=0.3, precision=precision, precond=mg)
    if kind == "step":
        nx, ny, nz = _box(rng, 12, 80)
        return dict(kind="step", nx=nx, ny=ny, nz=nz, nu=nu, precision=precision, precond=mg)
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(4, 24), nmin=8, nmax=rng.randint(16, 32), nu=0.3,
                    shapes=rng.randint(0, 10 ** 6), precision=precision, precond=mg)
    if kind == "serve":
        return dict(kind="serve", count=rng.randint(3, 12), nmin=8, nmax=rng.randint(16, 40), nu=0.3,
                    shapes=rng.randint(0, 10 ** 6), precision=precision, precond=GAMG)
    nx, ny, nz = _box(rng, 8, 80)
    return dict(kind="ldu", nx=nx, ny=ny, nz=nz)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _opts(case, relax=0.0):
    return dict(solutionTolerance=TOL, alternativeTolerance=TOL, pcgTolerance=1e-2 * TOL, pcgRelTol=0.9,
                nCorrectors=100000, precision=case["precision"], preconditioner=case["precond"], relaxD=relax)


def _direction(rng):
    d = rng.normal(size=3)
    return d / np.linalg.norm(d)


def _young(rng):
    """E of the sweep and serving generators: log-normal, median 100 GPa, sigma 0.5."""
    return float(100e9 * np.exp(0.5 * rng.normal()))


def _solve_state(ctx, case, rng):
    pm = PolyMesh.box(case["nx"], case["ny"], case["nz"], (case["lx"], case["ly"], case["lz"]), case["jitter"],
                      int(rng.integers(1 << 30)), False)
    fixed, loaded = (0, 1) if case["load"] == "cantilever" else (4, 5)
    m = SolverMesh(ctx, pm, [cases.FIX if p == fixed else cases.TRAC for p in range(6)])
    m.set_material(_young(rng), case["nu"])
    for p in range(6):
        m.set_bc(p, (0.0, 0.0, 0.0))
    if case["load"] == "cantilever":
        m.set_bc(loaded, rng.uniform(1e5, 1e7) * np.array([0.0, -1.0, 0.0]) + rng.uniform(-1e4, 1e4, size=3))
    else:  # tension with some shear
        m.set_bc(loaded, rng.uniform(1e5, 1e7) * np.array([0.0, 0.0, 1.0]) + rng.uniform(-1e4, 1e4, size=3))
    if case["outer"]:
        opts = dict(cases.SMALL_OPTS, nCorrectors=case["outer"], pcgRelTol=case["rel_tol"],
                    precision=case["precision"], preconditioner=case["precond"])
    else:
        opts = dict(_opts(case, case["relax"]), pcgRelTol=case["rel_tol"])
    return dict(mesh=m, opts=opts)


def _roller_inputs(case, seed):
    """Points of the jittered unit cube (blockMesh numbering), E and the tension."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    g = np.arange(n + 1) / n
    pts = np.stack(np.meshgrid(g, g, g, indexing="ij"), axis=-1).transpose(2, 1, 0, 3).copy()  # [k, j, i]
    pts[1:-1, 1:-1, 1:-1] += rng.uniform(-0.15 / n, 0.15 / n, size=(n - 1, n - 1, n - 1, 3))
    return pts, _young(rng), float(rng.uniform(1e5, 1e7))


def _model_state(ctx, case, seed):
    pts, E, t = _roller_inputs(case, seed)
    n = case["n"]
    a = PolyMesh.box(n, n, n).addressing()
    pm = PolyMesh.from_arrays(pts.reshape(-1, 3), a["fOff"], a["fVerts"], a["owner"], a["neighbour"], n ** 3,
                              a["patchStart"], a["patchSize"])
    roller, free = dict(type="fixedDisplacementZeroShear"), dict(type="solidTraction")
    model = solid_model_new("linearGeometryTotalDisplacement", ctx, pm,
                            [roller, free, roller, free, roller, dict(type="solidTraction", traction=(0.0, 0.0, t))],
                            E, case["nu"], solver=_opts(case), ls_full_delta=True)
    return dict(model=model)


def _tets_state(ctx, case, rng):
    _, m, _, _, _ = cases.tet_inclusions(ctx, n=case["n"], seed=int(rng.integers(1 << 30)), inc_seed=3, nu=case["nu"],
                                         E_matrix=200e9, E_inc=20e9, rmin=0.1, rmax=0.2,
                                         traction=tuple(rng.uniform(1e6, 5e6) * np.array([0.0, 1.0, 0.2])))
    return dict(mesh=m, opts=_opts(case))


def _two_laws_state(ctx, case, rng):
    n = case["n"]
    pm = PolyMesh.box(n, n, n, (1.0, 1.0, 1.0), 0.1, int(rng.integers(1 << 30)), False)
    zone = (np.linalg.norm(pm.cell_centres() - 0.5, axis=1) < 0.3).astype(np.int32)
    E = np.where(zone == 1, 0.1, 1.0) * _young(rng)
    patches = [dict(type="solidTraction") for _ in range(6)]
    patches[4] = dict(type="fixedDisplacement", value=(0.0, 0.0, 0.0))
    patches[5] = dict(type="solidTraction", traction=(0.0, 0.0, float(rng.uniform(1e5, 1e7))))
    model = solid_model_new("linearGeometryTotalDisplacement", ctx, pm, patches, E, case["nu"], solver=_opts(case),
                            zones=zone)
    return dict(model=model)


def _step_state(ctx, case, rng):
    n = (case["nx"], case["ny"], case["nz"])
    L = tuple(0.01 * v for v in n)
    pm = PolyMesh.box(*n, L, 0.1, int(rng.integers(1 << 30)), False)
    m = SolverMesh(ctx, pm, [cases.FIX] + [cases.TRAC] * 5)
    m.set_material(_young(rng), case["nu"])
    m.set_density(7800.0)
    m.set_gravity((0.0, -9.81, 0.0))
    for p in range(6):
        m.set_bc(p, (0.0, 0.0, 0.0))
    m.set_bc(1, 1e6 * _direction(rng))
    # the two old-time fields of a beam in motion: a bending mode and its velocity over one step
    x = pm.cell_centres() / np.array(L)
    a = rng.uniform(0.5, 1.5, size=3) * 1e-6
    old = np.stack([a[0] * x[:, 0] * x[:, 1], -a[1] * x[:, 0] ** 2, a[2] * x[:, 0] * x[:, 2]], axis=1)
    return dict(mesh=m, old=old, old_old=old * (1.0 - 0.02 * rng.uniform(0.5, 1.5)),
                opts=dict(_opts(case), d2dt2=_abi.D2DT2_EULER, deltaT=5e-5))


def _boxes(ctx, case, rng):
    """Uneven boxes of the sweep generator's form: shapes from the case, jitter, E and loads from the seed."""
    shapes = np.random.default_rng(case["shapes"])
    out = []
    for _ in range(case["count"]):
        # uneven, but of moderate aspect: slender boxes take many times the outer iterations
        base = shapes.integers(case["nmin"], case["nmax"] + 1)
        n = [int(np.clip(round(base * shapes.uniform(0.75, 1.35)), case["nmin"], case["nmax"])) for _ in range(3)]
        nu = float(shapes.uniform(0.2, case["nu"]))
        spec = dict(n=tuple(n), L=tuple(0.01 * v for v in n), jitter=0.1, seed=int(rng.integers(1 << 30)),
                    E=_young(rng), nu=nu, traction=tuple(rng.uniform(1e5, 1e7) * _direction(rng)))
        out.append(cases.box_case(ctx, spec))
    return out


def _batch_state(ctx, case, rng):
    b = Batch(ctx)
    for _, m, _ in _boxes(ctx, case, rng):
        b.add(m)
    return dict(batch=b, opts=_opts(case, 0.8))


def _serve_state(ctx, case, rng):
    boxes = _boxes(ctx, case, rng)
    requests = [(m, bv) for _, m, bv in boxes]
    if len(boxes) > 4:  # every fifth request repeats an earlier mesh with another load
        for k in range(4, len(boxes), 5):
            _, m, bv = boxes[k - 4]
            requests[k] = (m, bv @ np.diag(rng.uniform(0.5, 1.5, size=3)))
    cells = sum((m.nCells + 63) // 64 * 64 for _, m, _ in boxes)
    server = Server(ctx, 3000 * cells + (1 << 26), max_slots=64, **_opts(case, 0.8))
    return dict(server=server, requests=requests, boxes=boxes)


def _ldu_inputs(case, seed):
    """A 7-point momentum-component matrix in LDU form (uneven face coefficients as of a jittered mesh, Dirichlet
    rows at one end), a displacement component and the source it solves."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    c = np.arange(nx * ny * nz, dtype=np.int64).reshape(nz, ny, nx)
    lower = np.concatenate([c[:, :, :-1].ravel(), c[:, :-1].ravel(), c[:-1].ravel()])
    upper = np.concatenate([c[:, :, 1:].ravel(), c[:, 1:].ravel(), c[1:].ravel()])
    order = np.lexsort((upper, lower))  # upper-triangular order
    lower, upper = lower[order], upper[order]
    a = 1e9 * np.exp(0.2 * rng.normal(size=lower.size))
    diag = np.bincount(lower, a, c.size) + np.bincount(upper, a, c.size)
    diag[c[:, :, 0].ravel()] += 2e9
    i = (np.arange(nx) + 0.5) / nx
    k = (np.arange(nz) + 0.5) / nz
    psi = 1e-5 * np.broadcast_to((i ** 2)[None, None, :] * (1.0 + 0.3 * np.sin(3.0 * k))[:, None, None], c.shape)
    psi = (psi + 1e-7 * rng.normal(size=c.shape)).ravel()
    src = diag * psi - np.bincount(lower, a * psi[upper], c.size) - np.bincount(upper, a * psi[lower], c.size)
    return lower, upper, diag, -a, src, psi


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    ctx = s4f.Context(0)
    kind = case["kind"]
    if kind == "ldu":
        lower, upper, diag, a, src, _ = _ldu_inputs(case, seed)
        state = dict(ldu=LduSolver(ctx, case["nx"] * case["ny"] * case["nz"], lower, upper), diag=diag, upper=a, src=src,
                     psi=np.zeros_like(src))
    elif kind == "model":
        state = _model_state(ctx, case, seed)
    else:
        state = dict(solve=_solve_state, tets=_tets_state, two_laws=_two_laws_state, step=_step_state,
                     batch=_batch_state, serve=_serve_state)[kind](ctx, case, rng)
    state["ctx"] = ctx
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    if "ldu" in state:
        psi, _ = state["ldu"].solve(state["diag"], state["upper"], state["src"], state["psi"], tolerance=1e-12,
                                    max_iter=5000)
        return psi
    if "batch" in state:
        return [dict(D=r["D"], sigma=r["sigma"]) for r in state["batch"].solve(**state["opts"])]
    if "server" in state:
        srv = state["server"]
        ids = [srv.submit(m, bv) for m, bv in state["requests"]]
        done = {}
        while len(done) < len(ids):
            rid = srv.poll(wait_ms=1000)
            if rid is not None:
                r = srv.result(rid)
                done[rid] = dict(D=r["D"], sigma=r["sigma"])
        return [done[i] for i in ids]
    if "model" in state:
        model = state["model"]
        model.evolve()
        out = dict(D=model.D, sigma=model.sigma, gradD=model.gradD)
        if model.mesh.nCells and getattr(model.mesh, "zones", None) is not None:
            out.update(model.write_fields())
        return out
    m = state["mesh"]
    if "old" in state:
        m.set_old_time(state["old"], state["old_old"])
    r = m.solve(**state["opts"])
    return dict(D=r["D"], sigma=r["sigma"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and exact values
# ---------------------------------------------------------------------------

def _cells(case):
    kind = case["kind"]
    if kind in ("model", "two_laws"):
        return case["n"] ** 3
    if kind == "tets":
        return 6 * case["n"] ** 3
    if kind in ("batch", "serve"):
        return case["count"] * (0.5 * (case["nmin"] + case["nmax"])) ** 3
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """Each input read once and each result written once: the face geometry and coefficients (area vector, weight,
    matrix and Rhie-Chow coefficient, both cells), the cell data (centre, least-squares inverse, diagonal), D and
    sigma.  Operations: one residual, gradient and matrix product."""
    C = _cells(case)
    if case["kind"] == "ldu":
        return dict(bytes=C * (3 * (8 + 8) + 8 + 8 + 8 + 8), flops=C * 13)
    faces = 2 if case["kind"] == "tets" else 3
    return dict(bytes=C * (faces * (24 + 8 + 8 + 8 + 8) + 24 + 48 + 8 + 24 + 48), flops=C * (faces * 300 + 200))


def _cell_centres(p):
    """OpenFOAM cell centres of a structured hex block with points p[k, j, i]."""
    def corner(i, j, k):
        n0, n1, n2 = p.shape[0] - 1, p.shape[1] - 1, p.shape[2] - 1
        return p[k:n0 + k, j:n1 + j, i:n2 + i]
    v = [corner(*b) for b in ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))]
    centres, areas = [], []
    for q in ((0, 4, 7, 3), (1, 2, 6, 5), (0, 1, 5, 4), (3, 7, 6, 2), (0, 3, 2, 1), (4, 5, 6, 7)):
        w = [v[t] for t in q]
        mid = sum(w) / 4.0
        num, den, area = 0.0, 0.0, 0.0
        for t in range(4):
            a, b = w[t], w[(t + 1) % 4]
            n = np.cross(b - a, mid - a)
            mag = np.linalg.norm(n, axis=-1, keepdims=True)
            num, den, area = num + mag * (a + b + mid), den + mag, area + n
        centres.append(num / den / 3.0)
        areas.append(0.5 * area)
    est = sum(centres) / 6.0
    num, den = 0.0, 0.0
    for c, s in zip(centres, areas):
        vol = np.sum(s * (c - est), axis=-1, keepdims=True)
        num, den = num + vol * (0.75 * c + 0.25 * est), den + vol
    return (num / den).reshape(-1, 3)


def exact(case, seed):
    """The rollers' uniform uniaxial strain and the linear system's manufactured solution; the other solves have no
    closed form."""
    if case["kind"] == "ldu":
        return _ldu_inputs(case, seed)[-1]
    if case["kind"] != "model":
        return None
    pts, E, t = _roller_inputs(case, seed)
    x = _cell_centres(pts)
    e = np.array([-case["nu"] * t / E, -case["nu"] * t / E, t / E])
    sigma = np.zeros((len(x), 6))
    sigma[:, 5] = t
    return dict(D=x * e, sigma=sigma, gradD=np.tile(np.diag(e).ravel(), (len(x), 1)))
