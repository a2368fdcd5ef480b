"""Instances of a batch or of a server do not reach one another: whatever the
first one holds (infinities and NaN of a diverged solve, vectors that its PCG
never wrote), the others' results are bitwise those of their solves alone.  The
first instance owns row 0 of every multigrid level, which an empty slot of
another instance's row must not read."""
import time

import numpy as np
import pytest

from tests._cases import E_STEEL, NU_STEEL

pytestmark = pytest.mark.gpu

# outer iterations capped; no stall test: a diverging member would switch the whole batch to FP64
CAPPED = dict(solutionTolerance=1e-14, alternativeTolerance=1e-14, pcgTolerance=1e-16, pcgRelTol=0.1, nCorrectors=6,
              mixedStallWindow=-1)
# three and more levels beside instances that pass through the deeper ones; a partial last slice
SIZES = [(28, 25, 24), (9, 8, 8), (23, 11, 9)]


@pytest.fixture(scope="module")
def ctx():
    from solids4foam_amd import Context
    c = Context(0)
    yield c
    c.close()


def _box(ctx, n, seed, traction=(1e6, -2e6, 5e5)):
    from solids4foam_amd import PolyMesh, SolverMesh, cases
    pm = PolyMesh.box(*n, L=tuple(0.1 * v for v in n), jitter=0.1, seed=seed)
    m = SolverMesh(ctx, pm, [cases.FIX] + [cases.TRAC] * 5)
    m.set_material(E_STEEL, NU_STEEL)
    bv = np.zeros((pm.nBoundaryFaces, 3))
    bv[pm.patch_faces(1)] = traction
    for p in range(6):
        m.set_bc(p, bv[pm.patch_faces(p)])
    return m, bv


def _equal(r, a):
    return all(np.isfinite(r[k]).all() and np.array_equal(r[k], a[k]) for k in ("D", "sigma")) and \
        r["nOuter"] == a["nOuter"]


def _check_batch(ctx, precond, precision, tets=False):
    # the first member's load overflows the sums of its first PCG iteration; then
    # it has none: its PCG never runs, and its vectors keep what the first solve left
    from solids4foam_amd.batch import Batch
    print(f"[isolation] batch precond={precond} precision={precision}", flush=True)
    opts = dict(CAPPED, precision=precision, preconditioner=precond, pcgMaxIter=40)
    first, _ = _box(ctx, (12, 11, 10), 1, traction=(1e250, 1e250, 1e250))
    others = [_box(ctx, n, 2 + i)[0] for i, n in enumerate(SIZES)]
    if tets:  # no single slot count: the sequences with finalize kernels
        from solids4foam_amd import cases
        others.append(cases.tet_inclusions(ctx, n=4, seed=3)[1])
    alone = [m.solve(**opts) for m in others]
    b = Batch(ctx)
    for m in [first] + others:
        b.add(m)
    got = b.solve(**opts)
    assert not np.isfinite(got[0]["D"]).all() and not got[0]["converged"]
    for i, a in enumerate(alone):
        assert _equal(got[1 + i], a), ("diverging first", i)
    first.set_bc(1, (0.0, 0.0, 0.0))
    got = b.solve(**opts)
    assert got[0]["converged"] and not got[0]["D"].any()
    for i, a in enumerate(alone):
        assert _equal(got[1 + i], a), ("unloaded first", i)
    b.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_batch_multigrid(ctx, precision):
    from solids4foam_amd import PRECOND_GAMG
    _check_batch(ctx, PRECOND_GAMG, precision)


@pytest.mark.parametrize("precision", [0, 1])
def test_server_multigrid(ctx, precision):
    # the diverging request keeps its PCG busy with NaN while the others join it on the map
    from solids4foam_amd import PRECOND_GAMG, _abi
    from solids4foam_amd.serve import Server
    print(f"[isolation] server precision={precision}", flush=True)
    opts = dict(CAPPED, precision=precision, preconditioner=PRECOND_GAMG, pcgMaxIter=2000)
    first = _box(ctx, (12, 11, 10), 1, traction=(1e250, 1e250, 1e250))
    others = [_box(ctx, n, 2 + i) for i, n in enumerate(SIZES)]
    alone = [m.solve(**opts) for m, _ in others]
    srv = Server(ctx, 1 << 30, max_slots=8, **opts)
    ids = [srv.submit(m, bv) for m, bv in [first] + others]
    got = {}
    t0 = time.time()
    while len(got) < len(ids) and time.time() - t0 < 60:
        rid = srv.poll(100)
        if rid is not None:
            got[rid] = srv.result(rid)
    srv.close()
    assert len(got) == len(ids)
    assert got[ids[0]]["status"] == _abi.S4F_ERR_DIVERGED
    for i, (rid, a) in enumerate(zip(ids[1:], alone)):
        assert _equal(got[rid], a), i


@pytest.mark.parametrize("precision", [0, 1])
def test_batch_smoothed_multigrid(ctx, precision):
    # weighted restriction of the first level
    from solids4foam_amd import PRECOND_GAMG_SMOOTHED
    _check_batch(ctx, PRECOND_GAMG_SMOOTHED, precision)


@pytest.mark.parametrize("precond", [0, 2, 3])
def test_batch_turns_merged(ctx, precond):
    # an instance over the line of merged launches leaves first (no load): the
    # others go on in merged launches, on a hierarchy that still holds its rows
    from solids4foam_amd.batch import Batch
    print(f"[isolation] batch turns merged precond={precond}", flush=True)
    opts = dict(CAPPED, precision=0, preconditioner=precond, pcgMaxIter=40, nCorrectors=40)
    large, _ = _box(ctx, (64, 41, 25), 1, traction=(0.0, 0.0, 0.0))
    large.set_tiles(65536, 1)  # a tile per slice: 1,025
    others = [_box(ctx, n, 2 + i)[0] for i, n in enumerate(SIZES)]
    alone = [m.solve(**opts) for m in others]
    b = Batch(ctx)
    for m in others[:1] + [large] + others[1:]:
        b.add(m)
    got = b.solve(**opts)
    assert got[1]["converged"] and got[1]["nOuter"] < 5
    del got[1]
    for i, (r, a) in enumerate(zip(got, alone)):
        assert r["nOuter"] == 40 and _equal(r, a), i
    b.close()


@pytest.mark.parametrize("tets", [False, True])
@pytest.mark.parametrize("precond", [0, 2, 3])
def test_batch_sequences(ctx, precond, tets):
    _check_batch(ctx, precond, 0, tets)
