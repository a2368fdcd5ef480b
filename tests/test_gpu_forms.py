"""The single-kernel entry points run the kernels that a solve of the mesh
launches: up to 1,024 tiles of one slot count the merged ones, above those with
finalize kernels beside them."""
import numpy as np
import pytest

from tests._cases import E_STEEL, NU_STEEL, cube_tension_bc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from solids4foam_amd import Context
    c = Context(0)
    yield c
    c.close()


def _mesh(ctx, n, tets, tiles):
    from solids4foam_amd import PolyMesh, SolverMesh
    pm = PolyMesh.box(*n, L=(1.0, 1.0, 1.0), jitter=0.15, seed=3, tets=tets)
    sl = [pm.patch_faces(p) for p in range(6)]
    pt, bv = cube_tension_bc(pm.nBoundaryFaces, sl)
    m = SolverMesh(ctx, pm, pt, ls_full_delta=tets)
    m.set_material(E_STEEL, NU_STEEL)
    for p in range(6):
        m.set_bc(p, bv[sl[p]])
    if tiles:
        m.set_tiles(*tiles)
    return m, pt, bv


# merged: a partial slice, tiles of several slices, the last merged tile count; then one tile more
FORMS = [((9, 7, 6), False, None), ((33, 32, 31), False, (20, 4)), ((64, 32, 32), False, (65536, 1)),
         ((64, 41, 25), False, (65536, 1)), ((5, 4, 4), True, None), ((23, 22, 22), True, (65536, 1))]


@pytest.mark.parametrize("n,tets,tiles", FORMS)
def test_residual(ctx, oracle_mod, n, tets, tiles):
    # sums of at most six faces' terms in FP64, against the oracle's in another order
    print(f"[forms] residual {n} tets={tets} tiles={tiles}", flush=True)
    m, pt, bv = _mesh(ctx, n, tets, tiles)
    om = oracle_mod.Mesh.box(*n, L=(1.0, 1.0, 1.0), jitter=0.15, seed=3, tets=tets)
    oc = oracle_mod.Case(om, E_STEEL, NU_STEEL, pt, bv, ls_full_delta=tets)
    for _ in range(2):
        oc.iterate(precond=oracle_mod.PRECOND_DIAGONAL)
    C, B = om.nCells, om.nBoundaryFaces
    D, G, sb = oc.get("D").reshape(C, 3), oc.get("G").reshape(C, 9), oc.get("sigmab").reshape(B, 6)
    oc.op("residual")
    R = oc.get("R").reshape(C, 3)
    assert np.abs(m.residual(D, G, sb) - R).max() < 1e-10 * np.abs(R).max()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,tets,tiles,merged", [FORMS[0] + (True,), FORMS[2] + (True,), FORMS[3] + (False,),
                                                 FORMS[4] + (True,)])
def test_kernel_times(ctx, n, tets, tiles, merged, precision):
    # a merged sequence launches no finalize kernel; the replays leave the mesh as it was
    from solids4foam_amd import autotune
    print(f"[forms] kernel times {n} tets={tets} precision={precision}", flush=True)
    m, _, _ = _mesh(ctx, n, tets, tiles)
    opts = dict(precision=precision, preconditioner=3, nCorrectors=3, pcgRelTol=0.1)
    a = m.solve(**opts)
    t = {k: autotune.kernel_ms(m, k, precision, 3) for k in range(9)}
    assert (t.pop(3) == 0.0) == merged
    assert all(v > 0.0 for v in t.values())
    b = m.solve(**opts)
    assert np.array_equal(a["D"], b["D"]) and np.array_equal(a["sigma"], b["sigma"])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,tets", [((5, 4, 3), False), ((3, 3, 2), True)])
def test_product_of_an_infinite_value(ctx, n, tets, mixed):
    # an infinite entry reaches its own row and its neighbours', as infinity: an
    # empty or boundary slot adds nothing, also where the row's value is infinite
    print(f"[forms] infinite value {n} tets={tets} mixed={mixed}", flush=True)
    m, _, _ = _mesh(ctx, n, tets, None)
    C = m.nCells
    for cell in (0, C // 2, C - 1):
        x = np.zeros((C, 3))
        x[cell] = 1.0
        reach = m.spmv3(x, mixed=mixed) != 0.0
        x[cell] = np.inf
        y = m.spmv3(x, mixed=mixed)
        assert reach[cell].all() and not np.isnan(y).any()
        assert np.array_equal(np.isinf(y), reach) and (y[cell] > 0).all()
