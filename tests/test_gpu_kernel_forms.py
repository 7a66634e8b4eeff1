"""The device kernels' forms held to each other at the sizes where a form can
go wrong: the last, partly filled wavefront or tile, cells of every face
count, the smallest meshes, both precisions. Where both forms add the same
terms in the same order the bar is equality."""
import numpy as np
import pytest

from myjoe_amd import cases, joemi
from oracle.oracle import Oracle
from tests.helpers import compare

pytestmark = pytest.mark.gpu


def box(n, frac, scheme="HLLC", kind="inviscid", **kw):
    """A split box of n^3 hexes, frac of them split into tetrahedra."""
    mm, joe = cases.box_case(n, frac=frac, seed=n, scheme=scheme, **kw)
    if kind != "inviscid":
        joe = joe.replace("MU_REF = 0.0", "MU_REF = 0.01\nMU_MODE = POWERLAW\nMU_POWER_LAW = 0.7")
    if kind == "sst":
        joe = cases.with_sst(joe, 0.001, 5.0, cases.SST_BOX)
    if kind in ("coupled", "coupled_sa"):
        joe = cases.coupled(joe)
    if kind == "coupled_sa":
        joe = cases.with_sa(joe, 0.006, cases.SA_BOX)
    return joemi.Mesh.from_faces(mm), joe


def values(mesh, joe, names, precision=joemi.JM_FP64, implicit=True, seed=5):
    s = joemi.Solver(mesh, joe, precision)
    s.set_state(*cases.random_state(mesh.ncv, seed))
    s.calc_rhs(implicit)
    return {k: s.get(k) for k in names}


# 1 cell .. several wavefronts; frac 0: hexes only (ten cells of six faces per
# wavefront), 1: tetrahedra only (sixteen of four), between: both
@pytest.mark.parametrize("precision", [joemi.JM_FP64, joemi.JM_MIXED])
@pytest.mark.parametrize("n,frac", [(1, 0.0), (1, 1.0), (2, 0.5), (3, 0.0), (5, 0.5), (4, 1.0)])
@pytest.mark.parametrize("scheme,kind", [("HLLC", "inviscid"), ("ROE", "inviscid"), ("HLLC", "laminar"),
                                         ("HLLC", "coupled"), ("HLLC", "coupled_sa")])
def test_jacobian_per_entry_equals_per_cell(n, frac, precision, scheme, kind):
    print(f"jacobian forms n={n} frac={frac} precision={precision} {scheme} {kind}", flush=True)
    mesh, joe = box(n, frac, scheme, kind)
    a = values(mesh, joe + "GPU_JAC_KERNEL = ENTRY\n", ["A"], precision)["A"]
    b = values(mesh, joe + "GPU_JAC_KERNEL = CELL\n", ["A"], precision)["A"]
    assert np.array_equal(a, b, equal_nan=True)


# the block BiCGStab against its own stop test: 1 cell .. several blocks of
# either launch shape with the true residual, and on both sides of the size
# from which it takes the recurrence's and confirms it (14k cells); its sums
# finished from 256 and 257 partials (13056 cells, one more), 1024 and 1025
# (52224); a zero and a near guess, tolerances it reaches and one it cannot
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 1), (7, 3, 2), (4, 13, 1), (8, 8, 8), (23, 23, 23), (25, 25, 25),
                                  (3, 71, 73), (64, 12, 17), (7, 7, 267), (64, 24, 34), (11, 47, 102)])
def test_block_solver_true_residual_at_the_stop(dims):
    print(f"block solver {dims}", flush=True)
    n = int(np.prod(dims))
    idx = np.arange(n).reshape(dims)
    r, c = [np.arange(n)], [np.arange(n)]
    for ax in range(3):
        a = np.moveaxis(idx, ax, 0)
        for x, y in ((a[:-1], a[1:]), (a[1:], a[:-1])):
            r.append(x.ravel())
            c.append(y.ravel())
    row, nv = np.concatenate(r), np.concatenate(c)
    order = np.argsort(row, kind="stable")  # the diagonal stays first in its row
    row, nv = row[order], nv[order].astype(np.int32)
    ni = np.searchsorted(row, np.arange(n + 1)).astype(np.int32)
    g = np.random.default_rng(n)
    A = 0.1 * g.standard_normal((len(nv), 5, 5)) - 0.6 * np.eye(5)
    A[ni[:-1]] += 5.0 * np.eye(5)
    inv = np.linalg.inv(A[ni[:-1]])

    def mul(x):
        return np.add.reduceat(np.einsum("kij,kj->ki", A, x[nv]), ni[:-1], axis=0)

    x = g.standard_normal((n, 5))
    rhs = mul(x)
    t = joemi.DeviceArray
    d = [t(v) for v in (ni, nv, A, rhs)]

    def resid(phi):  # the reference's stop measure
        return np.max(np.abs(np.einsum("cij,cj->ci", inv, rhs - mul(phi))))

    # from the near guess 1e-10 would be a residual below 1e-12, where the
    # solver's absolute guards (t.t + 1e-20) stall it
    zero, near = np.zeros((n, 5)), x + 1e-3 * g.standard_normal((n, 5))
    for guess, rels in ((zero, (1e-2, 1e-6, 1e-10)), (near, (1e-2, 1e-6))):
        for rel in rels:
            phi = t(guess)
            it, st = joemi.block_bcgstab(*d, phi, zero_abs=1e-300, zero_rel=rel, max_iter=60)
            assert st == 1 and it >= 1
            # the device's test is taken on this residual up to its rounding
            # (a few dozen sums of terms of size 5: 1e-13)
            assert resid(phi.numpy()) <= rel * (resid(guess) + 1e-12) * (1 + 1e-6) + 1e-13
        phi = t(guess)
        it, st = joemi.block_bcgstab(*d, phi, zero_abs=0.0, zero_rel=1e-30, max_iter=60)
        # stalled by those guards, |t| near 1e-10: at the solution to ten times that
        assert (st == 1 and it <= 60) or (st == 0 and it == 61)  # its limit, not before
        assert np.max(np.abs(phi.numpy() - x)) <= 1e-9 * np.max(np.abs(x))


# the scalar rows per entry (their off-diagonal entries written from the other
# side of each face) against the per-cell form: the segregated SST rows and
# row 5 of the coupled SA blocks (the latter in test_jacobian_... too)
@pytest.mark.parametrize("n,frac", [(1, 1.0), (2, 0.5), (3, 0.0), (5, 0.5), (4, 1.0)])
def test_sst_rows_per_entry_equal_per_cell(n, frac):
    print(f"sst rows n={n} frac={frac}", flush=True)
    mesh, joe = box(n, frac, "HLLC", "sst")
    names = ["ASCAL", "RHS_KINE", "RHS_OMEGA", "A"]
    a = values(mesh, joe + "GPU_SCAL_KERNEL = ENTRY\n", names)
    b = values(mesh, joe + "GPU_SCAL_KERNEL = CELL\n", names)
    for k in names:
        assert np.array_equal(a[k], b[k], equal_nan=True), k


# the gradient per cell and field, the same with the cells in another thread
# order, and the gradient by tiles, against the per-entry form
@pytest.mark.parametrize("grad", ["LEASTSQUARES", "GREENGAUSS"])
@pytest.mark.parametrize("n,frac", [(1, 0.0), (1, 1.0), (2, 0.5), (3, 0.0), (5, 0.5), (4, 1.0), (9, 0.5)])
def test_gradient_forms_agree(n, frac, grad):
    print(f"gradient forms n={n} frac={frac} {grad}", flush=True)
    mesh, joe = box(n, frac, grad=grad)
    names = ["GRAD_RHO", "GRAD_P", "GRAD_U", "ALPHA_RHO", "RHS_RHO", "RHS_RHOU", "RHS_RHOE"]
    ref = values(mesh, joe + "GPU_GRAD_KERNEL = ENTRY\n", names, implicit=False)
    cell = "GPU_GRAD_KERNEL = CELL\n"
    for keys in (cell + "GPU_TILE_KERNELS = NEVER\n", cell + "GPU_TILE_KERNELS = ALWAYS\n",
                 cell + "GPU_TILE_KERNELS = NEVER\nGPU_GRAD_THREAD_ORDER = SORTED\n"):
        got = values(mesh, joe + keys, names, implicit=False)
        for k in names:
            assert np.array_equal(got[k], ref[k], equal_nan=True), k


# the inviscid flux (every option of it, both time steps) by entry, by tiles
# and as the size decides (the last three by tiles) against the per-cell form
@pytest.mark.parametrize("n,frac", [(1, 0.0), (1, 1.0), (2, 0.5), (3, 0.0), (5, 0.5), (4, 1.0), (9, 0.5),
                                    (36, 0.0), (24, 0.5), (20, 1.0)])
@pytest.mark.parametrize("scheme", ["HLLC", "ROE", "AUSM"])
@pytest.mark.parametrize("second", [True, False])
@pytest.mark.parametrize("extra", ["", "TIME_STEP = SUM_BASED\n", "GRAVITY 0.1 -0.2 0.3\n"])
def test_flux_forms_agree(n, frac, scheme, second, extra):
    print(f"flux forms n={n} frac={frac} {scheme} {second} {extra!r}", flush=True)
    mesh, joe = box(n, frac, scheme, second_order=second)
    names = ["RHS_RHO", "RHS_RHOU", "RHS_RHOE", "LOCAL_DT"]
    b = values(mesh, joe + extra + "GPU_FLUX_KERNEL = CELL\n", names, implicit=False)
    for tiles in ("NEVER", "ALWAYS", "AUTO"):
        a = values(mesh, joe + extra + f"GPU_FLUX_KERNEL = ENTRY\nGPU_TILE_KERNELS = {tiles}\n", names, implicit=False)
        for k in names:
            assert np.array_equal(a[k], b[k], equal_nan=True), (tiles, k)


def duplicate_pairs(mm, every=5):
    """Every few internal quadrilaterals as two triangles between the same
    cells: duplicate neighbour pairs."""
    nodes, cells, zone, ptr, quads = [], [], [], [0], 0
    for f in range(mm.nfa):
        parts = [mm.face_nodes[mm.face_ptr[f]:mm.face_ptr[f + 1]]]
        if mm.face_cells[f, 1] >= 0 and len(parts[0]) == 4:
            quads += 1
            if quads % every == 0:
                parts = [parts[0][[0, 1, 2]], parts[0][[0, 2, 3]]]
        for nd in parts:
            nodes.append(nd)
            ptr.append(ptr[-1] + len(nd))
            cells.append(mm.face_cells[f])
            zone.append(mm.face_zone[f])
    mm.face_ptr, mm.face_nodes = np.array(ptr, mm.face_ptr.dtype), np.concatenate(nodes).astype(mm.face_nodes.dtype)
    mm.face_cells, mm.face_zone = np.array(cells, mm.face_cells.dtype), np.array(zone, mm.face_zone.dtype)
    return mm


# the tile forms under every option that reaches them (schemes and the coupled
# flux, both gradients, viscous runs (gradient only), every SYMM_BC, every
# boundary kind, duplicate neighbour pairs): the same bits as without tiles
TILE_FIELDS = ["GRAD_RHO", "GRAD_P", "GRAD_U", "ALPHA_RHO", "RHS_RHO", "RHS_RHOU", "RHS_RHOE", "LOCAL_DT", "FLUX_FA",
               "COUNTERS"]


@pytest.mark.parametrize("n,frac,dup", [(1, 1.0, False), (5, 0.5, False), (13, 0.5, False), (7, 0.0, True),
                                        (9, 0.3, True)])
@pytest.mark.parametrize("kind", ["HLLC", "ROE", "AUSM", "coupled", "laminar", "coupled laminar"])
def test_tile_forms_under_every_option(n, frac, dup, kind):
    print(f"tile forms n={n} frac={frac} dup={dup} {kind}", flush=True)
    mm, _ = cases.box_case(n, frac=frac, seed=n)
    mesh = joemi.Mesh.from_faces(duplicate_pairs(mm) if dup else mm)
    scheme = kind if kind in ("ROE", "AUSM") else "HLLC"
    for grad in ("LEASTSQUARES", "GREENGAUSS"):
        for bcs in (cases.BOX_BCS, cases.BOX_BCS_ALT):
            for symm in ("ORIGINAL_NUMERIC", "NEW_NUMERIC", "ANALYTICAL"):
                for second in (True, False):
                    joe = cases.box_joe_in(scheme, second, grad, bcs=bcs, symm_bc=symm)
                    if "coupled" in kind:
                        joe = cases.coupled(joe, keep_symm_bc=True)
                    names = TILE_FIELDS
                    if "laminar" in kind:
                        joe = joe.replace("MU_REF = 0.0", "MU_REF = 0.01\nMU_MODE = POWERLAW\nMU_POWER_LAW = 0.7")
                        names = names + ["GRAD_ENTHALPY"]
                    a = values(mesh, joe + "GPU_TILE_KERNELS = ALWAYS\n", names, implicit=False)
                    b = values(mesh, joe + "GPU_TILE_KERNELS = NEVER\n", names, implicit=False)
                    for k in names:
                        assert np.array_equal(a[k], b[k], equal_nan=True), (grad, symm, second, k)


def test_duplicate_pairs_match_the_oracle():
    print("duplicate pairs", flush=True)
    for grad in ("LEASTSQUARES", "GREENGAUSS"):
        mm, joe = cases.box_case(5, frac=0.3, seed=2, grad=grad)
        nfa = mm.nfa
        mm = duplicate_pairs(mm)
        assert mm.nfa > nfa
        mesh = joemi.Mesh.from_faces(mm)
        o = Oracle(mesh.as_dump(), joe)
        o.set_state(*cases.random_state(mesh.ncv, 5))
        o.residual(True)
        names = TILE_FIELDS[:-1] + ["A"]
        for tiles in ("ALWAYS", "NEVER"):
            got = values(mesh, joe + f"GPU_TILE_KERNELS = {tiles}\n", names)
            for k in names:
                compare(got[k], o.get(k), 1e-12, f"duplicates:{tiles}:{k}")


def morton(x):
    """21 bits of every coordinate of the centroids, scaled by their largest
    extent, interleaved with x lowest."""
    lo = x.min(0)
    q = (np.minimum((x - lo) / (x.max(0) - lo).max(), 0.99999999) * (1 << 21)).astype(np.uint64)
    key = np.zeros(len(x), np.uint64)
    for b in range(21):
        for i in range(3):
            key |= ((q[:, i] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + i)
    return key


# cells along the Morton curve, equal keys in their own order: either side of
# the size from which the sort goes by digits (65536), with the centroids as
# they are and moved to the corners of an 8^3 grid, so that many share a key
@pytest.mark.parametrize("n,grid", [(2, None), (40, None), (41, None), (40, 8), (41, 8)])
def test_cell_order_is_the_stable_morton_order(n, grid):
    print(f"cell order n={n} grid={grid}", flush=True)
    mm, joe = cases.box_case(n, frac=0.0, seed=n)
    dump = joemi.Mesh.from_faces(mm).as_dump()
    x = dump["X_CV"].reshape(-1, 3)
    if grid:
        x[:] = np.floor(x * grid) / grid
    mesh = joemi.Mesh.from_ugp(dump)
    pos = joemi.Solver(mesh, joe + "GPU_CELL_ORDER = MORTON\n").get("CELL_ORDER").astype(np.int64)
    assert np.array_equal(np.argsort(pos), np.argsort(morton(x[:mesh.ncv]), kind="stable"))
