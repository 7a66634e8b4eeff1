"""The device kernels' forms held to each other at the sizes where a form can
go wrong: the last, partly filled wavefront or tile, cells of every face
count, the smallest meshes, both precisions. Where both forms add the same
terms in the same order the bar is equality."""
import numpy as np
import pytest

from myjoe_amd import cases, joemi

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
