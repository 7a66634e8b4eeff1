"""runBackwardEulerCoupled (TIME_INTEGRATION = BACKWARD_EULER_COUPLED), HLLC,
inviscid, laminar, and with the Spalart-Allmaras scalar in 6x6 blocks:
calcRhsCoupled's residual and Jacobian blocks (JoeWithModels.cpp:4596-5825,
UgpWithCvCompFlow.cpp:1808-2287, 3040-3274; TurbModel_SA.h:359-434).

Pinned against the reference's own calcRhsCoupled (tests/golden/coupled_*.npz,
written by make_golden.py through the harness's rhs-coupled mode). The
reference's coupled loop solves with PETSc GMRES, absent here; this build
runs the same loop with its block-Jacobi BiCGStab, so the loop is pinned by
what the mathematics fixes: the coupled and segregated fluxes are the same
function written two ways (h = gamma R T / (gamma - 1) with T = p / (rho R)
against gamma / (gamma - 1) p / rho), so both loops reach the same steady
state.
"""
import glob
import os

import numpy as np
import pytest

from myjoe_amd import cases, joemi
from tests.test_oracle_golden import GOLD, joe_text, load, mesh_for, parse_joe_in

COUPLED = sorted(os.path.basename(p)[:-4] for p in glob.glob(os.path.join(GOLD, "coupled_*.npz")))
FIELDS = ["PRESS", "VEL", "RHO_BFA", "VEL_BFA", "P_BFA", "T_BFA", "H_BFA", "LOCAL_DT", "GRAD_RHO", "GRAD_P",
          "GRAD_U", "RHS_RHO", "RHS_RHOU", "RHS_RHOE", "A"]
VISC_FIELDS = ["GRAD_ENTHALPY", "MUL_FA"]
# with the Spalart-Allmaras scalar in the coupled system (6x6 blocks): its
# residual row, boundary values, limited gradient, diffusivity, eddy
# viscosity and model fields
SA_FIELDS = ["RHS_NUSA", "NUSA_BFA", "GRAD_NUSA", "DIFF_NUSA", "MUT_FA", "WALL_DIST", "STR_MAG", "VORT_MAG"]


def _mesh_key(fixture):
    return fixture[len("coupled_"):]


def test_coupled_fixture_set_complete():
    # both geometries, every SYMM_BC mode (and the key absent), every boundary
    # kind the coupled face loop distinguishes, Green-Gauss, first order
    assert len(COUPLED) >= 6
    kinds, symm = set(), set()
    for f in COUPLED:
        P = parse_joe_in(joe_text(load(f)))
        assert P["TIME_INTEGRATION"][0][1] == "BACKWARD_EULER_COUPLED"
        for z in ("inlet", "outlet", "wall", "farfield", "symm", "bump_wall", "top", "zsym"):
            if z in P:
                kinds.add(P[z][0][1])
        symm.add(P["SYMM_BC"][0][1] if "SYMM_BC" in P else None)
    assert kinds >= {"CBC", "CBC_SUBSONIC_INLET", "CBC_SUBSONIC_OUTLET", "WALL", "FARFIELD", "NEUMANN", "SYMMETRY"}
    assert symm == {None, "ORIGINAL_NUMERIC", "NEW_NUMERIC", "ANALYTICAL"}
    assert any("first" in f for f in COUPLED) and any("gg" in f for f in COUPLED)
    assert any("bump" in f for f in COUPLED)
    # laminar: both viscosity laws, first order, the alternate boundary kinds
    visc = [f for f in COUPLED if "visc" in f]
    assert any("_pl" in f for f in visc) and any("_su" in f for f in visc)
    assert any("first" in f for f in visc) and any("alt" in f for f in visc)


@pytest.mark.parametrize("fixture", COUPLED)
def test_oracle_coupled_bit_exact(fixture):
    from oracle.oracle import Oracle

    g = load(fixture)
    o = Oracle(mesh_for(_mesh_key(fixture)), joe_text(g))
    o.set_state(g["RHO"], g["RHOU"], g["RHOE"])
    sa = "_sa" in fixture
    if sa:
        o.set_scalar(g["NUSA"])
    o.residual(True)
    for k in FIELDS + (VISC_FIELDS if "visc" in fixture else []) + (SA_FIELDS if sa else []):
        if k not in g:
            assert "first" in fixture and k.startswith("GRAD"), k
            continue
        got = o.get(k)
        assert got.shape == g[k].shape, k
        nbad = int(np.sum(got != g[k]))
        assert nbad == 0, f"{fixture}:{k}: {nbad} of {got.size} differ"


def test_coupled_forms_differ_from_segregated_by_rounding_only():
    # the same state through the segregated restatement: residuals agree to
    # rounding (the two energy forms are one function), but not bit for bit,
    # and the Jacobians differ in the last bits too (so a coupled path that
    # fell back to the segregated forms fails the bit-exact test above)
    from oracle.oracle import Oracle

    g = load("coupled_box4_hllc")
    seg = joe_text(g).replace("BACKWARD_EULER_COUPLED", "BACKWARD_EULER").replace("PETSC_GMRES", "BCGSTAB")
    o = Oracle(mesh_for("box4_hllc"), seg)
    o.set_state(g["RHO"], g["RHOU"], g["RHOE"])
    o.residual(True)
    for k in ("RHS_RHO", "RHS_RHOU", "RHS_RHOE", "A"):
        a, b = o.get(k), g[k]
        scale = np.max(np.abs(b))
        assert np.max(np.abs(a - b)) <= 1e-12 * scale, k
    assert not np.array_equal(o.get("RHS_RHOE"), g["RHS_RHOE"])
    assert not np.array_equal(o.get("A"), g["A"])


def _bump_pair(nsteps):
    mm, joe = cases.bump_case(24, 8, nsteps=nsteps)
    return mm, joe, cases.coupled(joe)


def _uniform(ncv):
    # the bump's initial condition: rho = p = 1, u = (U_BUMP, 0, 0)
    u = cases.U_BUMP
    rhou = np.zeros((ncv, 3))
    rhou[:, 0] = u
    return np.ones(ncv), rhou, np.full(ncv, 1.0 / 0.4 + 0.5 * u * u)


def test_coupled_loop_reaches_the_segregated_steady_state():
    # both loops run to the L1 floor on the bump; the steady state is the
    # discretisation's, which the two flux forms share
    from oracle.oracle import Oracle

    mm, seg, cpl = _bump_pair(1200)
    mesh = joemi.Mesh.from_faces(mm)
    states = []
    for joe in (seg, cpl):
        o = Oracle(mesh.as_dump(), joe)
        o.set_state(*_uniform(mesh.ncv))
        n, hist = o.run(1200)
        assert hist[-1, 4] < 1e-6 * hist[0, 4]
        states.append(o.state())
    for a, b, k in zip(states[0], states[1], ("rho", "rhou", "rhoE")):
        assert np.max(np.abs(a - b)) <= 1e-8 * np.max(np.abs(a)), k


@pytest.mark.parametrize("edit,needle", [
    (lambda s: s.replace("SPACE_INTEGRATION = HLLC", "SPACE_INTEGRATION = ROE"), "HLLC only"),
    (lambda s: s + "GPU_FLUX_KERNEL = CELL\n", "GPU_FLUX_KERNEL"),
    (lambda s: s.replace("PETSC_GMRES", "LU"), "LINEAR_SOLVER_NS"),
])
def test_coupled_input_checked_before_device(edit, needle):
    mm, joe = cases.box_case(2, seed=0)
    mesh = joemi.Mesh.from_faces(mm)
    with pytest.raises(joemi.JoemiError) as e:
        joemi.Solver(mesh, edit(cases.coupled(joe)))
    assert e.value.status == 5, str(e.value)
    assert needle in str(e.value)


# the SA fields the device keeps (MUT_FA and DIFF_NUSA are formed per face
# where they are used, and pinned through the residual and the blocks)
SA_DEVICE_FIELDS = ["RHS_NUSA", "NUSA_BFA", "GRAD_NUSA", "WALL_DIST", "STR_MAG", "VORT_MAG"]


@pytest.mark.gpu
@pytest.mark.parametrize("fixture", COUPLED)
def test_gpu_coupled_matches_reference(fixture):
    # the HIP path against calcRhsCoupled's outputs, at the residual bar of
    # the segregated fixtures (1e-12 relative); with SA, A is [nnz][6][6]
    from tests.helpers import compare
    from tests.test_mesh_golden import MESHES

    print(f"coupled {fixture}", flush=True)
    g = load(fixture)
    mesh = joemi.Mesh.from_faces(MESHES[_mesh_key(fixture).split("_")[0]]())
    sa = "_sa" in fixture
    exact = total = 0
    for extra in ("", "GPU_TILE_KERNELS = ALWAYS\n"):  # by size, and by tiles
        s = joemi.Solver(mesh, joe_text(g) + extra)
        s.set_state(g["RHO"], g["RHOU"], g["RHOE"])
        if sa:
            s.set_scalar(g["NUSA"])
        s.calc_rhs(True)
        for k in FIELDS + (["GRAD_ENTHALPY", "MUL_FA"] if "visc" in fixture else []) + \
                (SA_DEVICE_FIELDS + ["MUT_FA"] if sa else []):
            if k not in g:
                continue
            e, n = compare(s.get(k), g[k], 1e-12, f"{fixture}:{extra.strip()}:{k}")
            exact += e
            total += n
    print(f"{fixture}: {exact}/{total} bit-exact")


@pytest.mark.gpu
@pytest.mark.parametrize("visc", [False, True])
def test_gpu_coupled_steps_track_oracle(visc):
    # the coupled loop on the device against the oracle's, 40 steps (the
    # trajectory bars of the segregated loop: L1 history 1e-7, state 1e-9)
    from oracle.oracle import Oracle
    from tests.helpers import compare

    print(f"coupled steps visc={visc}", flush=True)
    mm, _, cpl = _bump_pair(40)
    if visc:
        cpl = cpl.replace("MU_REF = 0.0", "MU_REF = 0.002\nMU_MODE = POWERLAW")
    mesh = joemi.Mesh.from_faces(mm)
    o = Oracle(mesh.as_dump(), cpl)
    s = joemi.Solver(mesh, cpl)
    o.set_state(*_uniform(mesh.ncv))
    s.set_state(*_uniform(mesh.ncv))
    n_o, hist_o = o.run(40)
    n_g, hist_g = s.run(40)
    assert n_o == n_g == 40
    compare(hist_g, hist_o, 1e-7, "coupled L1 history")
    for a, b, k in zip(s.state(), o.state(), ("rho", "rhou", "rhoE")):
        compare(a, b, 1e-9, k)


@pytest.mark.gpu
def test_gpu_coupled_graph_step_equals_eager_step():
    print("coupled graph step", flush=True)
    mm, _, cpl = _bump_pair(10)
    mesh = joemi.Mesh.from_faces(mm)
    a = joemi.Solver(mesh, cpl)
    b = joemi.Solver(mesh, cpl)
    a.init_uniform()
    b.init_uniform()
    for k in range(10):
        ia, ib = a.step(), b.step_graph()
        assert list(ia.resid) == list(ib.resid), k
    for x, y in zip(a.state(), b.state()):
        assert np.array_equal(x, y)


def _sa_bump(nsteps):
    mm, joe = cases.bump_case(24, 8, nsteps=nsteps)
    visc = "MU_REF = 0.002\nMU_MODE = POWERLAW\nMU_POWER_LAW = 0.76\nPR = 0.72"
    return mm, cases.coupled(cases.with_sa(joe.replace("MU_REF = 0.0", visc), 0.006, cases.SA_BUMP))


def test_oracle_coupled_sa_converges():
    # the coupled loop with the scalar on the bump: the energy residual falls
    # by 1e-8 and nuSA stays inside the model's clip bounds
    from oracle.oracle import Oracle

    mm, joe = _sa_bump(1200)
    mesh = joemi.Mesh.from_faces(mm)
    o = Oracle(mesh.as_dump(), joe)
    o.set_state(*_uniform(mesh.ncv))
    n, hist = o.run(1200)
    assert n == 1200 and hist.shape[1] == 6
    assert hist[-1, 4] < 1e-7 * hist[0, 4]
    assert hist[-1, 5] < 1e-7 * hist[0, 5]
    nu = o.get("NUSA")
    assert np.all(nu >= 1e-10) and np.all(nu <= 1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [joemi.JM_FP64, joemi.JM_MIXED])
def test_gpu_coupled_sa_steps_track_oracle(precision):
    # 40 coupled steps with the scalar in the 6x6 system. FP64: the
    # trajectory bars of the segregated loop (L1 history 1e-7, state 1e-9);
    # mixed (FP32 blocks, preconditioner and Krylov) follows a different
    # inexact-Newton path, so only its L1 history is held, loosely
    from oracle.oracle import Oracle
    from tests.helpers import compare

    print(f"coupled SA steps precision={precision}", flush=True)
    mm, joe = _sa_bump(40)
    mesh = joemi.Mesh.from_faces(mm)
    o = Oracle(mesh.as_dump(), joe)
    s = joemi.Solver(mesh, joe, precision)
    o.set_state(*_uniform(mesh.ncv))
    s.init_uniform()
    n_o, hist_o = o.run(40)
    n_g, hist_g = s.run(40)
    assert n_o == n_g == 40
    if precision == joemi.JM_FP64:
        compare(hist_g[:, :5], hist_o[:, :5], 1e-7, "coupled SA L1 history")
        for a, b, k in zip(s.state(), o.state(), ("rho", "rhou", "rhoE")):
            compare(a, b, 1e-9, k)
        compare(s.get("NUSA"), o.get("NUSA"), 1e-9, "nuSA")
    else:
        compare(hist_g[:, 4], hist_o[:, 4], 1e-2, "coupled SA mixed energy L1")


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [joemi.JM_FP64, joemi.JM_MIXED])
def test_gpu_coupled_sa_steady_state_matches_oracle(precision):
    # both precisions reach the oracle's coupled steady state to 1e-8 of each
    # variable's largest magnitude; in the coupled system nuSA converges with
    # the mean flow (no scalar-solve stop band), so it is held to the same bar
    from oracle.oracle import Oracle

    print(f"coupled SA steady precision={precision}", flush=True)
    nsteps = 1500
    mm, joe = _sa_bump(nsteps)
    mesh = joemi.Mesh.from_faces(mm)
    o = Oracle(mesh.as_dump(), joe)
    o.set_state(*_uniform(mesh.ncv))
    n, rhist = o.run(nsteps)
    assert rhist[-1, 4] < 1e-7 * rhist[0, 4]
    s = joemi.Solver(mesh, joe, precision)
    s.init_uniform()
    n_g, hist = s.run(nsteps)
    assert n_g == nsteps
    ref = dict(zip(("rho", "rhou", "rhoE"), o.state()))
    ref["nuSA"] = o.get("NUSA")
    got = dict(zip(("rho", "rhou", "rhoE"), s.state()))
    got["nuSA"] = s.get("NUSA")
    worst = {k: float(np.max(np.abs(got[k] - b)) / np.max(np.abs(b))) for k, b in ref.items()}
    print("coupled SA steady", precision, {k: f"{v:.1e}" for k, v in worst.items()}, flush=True)
    for k, v in worst.items():
        assert v <= 1e-8, (precision, k, v)
