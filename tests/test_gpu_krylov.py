"""The BiCGStab's residual by its recurrence (GPU_KRYLOV_RESIDUAL =
RECURRENCE, the default): r = s - omega t, where the reference recomputes
rhs - A phi every iteration (UgpWithCv.cpp:2812-2846), one product with A
fewer per iteration. It changes the linear solves' path only: a
mixed-precision steady solve reaches the same steady state as with the true
residual (GPU_KRYLOV_RESIDUAL = TRUE). FP64 solves take it from 16 MB of A on
and confirm the stop test on the true residual; smaller ones take the
reference's form whatever the key says."""
import numpy as np
import pytest

from myjoe_amd import cases, joemi

pytestmark = pytest.mark.gpu


def test_recurrence_residual_reaches_the_same_steady_state():
    print("krylov recurrence steady", flush=True)
    mm, joe = cases.bump_case(24, 8, nsteps=1200)
    mesh = joemi.Mesh.from_faces(mm)
    states = []
    for text in (joe + "GPU_KRYLOV_RESIDUAL = TRUE\n", joe):
        s = joemi.Solver(mesh, text, joemi.JM_MIXED)
        s.init_uniform()
        n, hist = s.run(1200)
        assert hist[-1, 4] < 1e-6 * hist[0, 4]
        states.append(s.state())
    for a, b, k in zip(states[0], states[1], ("rho", "rhou", "rhoE")):
        d = float(np.max(np.abs(a - b)) / np.max(np.abs(a)))
        print("recurrence steady", k, f"{d:.1e}", flush=True)
        assert d <= 1e-8, (k, d)


def test_recurrence_key_leaves_the_fp64_solve_alone():
    # 192 cells: below the size from which FP64 solves take the recurrence
    mm, joe = cases.bump_case(24, 8, nsteps=5)
    mesh = joemi.Mesh.from_faces(mm)
    out = []
    for text in (joe + "GPU_KRYLOV_RESIDUAL = TRUE\n", joe):
        s = joemi.Solver(mesh, text, joemi.JM_FP64)
        s.init_uniform()
        s.run(5)
        out.append(s.state())
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)


def test_batched_server_takes_the_recurrence_for_fp32_solves():
    # the batched FP32 BiCGStab takes the recurrence: a mixed request asking
    # for the true residual is refused, an FP64 one served
    mm, joe = cases.bump_case(24, 8, nsteps=5)
    mesh = joemi.Mesh.from_faces(mm)
    srv = joemi.Server(1 << 30, 2, batched=True)
    with pytest.raises(joemi.JoemiError) as e:
        srv.submit(mesh, joe + "GPU_KRYLOV_RESIDUAL = TRUE\n", joemi.JM_MIXED)
    assert e.value.status == 5 and "RECURRENCE" in str(e.value)
    t = srv.submit(mesh, joe + "GPU_KRYLOV_RESIDUAL = TRUE\n", joemi.JM_FP64)
    srv.wait(t)
    srv.release(t)
    srv.close()


# FP64 solves of 16 MB and more take the recurrence's residual and confirm the
# stop test on the true one. A tolerance the confirmation passes at once, two
# near the rounding of the true residual, where the recurrence meets the test
# and the confirmation fails and the chunk's other launches do nothing, and
# limits that are reached before: the ordinary step, the graph step and both
# servers do the same iterations, and a solve that does not converge ends at
# its limit, not before. (The geometry is scaled so that the solver's absolute
# guards, 1e-20 beside t.t, lie below the rounding.)
@pytest.mark.parametrize("max_iter,rel", [(30, 1e-2), (60, 1e-15), (60, 3e-16), (7, 1e-12), (1, 1e-2), (0, 1e-2)])
def test_confirmed_solves_end_at_the_same_iteration(max_iter, rel):
    print(f"confirmed solves {max_iter} {rel}", flush=True)
    n = 3
    mm, joe = cases.bump_case(240, 80, nsteps=n, ls=f"MAX_ITER={max_iter} ABS_RESID=1.0e-300 REL_RESID={rel}")
    mm.x_no *= 1e4
    mesh = joemi.Mesh.from_faces(mm)
    info, state = [], []
    for graph in (False, True):
        s = joemi.Solver(mesh, joe)
        s.init_uniform()
        steps = [s.step_graph() if graph else s.step() for _ in range(n)]
        info.append([(i.lin_iters, i.lin_status, list(i.resid)) for i in steps])
        state.append(s.state())
    print(info[0], flush=True)
    assert info[0] == info[1]
    for it, st, _ in info[0]:
        # a solve at its limit has counted one iteration more (limit 0: one is done)
        assert st == 1 or (st == 0 and it == max_iter + 1) or (st == 2 and max_iter == 0 and it == 1)
    for batched in (False, True):
        srv = joemi.Server(1 << 30, 2, batched=batched)
        t = srv.submit(mesh, joe)
        srv.wait(t)
        st, rep = srv.result(t)
        assert rep.status == joemi.Server.DONE and rep.steps == n and list(rep.resid) == info[0][-1][2]
        state.append(st)
        srv.release(t)
        srv.close()
    for other in state[1:]:
        for a, b in zip(state[0], other):
            assert np.array_equal(a, b)


# above that size the key decides: TRUE is the reference's form in every kind
# of step, so its iterates part from the recurrence's by rounding (a tolerance
# that takes some twenty iterations), and only by that
def test_fp64_solves_take_the_true_residual_when_asked():
    print("fp64 true residual", flush=True)
    mm, joe = cases.bump_case(240, 80, nsteps=2, ls="MAX_ITER=60 ABS_RESID=1.0e-300 REL_RESID=1e-11")
    mm.x_no *= 1e4
    mesh = joemi.Mesh.from_faces(mm)
    out = {}
    for text in (joe + "GPU_KRYLOV_RESIDUAL = TRUE\n", joe):
        states = []
        for graph in (False, True):
            s = joemi.Solver(mesh, text)
            s.init_uniform()
            for _ in range(2):
                info = s.step_graph() if graph else s.step()
                assert info.lin_status == 1 and info.lin_iters > 10
            states.append(s.state())
        srv = joemi.Server(1 << 30, 2, batched=True)
        t = srv.submit(mesh, text)
        srv.wait(t)
        states.append(srv.result(t)[0])
        srv.release(t)
        srv.close()
        for other in states[1:]:
            for a, b in zip(states[0], other):
                assert np.array_equal(a, b)
        out[text] = np.concatenate([np.ravel(x) for x in states[0]])
    a, b = out.values()
    d = np.max(np.abs(a - b)) / np.max(np.abs(a))
    print(f"true against recurrence {d:.1e}", flush=True)
    # both stop on a true residual 1e-11 below the first
    assert 0.0 < d <= 1e-10
