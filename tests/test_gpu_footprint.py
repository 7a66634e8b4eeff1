"""jm_ctx_footprint and the server's admission count against the bytes that a
context's buffers hold after a step, for the options that add buffers: neither
may be less, or the server admits past the budget it was given."""
import pytest

from myjoe_amd import cases, joemi

pytestmark = pytest.mark.gpu

LAMINAR = ("MU_REF = 0.0", "MU_REF = 0.01\nMU_MODE = POWERLAW\nMU_POWER_LAW = 0.7")
# name: (gradient, the Joe.in's change, added keys)
OPTIONS = {
    "inviscid": ("LEASTSQUARES", None, ""),
    "greengauss": ("GREENGAUSS", None, ""),
    "tiles": ("GREENGAUSS", None, "GPU_TILE_KERNELS = ALWAYS\n"),
    "face": ("LEASTSQUARES", None, "GPU_FLUX_KERNEL = FACE\nGPU_GRAD_THREAD_ORDER = SORTED\n"),
    "sum": ("LEASTSQUARES", None, "TIME_STEP = SUM_BASED\n"),
    "laminar": ("LEASTSQUARES", LAMINAR, ""),
    "laminar greengauss": ("GREENGAUSS", LAMINAR, "TIME_STEP = SUM_BASED\nGPU_TILE_KERNELS = ALWAYS\n"),
    "ilu": ("LEASTSQUARES", None, "GPU_PRECONDITIONER = ILU0\n"),
    "sa": ("LEASTSQUARES", LAMINAR, "sa"),
    "coupled sa": ("GREENGAUSS", LAMINAR, "coupled sa"),
    "sst": ("GREENGAUSS", LAMINAR, "sst"),
}


@pytest.mark.parametrize("precision", [joemi.JM_FP64, joemi.JM_MIXED])
@pytest.mark.parametrize("n,frac", [(6, 0.5), (19, 0.5), (27, 0.0), (16, 1.0)])
def test_footprint_covers_what_a_context_holds(n, frac, precision):
    for name, (grad, change, extra) in OPTIONS.items():
        print(f"footprint n={n} frac={frac} precision={precision} {name}", flush=True)
        mm, joe = cases.box_case(n, frac=frac, seed=n, grad=grad)
        joe = joe.replace("NSTEPS = 10", "NSTEPS = 1")
        if change:
            joe = joe.replace(*change)
        if "coupled" in extra:
            joe = cases.coupled(joe)
        if "sa" in extra.split():
            joe = cases.with_sa(joe, 0.006, cases.SA_BOX)
        elif extra == "sst":
            joe = cases.with_sst(joe, 0.001, 5.0, cases.SST_BOX)
        else:
            joe += extra
        mesh = joemi.Mesh.from_faces(mm)
        s = joemi.Solver(mesh, joe, precision)
        s.init_uniform()
        s.step()
        held = int(s.get("DEVICE_BYTES")[0])
        del s
        turbulent = name.endswith(("sa", "sst"))
        if name != "ilu" and not turbulent:
            assert held <= mesh.footprint(precision)
        # a server refuses a request that holds more than its budget
        srv = joemi.Server(held - 1, 1)
        with pytest.raises(joemi.JoemiError) as e:
            srv.submit(mesh, joe, precision)
        assert "budget" in str(e.value)
        srv.close()
        if turbulent or name == "ilu":  # not in graph steps
            continue
        # and charges no more than the tiles' bound and the constant above it
        srv = joemi.Server(int(1.06 * held) + (2 << 20), 1)
        t = srv.submit(mesh, joe, precision)
        srv.wait(t)
        assert srv.result(t)[1].status == joemi.Server.DONE
        srv.release(t)
        srv.close()


def test_a_context_keeps_no_lists_for_kernels_it_does_not_run():
    print("lists kept", flush=True)

    def held(n, joe):
        mesh = joemi.Mesh.from_faces(cases.box_case(n, frac=0.5, seed=n)[0])
        return mesh, int(joemi.Solver(mesh, joe).get("DEVICE_BYTES")[0])

    joe = cases.box_joe_in("HLLC")
    never, always = "GPU_TILE_KERNELS = NEVER\n", "GPU_TILE_KERNELS = ALWAYS\n"
    for text in (joe, joe.replace(*LAMINAR)):  # a mesh too small for tiles
        assert held(9, text)[1] == held(9, text + never)[1] < held(9, text + always)[1]
    # a mesh that takes them: a viscous run keeps no face evaluations (16
    # bytes each, at least two per cell), nor does the per-cell flux
    mesh, flux = held(26, joe)
    rest = held(26, joe + never)[1]
    assert flux - rest > 32 * mesh.ncv
    for text in (joe.replace(*LAMINAR), joe + "GPU_FLUX_KERNEL = CELL\n"):
        assert 0 < held(26, text)[1] - held(26, text + never)[1] < 32 * mesh.ncv
