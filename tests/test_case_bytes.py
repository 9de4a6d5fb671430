"""Device memory of a case: the sweep's arrays of blocks thinner than a pencil
against the same case without a sweep, and what admission reserves against what
the case then holds."""
import pytest

from aither_amd import Server, cases


def vortex(tmp_path, dims, solver, sweeps=1):
    ni, nj, nk = dims
    return cases.vortex_case(str(tmp_path), n=max(dims), iterations=4, ni=ni, nj=nj, nk=nk, solver=solver, sweeps=sweeps)


# the sweep's arrays (40 doubles a cell with the scalar solver) take about as much
# as all others, in steps of a power of two of lanes, so a thin block's share is
# that of a cube within the rounding (the Jacobi solver has every array but those)
@pytest.mark.parametrize("dims", [(128, 128, 1), (128, 1, 128), (1, 128, 128), (128, 96, 2), (96, 3, 128), (5, 128, 96),
                                  (1, 1, 512), (512, 1, 1), (48, 48, 48)])
@pytest.mark.parametrize("sweep,jacobi", [("lusgs", "dplur"), ("blusgs", "bdplur")])
@pytest.mark.parametrize("precision", [0, 1])
def test_sweep_arrays_of_thin_blocks(tmp_path, dims, sweep, jacobi, precision):
    fixed = Server.estimate(vortex(tmp_path, (1, 1, 2), jacobi), precision)
    a = Server.estimate(vortex(tmp_path, dims, sweep), precision) - fixed
    b = Server.estimate(vortex(tmp_path, dims, jacobi), precision) - fixed
    print(dims, sweep, precision, a, b, a / b, flush=True)
    assert a <= 2.5 * b


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(65, 33, 1), (33, 1, 65), (1, 65, 33), (40, 3, 40), (21, 22, 23), (1, 1, 200)])
@pytest.mark.parametrize("solver,sweeps", [("lusgs", 1), ("lusgs", 2), ("blusgs", 1), ("blusgs", 2), ("dplur", 1),
                                           ("bdplur", 2)])
@pytest.mark.parametrize("precision", [0, 1])
def test_admission_reserves_what_a_case_holds(tmp_path, dims, solver, sweeps, precision):
    path = vortex(tmp_path, dims, solver, sweeps)
    print("case bytes", dims, solver, sweeps, precision, flush=True)
    with Server(max_slots=2, precision=precision) as srv:
        slot = srv.admit(path, 1e-200, 10)
        assert srv.info(slot).device_bytes <= Server.estimate(path, precision)
