"""Device memory of a case: the sweep's arrays of blocks thinner than a pencil
against the same case without a sweep, and what admission reserves against what
the case then holds."""
import numpy as np
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


@pytest.mark.gpu
@pytest.mark.parametrize("solver,sweeps", [("lusgs", 1), ("lusgs", 2), ("blusgs", 1), ("blusgs", 2)])
@pytest.mark.parametrize("precision", [0, 1])
def test_case_too_large_with_the_sweep_arrays(tmp_path, solver, sweeps, precision):
    """Four fifths of a case's bytes are enough without the pencil sweep's
    arrays: an empty server takes it so, alone and with a small case beside it,
    and both end as with the arrays."""
    for d in ("a", "b"):
        (tmp_path / d).mkdir()
    large, small = vortex(tmp_path / "a", (33, 32, 31), solver, sweeps), vortex(tmp_path / "b", (5, 6, 4), solver, sweeps)
    need = Server.estimate(large, precision)
    budget = 0.8 * need
    print("too large with the arrays", solver, sweeps, precision, need, budget, flush=True)
    out = []
    for b in (0.0, budget):
        with Server(max_slots=4, precision=precision, hbm_budget=b) as srv:
            first = srv.admit(large, 1e-200, 2 ** 30)
            assert first is not None
            if b:
                assert srv.info(first).device_bytes <= srv.memory()[0] <= budget
                # the same again does not fit beside it, with or without them
                assert srv.admit(large, 1e-200, 2 ** 30) is None
            srv.step(3)
            W = [srv.state(first)]
            second = srv.admit(small, 1e-200, 2 ** 30)
            assert second is not None
            srv.step(2)
            W += [srv.state(first), srv.state(second)]
            srv.retire(first)  # the small case alone, with the arrays
            srv.step(2)
            out.append(W + [srv.state(second)])
    assert all(np.array_equal(x, y) for x, y in zip(*out))
