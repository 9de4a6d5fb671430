"""The pencil sweep against the one-launch-per-hyperplane sweep, through the
C ABI: bit for bit on blocks whose longest axis is i, j or k (the axis the
pencils run along), whose other sides are one cell, a full pencil, or a
remainder, with one and several sweeps, both operator precisions and the
viscous terms; and after the operator precision changes between solves."""
import numpy as np
import pytest

from aither_amd import Solver, cases

pytestmark = pytest.mark.gpu


def run(path, order, precisions):
    s = Solver(path)
    s.set_sweep_ordering(order)
    out = []
    for nn, p in enumerate(precisions):
        s.set_implicit_precision(p)
        s.begin_step(nn)
        n = s.iterate(nn, 0)
        out += [s.update_vector(), np.array(n.l2[:5])]
    out.append(s.get_state())
    s.close()
    return out


@pytest.mark.parametrize("dims", [(31, 8, 9), (9, 33, 16), (8, 17, 40), (1, 1, 5), (7, 1, 2), (8, 8, 8), (25, 24, 23)])
@pytest.mark.parametrize("sweeps,precisions", [(1, (0, 0, 0)), (1, (1, 1, 1)), (2, (0, 0, 0)), (3, (1, 1)),
                                               (1, (0, 1, 0, 0, 1)), (2, (1, 0, 1, 0))])
def test_pencil_equals_hyperplane(tmp_path, dims, sweeps, precisions):
    ni, nj, nk = dims
    path = cases.vortex_case(str(tmp_path), n=max(dims), iterations=4, ni=ni, nj=nj, nk=nk, sweeps=sweeps)
    print("pencil", dims, sweeps, precisions, flush=True)
    a, b = run(path, Solver.PENCIL, precisions), run(path, Solver.HYPERPLANE, precisions)
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("sweeps,precisions", [(1, (0, 0)), (2, (1, 1)), (2, (0, 1, 0))])
def test_viscous_pencil_equals_hyperplane(tmp_path, sweeps, precisions):
    path = cases.bump_case(str(tmp_path), seed=4, n=13, iterations=4, viscous=True, visc_recon="centralFourth")[0]
    text = open(path).read().replace("matrixSweeps: 1", f"matrixSweeps: {sweeps}")
    open(path, "w").write(text)
    print("viscous pencil", sweeps, precisions, flush=True)
    a, b = run(path, Solver.PENCIL, precisions), run(path, Solver.HYPERPLANE, precisions)
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("between", ["state", "level", "order"])
@pytest.mark.parametrize("precision", [0, 1])
def test_changes_between_residual_and_relax(tmp_path, precision, between):
    """The residual stage writes the sweep's inputs; a relax after the state,
    the stored solution or the order changed forms them again."""
    path = cases.vortex_case(str(tmp_path), n=13, iterations=2, ni=21, nj=9, nk=13)
    print("pencil, change before the relax", precision, between, flush=True)
    out = []
    for order in (Solver.PENCIL, Solver.HYPERPLANE):
        s = Solver(path)
        s.set_implicit_precision(precision)
        s.set_sweep_ordering(Solver.TILED if between == "order" else order)
        s.begin_step(0)
        s.assign_ghost_cells()
        s.calc_residual()
        if between == "state":
            s.set_state(1.01 * s.get_state())
        elif between == "level":
            s.relax()
            s.update(0)
            s.begin_step(1)
        s.set_sweep_ordering(order)
        s.relax()
        out.append(s.update_vector())
        s.close()
    assert np.abs(out[0]).max() > 0
    assert np.array_equal(out[0], out[1])
