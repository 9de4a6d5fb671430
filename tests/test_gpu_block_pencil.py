"""The block LU-SGS pencil sweep against the one-launch-per-hyperplane sweep,
through the C ABI, bit for bit: blocks whose longest axis is i, j or k (the
axis the pencils run along, and the split of the block diagonal's tiles),
whose other sides are one cell, a full pencil or a remainder; one and several
sweeps, both operator precisions and changes between them, the viscous terms;
the two block pencil orders; and a state set between the residual and the
relax."""
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


def same(path, precisions):
    a, b = run(path, Solver.PENCIL, precisions), run(path, Solver.HYPERPLANE, precisions)
    assert np.abs(a[0]).max() > 0
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("dims", [(35, 8, 9), (9, 33, 16), (8, 17, 40), (33, 7, 1), (7, 1, 2), (8, 8, 8), (25, 24, 23)])
@pytest.mark.parametrize("sweeps,precisions", [(1, (0, 0)), (1, (1, 1)), (2, (0, 0)), (3, (1, 1)), (1, (0, 1, 0)),
                                               (2, (1, 0, 1))])
def test_block_pencil_equals_hyperplane(tmp_path, dims, sweeps, precisions):
    ni, nj, nk = dims
    path = cases.vortex_case(str(tmp_path), n=max(dims), iterations=4, ni=ni, nj=nj, nk=nk, sweeps=sweeps,
                             solver="blusgs")
    print("block pencil", dims, sweeps, precisions, flush=True)
    same(path, precisions)


@pytest.mark.parametrize("recon", ["central", "centralFourth"])
@pytest.mark.parametrize("sweeps,precisions", [(1, (0, 0)), (1, (1, 1)), (2, (0, 1, 0))])
def test_viscous_block_pencil_equals_hyperplane(tmp_path, recon, sweeps, precisions):
    path = cases.bump_case(str(tmp_path), seed=4, n=13, iterations=4, viscous=True, visc_recon=recon)[0]
    text = open(path).read().replace("matrixSweeps: 1", f"matrixSweeps: {sweeps}")
    open(path, "w").write(text.replace("matrixSolver: lusgs", "matrixSolver: blusgs"))
    print("viscous block pencil", recon, sweeps, precisions, flush=True)
    same(path, precisions)


@pytest.mark.parametrize("solver", ["vortex", "channel"])
def test_state_set_between_residual_and_relax(tmp_path, solver):
    """The relax uses the state as it is then (the viscous stage of the FP64
    operator hands its right-hand side on, so the channel runs FP32)."""
    if solver == "vortex":
        path, precision = cases.vortex_case(str(tmp_path), n=11, iterations=2, solver="blusgs"), 0
    else:
        path, precision = cases.channel_case(str(tmp_path), refine=0.125, steps=1, subits=2)[0], 1
    print("state set before the relax", solver, flush=True)
    out = []
    for order in (Solver.ROWS, Solver.HYPERPLANE):
        s = Solver(path)
        s.set_sweep_ordering(order)
        s.set_implicit_precision(precision)
        s.begin_step(0)
        s.assign_ghost_cells()
        s.calc_residual()
        for b in range(s.info.num_blocks):
            s.set_state(1.01 * s.get_state(b), b)
        s.relax()
        out.append([s.update_vector(b) for b in range(s.info.num_blocks)])
        s.close()
    assert np.abs(out[0][0]).max() > 0
    assert all(np.array_equal(x, y) for x, y in zip(*out))
