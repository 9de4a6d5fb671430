"""The block LU-SGS pencil sweep against the one-launch-per-hyperplane sweep,
through the C ABI, bit for bit, where a pencil meets a connection or a viscous
term: blocks joined in rotated orientations (each axis the longest of some
block, cut faces on both sides of both cut axes and at the pencils' ends), a
spanwise periodic channel of eight blocks, viscous blocks whose pencils run
along i, j or k and whose other axes are one cell, a full pencil or a remainder;
one and several sweeps, both operator precisions."""
import os

import numpy as np
import pytest

from aither_amd import Solver, cases
import conn_cases as cc

pytestmark = pytest.mark.gpu


def run(path, order, precision, steps, subits=1):
    s = Solver(path)
    s.set_implicit_precision(precision)
    s.set_sweep_ordering(order)
    out = []
    for nn in range(steps):
        s.begin_step(nn)
        for mm in range(subits):
            n = s.iterate(nn, mm)
            out.append(np.array(list(n.l2[:5]) + [n.linf, n.matrix_resid]))
    out += [f(b) for b in range(s.info.num_blocks) for f in (s.update_vector, s.get_state)]
    s.close()
    return out


def same(path, precision, steps=3, subits=1):
    a, b = (run(path, o, precision, steps, subits) for o in (Solver.PENCIL, Solver.HYPERPLANE))
    assert np.abs(a[-2]).max() > 0
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


# the cut normal to a block's longest axis, or along it, on blocks with full
# and partial pencils
@pytest.mark.parametrize("n,cut", [((6, 5, 8), 4), ((9, 5, 22), 17), ((19, 9, 8), 3)])
@pytest.mark.parametrize("q", [0, 97, 211, 350, 463, 575])
@pytest.mark.parametrize("eq", ["euler", "navierStokes"])
@pytest.mark.parametrize("sweeps,precision", [(1, 0), (1, 1), (2, 0), (2, 1)])
def test_connections(tmp_path, n, cut, q, eq, sweeps, precision):
    r0, r1 = cc.orientation_set()[q]
    path, _ = cc.write_pair(str(tmp_path), "cut", r0, r1, cut=cut, n=n, timeint="implicitEuler", eq=eq,
                            scale=1e-3 if eq == "navierStokes" else 1.0, solver="blusgs", sweeps=sweeps)
    print("block orders, connection", n, cut, q, eq, sweeps, precision, flush=True)
    same(path, precision)


@pytest.mark.parametrize("sweeps,precision", [(1, 0), (1, 1), (2, 0), (2, 1)])
def test_channel(tmp_path, sweeps, precision):
    path = cases.channel_case(str(tmp_path), refine=0.25, steps=2, subits=3, sweeps=sweeps)[0]
    print("block orders, channel", sweeps, precision, flush=True)
    same(path, precision, steps=2, subits=3)


def write_plate(outdir, dims, wall, sweeps, solver="blusgs"):
    """A laminar box of `dims` cells with a no-slip wall on the lower face of
    axis `wall`, free stream along the other two"""
    ni, nj, nk = dims
    i, j, k = np.meshgrid(*[np.arange(n + 1) for n in dims], indexing="ij")
    h = 2e-5
    x, y, z = h * i, h * (j + 0.01 * j * j), h * (k + 0.1 * np.sin(0.4 * i))
    cases.write_plot3d(os.path.join(outdir, "plate.xyz"), [(x, y, z)])
    xc, yc, zc = cases.cell_centres(x, y, z)
    s = 1.0 / (h * max(dims))
    rho, u, v, w, p = cc.state(0.3 * s * xc, 0.3 * s * yc, 0.3 * s * zc)
    cases.write_cloud(os.path.join(outdir, "plate.cloud"), xc, yc, zc, rho, u, v, w, p)
    types = {q: ("characteristic", 1) for q in cc.SURF_NAMES}
    types[cc.SURF_NAMES[2 * wall]] = ("viscousWall", 3)
    text = cc._inp("plate", [cases._surfaces_box(ni, nj, nk, types)], "thirdOrder", "implicitEuler", solver, sweeps,
                   eq="navierStokes")
    path = os.path.join(outdir, "plate.inp")
    with open(path, "w") as f:
        f.write(text.replace("boundaryStates: <", "boundaryStates: <viscousWall(tag=3), "))
    return path


@pytest.mark.parametrize("dims", [(33, 9, 8), (9, 33, 8), (8, 9, 33), (17, 9, 1), (17, 1, 9), (1, 17, 9), (9, 17, 1),
                                  (9, 1, 17), (1, 9, 17), (20, 2, 3), (3, 20, 2), (2, 3, 20)])
@pytest.mark.parametrize("solver", ["lusgs", "blusgs"])
@pytest.mark.parametrize("sweeps,precision", [(1, 0), (1, 1), (2, 0), (2, 1)])
def test_viscous_axes(tmp_path, dims, solver, sweeps, precision):
    wall = next(d for d in (1, 2, 0) if dims[d] > 1)
    path = write_plate(str(tmp_path), dims, wall, sweeps, solver)
    print("orders, viscous", dims, solver, sweeps, precision, flush=True)
    same(path, precision)


# one block for each tile the block diagonal may be cut into, with remainders
@pytest.mark.parametrize("dims", [(40, 16, 3), (9, 33, 9), (40, 3, 64), (33, 1, 9), (300, 1, 1), (9, 33, 1), (1, 40, 9),
                                  (1, 300, 1), (9, 9, 25), (1, 9, 33), (1, 1, 300)])
@pytest.mark.parametrize("eq", ["euler", "navierStokes"])
def test_diagonal_tiles(tmp_path, dims, eq):
    if eq == "euler":
        ni, nj, nk = dims
        path = cases.vortex_case(str(tmp_path), n=max(dims), iterations=4, ni=ni, nj=nj, nk=nk, solver="blusgs")
    else:
        path = write_plate(str(tmp_path), dims, next(d for d in (1, 2, 0) if dims[d] > 1), 1)
    print("block diagonal's tiles", dims, eq, flush=True)
    same(path, 0)


@pytest.mark.parametrize("solver", ["lusgs", "blusgs"])
@pytest.mark.parametrize("sweeps,precision", [(1, 0), (2, 0), (1, 1), (2, 1)])
def test_thin_and_thick_blocks_in_one_launch(tmp_path, solver, sweeps, precision):
    """Cases whose records hold one step, two, eight and sixty-four, side by side
    in a server and each alone"""
    from aither_amd import Server
    paths = []
    for q, (ni, nj, nk) in enumerate([(20, 19, 18), (33, 1, 40), (1, 1, 50), (4, 30, 9), (17, 2, 2)]):
        (tmp_path / str(q)).mkdir()
        paths.append(cases.vortex_case(str(tmp_path / str(q)), n=max(ni, nj, nk), iterations=4, ni=ni, nj=nj, nk=nk,
                                       solver=solver, sweeps=sweeps))
    print("thin and thick blocks", solver, sweeps, precision, flush=True)

    def states(some):
        with Server(max_slots=8, precision=precision) as srv:
            slots = [srv.admit(p, 1e-200, 2 ** 30) for p in some]
            srv.step(4)
            return [srv.state(s) for s in slots]
    alone = [states([p])[0] for p in paths]
    assert all(np.all(np.isfinite(a)) for a in alone)
    assert all(np.array_equal(a, b) for a, b in zip(states(paths), alone))
