"""The range in which the device's quotients and square roots (by a refined
reciprocal, without a scaling of the operands) are exact, through the face-flux
entry point."""
import numpy as np
import pytest

import aither_amd
import pyoracle

pytestmark = pytest.mark.gpu
N = 512


def states(seed):
    rng = np.random.default_rng(seed)
    W = [np.empty((N, 5)) for _ in range(2)]
    for w in W:
        w[:, 0] = rng.uniform(0.3, 3.0, N)
        w[:, 4] = rng.uniform(0.3, 3.0, N) / 1.4
        w[:, 1:4] = rng.normal(size=(N, 3)) * rng.uniform(0.01, 2.0, (N, 1))
    n = rng.normal(size=(N, 3))
    return W[0], W[1], n / np.linalg.norm(n, axis=1, keepdims=True)


def oracle(flux, L, R, n):
    gas = pyoracle.Gas(R=1 / 1.4, n=2.5)
    fn = pyoracle.lib().orc_roe_flux if flux == 0 else pyoracle.lib().orc_ausm_flux
    F = np.empty((N, 5))
    for q in range(N):
        fn(pyoracle.ctypes.byref(gas), pyoracle.P(L[q].copy()), pyoracle.P(R[q].copy()), pyoracle.P(n[q].copy()),
           pyoracle.P(F[q]))
    return F


@pytest.mark.parametrize("flux", [0, 1])
@pytest.mark.parametrize("density", [-300, -60, 0, 60, 300])
@pytest.mark.parametrize("speed", [-150, -30, 0, 30, 150])
def test_scaled_states(flux, density, speed):
    """Density times 2^density and speeds times 2^speed.  Every operation of the
    Roe flux is correctly rounded, so it has the oracle's bits; every step of
    AUSMPW+ scales by a power of two, so its flux does (its cubes are the oracle's
    library's, not always correctly rounded)."""
    s, t = 2.0 ** density, 2.0 ** speed
    scale = np.array([s, t, t, t, s * t * t])
    L, R, n = states(flux)
    print("flux at scale", flux, density, speed, flush=True)
    G = aither_amd.eval_face_flux(flux, 1 / 1.4, 2.5, L * scale, R * scale, n)
    if flux == 0:
        assert np.array_equal(G, oracle(flux, L * scale, R * scale, n))
    else:
        F = aither_amd.eval_face_flux(flux, 1 / 1.4, 2.5, L, R, n)
        assert np.array_equal(G, F * np.array([s * t, s * t * t, s * t * t, s * t * t, s * t * t * t]))


@pytest.mark.parametrize("flux", [0, 1])
@pytest.mark.parametrize("speed", [0.0, 1e-310, 1e-200, 1e-160, 1e-120, 1e-60])
def test_vanishing_speeds(flux, speed):
    """Speeds whose squares are below the square root's exact range, or no
    normal numbers, against the oracle (tolerance of the flux parity test)."""
    L, R, n = states(10 + flux)
    L[:, 1:4] *= speed
    R[:, 1:4] *= speed
    R[::2] = L[::2]
    print("flux at vanishing speeds", flux, speed, flush=True)
    F, Fo = aither_amd.eval_face_flux(flux, 1 / 1.4, 2.5, L, R, n), oracle(flux, L, R, n)
    assert np.all(np.isfinite(F))
    assert np.abs(F - Fo).max() <= 1e-13 * np.abs(Fo).max()
