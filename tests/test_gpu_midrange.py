"""The Euler pass takes its divisions through shared reciprocals where the
operands lie in the middle of the exponent range, and evaluates everything
else in the general form: both give the oracle's bits.  The states below sit
on either side of every range test: densities and pressures far from one,
velocities down to denormals beside a front, zero and signed-zero components,
near-vacuum, and cells whose limiter and first-order fallback act.
"""
import numpy as np
import pytest

from _oracle import OracleSolver

pytestmark = pytest.mark.gpu
G = 1.4


@pytest.fixture(scope="module")
def em():
    import emergence_amd

    emergence_amd.load()
    return emergence_amd


def _state(n, kind, seed=5, ng=6):
    rng = np.random.default_rng(seed)
    rho = 1.0 + 0.3 * rng.random(n)
    vel = 0.4 * rng.standard_normal((3,) + n)
    p = 1.0 + 0.5 * rng.random(n)
    for d in range(3):
        if n[d] == 1:
            vel[d] = 0.0
    if kind == "fronts":  # quiescent gas: velocities fall from 1 to denormals and to zero
        vel *= 10.0 ** rng.integers(-330, 1, (3,) + n)
        vel[:, : n[0] // 3] = 0.0
    elif kind == "signed_zero":
        vel[1] = np.where(rng.random(n) < 0.5, 0.0, -0.0)
        vel[2] = -0.0
    elif kind == "small":  # below the mid range
        rho, p, vel = rho * 1e-34, p * 1e-40, vel * 1e-3
    elif kind == "large":  # smoothness indicators above it
        rho, p, vel = rho * 1e3, p * 1e37, vel * 1e17
    elif kind == "near_vacuum":
        hole = rng.random(n) < 0.1
        rho, p = np.where(hole, rho * 1e-12, rho), np.where(hole, p * 1e-14, p)
        vel *= 3.0
    elif kind == "cold":  # kinetic energy far above the internal one: the limiter's test is near its margin
        p = p * 1e-9
        vel = vel + 5.0
    elif kind == "outlier":  # gas at rest but for single cells far out: the product of two weight sums overflows
        # (seven cells apart along every axis, one component each, density 1: the pressure there is exactly zero)
        vel *= 0.0
        i, j, k = np.indices(n)
        comp = np.where((i + 3 * j + 5 * k) % 7 == 0, (i + j + k) % 3, -1)
        rho = np.where(comp >= 0, 1.0, rho)
        for d in range(3):
            vel[d][comp == d] = 2.0 ** 70
    u = np.zeros(tuple(v + 2 * ng if v > 1 else 1 for v in n) + (5,))
    g = [ng if v > 1 else 0 for v in n]
    ui = u[g[0]:g[0] + n[0], g[1]:g[1] + n[1], g[2]:g[2] + n[2]]
    ui[..., 0] = rho
    for d in range(3):
        ui[..., 1 + d] = rho * vel[d]
    ui[..., 4] = p / (G - 1.0) + 0.5 * rho * (vel ** 2).sum(0)
    return u


@pytest.mark.parametrize("mode", ["weno", "central"])
@pytest.mark.parametrize("n", [(67, 9, 1), (12, 10, 70), (1, 70, 5)])
@pytest.mark.parametrize("kind", ["fronts", "signed_zero", "small", "large", "near_vacuum", "cold", "outlier"])
def test_residual_bits_in_and_outside_the_mid_range(em, kind, n, mode):
    bc = [["outflow", "outflow"], ["periodic", "periodic"], ["reflect", "outflow"]]
    u = _state(n, kind)
    g = em.HipSolver(n, (0, 0, 0), (1, 1, 1), u, mode=mode, bc=bc)
    o = OracleSolver(n, (0, 0, 0), (1, 1, 1))
    o.set_u(u)
    o.set_opts(mode=mode)
    for d in range(3):
        for s in range(2):
            o.set_bc(d, s, bc[d][s])
    dt = o.dt_cfl()
    assert g.dt_cfl() == dt
    a, sa = g.rhs(dt)
    b, sb = o.rhs(dt)
    a, b = o.interior(a), o.interior(b)
    assert list(sa) == list(sb)
    assert np.array_equal(a, b, equal_nan=True), (kind, n, mode, int((a != b).sum()))
    v = ~np.isnan(a)
    assert np.array_equal(a[v].view(np.int64), b[v].view(np.int64)), "sign of a zero"


@pytest.mark.parametrize("n", [(67, 9, 1), (12, 10, 70), (1, 70, 5)])
@pytest.mark.parametrize("kind", ["fronts", "signed_zero", "small", "large", "near_vacuum", "cold", "outlier"])
def test_hybrid_residuals_in_and_outside_the_mid_range(em, kind, n):
    """Hybrid mode, where only part of a wave's lanes evaluate a midpoint.  The
    sensor's logarithms differ from the host's by an ulp, which moves a blend
    weight by at most 3 / (tol / 2) 16 ulp(ln) (below 1e-10 for |ln| < 128):
    the bar is that share of the largest residual."""
    bc = [["outflow", "outflow"], ["periodic", "periodic"], ["reflect", "outflow"]]
    u = _state(n, kind)
    g = em.HipSolver(n, (0, 0, 0), (1, 1, 1), u, mode="hybrid", bc=bc)
    o = OracleSolver(n, (0, 0, 0), (1, 1, 1))
    o.set_u(u)
    o.set_opts(mode="hybrid")
    for d in range(3):
        for s in range(2):
            o.set_bc(d, s, bc[d][s])
    dt = o.dt_cfl()
    a, sa = g.rhs(dt)
    b, sb = o.rhs(dt)
    a, b = o.interior(a), o.interior(b)
    assert list(sa) == list(sb)
    assert np.array_equal(np.isnan(a), np.isnan(b))
    for k in range(5):
        assert np.nanmax(np.abs(a[..., k] - b[..., k])) <= 1e-10 * np.nanmax(np.abs(b[..., k])), k


@pytest.mark.parametrize("eos", [(5.0 / 3.0, 0.0, 0.0, 0.0), (4.4, 0.6, 0.0, 0.1), (1.3, 0.2, 0.3, -0.1)])
def test_residual_bits_with_stiffened_and_covolume_gases(em, eos):
    n = (66, 11, 6)
    u = _state(n, "plain")
    o = OracleSolver(n, (0, 0, 0), (1, 1, 1), eos=eos)
    g = em.HipSolver(n, (0, 0, 0), (1, 1, 1), u, mode="weno", eos=eos)
    o.set_u(u)
    o.set_opts(mode="weno")
    dt = o.dt_cfl()
    a, sa = g.rhs(dt)
    b, sb = o.rhs(dt)
    assert list(sa) == list(sb)
    assert np.array_equal(o.interior(a), o.interior(b), equal_nan=True)
