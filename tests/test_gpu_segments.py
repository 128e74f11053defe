"""A Weno pass walks its pencils in segments of several tiles, each tile
taking over cells, midpoints and a face flux from the one before: residuals
equal the oracle's bit for bit on a mesh whose three axes are cut into
segments of several tiles with partial last tiles and segments, and for every
tile shape (small meshes are cut into single tiles)."""
import numpy as np
import pytest

from _oracle import OracleSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["weno", "central"])
def test_segments_of_several_tiles(mode):
    import emergence_amd as em

    n = (97, 130, 98)
    rng = np.random.default_rng(11)
    u = em.case_init(1, n, (0, 0, 0), (6.0, 6.0, 6.0), 6, [0.3, 7.0])
    u *= 1.0 + 0.05 * rng.standard_normal(u.shape)
    bc = [["outflow", "reflect"], ["periodic", "periodic"], ["reflect", "outflow"]]
    o = OracleSolver(n, (0, 0, 0), (6.0, 6.0, 6.0))
    o.set_u(u)
    o.set_opts(mode=mode)
    for d in range(3):
        for s in range(2):
            o.set_bc(d, s, bc[d][s])
    g = em.HipSolver(n, (0, 0, 0), (6.0, 6.0, 6.0), u, mode=mode, bc=bc)
    dt = o.dt_cfl()
    ref, so = o.rhs(dt)
    for cfg in range(10):
        g.set_tiles([cfg] * 3)
        got, sg = g.rhs(dt)
        assert list(sg) == list(so), cfg
        assert np.array_equal(o.interior(got), o.interior(ref)), cfg


def _bursts(n, ng=6, seed=2):
    """Cold gas with a tenth of its cells far from their neighbours: many first-order fallbacks."""
    rng = np.random.default_rng(seed)
    f = np.exp(rng.standard_normal(n) * (rng.random(n) < 0.1))
    vel = 0.5 * rng.standard_normal((3,) + n) * (rng.random((3,) + n) < 0.1)
    u = np.zeros(tuple(v + 2 * ng if v > 1 else 1 for v in n) + (5,))
    ui = u[tuple(slice(ng, ng + v) if v > 1 else slice(0, 1) for v in n)]
    ui[..., 0] = f
    for d in range(3):
        if n[d] > 1:
            ui[..., 1 + d] = f * vel[d]
    ui[..., 4] = 1e-5 * f / 0.4 + 0.5 * (ui[..., 1:4] ** 2).sum(-1) / f
    return u


@pytest.mark.parametrize("real", ["f64", "f32"])
def test_hybrid_fallbacks_do_not_depend_on_the_tiles(real):
    """A midpoint beside the end of a tile may be evaluated by the tile on
    either side alone; its fallback is counted once all the same."""
    import emergence_amd as em

    n = (130, 66, 70)
    u = _bursts(n)
    bc = [["outflow", "reflect"], ["periodic", "periodic"], ["reflect", "outflow"]]
    g = em.HipSolver(n, (0, 0, 0), (6.0, 6.0, 6.0), u, mode="hybrid", bc=bc, tol=5.0, real=real, precise=True)
    dt = g.dt_cfl()
    want = None
    if real == "f64":
        o = OracleSolver(n, (0, 0, 0), (6.0, 6.0, 6.0))
        o.set_u(u)
        o.set_opts(mode="hybrid", tol=5.0)
        for d in range(3):
            for s in range(2):
                o.set_bc(d, s, bc[d][s])
        want = list(o.rhs(dt)[1])
    for cfg in range(10):
        g.set_tiles([cfg] * 3)
        got = list(g.rhs(dt)[1])
        want = want or got
        assert got == want, cfg
        assert got[2] > 1000
