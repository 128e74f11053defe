"""A Weno or Central pass walks its pencils in segments of several tiles, each
tile taking over cells, midpoints and a face flux from the one before:
residuals equal the oracle's bit for bit on a mesh whose three axes are cut
into segments of several tiles with partial last tiles, for every tile shape
(smaller meshes are cut into single tiles), and the FP32, contracted and
ensemble passes follow."""
import numpy as np
import pytest

from _oracle import OracleSolver

pytestmark = pytest.mark.gpu


N = (97, 130, 98)
BOX = ((0, 0, 0), (6.0, 6.0, 6.0))
BC = [["outflow", "reflect"], ["periodic", "periodic"], ["reflect", "outflow"]]
# FP32 takes first-order fallbacks beside the exactly flat ghosts of an outflow boundary, which FP64 does not
PERIODIC = [["periodic", "periodic"]] * 3


def _tile_cfgs():
    import os
    import re

    src = os.path.join(os.path.dirname(__file__), "..", "emergence_amd", "csrc", "em_pass.h")
    with open(src) as f:
        body = re.search(r"kTileCfgs\[\] = \{(.*?)\};", f.read(), re.S).group(1)
    return [tuple(map(int, m)) for m in re.findall(r"\{(\d+), (\d+), (\d+)\}", body)]


def _tiles_of_a_segment(n, axis, shape):
    """Tiles of a segment along the axis, by the library's rule (Grid::cut_segments)."""
    t, p, nt = shape
    fast = 1 if axis == 2 else 2
    slow = 3 - axis - fast
    groups = -(-n[fast] // p) * n[slow]
    ntile = -(-n[axis] // t)
    return max(1, ntile // min(-(-2 * (256 * 16 * 64 // nt) // groups), ntile))


def _state(n=N):
    import emergence_amd as em

    rng = np.random.default_rng(11)
    u = em.case_init(1, n, *BOX, 6, [0.3, 7.0])
    return u * (1.0 + 0.05 * rng.standard_normal(u.shape))


_ORACLE = {}


def _oracle(mode, bc=BC):
    """dt, interior residual and counters of the oracle, once per mode."""
    key = mode, str(bc)
    if key not in _ORACLE:
        o = OracleSolver(N, *BOX)
        o.set_u(_state())
        o.set_opts(mode=mode)
        for d in range(3):
            for s in range(2):
                o.set_bc(d, s, bc[d][s])
        dt = o.dt_cfl()
        r, st = o.rhs(dt)
        _ORACLE[key] = dt, o.interior(r).copy(), list(st)
    return _ORACLE[key]


def test_the_mesh_is_cut_into_segments_of_several_tiles():
    """Shapes of at most 64 cells along an axis: two or three tiles a segment,
    the last tile of each pencil a partial one."""
    for shape in _tile_cfgs():
        for axis in range(3):
            if shape[0] <= 64:
                assert _tiles_of_a_segment(N, axis, shape) >= 2, (shape, axis)
                assert N[axis] % shape[0] != 0


@pytest.mark.parametrize("mode", ["weno", "central"])
def test_segments_of_several_tiles(mode):
    import emergence_amd as em

    dt, ref, so = _oracle(mode)
    g = em.HipSolver(N, *BOX, _state(), mode=mode, bc=BC)
    for cfg in range(10):
        g.set_tiles([cfg] * 3)
        got, sg = g.rhs(dt)
        assert list(sg) == so, cfg
        assert np.array_equal(g.interior(got), ref), cfg


@pytest.mark.parametrize("mode", ["weno", "central"])
@pytest.mark.parametrize("real, precise, bar", [("f64", False, 1e-12), ("f32", False, 1e-4), ("f32", True, 1e-4)])
def test_segments_in_the_other_arithmetics(real, precise, bar, mode):
    """The contracted and the FP32 passes against the oracle, to the bars of
    test_gpu_uniform.py and test_gpu_f32.py (relative to the largest
    residual); without contraction every shape gives the same bits."""
    import emergence_amd as em

    bc = PERIODIC if real == "f32" else BC
    dt, ref, _ = _oracle(mode, bc)
    scale = np.abs(ref).max()
    g = em.HipSolver(N, *BOX, _state(), mode=mode, bc=bc, real=real, precise=precise)
    first = None
    for cfg in range(10):
        g.set_tiles([cfg] * 3)
        got = g.interior(g.rhs(dt)[0])
        assert np.abs(got - ref).max() <= bar * scale, cfg
        if precise:
            first = got.copy() if first is None else first
            assert np.array_equal(got, first), cfg


@pytest.mark.parametrize("mode", ["weno", "central"])
def test_segments_in_an_ensemble(mode):
    """An ensemble of a box, a smaller box, a plane and a line (of both
    layouts along the shared axes) steps as its members alone, bit for bit."""
    import emergence_amd as em

    sizes = [N, (60, 40, 50), (130, 90, 1), (1, 300, 1)]
    us = [_state(n) for n in sizes]
    want = []
    for n, u in zip(sizes, us):
        g = em.HipSolver(n, *BOX, u, mode=mode, bc=BC)
        g.run_steps(2)
        want.append(g.interior(g.download()))
    for order in ([0, 1, 2, 3], [3, 2, 1, 0]):
        for cfg in (0, 4, 7, 9):
            e = em.HipEnsemble([sizes[i] for i in order], [us[i] for i in order], lo=[BOX[0]] * 4, hi=[BOX[1]] * 4,
                               mode=mode, bc=BC)
            e.set_tiles(cfg)
            e.run_steps(2)
            for k, i in enumerate(order):
                d = e.download(k)
                c = d[tuple(slice(6, 6 + v) if v > 1 else slice(0, 1) for v in sizes[i])]
                assert np.array_equal(c, want[i]), (cfg, sizes[i])


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
