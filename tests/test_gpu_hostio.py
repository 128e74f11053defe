"""States survive the way into the device layout and back bit for bit, and the
host-array residual equals the one on device arrays: on meshes that are
converted on the host (small, thin), on the device, and on the device in two
pieces (above 256 MiB in the host layout)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(40, 1, 1), (33, 47, 1), (1000, 4, 4), (2, 60, 80), (16, 16, 16), (500, 300, 1), (70, 60, 65), (190, 190, 190)]


def _interior(a, n, ng=6):
    return a[tuple(slice(ng, ng + v) if v > 1 else slice(0, 1) for v in n)]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("real", ["f64", "f32"])
def test_upload_and_download(real, n):
    import emergence_amd as em

    rng = np.random.default_rng(1)
    u = 1.0 + 0.1 * rng.random(tuple(v + 12 if v > 1 else 1 for v in n) + (5,))
    u[..., 4] += 2.0
    g = em.HipSolver(n, (0, 0, 0), (1, 1, 1), u, mode="central", real=real)
    want = _interior(u, n).astype(np.float32 if real == "f32" else np.float64)
    assert np.array_equal(_interior(g.download(), n), want)
    g.upload(2.0 * u)
    assert np.array_equal(_interior(g.download(), n), 2.0 * want)
    r, _ = g.rhs(1e-3)
    for lo, hi, axis in [(r[:6], r[-6:], 0), (r[:, :6], r[:, -6:], 1), (r[:, :, :6], r[:, :, -6:], 2)]:
        assert n[axis] == 1 or not (lo.any() or hi.any())  # ghosts are zero
    if real == "f64" and np.prod(n) < 1000000:
        # the same residual through the cotangent path's conversions
        w = em.HipSolver(n, (0, 0, 0), (1, 1, 1), 2.0 * u, mode="weno")
        lam = rng.standard_normal(u.shape)
        a, b = w.adjoint_rhs(1e-3, lam), w.adjoint_rhs(1e-3, 2.0 * lam)
        assert np.array_equal(2.0 * a, b) and _interior(a, n).any()


@pytest.mark.parametrize("n", [(40, 1, 1), (64, 48, 1), (1000, 4, 4), (60, 50, 55)])
@pytest.mark.parametrize("real", ["f64", "f32"])
def test_fiveeq_upload_and_download(real, n):
    import emergence_amd as em

    rng = np.random.default_rng(1)
    u = 0.4 + 0.1 * rng.random(tuple(v + 12 if v > 1 else 1 for v in n) + (7,))
    u[..., 5] = 1e7
    g = em.HipFiveEq(n, (0, 0, 0), (1, 1, 1), u, real=real)
    want = _interior(u, n).astype(np.float32 if real == "f32" else np.float64)
    d = g.download()
    assert np.array_equal(_interior(d, n), want)
    assert d.sum() == _interior(d, n).sum() or np.isclose(d.sum(), _interior(d, n).sum(), rtol=1e-12)


def _free_bytes():
    import ctypes as C

    from emergence_amd import DeviceArray

    free, total = C.c_size_t(), C.c_size_t()
    assert DeviceArray._rt().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_an_ensemble_holds_one_conversion_buffer():
    """Its instances' transfers, also from several threads, go through one
    buffer (each its own: 129 MB here)."""
    from concurrent.futures import ThreadPoolExecutor

    import emergence_amd as em

    sizes = [(512, 512, 1)] * 11 + [(300, 400, 1)]  # the largest comes first and again after smaller ones
    rng = np.random.default_rng(1)
    us = [1.0 + 0.1 * rng.random((n[0] + 12, n[1] + 12, 1, 5)) + 2.0 * (np.arange(5) == 4) for n in sizes]
    em.HipSolver((64, 64, 1), (0, 0, 0), (1, 1, 1), us[0][:76, :76], mode="central").rhs(1e-3)  # context and code
    before = _free_bytes()
    e = em.HipEnsemble(sizes, us, mode="central")
    used = before - _free_bytes()
    states = 4 * 40 * sum(n[0] * n[1] for n in sizes)
    assert used < states + 80e6, (used, states)
    with ThreadPoolExecutor(4) as pool:
        for _ in range(3):
            list(pool.map(lambda i: e.upload(i, (i + 2.0) * us[i]), range(len(sizes))))
            got = list(pool.map(e.download, range(len(sizes))))
            for i, n in enumerate(sizes):
                assert np.array_equal(_interior(got[i], n), (i + 2.0) * _interior(us[i], n)), i
