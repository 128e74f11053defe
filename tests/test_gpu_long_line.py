"""A line whose Hybrid pass in the ordinary 27 x 8 tiles would need more than
2^32 threads (of which a launch runs a part only, without an error): the
residual of a uniform flow is written, and zero, everywhere."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_uniform_flow_on_a_long_line(mode):
    import torch

    import emergence_amd as em

    lib = em.load()
    n = 470_000_000
    u = torch.empty(5, n, dtype=torch.float64, device="cuda")
    for k, w in enumerate([1.0, 0.5, 0.0, 0.0, 1.0 / 0.4 + 0.125]):
        u[k] = w
    out = torch.full_like(u, 7.0)
    stats = torch.zeros(4, dtype=torch.int64, device="cuda")
    rc = lib.em_rhs_noalloc((C.c_int64 * 3)(n, 1, 1), (C.c_double * 3)(0, 0, 0), (C.c_double * 3)(1, 1, 1),
                            (C.c_double * 4)(1.4, 0, 0, 0), (C.c_int32 * 6)(), (C.c_double * 30)(), mode, 1, 1e-3, 1, 0.0,
                            u.data_ptr(), out.data_ptr(), stats.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.em_last_error().decode()
    torch.cuda.synchronize()
    assert float(out.abs().max()) == 0.0
    assert stats.tolist() == [n + 1, n + 1 if mode == 1 else 0, 0, 0]
