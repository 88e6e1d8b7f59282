"""Fields read into pinned memory are copied there directly: the same values,
without the threads that copy a staged field on to pageable memory."""
import ctypes
import time

import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu


def pinned(nbytes):
    hip = ctypes.CDLL(ekpnp.LIB_PATH)  # the runtime that the library itself uses
    p = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes), 0) == 0
    return hip, p


@pytest.mark.parametrize("nx,ny", [(8, 4), (513, 512), (4096, 2049)])
def test_pinned_destination(nx, ny):
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny)], precision="fp32")
    f = np.random.default_rng(nx).standard_normal((6, ny, nx))
    s.set_fields(0, *f)
    hip, p = pinned(nx * ny * 8 + 64)
    dp = ctypes.POINTER(ctypes.c_double)
    dst = np.ctypeslib.as_array(ctypes.cast(p, dp), shape=(nx * ny + 8,))
    page = np.empty((ny, nx))

    def read(out):
        cpu = time.process_time()
        assert ekpnp.lib().ekpnp_get_field(s._ctx, 0, ekpnp.FIELDS["psi"], out.ctypes.data_as(dp)) == 0
        return time.process_time() - cpu

    for off in (0, 5):  # the start of the allocation, and a place inside it
        view = dst[off:off + nx * ny]
        t_pin = min(read(view) for _ in range(5))
        assert np.array_equal(view.reshape(ny, nx), f[5])
        t_page = min(read(page) for _ in range(5))
        assert np.array_equal(page, f[5])
        print(f"{nx}x{ny}: CPU time pinned {1e3 * t_pin:.3f} ms, pageable {1e3 * t_page:.3f} ms", flush=True)
        # 67 MB: four threads' copies (6 ms of CPU at 10 GB/s) against the wait for a 1.3 ms DMA
        if nx * ny > 8e6:
            assert t_pin < 0.5 * t_page
    s.close()
    hip.hipHostFree(p)
