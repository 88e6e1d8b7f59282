"""Reading a large field right after an asynchronous step() waits for the GPU
without keeping more than the calling thread busy."""
import time

import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu


def test_waiting_for_the_steps_keeps_one_core_busy_at_most():
    nx, ny = 4096, 1024
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny)], precision="fp32")
    s.initialization(ekpnp.COLD_NOISE, 1)
    s.init_equilibrium()
    s.step(64)
    first = s.get_field(0, "psi")  # the staging exists from here on
    assert first.nbytes >= 16 << 20
    s.step(8 * 512)  # about 0.9 s of GPU work
    wall, cpu = time.perf_counter(), time.process_time()
    psi = s.get_field(0, "psi")
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    print(f"read-back after queued steps: wall {wall:.3f} s, CPU {cpu:.3f} s", flush=True)
    assert np.isfinite(psi).all()
    assert wall > 0.2  # the steps were still under way
    # the caller may spin in the runtime's wait (1.0 of wall) and four threads
    # copy and map for some ms; three spinning helpers would make it 4.0
    assert cpu <= 1.5 * wall + 0.1
