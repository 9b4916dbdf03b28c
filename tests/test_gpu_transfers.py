"""Fields and tracers to the device and back through the context's pinned memory: one
kernel for small boxes, chunks over threads for large ones, with sizes on both sides of
the line and ragged last chunks.  FP64 comes back bit for bit, FP32-mixed as the rounded
value; tracers in the caller's order whatever their slots."""
import sys

import numpy as np
import pytest

import pandora_amd as pa

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("prec", [pa.PDR_FP64, pa.PDR_FP32_MIXED], ids=["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(8, 8, 8), (24, 40, 36), (48, 48, 48), (60, 48, 72), (128, 128, 120),
                                   (200, 192, 160)], ids=lambda s: "x".join(map(str, s)))
def test_state_round_trip(shape, prec):
    note(f"state round trip {shape} precision {prec}")
    nx, ny, nz = shape
    rng = np.random.default_rng(nx)
    with pa.Pandora(nx=nx, ny=ny, nz=nz, precision=prec) as g:
        for put, get in ((g.set_state, g.get_state), (g.set_rk, g.get_rk), (g.set_state, g.get_state)):
            a = [rng.standard_normal(g.shape) + 1j * rng.standard_normal(g.shape) for _ in range(3)]
            put(*a)
            for x, y in zip(get(), a):
                want = y if prec == pa.PDR_FP64 else y.astype(np.complex64).astype(np.complex128)
                np.testing.assert_array_equal(x, want)


@pytest.mark.parametrize("count", [1, 7, 43690, 43691, 100001, 400000])
def test_tracers_keep_the_callers_order(count):
    note(f"{count} tracers")
    rng = np.random.default_rng(count)
    x = rng.uniform(0.2, 6.0, size=(count, 3))
    with pa.Pandora(32, nu=0.01) as g:  # the state is zero: tracers stay where they are
        g.particle_stats_config(True, keep_initial=True)
        g.set_particles(x)
        np.testing.assert_array_equal(g.get_particles()[0], x)
        up = rng.standard_normal((count, 3))
        g.set_particles_aux(up, x[::-1])
        g.set_particle_sort(1)
        g.run(1, 2, 0.0)
        xp, uprk = g.get_particles()
        np.testing.assert_array_equal(xp, x)
        assert not uprk.any()
        assert not g.get_particles_aux()[0].any()  # the advance sets particle_up: at rest
        # (it also rounds particle_xp0: xp0 + x - x); into the permuted slots and back
        g.set_particles_aux(up, x[::-1])
        up2, x0 = g.get_particles_aux()
        np.testing.assert_array_equal(up2, up)
        np.testing.assert_array_equal(x0, x[::-1])
