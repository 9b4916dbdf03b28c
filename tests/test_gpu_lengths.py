"""Line lengths with a factor 5 or more factors 3, and boxes whose sides differ, on the
length-specialised kernels: each length once along x, y and z, against the FP64 oracle
(state <= 1e-12 norm-wise in FP64 and <= 1e-5 FP32-mixed, tracers <= 1e-11 / 1e-6,
real-space moments <= 1e-11), in a sheared frame with the time step of the remesh clock."""
import sys

import numpy as np
import pytest

import pandora_amd as pa
from conftest import rel

pytestmark = pytest.mark.gpu

LENGTHS = [24, 30, 36, 40, 60, 72, 80, 90, 100, 108, 120, 144, 150, 160, 180, 200, 216, 240, 250, 288, 300, 320, 360,
           400, 432, 480, 640, 960, 1280]


def note(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n", LENGTHS)
def test_length_along_each_axis(oracle_mod, n):
    for shape in ((n, 36, 24), (24, n, 36), (36, 24, n)):
        nx, ny, nz = shape
        note(f"{shape} BF_ROT shear + 500 tracers, 3 steps through a remesh, FP64 and FP32-mixed")
        kw = dict(f_type=2, rk3_timestep=1, deform_s=100.0, remesh_t=2, nu=1e-4 if n > 300 else 0.001)
        u = pa.init_field_host(nx, n, 0.02, 4.0, ny=ny, nz=nz)
        xp = np.random.default_rng(n).uniform(0.5, 5.5, size=(500, 3))
        o = oracle_mod.Oracle(nx=nx, ny=ny, nz=nz, **kw)
        o.set_state(*u)
        o.set_particles(xp)
        to = 0.0
        for s in range(1, 4):
            to = o.step(s, to)
        so, xo = o.get_state(), o.get_particles()[0]
        qo = o.rs_stats()
        for prec, tol, xtol in ((pa.PDR_FP64, 1e-12, 1e-11), (pa.PDR_FP32_MIXED, 1e-5, 1e-6)):
            with pa.Pandora(nx=nx, ny=ny, nz=nz, precision=prec, **kw) as g:
                assert g.kernel_forms()["specialised"] == 1
                g.set_state(*u)
                g.set_particles(xp)
                assert g.run(1, 3, 0.0) == to
                for a, b in zip(g.get_state(), so):
                    assert rel(a, b) < tol
                assert np.abs(g.get_particles()[0] - xo).max() < xtol
                if prec == pa.PDR_FP64:
                    for name, v in g.rs_stats().items():
                        assert v == pytest.approx(qo[name], rel=1e-11, abs=1e-13), name
        o.close()


@pytest.mark.parametrize("shape", [(64, 64, 64), (30, 24, 36), (100, 36, 24), (24, 100, 36), (512, 24, 30),
                                   (36, 24, 640)], ids=lambda s: "x".join(map(str, s)))
def test_convective_form_against_oracle(oracle_mod, shape):
    """NS_R_CONV with each derivative formed in its own pass: whole-plane and i-line y tiles,
    2, 4 and 8 rows per x tile, fused and separate z forward; tracers, moments, a remesh."""
    nx, ny, nz = shape
    note(f"{shape} R_CONV shear + 500 tracers, 4 steps through a remesh, FP64 and FP32-mixed")
    kw = dict(f_type=2, ns_deformed=2, rk3_timestep=1, deform_s=100.0, remesh_t=2, nu=1e-4)
    u = pa.init_field_host(nx, sum(shape), 0.02, 4.0, ny=ny, nz=nz)
    xp = np.random.default_rng(nx).uniform(0.5, 5.5, size=(500, 3))
    o = oracle_mod.Oracle(nx=nx, ny=ny, nz=nz, **kw)
    o.set_state(*u)
    o.set_particles(xp)
    to = 0.0
    for s in range(1, 5):
        to = o.step(s, to)
    so, xo = o.get_state(), o.get_particles()[0]
    qo = o.rs_stats()
    for prec, tol, xtol in ((pa.PDR_FP64, 1e-12, 1e-11), (pa.PDR_FP32_MIXED, 1e-5, 1e-6)):
        with pa.Pandora(nx=nx, ny=ny, nz=nz, precision=prec, **kw) as g:
            assert g.kernel_forms()["specialised"] == 1
            g.set_state(*u)
            g.set_particles(xp)
            assert g.run(1, 4, 0.0) == to
            for a, b in zip(g.get_state(), so):
                assert rel(a, b) < tol
            assert np.abs(g.get_particles()[0] - xo).max() < xtol
            if prec == pa.PDR_FP64:
                for name, v in g.rs_stats().items():
                    assert v == pytest.approx(qo[name], rel=1e-11, abs=1e-13), name
    o.close()
