"""Stages joined by one kernel (a stage's z forward pass, FormF and the next one's inverse z
pass) against the same stages called one by one, which join nothing, and against pdr_step."""
import sys

import numpy as np
import pytest

import pandora_amd as pa
from conftest import rel

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


CASES = {
    "iso": dict(nu=0.01, rk3_dt=0.005),
    "cfl": dict(nu=0.01, rk3_timestep=3, rk3_cfl=0.4),
    "bfrot": dict(f_type=2, rk3_timestep=1, deform_s=20.0, remesh_t=2, nu=0.005),
    "rrot": dict(f_type=2, ns_deformed=3, rk3_timestep=1, deform_s=20.0, remesh_t=2, nu=0.005),
    "spherical": dict(nu=0.01, rk3_dt=0.005, dealiasing=2),
    "forced": dict(nu=0.01, rk3_dt=0.005, force_tf=0.2, force_kf=2.5, force_sigma=0.7, force_stop=4, force_seed=3),
}


@pytest.mark.parametrize("prec", [pa.PDR_FP64, pa.PDR_FP32_MIXED], ids=["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(24, 24, 24), (32, 32, 64), (64, 64, 64), (36, 48, 96), (128, 24, 128)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", list(CASES))
def test_run_equals_single_stages(name, shape, prec):
    """Six steps through a remesh, with tracers: run, step by step and stage by stage agree to
    FP64 1e-13 / FP32-mixed 2e-6 (the joined kernel may contract multiply-adds differently)."""
    note(f"{name} {shape} precision {prec}")
    nx, ny, nz = shape
    kw = dict(CASES[name], nx=nx, ny=ny, nz=nz, precision=prec)
    u = pa.init_field_host(nx, 5, 0.1, 4.0, ny=ny, nz=nz)
    xp = np.random.default_rng(1).uniform(0.5, 5.5, size=(200, 3))
    out = []
    for way in ("run", "step", "stage"):
        with pa.Pandora(**kw) as g:
            g.set_state(*u)
            g.set_particles(xp)
            t = 0.0
            if way == "run":
                t = g.run(1, 6, t)
            else:
                dt = g.dt
                for s in range(1, 7):
                    if way == "step":
                        t = g.rk3_calc(s, t)
                        continue
                    t0 = t
                    for stage, frac in ((1, 1.0 / 3.0), (2, 3.0 / 4.0), (3, 1.0)):
                        dt = g.stage(stage, s, t, dt)
                        t = t0 + frac * dt
                        g.update_b(s, t)
            out.append((t, g.get_state() + g.get_rk(), g.get_particles()[0]))
    tol = 1e-13 if prec == pa.PDR_FP64 else 2e-6
    for t, fields, x in out[:2]:
        assert t == pytest.approx(out[2][0], rel=tol)
        for a, b in zip(fields, out[2][1]):
            assert rel(a, b) < tol
        assert np.abs(x - out[2][2]).max() < 10 * tol
