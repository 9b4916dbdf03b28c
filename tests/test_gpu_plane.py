"""The y and x passes of a z plane as one kernel (square planes of short lines, whole and
in two parts) against the oracle: every length that takes it, cubes and boxes of other
depth, all forms that run on it, tracers, moments, the CFL maximum, both precisions; and
against the separate passes, which the chunked plane pass still runs."""
import sys

import numpy as np
import pytest

import pandora_amd as pa
from conftest import rel

pytestmark = pytest.mark.gpu

LENGTHS = [24, 30, 32, 36, 40, 48, 60, 64, 72, 80, 90, 96, 100, 108]


def note(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


def _pair(oracle_mod, n, nz, prec, kw, tracers):
    u = pa.init_field_host(n, n + nz, 0.05, 4.0, ny=n, nz=nz)
    g = pa.Pandora(nx=n, ny=n, nz=nz, precision=prec, **kw)
    o = oracle_mod.Oracle(nx=n, ny=n, nz=nz, **kw)
    g.set_state(*u)
    o.set_state(*u)
    if tracers:
        xp = np.random.default_rng(n).uniform(0.5, 5.5, size=(tracers, 3))
        g.set_particles(xp)
        o.set_particles(xp)
    return g, o


@pytest.mark.parametrize("prec", [pa.PDR_FP64, pa.PDR_FP32_MIXED], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n", LENGTHS)
def test_plane_lengths_against_oracle(oracle_mod, n, prec):
    tol, xtol, mtol = (1e-12, 1e-11, 1e-11) if prec == pa.PDR_FP64 else (1e-5, 1e-6, 1e-3)
    for nz, kw in ((n, dict(f_type=2, rk3_timestep=1, deform_s=100.0, remesh_t=2, nu=1e-3)),
                   (36, dict(f_type=2, ns_deformed=3, rk3_timestep=1, deform_s=100.0, remesh_t=2, nu=1e-3)),
                   (24, dict(rk3_timestep=3, rk3_cfl=0.2, nu=1e-3))):
        note(f"{n}x{n}x{nz} {kw} precision {prec}, 3 steps, 300 tracers")
        g, o = _pair(oracle_mod, n, nz, prec, kw, 300)
        g.set_stage_stats(1)
        tg = to = 0.0
        for s in range(1, 4):
            if s == 2:  # the record of step 2 is of the state before it (step 3 remeshes first)
                mo = o.rs_stats()
            tg = g.rk3_calc(s, tg)
            if s == 2:
                mg = g.stage_stats()[3]
            to = o.step(s, to)
        assert tg == pytest.approx(to, rel=1e-12 if prec == pa.PDR_FP64 else 1e-5)
        for a, b in zip(g.get_state(), o.get_state()):
            assert rel(a, b) < tol
        assert np.abs(g.get_particles()[0] - o.get_particles()[0]).max() < xtol
        for rec, ref in ((g.rs_stats(), o.rs_stats()), (mg, mo)):
            for name, v in rec.items():
                if name.startswith(("rs_u", "rs_rms", "omega", "ucfl")):
                    scale = abs(ref["rs_u1u1"]) if name.startswith("rs_u") else 0.0
                    assert v == pytest.approx(ref[name], rel=mtol, abs=mtol * scale), name
        g.close()
        o.close()


@pytest.mark.parametrize("n", [32, 64, 96])
def test_plane_equals_separate_passes(monkeypatch, n):
    """FP64 <= 1e-14 and FP32 <= 2e-6 from the separate y, x and y passes over 5 steps."""
    note(f"{n}^3 isotropic, fused planes against the chunked plane pass")
    u = pa.init_field_host(n, 3, 0.5, 4.0)
    for prec, tol in ((pa.PDR_FP64, 1e-14), (pa.PDR_FP32_MIXED, 2e-6)):
        out = []
        for mb in (None, "0.3"):
            if mb:
                monkeypatch.setenv("PDR_ZCHUNK_MB", mb)
            else:
                monkeypatch.delenv("PDR_ZCHUNK_MB", raising=False)
            with pa.Pandora(n, nu=0.01, precision=prec) as g:
                assert (g.kernel_forms()["zchunk"] == n) == (mb is None)
                g.set_state(*u)
                g.run(1, 5, 0.0)
                out.append(g.get_state())
        for a, b in zip(*out):
            assert rel(a, b) < tol
