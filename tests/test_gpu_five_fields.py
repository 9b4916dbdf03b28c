"""Boxes large enough that the inverse y pass forms the last vorticity component (five fields
through the z pass): against the FP64 oracle (state <= 1e-12 norm-wise in FP64 and <= 1e-5
FP32-mixed, as for every length), and where a frame set by hand puts k3 into that component
(six fields again) against the runtime-radix kernels."""
import sys

import numpy as np
import pytest

import pandora_amd as pa
from conftest import rel

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


FORMS = {"iso": dict(rk3_dt=0.002), "bfrot": dict(f_type=2, rk3_timestep=1, deform_s=100.0, remesh_t=2),
         "rrot": dict(f_type=2, ns_deformed=3, rk3_timestep=1, deform_s=100.0, remesh_t=2)}


@pytest.mark.parametrize("shape", [(128, 24, 384), (100, 30, 512), (32, 36, 1024)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", list(FORMS))
def test_five_fields_against_oracle(oracle_mod, form, shape):
    nx, ny, nz = shape
    note(f"{form} {shape}, 3 steps, FP64 and FP32-mixed")
    kw = dict(FORMS[form], nu=1e-4)
    u = pa.init_field_host(nx, 7, 0.02, 4.0, ny=ny, nz=nz)
    o = oracle_mod.Oracle(nx=nx, ny=ny, nz=nz, **kw)
    o.set_state(*u)
    to = 0.0
    for s in range(1, 4):
        to = o.step(s, to)
    so, qo = o.get_state(), o.rs_stats()
    o.close()
    for prec, tol in ((pa.PDR_FP64, 1e-12), (pa.PDR_FP32_MIXED, 1e-5)):
        with pa.Pandora(nx=nx, ny=ny, nz=nz, precision=prec, **kw) as g:
            assert g.kernel_forms()["specialised"] == 1
            g.set_state(*u)
            assert g.run(1, 3, 0.0) == to
            for a, b in zip(g.get_state(), so):
                assert rel(a, b) < tol
            if prec == pa.PDR_FP64:
                for name, v in g.rs_stats().items():
                    assert v == pytest.approx(qo[name], rel=1e-11, abs=1e-13), name


@pytest.mark.parametrize("prec,tol", [(pa.PDR_FP64, 1e-12), (pa.PDR_FP32_MIXED, 1e-5)], ids=["fp64", "fp32"])
@pytest.mark.parametrize("skew", [0.0, 0.25])
def test_frame_set_by_hand(monkeypatch, skew, prec, tol):
    """NS_R_ROT takes every entry of bmat into its curl; with bmat(3, 1) the last vorticity
    component has k3 in it."""
    nx, ny, nz = 128, 24, 384
    note(f"bmat(3, 1) = {skew}, precision {prec}")
    u = pa.init_field_host(nx, 3, 0.02, 4.0, ny=ny, nz=nz)
    out = []
    for generic in ("0", "1"):
        monkeypatch.setenv("PDR_GENERIC_KERNELS", generic)
        kw = dict(FORMS["rrot"], nu=1e-4, nx=nx, ny=ny, nz=nz, precision=prec)
        with pa.Pandora(**kw) as g:
            b, bi = np.eye(3), np.eye(3)
            b[2, 0] = skew
            g.set_frame(b.T, bi.T)
            g.set_state(*u)
            g.run(1, 1, 0.0)
            out.append(g.get_state())
    for a, b in zip(*out):
        assert rel(a, b) < tol
