"""The z passes of lines from 256 points, whose kernels differ in how they form their indices
with the length, the forcing and the number of workgroups: boxes of few and of many z lines
against the runtime-radix kernels (FP64 <= 1e-12, FP32-mixed <= 1e-5 of the state, the bounds
of the comparison with the oracle)."""
import sys

import pytest

import pandora_amd as pa
from conftest import rel

pytestmark = pytest.mark.gpu

FORCED = dict(rk3_dt=0.002, force_tf=0.2, force_kf=2.5, force_sigma=0.7, force_stop=1000, force_seed=3)
FORMS = {"bfrot": dict(f_type=2, rk3_timestep=1, deform_s=100.0, remesh_t=2), "forced": FORCED,
         "deformed": dict(FORCED, f_type=5, b110=2)}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("nxy", [(24, 30), (192, 160)], ids=["few", "many"])
@pytest.mark.parametrize("nz", [256, 288, 300, 360, 384, 480, 512])
def test_z_passes_against_runtime_radix(monkeypatch, nz, nxy, form):
    nx, ny = nxy
    print(f"[gpu case] {nx}x{ny}x{nz} {form}, 2 steps, FP64 and FP32-mixed", flush=True)
    sys.stdout.flush()
    u = pa.init_field_host(nx, nz, 0.02, 4.0, ny=ny, nz=nz)
    for prec, tol in ((pa.PDR_FP64, 1e-12), (pa.PDR_FP32_MIXED, 1e-5)):
        out = []
        for generic in (0, 1):
            monkeypatch.setenv("PDR_GENERIC_KERNELS", str(generic))
            with pa.Pandora(nx=nx, ny=ny, nz=nz, precision=prec, nu=1e-4, **FORMS[form]) as g:
                assert g.kernel_forms()["specialised"] == 1 - generic
                g.set_state(*u)
                g.run(1, 2, 0.0)
                out.append(g.get_state())
        for a, b in zip(*out):
            assert rel(a, b) < tol
