"""The passes that a box's steps take together (pdr_kernel_routes) at the sizes where the rule
changes, each against the FP64 oracle: fused planes over four workgroups down to one, a
workgroup with several of a plane's parts among them, whose results the joined z pass adds;
boxes too deep for them; and five or six fields through z."""
import sys

import numpy as np
import pytest

import pandora_amd as pa
from conftest import rel

pytestmark = pytest.mark.gpu

F64, F32 = pa.PDR_FP64, pa.PDR_FP32_MIXED
# (nx = ny, nz, precision): groups, parts, joined
PLANES = [
    (32, 32, F64, 4, 4, 1),
    (32, 72, F32, 4, 4, 1),
    (48, 96, F64, 3, 4, 1),    # a group has two of the four parts
    (60, 100, F32, 3, 4, 1),
    (60, 128, F32, 2, 4, 1),   # each has two
    (64, 80, F32, 4, 4, 1),
    (24, 256, F64, 1, 1, 0),   # a plane whole, its result in place
    (30, 128, F32, 1, 1, 1),
    (64, 96, F64, 0, 0, 1),    # too deep for planes in parts
    (64, 128, F64, 0, 0, 0),
    (48, 192, F32, 0, 0, 0),
]


def note(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


def _compare(oracle_mod, nx, ny, nz, prec, kw, steps, tracers, routes):
    u = pa.init_field_host(nx, nx + 3 * nz, 0.02, 4.0, ny=ny, nz=nz)
    xp = np.random.default_rng(nz).uniform(0.5, 5.5, size=(tracers, 3))
    o = oracle_mod.Oracle(nx=nx, ny=ny, nz=nz, **kw)
    o.set_state(*u)
    o.set_particles(xp)
    to = 0.0
    for s in range(1, steps + 1):
        to = o.step(s, to)
    tol, xtol = (1e-12, 1e-11) if prec == F64 else (1e-5, 1e-6)
    with pa.Pandora(nx=nx, ny=ny, nz=nz, precision=prec, **kw) as g:
        r = g.kernel_routes()
        assert {k: r[k] for k in routes} == routes
        g.set_state(*u)
        g.set_particles(xp)
        tg = g.run(1, steps, 0.0)
        assert tg == pytest.approx(to, rel=1e-12 if prec == F64 else 1e-5)
        for a, b in zip(g.get_state(), o.get_state()):
            assert rel(a, b) < tol
        assert np.abs(g.get_particles()[0] - o.get_particles()[0]).max() < xtol
        mo, mg = o.rs_stats(), g.rs_stats()
        for name in ("rs_u1u1", "rs_u2u2", "rs_u3u3", "rs_rmsvort1", "rs_rmsvort2", "rs_rmsvort3", "ucfl"):
            assert mg[name] == pytest.approx(mo[name], rel=1e-11 if prec == F64 else 1e-3), name
    o.close()


FORMS = {"bfrot": dict(f_type=2, rk3_timestep=1, deform_s=100.0, remesh_t=2, nu=1e-3),
         "iso_cfl": dict(rk3_timestep=3, rk3_cfl=0.2, nu=1e-3)}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("n,nz,prec,groups,parts,joined", PLANES,
                         ids=[f"{c[0]}x{c[0]}x{c[1]}-{'fp32' if c[2] else 'fp64'}" for c in PLANES])
def test_planes_over_workgroups(oracle_mod, form, n, nz, prec, groups, parts, joined):
    note(f"{n}x{n}x{nz} {form} precision {prec}: {groups} groups of {parts} parts, joined {joined}; 4 steps, 300 tracers")
    _compare(oracle_mod, n, n, nz, prec, FORMS[form], 4, 300,
             dict(plane_groups=groups, plane_parts=parts, joined=joined, z_fields=6))


@pytest.mark.parametrize("shape,prec,fields", [((128, 24, 384), F64, 5), ((128, 24, 384), F32, 5), ((100, 30, 512), F64, 5),
                                               ((32, 36, 1024), F32, 5), ((32, 36, 1024), F64, 6), ((128, 24, 128), F64, 6),
                                               # short z lines in boxes of too many for the joined pass
                                               ((192, 192, 96), F64, 6), ((192, 192, 96), F32, 6), ((512, 48, 96), F64, 5),
                                               ((512, 60, 128), F32, 5)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_fields_through_z(oracle_mod, shape, prec, fields):
    note(f"{shape} bfrot precision {prec}: {fields} fields through z; 3 steps")
    _compare(oracle_mod, *shape, prec, FORMS["bfrot"], 3, 100, dict(plane_groups=0, joined=0, z_fields=fields))
