"""Every line length an ensemble takes, three members of each at a time in uneven order, so
that each runs its own chain of launches (planes as one kernel and joined stages up to 64
points, the separate passes above): one run of several steps, runs of one step and a run
after a new state, against the same members stepped one by one."""
import sys

import numpy as np
import pytest

import pandora_amd as pa
from conftest import rel

pytestmark = pytest.mark.gpu

KW = dict(nu=0.01, rk3_timestep=2, rk3_dt=0.005)
ORDER = [64, 32, 256, 48, 128, 32, 96, 192, 64, 48, 32]


def note(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("prec", [pa.PDR_FP64, pa.PDR_FP32_MIXED], ids=["fp64", "fp32"])
def test_lengths_against_single_boxes(prec):
    note(f"ensemble of {ORDER}, precision {prec}")
    tol = 1e-6 if prec == pa.PDR_FP32_MIXED else 1e-13
    ens = [pa.Pandora(n, precision=prec, **KW) for n in ORDER]
    one = [pa.Pandora(n, precision=prec, **KW) for n in ORDER]
    e = pa.Ensemble(ens)
    t = np.zeros(len(ORDER))
    for seed, chunks in ((1, (4, 1, 1)), (2, (1, 2))):
        for g, o, n in zip(ens, one, ORDER):
            u = pa.init_field_host(n, seed + n, 0.5, 4.0)
            g.set_state(*u)
            o.set_state(*u)
        for steps in chunks:
            t = e.run(1, steps, t)
        for g, o in zip(ens, one):
            o.run(1, sum(chunks), 0.0)
            for a, b in zip(g.get_state(), o.get_state()):
                assert rel(a, b) < tol
    assert np.allclose(t, 9 * KW["rk3_dt"], rtol=1e-14)
    e.close()
    for g in ens + one:
        g.close()
