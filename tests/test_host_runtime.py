"""The library's host code on a stand-in for the HIP runtime (tests/host_runtime): what an
entry point does when a runtime call fails, and what it asks the runtime for.  Each case runs
in a process of its own, where the stand-in is loaded first; no GPU is used, kernels do not
run, so values are checked only where copies alone carry them."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PROLOGUE = """
import ctypes as C, os, sys
S = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
S.stand_in_fail.argtypes = [C.c_char_p, C.c_longlong, C.c_int]
S.stand_in_count.argtypes, S.stand_in_count.restype = [C.c_char_p], C.c_longlong
S.stand_in_bytes.argtypes, S.stand_in_bytes.restype = [C.c_int], C.c_longlong
S.stand_in_loaded_kernels.restype = C.c_longlong
sys.path.insert(0, {pkg!r})
import numpy as np
import pandora_amd as pa

def fail(call, nth=1, error=999):
    S.stand_in_fail(call.encode(), nth, error)
def count(call):
    return S.stand_in_count(call.encode())
def raises(f, *a):
    try:
        f(*a)
    except pa.PdrError as e:
        return e.code
    return 0
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("host_runtime") / "libhip_stand_in.so")
    subprocess.run(["g++", "-O1", "-Wall", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "host_runtime", "hip_stand_in.cpp"), "-o", lib], check=True)
    return lib


def _run(lib, body, **env):
    code = PROLOGUE.format(lib=lib, pkg=os.path.join(os.path.dirname(HERE), "pandora-2.0_amd")) + textwrap.dedent(body)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                       env={**os.environ, **env})
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


@pytest.mark.parametrize("call", ["hipGraphInstantiate", "hipStreamBeginCapture", "hipStreamCreateWithFlags"])
@pytest.mark.parametrize("tune", [False, True], ids=["set_split", "autotune"])
def test_ensemble_keeps_its_graphs_when_a_rebuild_fails(stand_in, call, tune):
    """Every step that a run reports has been queued, whichever call of whichever rebuild fails."""
    _run(stand_in, f"""
    sizes = [32, 96, 32, 128]
    e = pa.Ensemble([pa.Pandora(n, rk3_timestep=2, rk3_dt=0.25) for n in sizes])
    for nth in range(1, 60):
        fail({call!r}, nth)
        rc = raises(e.autotune, 1) if {tune} else raises(e.set_split, 1, 1)
        fail({call!r}, 0)
        before = count("hipGraphLaunch")
        assert list(e.run(1, 5, [0.0] * 4)) == [1.25] * 4
        assert count("hipGraphLaunch") - before == 5 * 3  # a graph a step for each of the three lengths
        if rc == 0:
            break
    assert nth > (8 if {tune} else 2)  # the failing cases came first
    """)


@pytest.mark.parametrize("n,prec", [(32, "PDR_FP64"), (32, "PDR_FP32_MIXED"), (96, "PDR_FP64"), (96, "PDR_FP32_MIXED")])
def test_transfers_without_pinned_memory(stand_in, n, prec):
    """Small states and states of several chunks, velocity and RK registers, four times over: they
    arrive whole where the host has no pinned memory left, and the box is usable afterwards."""
    _run(stand_in, f"""
    fail("hipHostMalloc", 1, 2)
    g = pa.Pandora({n}, precision=pa.{prec})
    rng = np.random.default_rng(1)
    for rep in range(4):
        u = [(rng.integers(-99, 99, g.shape) + 1j * rng.integers(-99, 99, g.shape)).astype(complex) for _ in range(3)]
        g.set_state(*u)
        assert all((a == b).all() for a, b in zip(g.get_state(), u))
        g.set_rk(*u[::-1])
        assert all((a == b).all() for a, b in zip(g.get_rk(), u[::-1]))
        g.run(rep + 1, 1, 0.0)  # launches that look at the runtime's last error
    assert count("hipHostMalloc") > 0 and S.stand_in_bytes(1) == 0
    """)


@pytest.mark.parametrize("n,prec", [(32, "PDR_FP64"), (32, "PDR_FP32_MIXED"), (96, "PDR_FP64"), (96, "PDR_FP32_MIXED")])
def test_transfers_with_another_device_current(stand_in, n, prec):
    """A program with boxes on two devices reads each whichever device is current, and finds the
    device that it had made current afterwards."""
    _run(stand_in, f"""
    boxes = []
    for dev in (0, 1):
        assert S.hipSetDevice(dev) == 0
        boxes.append(pa.Pandora({n}, precision=pa.{prec}))
        boxes[-1].set_particle_sort(0)
        boxes[-1].set_particles(np.linspace(0.1, 6.0, 3 * 70000).reshape(-1, 3))
    for dev in (1, 0):
        assert S.hipSetDevice(dev) == 0
        for g in boxes:
            u = [np.full(g.shape, 2.0 + k - 3.0j) for k in range(3)]
            g.set_state(*u)
            for rep in range(4):
                v = g.get_state()
                if {n} == 96:  # a small state's later downloads are a kernel's work
                    assert all((a == b).all() for a, b in zip(v, u))
                g.get_particles()
            assert S.stand_in_device() == dev
    """)


@pytest.mark.parametrize("prec", ["PDR_FP64", "PDR_FP32_MIXED"])
@pytest.mark.parametrize("mb,streams", [(1, 1), (2, 1), (2, 2)])
def test_chunked_box_holds_a_chunk(stand_in, prec, mb, streams):
    """The x-pencil buffers of a chunked box are one chunk (two with two in flight), the rest of
    the device memory is that of the whole-box run less its x-pencil buffer."""
    _run(stand_in, f"""
    n = (144, 128, 120)
    csz = 16 if pa.{prec} == pa.PDR_FP64 else 8
    plane = 6 * n[1] * (-(-(n[0] // 3 + 1) // 16) * 16) * csz
    size = {{}}
    for chunked in (False, True):
        if chunked:
            os.environ["PDR_ZCHUNK_MB"], os.environ["PDR_ZSTREAMS"] = "{mb}", "{streams}"
        g = pa.Pandora(nx=n[0], ny=n[1], nz=n[2], precision=pa.{prec})
        size[chunked] = int(g.sizes()[6])
        assert S.stand_in_bytes(0) == size[chunked]
        zc = g.kernel_forms()["zchunk"]
        assert zc == (max(1, min(n[2], {mb} * 1048576 // plane)) if chunked else n[2])
        g.close()
    assert size[True] == size[False] - (n[2] - {streams} * zc) * plane
    """)


@pytest.mark.parametrize("shape", [(32, 32, 32), (48, 48, 48), (64, 64, 64), (96, 96, 96), (256, 256, 256), (120, 48, 96)],
                         ids=lambda s: "x".join(map(str, s)))
def test_a_box_loads_the_code_of_its_lengths(stand_in, shape):
    """The runtime loads a code object whole, some 60 us for each kernel in it, at the first
    launch: the steps of a box load at most 32 kernels for each of its different lengths."""
    _run(stand_in, f"""
    n = {shape}
    g = pa.Pandora(nx=n[0], ny=n[1], nz=n[2], precision=pa.PDR_FP32_MIXED)
    g.run(1, 3, 0.0)
    print(S.stand_in_loaded_kernels())
    assert 0 < S.stand_in_loaded_kernels() <= 32 * len(set(n))
    """)


def test_what_a_small_box_is_made_of(stand_in):
    """One stream, with tracers as well; one copy for the tables; no query of the free memory for
    a box whose x-pencil chunk is the whole box; all given back."""
    _run(stand_in, """
    calls = ("hipStreamCreateWithFlags", "hipMemcpy", "hipMemGetInfo")
    before = [count(k) for k in calls]
    g = pa.Pandora(32, rk3_timestep=2)
    assert [count(k) - b for k, b in zip(calls, before)] == [1, 1, 0]
    g.set_particle_sort(0)
    for n in (100, 70000):
        g.set_particles(np.linspace(0.1, 6.0, 3 * n).reshape(-1, 3))
        g.run(1, 2, 0.0)
        g.get_state()
    assert count("hipStreamCreateWithFlags") == 1
    g.close()
    assert S.stand_in_bytes(0) == 0 and S.stand_in_bytes(1) == 0
    assert count("hipStreamCreateWithFlags") == count("hipStreamDestroy")
    """)


def test_routes_of_a_box(stand_in):
    """pdr_kernel_routes and the x rows of pdr_kernel_forms where the rules change: the length that
    fused planes end at, the groups that a plane's parts are spread over, joined stages (none with
    a truncation of the state), five fields through z (not with a frame that puts k3 into the last
    vorticity component, nor with the y pass's fields split), chunks, the runtime-radix kernels."""
    _run(stand_in, """
    F64, F32 = pa.PDR_FP64, pa.PDR_FP32_MIXED
    def routes(nx, ny, nz, prec, **kw):
        with pa.Pandora(nx=nx, ny=ny, nz=nz, precision=prec, **kw) as g:
            return tuple(g.kernel_routes().values()) + (g.kernel_forms()["xrows"],)
    sheared = dict(f_type=2, rk3_timestep=1, deform_s=1.0, remesh_t=4)
    # groups, parts, joined, fields through z, x rows
    for args, kw, want in [
        ((32, 32, 32, F64), {}, (4, 4, 1, 6, 8)),
        ((64, 64, 64, F64), {}, (4, 4, 1, 6, 16)),
        ((30, 30, 30, F64), {}, (1, 1, 1, 6, 30)),
        ((72, 72, 72, F64), {}, (0, 0, 1, 6, 8)),
        ((48, 48, 96, F64), {}, (3, 4, 1, 6, 12)),
        ((48, 48, 100, F64), {}, (0, 0, 0, 6, 16)),
        ((64, 64, 72, F64), {}, (0, 0, 1, 6, 16)),
        ((64, 64, 80, F32), {}, (4, 4, 1, 6, 16)),
        ((64, 64, 96, F32), {}, (0, 0, 1, 6, 16)),
        ((60, 60, 128, F32), {}, (2, 4, 1, 6, 15)),
        ((60, 60, 144, F32), {}, (0, 0, 0, 6, 16)),
        ((24, 24, 256, F64), {}, (1, 1, 0, 6, 24)),
        ((24, 24, 640, F64), {}, (1, 1, 0, 6, 24)),
        ((64, 60, 64, F64), {}, (0, 0, 1, 6, 16)),
        ((96, 96, 96, F64), {}, (0, 0, 1, 6, 8)),
        ((128, 128, 96, F64), {}, (0, 0, 0, 6, 4)),
        ((128, 128, 96, F32), {}, (0, 0, 1, 6, 4)),
        ((192, 192, 96, F32), {}, (0, 0, 0, 6, 4)),
        ((512, 48, 96, F64), {}, (0, 0, 0, 5, 2)),
        ((512, 512, 80, F64), {}, (0, 0, 1, 6, 2)),
        ((64, 60, 64, F64), {}, (0, 0, 1, 6, 16)),
        ((32, 32, 32, F64), dict(dealiasing=2), (4, 4, 0, 6, 8)),
        ((32, 32, 32, F64), dict(sheared, ns_deformed=2), (0, 0, 0, 6, 8)),
        ((50, 50, 50, F64), {}, (0, 0, 0, 6, 0)),
        ((50, 50, 50, F64), dict(sheared, ns_deformed=2), (0, 0, 0, 18, 0)),
        ((256, 256, 256, F64), {}, (0, 0, 0, 5, 2)),
        ((128, 24, 384, F32), sheared, (0, 0, 0, 5, 4)),
        ((128, 24, 384, F32), dict(sheared, ns_deformed=3), (0, 0, 0, 5, 4)),
        ((128, 24, 128, F64), sheared, (0, 0, 0, 6, 4)),
    ]:
        assert routes(*args, **kw) == want, (args, kw, routes(*args, **kw), want)
    with pa.Pandora(nx=128, ny=24, nz=384, ns_deformed=3, **sheared) as g:
        assert g.kernel_routes()["z_fields"] == 5
        b = np.eye(3)
        b[2, 0] = 0.25
        g.set_frame(b.T, np.eye(3))
        assert g.kernel_routes()["z_fields"] == 6
    os.environ["PDR_ZCHUNK_MB"] = "0.3"
    assert routes(32, 32, 32, F64) == (0, 0, 1, 6, 16)
    """)
