"""Build the MI355X RK3-step library (and the Fortran ISO_C_BINDING shim) in tree.

    python pandora-2.0_amd/build_lib.py

Outputs (git-ignored, shipped with the source tree):
    pandora-2.0_amd/lib/libpandora_amd.so     HIP kernels + C-ABI (include/pandora_amd.h)
    pandora-2.0_amd/lib/pdr_rk3_amd.o/.mod    Fortran shim module (if amdflang is present)
    pandora-2.0_amd/lib/pdr_fortran_driver    Fortran driver program using the shim
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
FSRC = os.path.join(PKG, "fortran")
LIB = os.path.join(PKG, "lib")
SO = os.path.join(LIB, "libpandora_amd.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FC = os.environ.get("PDR_FC", "/opt/rocm/bin/amdflang")
ARCH = "gfx950"


def spec_lengths():
    """The line lengths of PDR_SPEC_LENGTHS (pdr_spec.hpp)."""
    with open(os.path.join(CSRC, "pdr_spec.hpp")) as f:
        rows = re.search(r"#define PDR_SPEC_LENGTHS\(X\)((?:.*\\\n)*.*\n)", f.read()).group(1)
    return [int(n) for n in re.findall(r"X\((\d+)\)", rows)]


# (source, extra defines, object); the costliest first.  pdr_spec.hip is compiled once for
# each length and precision.
SOURCES = [("pdr_ens_passes.hip", [], "pdr_ens_passes.o")]
SOURCES += [("pdr_spec.hip", [f"-DPDR_SPEC_N={n}", f"-DPDR_SPEC_FP32={f}"], f"pdr_spec_{n}_f{32 if f else 64}.o")
            for n in sorted(spec_lengths(), reverse=True) for f in (0, 1)]
SOURCES += [(f"{s}.hip", [], f"{s}.o") for s in ("pdr_api", "pdr_kernels", "pdr_spec_dispatch", "pdr_host", "pdr_xfer", "pdr_stats",
                                                 "pdr_pstats", "pdr_sort", "pdr_ens")]


def _run(cmd, cwd=None):
    print("+", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True, cwd=cwd)


def build_hip(verbose: bool = True) -> str:
    """Compile every HIP source (in parallel, one hipcc per object) and link the library."""
    from concurrent.futures import ThreadPoolExecutor

    os.makedirs(LIB, exist_ok=True)
    cmds, objs = [], []
    for src, defines, name in SOURCES:
        obj = os.path.join(LIB, name)
        cmds.append([HIPCC, *defines, f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-c",
                     # no packed-FP32 instructions: some of their forms have given wrong results on gfx950
                     "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                     "-Wall", "-Wno-unused-parameter", "-Wno-unused-command-line-argument",
                     "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                     os.path.join(CSRC, src), "-o", obj])
        objs.append(obj)
    jobs = max(1, min(len(cmds), int(os.environ.get("MAX_JOBS", "0") or 0) or (os.cpu_count() or 1)))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        for f in [ex.submit(_run, cmd) for cmd in cmds]:
            f.result()
    tmp = SO + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs)
    os.replace(tmp, SO)
    return SO


def build_fortran() -> bool:
    """Compile the ISO_C_BINDING shim and its driver with amdflang, if present."""
    if not os.path.exists(FC) or not os.path.isdir(FSRC):
        print(f"[build] Fortran compiler {FC} not found; shim not built", flush=True)
        return False
    os.makedirs(LIB, exist_ok=True)
    shim = os.path.join(FSRC, "pdr_rk3_amd.f90")
    drv = os.path.join(FSRC, "pdr_fortran_driver.f90")
    _run([FC, "-O2", "-fPIC", "-c", shim, "-o", os.path.join(LIB, "pdr_rk3_amd.o"),
          "-module-dir", LIB])
    if os.path.exists(drv):
        _run([FC, "-O2", drv, os.path.join(LIB, "pdr_rk3_amd.o"), "-I", LIB,
              "-L", LIB, "-lpandora_amd", "-Wl,-rpath,$ORIGIN",
              "-o", os.path.join(LIB, "pdr_fortran_driver")])
    return True


def build() -> None:
    build_hip()
    build_fortran()


if __name__ == "__main__":
    build_hip()
    if "--no-fortran" not in sys.argv:
        build_fortran()
