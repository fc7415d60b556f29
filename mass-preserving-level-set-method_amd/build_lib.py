"""Build recipe of the gfx950 library (and of the Fortran driver that links it).

    python mass-preserving-level-set-method_amd/build_lib.py

hipcc cross-compiles for gfx950 without a GPU.  Packed-FP32 instructions are
switched off for all device code (-packed-fp32-ops).
"""
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "liblsmp.so")
FDIR = os.path.join(HERE, "fortran")
DRIVER = os.path.join(LIB_DIR, "lsmp_driver")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]
SOURCES = ["lsmp_kernels.hip", "lsmp_host.hip", "lsmp_learn.hip", "lsmp_metrics.hip", "lsmp_clsvof.hip",
           "lsmp_noalloc.hip", "lsmp_redis.hip", "lsmp_redis2d.hip", "lsmp_redis_box.hip", "lsmp_adv_tile.hip", "lsmp_energy.hip"]


def _run(cmd, cwd=None):
    r = subprocess.run(cmd, cwd=cwd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops' is not a recognized feature" not in l
                    and "(ignoring feature)" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{out}")
    return out


def build_library(verbose=False):
    """Each translation unit compiles in its own hipcc process (in parallel),
    then one link step makes the shared library."""
    from concurrent.futures import ThreadPoolExecutor

    os.makedirs(LIB_DIR, exist_ok=True)
    obj_dir = os.path.join(LIB_DIR, "obj")
    os.makedirs(obj_dir, exist_ok=True)
    cflags = [f for f in HIP_FLAGS if f != "-shared"]
    objs = [os.path.join(obj_dir, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    with ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        outs = list(ex.map(lambda so: _run([HIPCC] + cflags + ["-c", os.path.join(CSRC, so[0]), "-o", so[1]]),
                           zip(SOURCES, objs)))
    tmp = LIB + ".tmp"
    outs.append(_run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs))
    os.replace(tmp, LIB)
    out = "\n".join(o for o in outs if o.strip())
    if verbose and out.strip():
        print(out)
    return LIB


def build_driver(verbose=False):
    """The Fortran driver (ISO_C_BINDING) that replaces the reference's
    main.f90 time loop around the library.  Skipped when flang is absent."""
    flang = shutil.which("flang") or shutil.which("amdflang")
    srcs = [os.path.join(FDIR, f) for f in ("lsmp_mod.f90", "lsmp_cases.f90", "lsmp_driver.f90")]
    if not flang or not all(os.path.exists(s) for s in srcs):
        return None
    mod = os.path.join(LIB_DIR, "mod")
    os.makedirs(mod, exist_ok=True)
    cmd = [flang, "-O2", "-J", mod] + srcs + ["-o", DRIVER, "-L" + LIB_DIR, "-llsmp",
                                             "-Wl,-rpath,$ORIGIN"]
    out = _run(cmd)
    if verbose and out.strip():
        print(out)
    return DRIVER


if __name__ == "__main__":
    print(build_library(verbose=True))
    d = build_driver(verbose=True)
    if d:
        print(d)
    sys.exit(0)
