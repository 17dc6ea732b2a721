"""Builds ``libwalrus_hip.so`` (HIP kernels + C ABI) for gfx950 with hipcc, in-tree.

Run ``python -m thewalrus_amd._build`` (or ``__graft_entry__.build()``).  Each ``.hip`` source
is compiled separately and linked into one shared library next to this file.
"""
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
LIB = os.path.join(HERE, "libwalrus_hip.so")
OBJDIR = os.path.join(HERE, "_obj")

SOURCES = ["capi.hip", "sieve_generic.hip", "sieve_pm1.hip", "sieve_pm1m.hip", "sieve_pm1s.hip", "sieve_call.hip", "sieve_sym.hip", "sieve_rep4.hip", "sieve_lhb.hip", "montrealer.hip", "hermite.hip"]

HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-variable",
    # keep packed FP32 instructions out of the device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + INCLUDE,
    "-I" + CSRC,
]


def _compile(src, objdir=OBJDIR, defines=()):
    obj = os.path.join(objdir, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + FLAGS + ["-D" + d for d in defines] + ["-c", os.path.join(CSRC, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s\n%s" % (src, res.stdout, res.stderr))
    return obj


def build(verbose=False, out=LIB, defines=()):
    """Compile every HIP source and link the shared library; returns its path.

    ``defines`` (e.g. ``["WH_PM1_KUNROLL=4"]``) build a variant into ``out``."""
    objdir = OBJDIR if out == LIB else out + ".obj"
    os.makedirs(objdir, exist_ok=True)
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with ThreadPoolExecutor(max_workers=min(4, len(srcs))) as ex:
        objs = list(ex.map(lambda s: _compile(s, objdir, defines), srcs))
    tmp = out + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n%s\n%s" % (res.stdout, res.stderr))
    os.replace(tmp, out)
    if verbose:
        print("built", out)
    return out


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
