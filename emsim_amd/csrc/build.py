"""Build the gfx950 HIP library ``emsim_amd/backend/hip_ext/libemsim_hip.so``.

Usage: python emsim_amd/csrc/build.py [--verbose]

hipcc cross-compiles for gfx950 without a GPU present.  Packed-FP32 VALU
instructions are disabled for all device code.
"""
import os
import subprocess
import sys
import time
from pathlib import Path

HERE = Path(__file__).resolve().parent
PKG = HERE.parent
OUT_DIR = PKG / "backend" / "hip_ext"
LIB = OUT_DIR / "libemsim_hip.so"
SOURCES = [HERE / "emsim_hip.hip", HERE / "fno.hip"]
DEPS = SOURCES + sorted(HERE.glob("*.hpp")) + [PKG.parent / "include" / "emsim_hip.h"]

ARCH = os.environ.get("EMSIM_HIP_ARCH", "gfx950")

FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (Path(cand).exists() or cand == "hipcc"):
            return cand
    raise RuntimeError("hipcc not found")


def build(verbose: bool = False) -> Path:
    OUT_DIR.mkdir(parents=True, exist_ok=True)
    tmp = LIB.with_suffix(".so.tmp")
    t0 = time.time()
    objs = [OUT_DIR / (src.stem + ".o") for src in SOURCES]
    cmds = [[hipcc(), *FLAGS, "-c", str(src), "-o", str(obj)] for src, obj in zip(SOURCES, objs)]
    if verbose:
        for cmd in cmds:
            print(" ".join(cmd), flush=True)
    procs = [subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
             for cmd in cmds]
    outs = [proc.communicate()[0] for proc in procs]
    for proc, out in zip(procs, outs):
        if proc.returncode != 0:
            sys.stderr.write(out)
            raise RuntimeError(f"hipcc failed with exit code {proc.returncode}")
    res = subprocess.run([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs),
                          "-o", str(tmp)], capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"hipcc link failed with exit code {res.returncode}")
    for obj in objs:
        obj.unlink()
    os.replace(tmp, LIB)
    if verbose:
        noise = [ln for out in outs for ln in out.splitlines() if "packed-fp32-ops" not in ln]
        if noise:
            print("\n".join(noise))
        print(f"built {LIB} in {time.time() - t0:.1f}s", flush=True)
    return LIB


if __name__ == "__main__":
    build(verbose="--verbose" in sys.argv or "-v" in sys.argv)
