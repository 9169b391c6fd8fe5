"""Builds the gfx950 HIP library ``libaship.so`` in-tree with hipcc."""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libaship.so")
SOURCES = ["aship.hip", "generic.hip", "generic_columns_short.hip", "generic_columns_8.hip",
           "generic_columns_16.hip", "generic_columns_32.hip"]

# Packed-FP32 VALU forms are disabled for every HIP translation unit.
HIPCC_FLAGS = [
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the HIP library cannot be built")


def build(verbose: bool = False) -> str:
    """Compiles the library (always, even if one exists) and returns its path.

    The translation units compile side by side and are linked into ``libaship.so``."""
    inc = ["-I", os.path.join(HERE, "..", "include")]
    with tempfile.TemporaryDirectory(prefix="aship_build_") as objdir:
        objs, procs = [], []
        for src in SOURCES:
            objs.append(os.path.join(objdir, src + ".o"))
            cmd = [hipcc()] + HIPCC_FLAGS + inc + ["-c", os.path.join(CSRC, src), "-o", objs[-1]]
            if verbose:
                print(" ".join(cmd), file=sys.stderr)
            procs.append(subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True))
        logs = [(p.communicate()[0], p.returncode) for p in procs]
        if any(rc != 0 for _, rc in logs):
            raise RuntimeError("hipcc failed:\n" + "".join(text for text, rc in logs if rc != 0))
        tmp = LIB + ".tmp"
        cmd = [hipcc(), "--offload-arch=gfx950", "-shared"] + objs + ["-o", tmp]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("hipcc failed to link:\n" + r.stdout + r.stderr)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
