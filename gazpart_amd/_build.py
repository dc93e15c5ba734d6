"""Compile the HIP library for gfx950 in-tree (gazpart_amd/libgazpart_gpu.so)."""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc", "gp_lib.hip")
SRCS = [SRC, os.path.join(HERE, "csrc", "gp_dns.hip")]
LIBS = ["-L/opt/rocm/lib", "-lrocfft", "-Wl,-rpath,/opt/rocm/lib"]
OUT = os.path.join(HERE, "libgazpart_gpu.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed FP32 instructions are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def build(verbose: bool = False) -> str:
    # one object a source, side by side, then the link
    objs = [os.path.join(HERE, os.path.basename(s)[:-4] + ".o") for s in SRCS]
    cmds = [[HIPCC, *FLAGS, "-c", s, "-o", o] for s, o in zip(SRCS, objs)]
    procs = []
    for c in cmds:
        if verbose:
            print(" ".join(c), file=sys.stderr)
        procs.append(subprocess.Popen(c, stderr=subprocess.PIPE, text=True))
    errs = [p.communicate()[1] for p in procs]
    for p, e in zip(procs, errs):
        if p.returncode != 0:
            raise RuntimeError(f"hipcc failed:\n{e[-4000:]}")
    link = [HIPCC, "--offload-arch=gfx950", "-shared", *objs, *LIBS, "-o", OUT + ".tmp"]
    r = subprocess.run(link, capture_output=True, text=True)
    for o in objs:
        os.remove(o)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed:\n{r.stderr[-4000:]}")
    os.replace(OUT + ".tmp", OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
