"""Builds libkge_mi355.so from cuke_amd/csrc/*.hip with hipcc for gfx950, and beside it _host.so, the
Python binding's native host path (csrc/host.cpp, g++ against the installed torch's headers).

Both are built in-tree (cuke_amd/) so that they travel with the source tree; nothing is compiled at
import time.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "csrc", "build")
LIB = os.path.join(HERE, "libkge_mi355.so")
HOST = os.path.join(HERE, "_host.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-attributes",
] + os.environ.get("KGE_EXTRA_HIPCC_FLAGS", "").split()


def sources() -> list[str]:
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str, force: bool) -> str:
    obj = os.path.join(OBJ, src[:-4] + ".o")
    deps = [os.path.join(CSRC, src), os.path.join(HERE, "..", "include", "kge_mi355.h")] + \
        [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hpp")]
    if not force and os.path.exists(obj) and all(os.path.getmtime(obj) > os.path.getmtime(d) for d in deps):
        return obj
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    msgs = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                     if "packed-fp32-ops" not in l and l.strip())
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{msgs}")
    if msgs:
        print(msgs, file=sys.stderr)
    return obj


def _compile_host(force: bool) -> str:
    import sysconfig
    from importlib.util import find_spec
    torch = os.path.dirname(find_spec("torch").origin)
    src, obj = os.path.join(CSRC, "host.cpp"), os.path.join(OBJ, "host.o")
    deps = [src, os.path.join(HERE, "..", "include", "kge_mi355.h")]
    if not force and os.path.exists(obj) and all(os.path.getmtime(obj) > os.path.getmtime(d) for d in deps):
        return obj
    inc = [f"-I{torch}/include", f"-I{torch}/include/torch/csrc/api/include", f"-I{sysconfig.get_paths()['include']}",
           "-I/opt/rocm/include"]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM", *inc, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed on host.cpp:\n" + r.stdout + r.stderr)
    return obj


def _link_host(obj: str) -> None:
    from importlib.util import find_spec
    lib = os.path.join(os.path.dirname(find_spec("torch").origin), "lib")
    cmd = ["g++", "-shared", "-o", HOST, obj, f"-L{lib}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", "-lamdhip64",
           f"-L{HERE}", "-l:libkge_mi355.so", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link of _host.so failed:\n" + r.stdout + r.stderr)


def build(force: bool = True, jobs: int = 8) -> str:
    os.makedirs(OBJ, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(_compile_host, force)
        objs = list(ex.map(lambda s: _compile(s, force), sources()))
        host_obj = host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    _link_host(host_obj)
    return LIB


if __name__ == "__main__":
    print(build(force="--incremental" not in sys.argv))
