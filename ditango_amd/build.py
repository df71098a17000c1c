"""Build libditango_hip.so (gfx950) in-tree with hipcc.

``python -m ditango_amd.build`` compiles every translation unit under
``ditango_amd/csrc`` and links ``ditango_amd/lib/libditango_hip.so`` (the drop-in
library), ``ditango_amd/lib/_ditango_host.so`` (the Python extension module of ``csrc/host_binding.cpp``, host code
only) and ``ditango_amd/lib/libditango_probes.so`` (the benchmark's measurement
aids, a library of its own that only ``bench.py`` loads).  hipcc
cross-compiles for gfx950 without a GPU.  Packed-FP32 instruction selection is
switched off for all device code (``-target-feature -packed-fp32-ops``).
"""
from __future__ import annotations

import json
import os
import re
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
LIB_DIR = PKG / "lib"
LIB_PATH = LIB_DIR / "libditango_hip.so"
HOST_PATH = LIB_DIR / "_ditango_host.so"             # Python extension: the host side of the launches (csrc/host_binding.cpp)
PROBES_PATH = LIB_DIR / "libditango_probes.so"
DEMO_PATH = LIB_DIR / "dt_capi_demo"
RESOURCES_PATH = LIB_DIR / "kernel_resources.json"   # per-kernel registers / scratch / occupancy of the last build
SOURCES = ["attn_fwd.hip", "attn_f32.hip", "state_ops.hip", "producer.hip", "qkv.hip", "capi.hip"]
PROBE_SOURCES = ["probes.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
COMMON = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{ROOT / 'include'}", f"-I{CSRC}",
]


def _run(cmd):
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(map(str, cmd)) + "\n" + res.stdout + res.stderr)
    return res


def parse_resource_remarks(text: str) -> dict:
    """``{kernel symbol: {"VGPRs": n, "ScratchSize [bytes/lane]": n, ...}}`` from the compiler's
    ``-Rpass-analysis=kernel-resource-usage`` remarks."""
    out, cur = {}, None
    for line in text.splitlines():
        m = re.search(r"remark:\s+Function Name: (\S+)", line)
        if m:
            cur = out.setdefault(m.group(1), {})
            continue
        m = re.search(r"remark:\s+([A-Za-z][^:]*): (-?\d+)", line)
        if m and cur is not None:
            cur[m.group(1).strip()] = int(m.group(2))
    return out


def build_lib(verbose: bool = False, extra_flags=()) -> Path:
    """Compile and link the library unconditionally; returns its path."""
    LIB_DIR.mkdir(exist_ok=True)
    objs = []

    resources = {}

    def compile_one(src):
        obj = LIB_DIR / (Path(src).stem + ".o")
        # the resource remarks (registers, scratch, occupancy per kernel) come with the compilation at no cost
        cmd = [HIPCC, *COMMON, *extra_flags, "-Rpass-analysis=kernel-resource-usage", "-c", str(CSRC / src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        resources[src] = parse_resource_remarks(_run(cmd).stderr)
        return obj

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    host_obj = LIB_DIR / "host_binding.o"
    host_compile = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-DTORCH_EXTENSION_NAME=_ditango_host",
                    f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{ROOT / 'include'}",
                    f"-I{sysconfig.get_paths()['include']}", *(f"-I{d}" for d in include_paths()),
                    "-c", str(CSRC / "host_binding.cpp"), "-o", str(host_obj)]
    host_link = [host_compile[0], "-shared", str(host_obj), *(f"-L{d}" for d in library_paths()), "-ltorch", "-ltorch_cpu",
                 "-lc10", "-ltorch_python", f"-L{LIB_DIR}", "-lditango_hip", "-Wl,-rpath,$ORIGIN", "-o", str(HOST_PATH)]
    if verbose:
        print(" ".join(host_compile), flush=True)
    with ThreadPoolExecutor(max_workers=7) as ex:
        host = ex.submit(_run, host_compile)
        all_objs = list(ex.map(compile_one, SOURCES + PROBE_SOURCES))
        host.result()
    objs, probe_objs = all_objs[:len(SOURCES)], all_objs[len(SOURCES):]
    # a version script keeps everything but the C entry points out of the dynamic symbol table
    for out, members, exports in ((LIB_PATH, objs, "exports_hip.map"), (PROBES_PATH, probe_objs, "exports_probes.map")):
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", f"-Wl,--version-script={CSRC / exports}",
               *map(str, members), "-o", str(out)]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)
    if verbose:
        print(" ".join(host_link), flush=True)
    _run(host_link)
    RESOURCES_PATH.write_text(json.dumps(resources, indent=1, sort_keys=True) + "\n")
    # a host program that uses nothing but the C header and the HIP runtime (tests/test_capi_demo_gpu.py runs it)
    cmd = [HIPCC, "-O2", "-std=c++17", "-Wno-unused-result", f"-I{ROOT / 'include'}", str(CSRC / "capi_demo.cpp"),
           f"-L{LIB_DIR}", "-lditango_hip", "-Wl,-rpath,$ORIGIN", "-o", str(DEMO_PATH)]
    if verbose:
        print(" ".join(cmd), flush=True)
    _run(cmd)
    return LIB_PATH


if __name__ == "__main__":
    path = build_lib(verbose=True)
    print(f"built {path}")
    sys.exit(0)
