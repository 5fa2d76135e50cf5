"""Builds libdmgx.so (HIP kernels for gfx950 + C++ host + the C ABI) in-tree.

Usage: python dmg-md_amd/build.py   (or __graft_entry__.build())
"""
from __future__ import annotations

import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libdmgx.so")
SOURCES = ["kernels.hip", "descriptor.hip", "neighbor.hip", "nep_model.cpp", "ensemble.cpp", "engine.cpp", "serve.cpp",
           "frontend.cpp", "noalloc.hip", "capi.cpp"]
DESCRIPTOR_GROUPS = 12  # descriptor_instances.hip is compiled once per group
ARCH = os.environ.get("DMGX_OFFLOAD_ARCH", "gfx950")


def compile_commands(out_dir: str) -> list:
    """(command, object) per translation unit."""
    hipcc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    flags = [
        hipcc, f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-c",
        # packed FP32 (v_pk_*_f32) stays off: scalar FP32 only
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-Wno-unused-command-line-argument", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
    ]
    units = [(["-DDMGX_DESCRIPTOR_GROUP=%d" % g], "descriptor_instances.hip", "descriptor_%d.o" % g)
             for g in range(DESCRIPTOR_GROUPS)]
    units += [([], s, s.replace(".", "_") + ".o") for s in SOURCES]
    return [(flags + d + [os.path.join(CSRC, s), "-o", os.path.join(out_dir, o)], os.path.join(out_dir, o))
            for d, s, o in units]


def link_command(objects: list, out: str) -> list:
    hipcc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    return [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,-z,defs", *objects, "-o", out]


CLI = os.path.join(HERE, "dmgx-run")


def cli_command(out: str = CLI) -> list:
    """The dmgx-run executable: a thin C++ caller of dmgx_run_directory."""
    return ["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "include"), os.path.join(CSRC, "dmgx_run.cpp"),
            "-L", HERE, "-ldmgx", "-Wl,-rpath,$ORIGIN", "-o", out]


def _run(cmd: list, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed building {cmd[-1]}")


def build(verbose: bool = False) -> str:
    with tempfile.TemporaryDirectory(prefix="dmgx_build_") as d:
        units = compile_commands(d)
        workers = min(len(units), int(os.environ.get("MAX_JOBS", 0)) or os.cpu_count() or 1, 16)
        with ThreadPoolExecutor(workers) as pool:
            list(pool.map(lambda u: _run(u[0], verbose), units))
        _run(link_command([o for _, o in units], LIB + ".tmp"), verbose)
    os.replace(LIB + ".tmp", LIB)
    _run(cli_command(CLI + ".tmp"), verbose)
    os.replace(CLI + ".tmp", CLI)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
