"""Build the in-tree HIP library ``libposidonius_hip.so`` for gfx950.

``python -m posidonius_amd.build`` (or ``__graft_entry__.build()``) compiles
``csrc/posidonius_hip.hip`` with hipcc.  Flags:

* ``-ffp-contract=off``: every multiply and add rounds separately, as in the
  reference (Rust never fuses), which is what makes bitwise parity with the
  CPU oracle possible;
* ``-Xclang -target-feature -Xclang -packed-fp32-ops``: no packed-FP32
  instructions are generated;
* ``--offload-arch=gfx950``: MI355X only;
* ``-mllvm -amdgpu-sched-strategy=iterative-maxocc``: the machine scheduler
  variant that measured fastest for the step kernel (3.15e8 vs 3.01e8
  system-steps/s with the default strategy on the 65,536-system ensemble).
  Scheduling reorders instructions only; results are bitwise unchanged;
* ``-save-temps=obj``: the device listing is kept for `partial_spills`.
"""
from __future__ import annotations

import glob
import os
import re
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc", "posidonius_hip.hip")
HEADERS = [*(os.path.join(HERE, "csrc", h) for h in ("whfast_step.hpp", "whfast_fixed.hpp", "adjoint_math.hpp",
                                                     "adjoint_kernels.hpp", "adjoint_sweep.hpp", "crmath.hpp")),
           os.path.join(os.path.dirname(HERE), "include", "posidonius_hip.h")]
OUT = os.path.join(HERE, "libposidonius_hip.so")
ARCH = os.environ.get("POSIDONIUS_OFFLOAD_ARCH", "gfx950")


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def partial_spills(listing: str) -> list[str]:
    """Vector registers saved or copied where a divergent branch has joined but
    its lanes are still switched off, as "kernel label: instruction".

    The register allocator of ROCm 7.2 can put a spill at the top of a join
    block, before the ``s_or_b64 exec, exec`` that restores the lanes that
    skipped the branch: those lanes never store the value and later reload what
    the slot held.  (It did for the number of the lane's system at
    ``act && (...)`` in whfast_fixed_kernel with one wavefront a set: a system
    stopped before the launch stored its time over another's, or out of range.)
    Nothing in the source is wrong then, so the listing is looked through: a
    label that an ``s_cbranch_execz`` jumps to, then vector instructions before
    the restore.  A region that two branches leave early may also end so, but
    after arithmetic of its own, which a join has none of.
    """
    found = []
    for m in re.finditer(r"^(_Z\w+):.*?$(.*?)^\.Lfunc_end", listing, re.M | re.S):
        joins = set(re.findall(r"s_cbranch_execz (\.LBB\w+)", m[2]))
        label, early = None, []
        for line in m[2].splitlines():
            code = line.split(";")[0].strip()
            if q := re.match(r"(\.LBB\w+):", line):
                label, early = (q[1] if q[1] in joins else None), []
            elif not label or not code:
                continue
            elif re.match(r"s_or_b64 exec, exec", code):
                found += [f"{m[1]} {label}: {e}" for e in early]
                label = None
            elif re.match(r"s_c?branch|s_endpgm|s_\w+ exec\b|s_\w+_saveexec", code):
                label = None
            elif re.match(r"scratch_|v_accvgpr_|v_mov_b(32|64)\w* [va]\S+, [va]", code):
                early.append(line.strip())
            elif re.match(r"v_(?!readlane|writelane|readfirstlane)|global_|flat_|ds_|buffer_", code):
                label = None
    return found


def build_library(verbose: bool = False, extra_flags=None) -> str:
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-shared",
           "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-mllvm", "-amdgpu-sched-strategy=iterative-maxocc",
           "-Wall", "-Wno-unused-function",
           "-I", os.path.join(os.path.dirname(HERE), "include"), "-save-temps=obj", SRC]
    if extra_flags:
        cmd[1:1] = list(extra_flags)
    with tempfile.TemporaryDirectory() as temps:
        built = os.path.join(temps, os.path.basename(OUT))
        cmd += ["-o", built]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
        listings = glob.glob(os.path.join(temps, "*amdgcn*.s"))
        if not listings:
            raise RuntimeError("no device listing in " + temps)
        for path in listings:
            with open(path) as f:
                if found := partial_spills(f.read()):
                    raise RuntimeError("registers spilled under a partial mask:\n" + "\n".join(found))
        shutil.copy(built, OUT + ".tmp")
    os.replace(OUT + ".tmp", OUT)
    return OUT


CLI_SRC = os.path.join(HERE, "host", "posidonius_cli.cpp")
CLI_OUT = os.path.join(HERE, "posidonius-hip")


def build_cli(verbose: bool = False) -> str:
    """The `posidonius-hip start|resume` host, linked against the library."""
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(os.path.dirname(HERE), "include"), CLI_SRC,
           "-o", CLI_OUT + ".tmp", "-L", HERE, "-lposidonius_hip", "-Wl,-rpath,$ORIGIN",
           "-L", os.path.join(rocm, "lib"), "-Wl,-rpath," + os.path.join(rocm, "lib")]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(CLI_OUT + ".tmp", CLI_OUT)
    return CLI_OUT


if __name__ == "__main__":
    print(build_library(verbose=True, extra_flags=sys.argv[1:]))
    print(build_cli(verbose=True))
