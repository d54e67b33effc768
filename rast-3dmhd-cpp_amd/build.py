"""Builds libmhd3d.so (HIP, gfx950) in-tree: rast-3dmhd-cpp_amd/lib/libmhd3d.so.

Every source under csrc/ (.hip device + host code, .cpp host code) is compiled
to an object in parallel, then the objects are linked into one library.
"""
import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
SOURCES = [os.path.join(CSRC, f)
           for f in ("mhd3d.hip", "mixed.hip", "mixed_ensemble.hip", "ext_stream.hip", "ext_mixed.hip", "dumpio.cpp",
                     "static_state.cpp")]
OUT_DIR = os.path.join(HERE, "lib")
OBJ_DIR = os.path.join(HERE, "lib", "obj")
OUT = os.path.join(OUT_DIR, "libmhd3d.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # parity: no contraction into FMA, same rounding as the reference's x86-64 build
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
    # the 2-wave one-barrier variants of the FP64 MHD stage kernels (kept for
    # the autotuner) need more registers than 2 waves allow; the compiler
    # builds them for 1 wave and says so for each
    "-Wno-pass-failed",
]
# per-source additions: the mixed form's single-domain FP32 kernels measured
# fastest with the instruction-level-parallelism scheduler (MI355X,
# 512x512x256 MHD stage kernel 3.28 ms against 3.35 ms with the default one);
# the ensemble's FP32 kernels (mixed_ensemble.hip) keep the default
SOURCE_FLAGS = {
    "mixed.hip": ["-mllvm", "-amdgpu-sched-strategy=max-ilp"],
}

# The compiler's report of each kernel's registers, for check_walls.
USAGE = "kernel-resource-usage"
USAGE_FLAGS = ["-Rpass-analysis=" + USAGE, "-fno-caret-diagnostics"]

# stage_stream_kernel with the wall points (its last template argument true),
# the stage launch that also takes the walls and closes the step: its builds in
# each source -- hydro and magnetic, with and without rotation, three stages.
WALLS = re.compile(r"stage_stream_kernelI[df](?:Lb[01]E){2}Li\dELi\dE(?:Lb[01]E){3}Li\d+ELb[01]ELb1EE")
WALL_KERNELS = {"mhd3d.hip": 12, "mixed.hip": 12}


def kernel_usage(text):
    """{kernel: {"VGPRs": n, "AGPRs": n, ...}} from the compiler's remarks."""
    out, cur = {}, None
    for line in text.splitlines():
        m = re.search(r"remark:\s*(.+?): (\S+) \[-Rpass-analysis=" + USAGE, line)
        if not m:
            continue
        if m.group(1) == "Function Name":
            cur = out.setdefault(m.group(2), {})
        elif cur is not None and m.group(2).isdigit():
            cur[re.sub(r" \[.*", "", m.group(1))] = int(m.group(2))
    return out


def check_walls(usage):
    """Number of kernels with the wall points in `usage`; refuses one whose
    values do not fit the vector registers.  While that launch was being
    written, a build of a variant that kept values in accumulation registers
    flagged finite states as non-finite.  The same variant of the present
    source does not, so the cause is not known, and 251 of 256 registers in the
    FP64 magnetic stage 3 are too close to leave it to the next compiler."""
    walls = {k: u for k, u in usage.items() if WALLS.search(k)}
    for k, u in walls.items():
        over = {r: u[r] for r in ("AGPRs", "ScratchSize", "VGPRs Spill") if u[r] != 0}
        if over:
            raise RuntimeError(f"{k}: {over}: the stage launch with the walls must fit the vector registers")
    return len(walls)


def _compile(src, extra, verbose):
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, *SOURCE_FLAGS.get(os.path.basename(src), []), *extra, "-c", src, "-o", obj]
    if src.endswith(".cpp"):
        cmd = [HIPCC, "-O3", "-std=c++17", "-fPIC", "-Wno-unused-result", *extra, "-c", src, "-o", obj]
    else:
        cmd += USAGE_FLAGS
    if verbose:
        print(" ".join(cmd), flush=True)
    run = subprocess.run(cmd, stderr=subprocess.PIPE, text=True)
    include = []   # the "In file included from" lines of a diagnostic go with it
    for line in run.stderr.splitlines():
        if line.startswith("In file included from"):
            include.append(line)
            continue
        if USAGE not in line:
            print(*include, line, sep="\n", file=sys.stderr, flush=True)
        include = []
    run.check_returncode()
    n, want = check_walls(kernel_usage(run.stderr)), WALL_KERNELS.get(os.path.basename(src), 0)
    if n != want:
        raise RuntimeError(f"{src}: {n} stage kernels with the walls in the compiler's report, not {want}")
    return obj


def build(verbose=False, extra=()):
    os.makedirs(OBJ_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        objs = list(ex.map(lambda s: _compile(s, list(extra), verbose), SOURCES))
    tmp = OUT + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    build(verbose=True, extra=sys.argv[1:])
