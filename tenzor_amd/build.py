"""Build libtenzor_hip.so (gfx950) in-tree with hipcc.

Every source under tenzor_amd/csrc is compiled as HIP for gfx950 only and
linked into tenzor_amd/libtenzor_hip.so, which travels with the repository
snapshot to the GPU box.  `python -m tenzor_amd.build` rebuilds it.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libtenzor_hip.so"
SOURCES = ["runtime.cpp", "safetensors.cpp", "ew.hip", "gemm.hip", "gemm_pipe.hip", "ew_jit.cpp", "attention.hip", "arctic.hip",
           "tokenizer.cpp", "embed.hip", "tenzor_file.cpp", "gemm_fp.hip", "mlp.hip", "linear_small.hip"]

# -ffp-contract=off: every multiply and add rounds separately unless a kernel
# asks for an FMA explicitly (bit-exact elementwise chains).
# -packed-fp32-ops off: no v_pk_*_f32 in generated code.
# -amdgpu-mfma-vgpr-form: MFMA accumulators live in ordinary VGPRs; with the
# accumulation-register form the compiler copied every accumulator between
# the two register files around each pipeline stage of the GEMM.
HIPFLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
    "-Wall",
    "-Wno-unused-result",
    "-Wno-unused-function",
    "-Wno-inline-asm",  # M0 is written by the direct-to-LDS load asm on purpose
]


# Per-source additions.  attention.hip: its scores are finite or -inf by
# construction, and with NaNs honoured every fmaxf of an MFMA or permlane
# result gets an extra quieting v_max per operand.
EXTRA_FLAGS = {"attention.hip": ["-fno-honor-nans"]}


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; cannot build libtenzor_hip.so")
    return exe


def scratch_spills(remarks: str) -> list[tuple[str, int]]:
    """(kernel, bytes per lane) for every kernel the compiler's
    kernel-resource-usage remarks report with a non-zero scratch size."""
    out, name = [], None
    for line in remarks.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            continue
        m = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if m and name and int(m.group(1)) > 0:
            out.append((name, int(m.group(1))))
    return out


def _compile(src: str) -> Path:
    obj = BUILD / (Path(src).stem + ".o")
    cmd = [hipcc(), "-x", "hip", *HIPFLAGS, *EXTRA_FLAGS.get(src, []), "-Rpass-analysis=kernel-resource-usage", "-c",
           str(CSRC / src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"compile of {src} failed:\n{res.stderr}")
    # The pipelined GEMM tracks its direct-to-LDS loads with explicit vmcnt
    # counts; compiler spill traffic would be vector memory ops it does not
    # plan for, so no kernel may spill to scratch.
    spills = scratch_spills(res.stderr)
    if spills:
        raise RuntimeError(f"{src}: kernels spill to scratch: {spills}")
    return obj


def build(jobs: int | None = None, verbose: bool = False) -> Path:
    """Compile every source and link the shared library; returns its path."""
    BUILD.mkdir(exist_ok=True)
    jobs = jobs or min(len(SOURCES), os.cpu_count() or 4, 8)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs),
           "-L/opt/rocm/lib", "-lhiprtc"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


def build_host_tests(verbose: bool = False) -> Path:
    """Compile the C++ host-API parity test (tests/cpp/test_host_api.cpp)
    against the built library and the CPU oracle (its checker)."""
    root = Path(__file__).resolve().parent.parent
    src = root / "tests" / "cpp" / "test_host_api.cpp"
    exe = root / "tests" / "cpp" / "test_host_api"
    cmd = ["g++", "-std=c++17", "-O2", "-Wall", str(src), "-o", str(exe),
           f"-L{root / 'tenzor_amd'}", "-ltenzor_hip", f"-L{root / 'oracle'}", "-loracle",
           "-Wl,-rpath,$ORIGIN/../../tenzor_amd:$ORIGIN/../../oracle"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"host test build failed:\n{res.stderr}")
    if verbose:
        print(f"built {exe}")
    return exe


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
