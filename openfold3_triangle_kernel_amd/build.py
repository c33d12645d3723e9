"""Build recipe for the gfx950 shared library ``libtpf_amd.so``.

Every HIP source under ``csrc/`` is compiled with hipcc for gfx950 only and
linked into one C-ABI shared library that sits next to this file.  The
library exports plain ``extern "C"`` entry points (declared in
``include/tpf_amd.h``); Python reaches them through ``ctypes``.  A second
library, the Python extension ``_tpf_host.so`` (``csrc/host/``), runs the two
operators' host path for plain tensors on top of the first.
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sysconfig
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_NAME = "libtpf_amd.so"
LIB_PATH = PKG_DIR / LIB_NAME
HOST_SRC = CSRC / "host" / "torch_host.cpp"
HOST_NAME = "_tpf_host"
HOST_PATH = PKG_DIR / f"{HOST_NAME}.so"
BUILD_DIR = PKG_DIR / "_build"
ARCH = "gfx950"

# Packed FP32 VALU ops are disabled for all device code (hipcc -O3 otherwise
# forms v_pk_* f32 instructions from ordinary float code).
DEVICE_FLAGS = [
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    # Keep MFMA accumulators in ordinary VGPRs (no v_accvgpr copies around
    # the softmax / epilogue code that reads them).
    "-mllvm",
    "-amdgpu-mfma-vgpr-form",
]


# Per-source extra flags.  attention.hip: the kernels never test for NaN
# and take scores that are finite or -inf, so fmaxf needs no NaN quieting
# (without the flag every v_max of an MFMA result is preceded by a
# canonicalising v_max: six VALU instructions per 32 x 32 score block).
FILE_FLAGS = {"attention.hip": ["-fno-honor-nans"]}


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found: the TurboPairFormer MI355X library needs ROCm's hipcc")


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.cpp"))


def build(verbose: bool = False, jobs: int | None = None) -> Path:
    """Compile every source and link ``libtpf_amd.so`` and ``_tpf_host.so`` (always
    rebuilds)."""
    import torch  # the host extension compiles against torch's headers

    hipcc = _hipcc()
    BUILD_DIR.mkdir(exist_ok=True)
    common = [
        "-O3",
        "-std=c++17",
        "-fPIC",
        f"--offload-arch={ARCH}",
        f"-I{CSRC}",
        f"-I{PKG_DIR.parent / 'include'}",
        "-Wno-unused-command-line-argument",
    ]
    objs = []
    cmds = []
    for src in sources():
        obj = BUILD_DIR / (src.stem + ".o")
        objs.append(obj)
        extra = (DEVICE_FLAGS + FILE_FLAGS.get(src.name, [])) if src.suffix == ".hip" else []
        lang = ["-x", "hip"] if src.suffix == ".hip" else []
        cmds.append([hipcc, *common, *extra, *lang, "-c", str(src), "-o", str(obj)])
    torch_dir = Path(torch.__file__).resolve().parent
    inc = torch_dir / "include"
    host_obj = BUILD_DIR / "torch_host.o"
    cmds.insert(0, [
        hipcc, "-O2", "-std=c++17", "-fPIC", f"-DTORCH_EXTENSION_NAME={HOST_NAME}",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DUSE_ROCM",
        "-D__HIP_PLATFORM_AMD__=1", f"-I{PKG_DIR.parent / 'include'}", f"-isystem{inc}",
        f"-isystem{inc / 'torch' / 'csrc' / 'api' / 'include'}",
        f"-isystem{sysconfig.get_paths()['include']}", "-Wno-unused-command-line-argument",
        "-c", str(HOST_SRC), "-o", str(host_obj)])  # first: the longest one

    def run(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed ({res.returncode}):\n{' '.join(cmd)}\n{res.stderr}")
        return res

    jobs = jobs or min(8, max(1, len(cmds)))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        list(pool.map(run, cmds))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    run([hipcc, "-shared", f"--offload-arch={ARCH}", "-fPIC", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, LIB_PATH)
    tmp = HOST_PATH.with_suffix(".so.tmp")
    run([hipcc, "-shared", "-fPIC", "-o", str(tmp), str(host_obj), f"-L{torch_dir / 'lib'}", "-lc10",
         "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", f"-L{PKG_DIR}", f"-l:{LIB_NAME}",
         "-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, HOST_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
