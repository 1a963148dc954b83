"""Build libmi_attn.so (the HIP kernels + C ABI) in-tree with hipcc for gfx950, and
_mi_torch.so (the op's autograd nodes in C++) beside it.

Each ``csrc/*.hip`` file is compiled to an object in parallel, then linked into
``machinelearning_amd/libmi_attn.so``. That library links only the HIP runtime: no
torch headers. ``csrc/autograd.cpp`` (host code over its C ABI) is compiled
against the installed torch's headers and links the library beside it.

    python -m machinelearning_amd.build_ext          # build (always recompiles)
"""

from __future__ import annotations

import concurrent.futures
import os
import pathlib
import shutil
import subprocess
import sys
import sysconfig

PKG = pathlib.Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIB = PKG / "libmi_attn.so"
TORCH_SRC = CSRC / "autograd.cpp"
TORCH_EXT = PKG / "_mi_torch.so"
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    # Packed FP32 VALU ops stay off: the compiler must not form v_pk_{add,mul,fma}_f32.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA accumulators in ordinary VGPRs: without this the backend picks the
    # AGPR form and copies every score / output tile between register files
    # (v_accvgpr_read/write) around the softmax, ~64 VALU ops per key tile.
    "-mllvm", "-amdgpu-mfma-vgpr-form",
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the HIP extension cannot be built")
    return exe


def sources() -> list[pathlib.Path]:
    return sorted(CSRC.glob("*.hip"))


def _compile(src: pathlib.Path, obj: pathlib.Path) -> None:
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{r.stderr}")


def _compile_torch(obj: pathlib.Path) -> None:
    from torch.utils import cpp_extension

    rocm = pathlib.Path(hipcc()).resolve().parents[1] / "include"
    inc = [*cpp_extension.include_paths(), str(rocm), "/opt/rocm/include",
           sysconfig.get_paths()["include"]]
    import torch
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden",
           f"-D_GLIBCXX_USE_CXX11_ABI={abi}", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           *[f"-I{d}" for d in dict.fromkeys(inc)], "-c", str(TORCH_SRC), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on {TORCH_SRC.name}:\n{r.stderr}")


def _link(cmd: list[str], out: pathlib.Path) -> None:
    tmp = out.with_suffix(".so.tmp")
    r = subprocess.run([*cmd, "-o", str(tmp)], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of {out.name} failed:\n{r.stderr}")
    os.replace(tmp, out)


def build(verbose: bool = False) -> pathlib.Path:
    """Compile every csrc/*.hip and the autograd nodes, link libmi_attn.so and
    _mi_torch.so. Returns the path of libmi_attn.so."""
    import torch

    objdir = PKG / "_build"
    objdir.mkdir(exist_ok=True)
    srcs = sources()
    objs = [objdir / (s.stem + ".o") for s in srcs]
    tobj = objdir / "torch_autograd.o"
    workers = min(len(srcs) + 1, max(1, (os.cpu_count() or 2)))
    with concurrent.futures.ThreadPoolExecutor(max_workers=workers) as ex:
        futs = [ex.submit(_compile_torch, tobj)]
        futs += [ex.submit(_compile, s, o) for s, o in zip(srcs, objs)]
        for f in futs:
            f.result()
    _link([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs)], LIB)
    tlib = pathlib.Path(torch.__file__).parent / "lib"
    _link(["g++", "-shared", str(tobj), f"-L{PKG}", f"-l:{LIB.name}", f"-L{tlib}", "-lc10",
           "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"], TORCH_EXT)
    if verbose:
        print(f"built {LIB} and {TORCH_EXT.name}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
