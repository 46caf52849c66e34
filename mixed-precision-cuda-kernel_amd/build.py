"""Builds libcherryq.so (HIP kernels + C ABI) for gfx950 with hipcc and cherryq_host.so (the host side of
the Python binding) with g++, in-tree.

    python build.py            # rebuild if any source is newer than the library
    python build.py --force

No CUDAExtension / hipify: the sources are HIP written for CDNA4 and are compiled directly.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
OBJ = HERE / "build"
LIB = HERE / "libcherryq.so"
PROBE_LIB = HERE / "libcherryq_probe.so"  # bench-only roofline reference kernels, not part of the product library
SOURCES = ["cq_api.hip", "cq_generic.hip", "cq_matvec.hip", "cq_stream.hip", "cq_stream_cu.hip", "cq_batch.hip", "cq_prompt.hip", "cq_f32.hip", "cq_decode.hip", "cq_prefill.hip", "cq_pack.hip", "cq_fakequant.hip", "cq_gemm.hip"]
HOST_LIB = HERE / "cherryq_host.so"  # host side of the Python binding (g++, linked against torch)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
]


def _deps():
    return list(CSRC.glob("*")) + [HERE.parent / "include" / "cherryq.h", Path(__file__)]


def built_for() -> str:
    """What the host library, which is bound to torch's ABI, says it was built for."""
    import torch
    return f"torch {torch.__version__}"


def needs_build() -> bool:
    if not LIB.exists() or not HOST_LIB.exists() or b"%s\0" % built_for().encode() not in HOST_LIB.read_bytes():
        return True
    t = min(LIB.stat().st_mtime, HOST_LIB.stat().st_mtime)
    return any(p.stat().st_mtime > t for p in _deps())


def host_command(source, output):
    """The compiler call for the host side of the Python binding."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    lib = Path(torch.__file__).resolve().parent / "lib"
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
            f'-DCHERRYQ_BUILT_FOR="{built_for()}"',
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            f"-I{HERE.parent / 'include'}", *(f"-isystem{p}" for p in (*include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"])),
            str(source), "-o", str(output), f"-L{lib}", "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-lc10_hip"]


def build_host():
    r = subprocess.run(host_command(CSRC / "cq_host.cpp", HOST_LIB), capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("host binding failed:\n" + r.stdout + r.stderr)


def build(force: bool = False, verbose: bool = False) -> Path:
    if not force and not needs_build():
        return LIB
    OBJ.mkdir(exist_ok=True)

    # cq_stream.hip: the dispatcher preloads the first six dwords of the kernel arguments (the
    # activation pointer, the stream pointer, K and the header size lead stream_kernel's list) into
    # scalar registers, which takes their load off the start-up chain of every workgroup
    # (4096 -> 11008: 6.67 -> 6.40 us, 4096 -> 4096: 4.38 -> 4.21 us)
    # cq_stream_cu.hip: likewise the first 14 dwords of stream_cu_kernel's list (pointers, shape and
    # record geometry: everything a wavefront needs for its first requests)
    # cq_prompt.hip: the products' loops begin at a line of the instruction cache; where they began elsewhere they took up to 1 % longer
    # (2048 rows of 4096 -> 11008: 181.5 -> 180.7 us)
    extra = {"cq_prompt.hip": ["-falign-loops=64"],
             "cq_stream.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=6"],
             "cq_stream_cu.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=14"]}

    def compile_one(src):
        out = OBJ / (src + ".o")
        cmd = [HIPCC, *FLAGS, *extra.get(src, []), "-c", str(CSRC / src), "-o", str(out)]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        msgs = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                         if "packed-fp32-ops" not in l and l.strip())
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{msgs}")
        if verbose and msgs:
            print(msgs)
        return out

    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        host = ex.submit(build_host)
        objs = list(ex.map(compile_one, SOURCES))
        host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", "-o", str(LIB), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    cmd = [HIPCC, *FLAGS, "-shared", "-o", str(PROBE_LIB), str(CSRC / "cq_probe.hip")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("probe library failed:\n" + r.stdout + r.stderr)
    return LIB


if __name__ == "__main__":
    p = build(force="--force" in sys.argv, verbose=True)
    print(f"built {p} ({p.stat().st_size} bytes)")
