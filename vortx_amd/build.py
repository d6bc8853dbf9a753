"""Build libvortx_hip.so in-tree.

Steps (no cmake):
  1. hipcc --genco --offload-arch=gfx950 for each kernel source in
     csrc/kernels/ -> _build/<name>.hsaco (gfx950 code objects);
  2. an assembler stub that .incbin's those code objects, so the shared
     library carries them and vx_init can hipModuleLoadData them;
  3. g++ for the host sources (HIP runtime API only), linked against
     libamdhip64;
  4. g++ for the CPython extension with the binding's fast calls (_pycall.*.so).

Every call recompiles everything (a build check, not an incremental build).
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
INCLUDE = os.path.join(os.path.dirname(PKG), "include")  # the public C ABI header
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libvortx_hip.so")
# named for the Python that it is built for: another one must not load it
PYCALL = os.path.join(PKG, "_pycall" + sysconfig.get_config_var("EXT_SUFFIX"))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
ARCH = "gfx950"

# module symbol -> kernel source
MODULES = {"vx_co_gemm": "gemm.hip", "vx_co_gemv_q": "gemv_q.hip", "vx_co_copy": "copy.hip",
           "vx_co_quantize": "quantize.hip", "vx_co_gemm_q": "gemm_q.hip",
           "vx_co_gemm_bf": "gemm_bf.hip"}
HOST_SOURCES = ["vx_host.cpp", "vx_layout.cpp", "vx_gguf.cpp"]

HIPCC_FLAGS = [
    "--genco", f"--offload-arch={ARCH}", "-O3", "-std=c++17",
    # packed-FP32 VALU ops (v_pk_fma_f32 and friends) stay disabled
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # leading scalar kernel arguments arrive preloaded in SGPRs (kernels
    # whose first argument is a struct are unaffected)
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
]


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout + r.stderr)
        raise RuntimeError(f"build step failed: {cmd[0]} ({r.returncode})")


def _hipcc() -> str:
    h = shutil.which("hipcc") or os.path.join(ROCM, "bin", "hipcc")
    if not os.path.exists(h):
        raise RuntimeError("hipcc not found")
    return h


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    hipcc = _hipcc()
    jobs = []
    for sym, src in MODULES.items():
        out = os.path.join(BUILD, os.path.splitext(src)[0] + ".hsaco")
        jobs.append([hipcc, *HIPCC_FLAGS, os.path.join(CSRC, "kernels", src), "-o", out])
    with cf.ThreadPoolExecutor(max_workers=len(jobs)) as ex:
        list(ex.map(_run, jobs))
    stub = os.path.join(BUILD, "vx_embed.S")
    with open(stub, "w") as f:
        f.write("/* generated by vortx_amd/build.py: embedded gfx950 code objects */\n")
        f.write('.section .rodata\n')
        for sym, src in MODULES.items():
            co = os.path.join(BUILD, os.path.splitext(src)[0] + ".hsaco")
            f.write(f".balign 4096\n.globl {sym}\n.type {sym}, @object\n{sym}:\n")
            f.write(f'.incbin "{co}"\n.globl {sym}_end\n{sym}_end:\n.byte 0\n')
        f.write('.section .note.GNU-stack,"",@progbits\n')
    tmp = LIB + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wextra",
           "-D__HIP_PLATFORM_AMD__", f"-I{INCLUDE}", f"-I{ROCM}/include",
           *[os.path.join(CSRC, s) for s in HOST_SOURCES], stub,
           f"-L{ROCM}/lib", "-lamdhip64", f"-Wl,-rpath,{ROCM}/lib", "-o", tmp]
    _run(cmd)
    os.replace(tmp, LIB)
    tmp = PYCALL + ".tmp"
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wextra", "-Wno-cast-function-type",
          "-Wno-missing-field-initializers", f"-I{INCLUDE}", f"-I{sysconfig.get_paths()['include']}",
          os.path.join(CSRC, "vx_pycall.cpp"), "-o", tmp])
    os.replace(tmp, PYCALL)
    untagged = os.path.join(PKG, "_pycall.so")  # from an older build
    if os.path.exists(untagged):
        os.remove(untagged)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
