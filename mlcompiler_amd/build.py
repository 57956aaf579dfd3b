"""Builds the in-tree native libraries of the package with hipcc for gfx950.

  libmlc_hip.so       HIP kernels + the C ABI declared in include/mlc_hip.h
  libhip_executor.so  the C++ HipExecutor class (mirror of the reference's
                      MetalExecutor paged-path methods) on top of that ABI
  _call.<abi>.so      HipExecutor's inner-loop calls into the ABI as a Python module, for the interpreter
                      and the numpy that build it
  libmlc_bench.so     native benchmark loops that call the ABI, plus a plain copy kernel
                      used to calibrate the HBM traffic counters
"""
from __future__ import annotations

import hashlib
import os
import shutil
import subprocess
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
LIB_PATH = os.path.join(CSRC, "libmlc_hip.so")
EXECUTOR_LIB_PATH = os.path.join(CSRC, "libhip_executor.so")
CALL_MODULE_PATH = os.path.join(PKG_DIR, "_call" + sysconfig.get_config_var("EXT_SUFFIX"))
CALL_STAMP_PATH = CALL_MODULE_PATH + ".stamp"         # what that module was built from and for
BENCH_LIB_PATH = os.path.join(CSRC, "libmlc_bench.so")
STAMP_PATH = os.path.join(CSRC, "libmlc_hip.stamp")   # hash of the sources the libraries were built from

# Packed FP32 instructions (v_pk_*_f32) are switched off on purpose: some of their forms have
# produced wrong results on the target machines.  hipcc's host pass prints a harmless
# "not a recognized feature" warning for the flag.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-fno-honor-nans",
    # the first 14 words of scalar kernel arguments arrive in registers with a wave (the Q4_0 matmul's first loads need no others)
    "-mllvm", "-amdgpu-kernarg-preload-count=14",
    "-Wno-inline-asm",  # the global->LDS load in paged_prefill_kernels.h names m0 as clobbered
]


# extra compiler flags for experiments (for example -DMLC_STREAM_PROBE: time stamps per workgroup)
HIPCC_FLAGS += os.environ.get("MLC_HIPCC_EXTRA", "").split()


def source_hash() -> str:
    """Hash over every source the native libraries are built from (and the flags)."""
    h = hashlib.sha256(" ".join(HIPCC_FLAGS).encode())
    files = [os.path.join(CSRC, n) for n in sorted(os.listdir(CSRC))
             if n.endswith((".h", ".hpp", ".hip", ".cpp"))]
    files.append(os.path.join(os.path.dirname(PKG_DIR), "include", "mlc_hip.h"))
    for f in files:
        h.update(os.path.basename(f).encode())
        with open(f, "rb") as fh:
            h.update(fh.read())
    return h.hexdigest()


def built_from_current_sources() -> bool:
    """True when the libraries exist and were built from the sources as they are now."""
    if not all(os.path.exists(p) for p in (LIB_PATH, EXECUTOR_LIB_PATH, BENCH_LIB_PATH, STAMP_PATH)):
        return False
    with open(STAMP_PATH) as fh:
        return fh.read().strip() == source_hash()


def call_module_identity() -> str:
    """What the call module is built from and for: its sources and numpy (the interpreter is in its name)."""
    import numpy
    h = hashlib.sha256()
    for f in (os.path.join(CSRC, "py_call.cpp"), os.path.join(os.path.dirname(PKG_DIR), "include", "mlc_hip.h")):
        with open(f, "rb") as fh:
            h.update(fh.read())
    return f"{h.hexdigest()} numpy {numpy.__version__}"


def call_module_is_current() -> bool:
    """True when the call module exists for this interpreter, from the sources and for the numpy of now."""
    if not all(os.path.exists(p) for p in (CALL_MODULE_PATH, CALL_STAMP_PATH)):
        return False
    with open(CALL_STAMP_PATH) as fh:
        return fh.read().strip() == call_module_identity()


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the HIP extension cannot be built")
    return exe


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError("build failed: " + " ".join(cmd) + "\n" + proc.stdout)


def build_call_module() -> None:
    import numpy
    if os.path.exists(CALL_STAMP_PATH):
        os.remove(CALL_STAMP_PATH)
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I" + sysconfig.get_paths()["include"],
          "-I" + numpy.get_include(), os.path.join(CSRC, "py_call.cpp"), "-o", CALL_MODULE_PATH,
          "-L" + CSRC, "-lmlc_hip", "-Wl,-rpath,$ORIGIN/csrc"])
    with open(CALL_STAMP_PATH, "w") as fh:
        fh.write(call_module_identity() + "\n")


def build_all(verbose: bool = False) -> None:
    """Compiles the decode-kernel variants and the runtime in parallel, then links them."""
    from concurrent.futures import ThreadPoolExecutor

    cc = hipcc()
    if os.path.exists(STAMP_PATH):
        os.remove(STAMP_PATH)   # no stamp while the libraries are being replaced
    obj_dir = os.path.join(CSRC, "build")
    os.makedirs(obj_dir, exist_ok=True)
    jobs = []
    for d in (64, 128):
        for h in (1, 2, 4, 8):
            obj = os.path.join(obj_dir, f"decode_d{d}_h{h}.o")
            jobs.append(([cc, *HIPCC_FLAGS, f"-DMLC_D={d}", f"-DMLC_HPW={h}", "-c",
                          os.path.join(CSRC, "paged_decode_inst.hip"), "-o", obj], obj))
    for d in (64, 128):
        obj = os.path.join(obj_dir, f"prefill_d{d}.o")
        jobs.append(([cc, *HIPCC_FLAGS, f"-DMLC_D={d}", "-c", os.path.join(CSRC, "paged_prefill_inst.hip"), "-o", obj], obj))
    tok_obj = os.path.join(obj_dir, "matmul_tokens.o")
    jobs.append(([cc, *HIPCC_FLAGS, "-c", os.path.join(CSRC, "matmul_tokens_inst.hip"), "-o", tok_obj], tok_obj))
    for ni in (1, 2, 4):
        obj = os.path.join(obj_dir, f"q4_matmul_ni{ni}.o")
        jobs.append(([cc, *HIPCC_FLAGS, f"-DMLC_Q4_NI={ni}", "-c", os.path.join(CSRC, "q4_matmul_inst.hip"), "-o", obj], obj))
    rt_obj = os.path.join(obj_dir, "mlc_hip.o")
    jobs.append(([cc, *HIPCC_FLAGS, "-c", os.path.join(CSRC, "mlc_hip.hip"), "-o", rt_obj], rt_obj))
    with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
        list(pool.map(lambda j: _run(j[0]), jobs))
    _run([cc, "--offload-arch=gfx950", "-shared", "-fPIC", *[j[1] for j in jobs], "-o", LIB_PATH])
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", os.path.join(CSRC, "hip_executor.cpp"),
          "-o", EXECUTOR_LIB_PATH, "-L" + CSRC, "-lmlc_hip", "-Wl,-rpath,$ORIGIN"])
    _run([cc, *HIPCC_FLAGS, "-shared", "-x", "hip", os.path.join(CSRC, "bench_loop.cpp"),
          "-o", BENCH_LIB_PATH, "-L" + CSRC, "-lmlc_hip", "-Wl,-rpath,$ORIGIN"])
    build_call_module()
    with open(STAMP_PATH, "w") as fh:
        fh.write(source_hash() + "\n")
    if verbose:
        print("built", LIB_PATH, EXECUTOR_LIB_PATH, BENCH_LIB_PATH, CALL_MODULE_PATH)


if __name__ == "__main__":
    build_all(verbose=True)
