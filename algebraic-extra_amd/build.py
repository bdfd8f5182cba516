"""Build libalgx.so (gfx950) and the torch operators over it in-tree.

    python algebraic-extra_amd/build.py            # compile every csrc/*.hip, link
    python algebraic-extra_amd/build.py --asm      # also write gfx950 ISA to _build/

Each translation unit is compiled separately (in parallel) and linked into
``algebraic_amd/libalgx.so`` next to the Python package that loads it;
``csrc/torch_ops.cpp`` is compiled against the installed torch's headers to the
extension module ``algebraic_amd/_ops.so``, which links that library.
"""

import argparse
import concurrent.futures as cf
import glob
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
OUT = os.path.join(HERE, "algebraic_amd", "libalgx.so")
OPS = os.path.join(HERE, "algebraic_amd", "_ops.so")
ARCH = "gfx950"
# Extra flags per translation unit: the MFMA kernels keep their accumulators in
# architectural VGPRs so the VALU reads them without accvgpr copies.
EXTRA = {
    "attn_fwd_mfma.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "attn_bwd_mfma.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "attn_fwd_ragged.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "attn_bwd_ragged.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "head.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "gemm_batched.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def flags():
    return [
        f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
        "-I", os.path.join(ROOT, "include"), "-I", CSRC,
        "-munsafe-fp-atomics",
        # Packed FP32 VALU forms stay disabled on this hardware pool.
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-Wno-unused-command-line-argument",
    ]


def _compile(src, asm):
    obj = os.path.join(BUILD, os.path.basename(src) + ".o")
    extra = EXTRA.get(os.path.basename(src), [])
    cmd = [hipcc()] + flags() + extra + ["-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"compile failed: {src}\n{res.stderr}")
    if asm:
        s = os.path.join(BUILD, os.path.basename(src) + ".s")
        subprocess.run([hipcc()] + flags() + extra + ["--cuda-device-only", "-S", src, "-o", s],
                       capture_output=True, text=True, check=True)
    return obj


def _compile_ops():
    torch = os.path.dirname(importlib.util.find_spec("torch").origin)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    obj = os.path.join(BUILD, "torch_ops.o")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_ops", "-I", os.path.join(ROOT, "include"),
           "-isystem", os.path.join(torch, "include"),
           "-isystem", os.path.join(torch, "include", "torch", "csrc", "api", "include"),
           "-isystem", os.path.join(rocm, "include"),
           "-isystem", sysconfig.get_paths()["include"],
           "-c", os.path.join(CSRC, "torch_ops.cpp"), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"compile failed: torch_ops.cpp\n{res.stderr}")
    return obj, os.path.join(torch, "lib")


def _link_ops(obj, torch_lib):
    tmp = OPS + ".tmp"
    cmd = [os.environ.get("CXX", "g++"), "-shared", "-o", tmp, obj, "-L", os.path.dirname(OUT),
           "-l:libalgx.so", "-L", torch_lib, "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
           "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed: _ops.so\n{res.stderr}")
    os.replace(tmp, OPS)


def build(asm=False, jobs=None):
    os.makedirs(BUILD, exist_ok=True)
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    jobs = jobs or min(8, len(sources) + 1, os.cpu_count() or 1)
    with cf.ThreadPoolExecutor(jobs) as ex:
        ops = ex.submit(_compile_ops)
        objs = list(ex.map(lambda s: _compile(s, asm), sources))
        ops_obj, torch_lib = ops.result()
    tmp = OUT + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-o", tmp] + objs
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed\n{res.stderr}")
    os.replace(tmp, OUT)
    _link_ops(ops_obj, torch_lib)
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--asm", action="store_true")
    ap.add_argument("-j", type=int, default=None)
    a = ap.parse_args()
    print(build(asm=a.asm, jobs=a.j))
    sys.exit(0)
