"""Compile the HIP/C++ sources of this package into libsqattn.so for gfx950, and
the Python binding of its hot entry points into _sqahost.so (where the headers of
torch and Python are there).

Every source of csrc/ is compiled by hipcc (-x hip) into _build/, then linked
into a shared library next to this file; binding/host.cpp is host code against
torch's C++ headers. Flags:
  -Xclang -target-feature -Xclang -packed-fp32-ops   no packed fp32 VALU ops
  -ffp-contract=fast-honor-pragmas is hipcc's default; code that must round
  every multiply and add on its own (the q4_0 quantizer, the K/Q producer)
  says #pragma clang fp contract(off): HIP's __fmul_rn/__fadd_rn are plain
  * and + and do not stop the fusion.
"""
import concurrent.futures
import glob
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "libsqattn.so")
HOST = os.path.join(HERE, "_sqahost.so")
ARCH = os.environ.get("SQA_OFFLOAD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

CFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-x", "hip",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result", "-I", os.path.join(ROOT, "include"),
]


def sources():
    csrc = os.path.join(HERE, "csrc")
    return sorted(glob.glob(os.path.join(csrc, "*.hip")) + glob.glob(os.path.join(csrc, "*.cpp")))


# Per-source extra flags. fa_prefill.hip: its MFMA accumulators are read and
# rescaled by VALU code, so keep every MFMA result in VGPRs (the AGPR form makes
# the register allocator copy the 128-register accumulator on every tile).
EXTRA_FLAGS = {
    "fa_prefill.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=true"],
}


def _compile(src, out):
    cmd = [HIPCC] + CFLAGS + EXTRA_FLAGS.get(os.path.basename(src), []) + ["-c", src, "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    errs = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{errs}")
    if errs.strip():
        sys.stderr.write(errs + "\n")
    return out


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n" + r.stderr)


def _torch_root():
    """torch's folder, or None where its C++ headers or Python's are missing (the
    package then runs without the binding, every call on the ctypes path)."""
    try:
        import torch
    except ImportError:
        return None
    root = os.path.dirname(torch.__file__)
    headers = (os.path.join(root, "include", "torch", "csrc", "autograd", "python_variable.h"),
               os.path.join(sysconfig.get_paths()["include"], "Python.h"))
    return root if all(os.path.exists(h) for h in headers) else None


def _compile_host(root, out):
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           sysconfig.get_paths()["include"], os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include")]
    _run([HIPCC, "-std=c++17", "-O2", "-fPIC", "-Wall", "-x", "c++", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"]
         + [f"-isystem{i}" for i in inc]
         + ["-c", os.path.join(HERE, "binding", "host.cpp"), "-o", out], "hipcc of binding/host.cpp")
    return [f"-L{os.path.join(root, 'lib')}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]


def build(verbose=False):
    bdir = os.path.join(HERE, "_build")
    os.makedirs(bdir, exist_ok=True)
    srcs = sources()
    outs = [os.path.join(bdir, os.path.basename(s) + ".o") for s in srcs]
    host, torch_root = os.path.join(bdir, "host.o"), _torch_root()
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        host_libs = ex.submit(_compile_host, torch_root, host) if torch_root else None
        list(ex.map(_compile, srcs, outs))
        host_libs = host_libs.result() if host_libs else None
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + outs, "link")
    os.replace(tmp, LIB)
    if host_libs:
        # finds libsqattn.so beside itself; torch's libraries are loaded with torch
        tmp = HOST + ".tmp"
        _run([HIPCC, "-shared", "-fPIC", "-o", tmp, host, f"-L{HERE}", "-l:libsqattn.so", "-Wl,-rpath,$ORIGIN"]
             + host_libs, "link of the binding")
        os.replace(tmp, HOST)
    elif os.path.exists(HOST):
        os.remove(HOST)  # of an earlier build, against an older library
    if verbose:
        print("built", LIB, HOST if host_libs else "(no headers of torch or Python: no native binding)")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
