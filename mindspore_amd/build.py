"""Builds libmi355x_int8.so (HIP kernels + C ABI) for gfx950 with hipcc.  Cross-compiles without a GPU."""
import os
import subprocess
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmi355x_int8.so")
DIAG_LIB = os.path.join(HERE, "libmi355x_diag.so")  # the benchmark's measurement aids, not part of the product
DEVICE_CALLS = os.path.join(HERE, "_device_calls.so")  # kernels.py's calls on torch device tensors
NATIVE_BENCH = os.path.join(HERE, "native_bench")
SOURCES = ["capi.hip", "gemm_i8.hip", "gemm_kblock.hip", "gemm_ring.hip", "gemm_split.hip", "gemm_anyrow.hip", "gemm_short.hip", "gemv_i8.hip", "conv_i8.hip", "conv_thin.hip", "conv_window.hip", "dynquant.hip", "host_copy.hip", "infer_shape.hip"]
# -ffp-contract=off: the float steps of DynamicQuant / dynamic MatMul and the host-side multiplier derivation are
# separately rounded operations in the reference and must not be fused.
FLAGS = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-result"]


def device_calls_command():
    """g++ command of the CPython extension (host code over torch's C++ API and the C ABI), or None where there is no torch with
    HIP: the library itself needs none, and kernels.py then takes host tensors only."""
    try:
        import torch
        if torch.version.hip is None:
            return None
        from torch.utils import cpp_extension as ext
    except ImportError:
        return None
    inc = ["-I" + p for p in ext.include_paths("cuda") + [sysconfig.get_paths()["include"]]]
    libs = ["-L" + p for p in ext.library_paths("cuda")]
    return (["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
             "-DUSE_ROCM=1"] + inc + [os.path.join(CSRC, "device_calls.cc"), "-o", DEVICE_CALLS] + libs +
            ["-lc10", "-ltorch_cpu", "-lc10_hip", "-ltorch_hip", "-ltorch", "-ltorch_python"])


def build_library(verbose=False):
    objs, procs = [], []
    cmd = device_calls_command()
    if cmd is None:
        print("no torch with HIP here: %s is not built" % os.path.basename(DEVICE_CALLS))
    else:
        procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    for src in SOURCES:
        obj = os.path.join(CSRC, src.replace(".hip", ".o"))
        cmd = ["hipcc"] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
        procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        objs.append(obj)
    for cmd, p in procs:
        out, _ = p.communicate()
        if verbose or p.returncode != 0:
            print(" ".join(cmd))
            print(out)
        if p.returncode != 0:
            raise RuntimeError("%s failed: %s" % (cmd[0], " ".join(cmd)))
    link = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    subprocess.check_call(link)
    subprocess.check_call(["hipcc"] + FLAGS + ["-shared", os.path.join(CSRC, "diag.hip"), "-o", DIAG_LIB])
    # the native benchmark host (a C++ caller of the C ABI, like a provider kernel)
    subprocess.check_call(["hipcc", "-O2", "-std=c++17", "-x", "hip", "--offload-arch=gfx950", "-Wno-unused-result",
                           os.path.join(CSRC, "native_bench.cc"), "-o", NATIVE_BENCH, "-L" + HERE, "-lmi355x_int8", "-lmi355x_diag",
                           "-Wl,-rpath,$ORIGIN"])
    return LIB


if __name__ == "__main__":
    print(build_library(verbose=True))
