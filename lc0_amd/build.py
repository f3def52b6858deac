"""Builds lc0_amd/liblc0mi.so (the C-ABI library: host C++ + gfx950 kernels) and, where g++ and Python's headers are there, the
extension of its Python mirror."""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "liblc0mi.so")
CALLS = os.path.join(HERE, "_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
SOURCES = ["weights.cc", "tables.cc", "network.cc", "capi.cc", "kernel_api.cc", "kernels.hip", "gemm_kernels.hip", "gemm_dma_half.hip",
           "gemm_dma_bf16.hip", "gemm_dma_f8.hip", "gemm_rowpanel.hip", "gemm_resident.hip", "gemm_norm.hip", "gemm_f32.hip", "smolgen_attention.hip", "smolgen_attention_few.hip", "encoder_narrow.hip", "encoder_narrow_f32.hip", "value_heads.hip", "resnet_kernels.hip", "resident_tower.hip", "resident_tower_f32.hip"]
# -packed-fp32-ops off: packed fp32 forms are not trusted on this hardware pool.
DEVICE_FLAGS = ["--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
FLAGS = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-result", "-Wno-unknown-warning-option"]


def build(verbose=False):
    objs = []
    build_dir = os.path.join(HERE, "build")
    os.makedirs(build_dir, exist_ok=True)
    procs = []
    for src in SOURCES:
        obj = os.path.join(build_dir, src.replace(".", "_") + ".o")
        cmd = ["hipcc"] + FLAGS + DEVICE_FLAGS + ["-x", "hip", "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        objs.append(obj)
    failed = False
    for src, p in procs:
        out, _ = p.communicate()
        lines = [l for l in out.splitlines() if "packed-fp32-ops" not in l and l.strip()]
        if p.returncode != 0:
            failed = True
            sys.stderr.write("\n".join(lines) + "\n")
        elif verbose and lines:
            print("\n".join(lines))
    if failed:
        raise RuntimeError("hipcc failed")
    cmd = ["hipcc", "-shared", "-fPIC", "--offload-arch=gfx950", "-o", LIB] + objs + ["-lz"]
    subprocess.check_call(cmd)
    build_calls()
    return LIB


def build_calls():
    """The extension that spares a Python program ctypes for the calls it makes per position. Nothing depends on it (the library serves
    C and C++ programs by itself, and backend.py does without), so a machine that cannot compile it gets a warning, and an
    extension of an earlier build does not stay beside the new library."""
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-shared", "-I" + sysconfig.get_path("include"),
           os.path.join(CSRC, "python_calls.cc"), "-o", CALLS, "-L" + HERE, "-l:liblc0mi.so", "-Wl,-rpath,$ORIGIN"]
    try:
        subprocess.check_call(cmd)
        return True
    except (OSError, subprocess.CalledProcessError) as e:
        if os.path.exists(CALLS):
            os.remove(CALLS)
        sys.stderr.write("warning: %s is not built (%s): Python programs go through ctypes\n" % (os.path.basename(CALLS), e))
        return False


if __name__ == "__main__":
    print(build(verbose=True))
