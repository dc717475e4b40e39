"""Build ``libmedvision_hip.so`` for gfx950 with hipcc (``python -m medvision_amd.build``).

hipcc cross-compiles without a GPU.  Objects go to ``medvision_amd/lib/obj``, the shared library to
``medvision_amd/lib/libmedvision_hip.so`` and the PyTorch binding of ``csrc/binding.cpp`` to
``medvision_amd/_native.so`` (in-tree, not tracked by git).
"""
import concurrent.futures
import glob
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libmedvision_hip.so")
# the same library with in-kernel time stamps in the tiled resampler (a measuring aid: `bench.py --timeline`)
TIMELINE_LIB_PATH = os.path.join(LIB_DIR, "libmedvision_hip_timeline.so")

# the host side of medvision_amd.ops (PyTorch's C++ API), linked against the library
NATIVE_PATH = os.path.join(HERE, "_native.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-munsafe-fp-atomics",
    # keep the compiler from forming packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]
# per-file additions, keyed by source file name
FILE_FLAGS = {
    # matrix-core accumulators in ordinary vector registers: the kernel packs and stores them right
    # away, and copies between the two register classes would outnumber its arithmetic
    "roi_pool.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), out))
    return out


def _native_object_command(obj):
    """Host code only: the compiler that ships with ROCm, PyTorch's headers."""
    import torch
    from torch.utils.cpp_extension import include_paths
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    return [os.path.join(rocm, "llvm", "bin", "clang++"), "-O2", "-std=c++17", "-fPIC", "-Wall",
            "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_native",
            "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
            *[f for d in (*include_paths(), os.path.join(rocm, "include"), sysconfig.get_paths()["include"])
              for f in ("-isystem", d)],
            "-c", os.path.join(CSRC, "binding.cpp"), "-o", obj]


def _native_link_command(obj):
    import torch
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return [HIPCC, "-shared", "-fPIC", "-o", NATIVE_PATH, obj, "-L" + torch_lib, "-lc10", "-lc10_hip", "-ltorch_cpu",
            "-ltorch_hip", "-ltorch", "-ltorch_python", "-L" + LIB_DIR, "-lmedvision_hip", "-Wl,-rpath,$ORIGIN/lib"]


def build(verbose=False, jobs=None):
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    obj_dir = os.path.join(LIB_DIR, "obj")
    os.makedirs(obj_dir, exist_ok=True)
    objs = [os.path.join(obj_dir, os.path.basename(s)[:-4] + ".o") for s in sources]
    commands = [[HIPCC, *FLAGS, *FILE_FLAGS.get(os.path.basename(src), []), "-c", src, "-o", obj]
                for src, obj in zip(sources, objs)]
    # instrumented twin: only roi_resample.hip differs
    tl_src = os.path.join(CSRC, "roi_resample.hip")
    tl_obj = os.path.join(obj_dir, "roi_resample_timeline.o")
    commands.append([HIPCC, *FLAGS, "-DMV_RESAMPLE_TIMELINE", "-c", tl_src, "-o", tl_obj])
    native_obj = os.path.join(obj_dir, "binding.o")
    commands.append(_native_object_command(native_obj))
    # longest first, so that the last one to finish is a short one
    commands.sort(key=lambda c: -os.path.getsize(c[c.index("-c") + 1]))
    with concurrent.futures.ThreadPoolExecutor(jobs or min(8, len(commands))) as pool:
        outs = list(pool.map(_run, commands))
    link = _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs])
    tl_objs = [tl_obj if os.path.basename(o) == "roi_resample.o" else o for o in objs]
    link += _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", TIMELINE_LIB_PATH, *tl_objs])
    link += _run(_native_link_command(native_obj))
    if verbose:
        for o in outs + [link]:
            if o.strip():
                print(o)
        print("built", LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
