"""The library's kernels and C ABI built for the CPU (x86-64): `build` compiles
them against the HIP stand-in of this folder, `use` puts that library and
guarded memory behind amrsolver_amd.level in a process of its own (an access out
of range ends it with status 99 and the kernel's name)."""
import concurrent.futures
import ctypes
import glob
import os
import subprocess
import types

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
CLANG = "/opt/rocm/llvm/bin/clang++"


def build(folder):
    csrc = os.path.join(ROOT, "amrsolver_amd", "csrc")
    # (vectorised straight-line code costs the compiler most of its time)
    flags = ["-O1", "-std=c++17", "-fPIC", "-mfma", "-ffp-contract=off", "-fno-vectorize", "-fno-slp-vectorize", "-w",
             "-I", HERE, "-I", os.path.join(ROOT, "include"), "-I", csrc, "-x", "c++", "-c"]
    sources = sorted(glob.glob(os.path.join(csrc, "*.hip"))) + [os.path.join(csrc, "capi.cpp"),
                                                                os.path.join(HERE, "runtime.cpp")]

    def compile_one(src):
        obj = os.path.join(folder, os.path.basename(src) + ".o")
        subprocess.run([CLANG, *flags, src, "-o", obj], check=True)
        return obj

    with concurrent.futures.ThreadPoolExecutor(8) as ex:
        objs = list(ex.map(compile_one, sources))
    lib = os.path.join(folder, "libamrsolver_cpu.so")
    subprocess.run([CLANG, "-shared", "-o", lib, *objs], check=True)
    return lib


def use(path):
    import numpy as np
    import torch
    lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
    lib.cpu_hip_malloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    lib.cpu_hip_free.argtypes = [ctypes.c_void_p]

    class Memory:
        def __init__(self, nbytes):
            p = ctypes.c_void_p()
            assert lib.cpu_hip_malloc(ctypes.byref(p), nbytes) == 0
            self.p = p.value

        def __del__(self):
            lib.cpu_hip_free(self.p)

    def zeros(shape, dtype=None, device=None):
        shape = (shape,) if isinstance(shape, int) else shape
        n = int(np.prod(shape))
        m = Memory(8 * n)
        buf = (ctypes.c_double * n).from_address(m.p)
        buf.memory = m
        a = np.frombuffer(buf, dtype=np.float64).reshape(shape)
        a[...] = 0.0
        return torch.from_numpy(a)

    stream = types.SimpleNamespace(cuda_stream=1)
    cuda = types.SimpleNamespace(is_available=lambda: True, set_device=lambda d: None, synchronize=lambda *a: None,
                                 current_stream=lambda *a: stream, Stream=lambda **k: stream, set_stream=lambda s: None)
    from amrsolver_amd import capi, level
    capi.LIBPATH = path
    level._torch = types.SimpleNamespace(zeros=zeros, empty=zeros, float64=torch.float64, from_numpy=torch.from_numpy,
                                         device=lambda *a: torch.device("cpu"), cuda=cuda, Tensor=torch.Tensor)
    return level
