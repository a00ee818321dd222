"""Builds the host runtime (scheduler, copies, scene set-up, autotuner) against hip_standin.cpp, which
queues work as a GPU would and runs it as late as the program allows, and lends it to Renderer."""
import contextlib
import ctypes as C
import os
import subprocess

import pytest

from cortexraytracercuda_amd import _abi as A
from cortexraytracercuda_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(HERE, "_build")
HOST = ["api.cpp", "serve.cpp", "tune.cpp", "host_stage.cpp", "scene_build.cpp", "bvh_gpu.hip"]


def _build():
    os.makedirs(OUT, exist_ok=True)
    lib = os.path.join(OUT, "libhost_standin.so")
    srcs = [os.path.join(B.CSRC, s) for s in HOST] + [os.path.join(HERE, "hip_standin.cpp")]
    heads = [os.path.join(d, f) for d in (B.CSRC, os.path.join(B.ROOT, "include")) for f in os.listdir(d) if f.endswith(".h")]
    newest = max(os.path.getmtime(p) for p in heads)
    objs, procs = [], []
    for s in srcs:
        o = os.path.join(OUT, os.path.basename(s) + ".o")
        objs.append(o)
        if os.path.exists(o) and os.path.getmtime(o) > max(newest, os.path.getmtime(s)):
            continue
        flags = ["-O1", "-std=c++17", "-fPIC", "-w", "-I" + os.path.join(B.ROOT, "include"), "-I" + B.CSRC]
        cc = [B.HIPCC, "--offload-host-only", "-x", "hip"] if s.endswith(".hip") else ["g++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include"]
        procs.append((o, subprocess.Popen(cc + flags + ["-c", s, "-o", o], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    for o, p in procs:
        out, _ = p.communicate()
        assert p.returncode == 0, out
    if procs or not os.path.exists(lib):
        # own symbols first; the runtime library only answers for what the stand-in leaves out
        nm = subprocess.run(["nm", "-u"] + objs, check=True, capture_output=True, text=True).stdout.split()
        binaries = ["-Wl,--defsym=%s=0" % n for n in nm if n.startswith("__hip_fatbin")]
        subprocess.run(["g++", "-shared", "-o", lib] + objs + binaries + ["-Wl,-Bsymbolic", "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64", "-lpthread"],
                       check=True)
    return lib


@pytest.fixture(scope="session")
def standin_lib():
    lib = C.CDLL(_build())
    for name, (args, res) in A._SIGS.items():
        fn = getattr(lib, name, None)
        if fn is not None:
            fn.argtypes, fn.restype = args, res
    for name in ("standin_allocated", "standin_launches", "standin_pending", "standin_ran"):
        getattr(lib, name).restype = C.c_uint64
    lib.standin_ran.argtypes = [C.c_uint64, C.POINTER(C.c_uint64)]
    lib.standin_memory_limit.argtypes = [C.c_uint64]
    return lib


@pytest.fixture
def standin(standin_lib, monkeypatch):
    """The library behind Renderer is the stand-in's for the length of a test."""
    monkeypatch.setattr(A, "_lib", standin_lib)
    standin_lib.standin_reset()
    yield standin_lib
    standin_lib.standin_reset()


@contextlib.contextmanager
def gate_closed(lib):
    lib.standin_gate(1)
    try:
        yield
    finally:
        lib.standin_gate(0)


def launches_that_ran(lib):
    out, k = [], 0
    v = (C.c_uint64 * 4)()
    while k < lib.standin_ran(k, v):
        out.append(dict(mode=v[0], requests=v[1], paths=v[2], samples=v[3]))
        k += 1
    return out
