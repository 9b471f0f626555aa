"""Runs code against libchimera_hip.so on the host model of the HIP runtime
(tests/host_hip) in a child process, without a GPU. `host_hip` is the fixture;
the code has `hip` (the model's controls), `capi` and the helpers below."""
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent

PRELUDE = """
import ctypes as C, sys
import numpy as np
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library, which takes it for its runtime
for name in ("used", "peak", "malloc"):
    getattr(hip, "host_hip_" + name).restype = C.c_size_t
from chimera_amd import capi

def capacity(n):
    hip.host_hip_set_capacity(C.c_size_t(n))

def context(max_batch=8, nprobe=8, k_refine=60):
    return capi.Context(None, nprobe, k_refine, 20, 3, max_batch=max_batch)

def build(ctx, docs, doc_len=100, clusters=2048, ex_bits=1):
    lens = np.full(docs, doc_len, np.int32)
    n = docs * doc_len
    ids, flips = np.arange(clusters, dtype=np.int64), np.zeros(64, np.uint8)
    capi.check(capi.lib().chimera_build_index_device(
        ctx.handle, C.c_void_p(4096), C.c_uint64(n), C.c_uint64(128), capi._ptr(lens), C.c_uint64(docs),
        C.c_uint64(clusters), C.c_uint64(ex_bits), capi._ptr(ids), capi._ptr(flips), C.byref(ctx.options),
        ctx.max_batch))
    ctx._set_shape(n, 128, clusters, ex_bits, lens)

def workspace():
    \"\"\"Bytes of the last index's search workspace: the last block but the
    status word's.\"\"\"
    assert hip.host_hip_malloc(0) == 4
    return hip.host_hip_malloc(1)

def zeros(nq):
    return np.zeros((nq, 32, 128), np.float32)

def fresh_peak(*args, **kw):
    \"\"\"Most memory that this build takes in a context of its own.\"\"\"
    ctx = context()
    hip.host_hip_reset_peak()
    base = hip.host_hip_used()
    build(ctx, *args, **kw)
    peak = hip.host_hip_peak() - base
    ctx.close()
    assert hip.host_hip_used() == base
    return peak
"""


@pytest.fixture(scope="session")
def host_hip(tmp_path_factory):
    so = tmp_path_factory.mktemp("host_hip") / "libamdhip64.so.7"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-w", str(HERE / "host_hip" / "host_hip.cpp"), "-o", str(so), "-Wl,-soname,libamdhip64.so.7"],
                   check=True, timeout=300)

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRELUDE + code, str(so)], cwd=HERE.parent, text=True,
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=300)
        assert p.returncode == 0, p.stdout
        return p.stdout

    return run
