"""The library's handling of device memory and of failing allocations, on the
CPU: a child process runs libchimera_hip.so on a model of the HIP runtime
(tests/host_hip), whose device memory has a set capacity and whose kernels do
nothing. What is checked is host code: what is allocated when, what a failure
leaves behind and in which order copies run."""
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


# 90,000 documents of 8-bit codes: blocks that 200,000 of 2-bit codes fit in,
# with a fifth of them unused
@pytest.mark.parametrize("docs,ex_bits", [(10_000, 1), (30_000, 1), (60_000, 1), (90_000, 7), (200_000, 1)])
def test_a_rebuild_needs_no_more_memory_than_a_first_build(host_hip, docs, ex_bits):
    # few CUs: the build's scratch is larger than the probe's record area
    host_hip(f"""
hip.host_hip_set_cus(4)
capacity(1 << 40)
need = max(fresh_peak(200_000), fresh_peak({docs}, ex_bits={ex_bits})) + (16 << 20)
ctx = context()
build(ctx, {docs}, ex_bits={ex_bits})
capacity(need)
build(ctx, 200_000)
assert hip.host_hip_used() <= need
assert ctx.search(zeros(8), 10)[0].shape == (8, 10)
""")


def test_the_probe_buffers_do_not_add_to_a_builds_scratch(host_hip):
    """Where the scratch does not fit the probe's record area, the probe's
    buffers (larger for larger batches) come after it."""
    host_hip("""
hip.host_hip_set_cus(4)
capacity(1 << 40)
peaks = []
for batch in (8, 256):
    ctx = context(max_batch=batch)
    hip.host_hip_reset_peak()
    build(ctx, 200_000, clusters=50_000)
    peaks.append(hip.host_hip_peak())
    assert hip.host_hip_used() < peaks[-1]  # the build is the peak, not what it leaves
    ctx.close()
assert abs(peaks[1] - peaks[0]) < 1 << 20, peaks
""")


def test_a_rebuild_plans_the_sub_batches_of_a_first_build(host_hip):
    """The queries per sub-batch come from the free memory, of which the
    blocks of the replaced index are part."""
    host_hip("""
capacity(20 << 30)
large, small = dict(docs=2_000_000, doc_len=3), dict(docs=20_000)

def plan(ctx):
    hip.host_hip_reset_launches()
    ctx.search(zeros(2048), 10)
    return hip.host_hip_launches(b"cand_count"), ctx.memory_usage()

fresh = context(max_batch=2048)
build(fresh, **large)
want = plan(fresh)
assert want[0] == 2  # the memory bounds them
fresh.close()
ctx = context(max_batch=2048)
build(ctx, **large)
build(ctx, **small)
build(ctx, **large)
assert plan(ctx) == want
build(ctx, **large)
assert plan(ctx) == want
build(ctx, docs=3_000_000, doc_len=2)
other = plan(ctx)
ctx.close()
fresh = context(max_batch=2048)
build(fresh, docs=3_000_000, doc_len=2)
assert plan(fresh)[0] == other[0]
""")


@pytest.mark.parametrize("refuse", ["host_hip_refuse_malloc(C.c_size_t(4 * ctx.n), C.c_size_t(4 * ctx.n))",
                                    "host_hip_refuse_host(1)"], ids=["positions", "ring"])
def test_a_download_that_falls_back_leaves_no_error(host_hip, refuse):
    """Without room for the token positions, or without pinned memory, the
    download takes another way; the error it met is not the next call's."""
    host_hip(f"""
ctx = context()
build(ctx, 20_000)
want = ctx.download()
ctx.close()
ctx = context()
build(ctx, 20_000)
hip.{refuse}
got = ctx.download()
assert all(np.array_equal(got[k], want[k]) for k in want)
assert ctx.search(zeros(8), 10)[0].shape == (8, 10)
""")


def test_a_search_without_a_device_view_of_its_staging_buffer(host_hip):
    host_hip("""
ctx = context()
build(ctx, 20_000)
hip.host_hip_refuse_pointer(1)
assert ctx.search(zeros(2), 10)[0].shape == (2, 10)
assert ctx.search(zeros(2), 10)[0].shape == (2, 10)
""")


def test_a_failed_build_leaves_no_error_to_other_contexts(host_hip):
    host_hip("""
ctx, other = context(), context()
build(ctx, 20_000)
capacity(hip.host_hip_used() + (64 << 20))
try:
    build(other, 200_000)
    raise AssertionError("no room for it")
except capi.ChimeraError as e:
    assert e.code == capi.ERR_HIP and "out of memory" in str(e)
assert ctx.search(zeros(8), 10)[0].shape == (8, 10)
try:
    ctx.alloc(1 << 40)
    raise AssertionError("no room for it")
except capi.ChimeraError as e:
    assert e.code == capi.ERR_HIP and "out of memory" in str(e)
assert ctx.search(zeros(8), 10)[0].shape == (8, 10)
""")


@pytest.mark.parametrize("threads", [0, 3])
def test_a_download_with_too_few_threads_keeps_the_order(host_hip, threads):
    """Without threads for every slot of the ring the rest is copied by the
    caller, after the kernel that makes the token positions."""
    host_hip(f"""
import resource
ctx = context()
build(ctx, 20_000)
want = ctx.download()
assert want["token_to_cluster_pos"].any()
stack, libc = 4 << 30, C.CDLL(None)
attr = (C.c_char * 64)()
assert libc.pthread_attr_init(attr) == 0
assert libc.pthread_attr_setstacksize(attr, C.c_size_t(stack)) == 0
assert libc.pthread_setattr_default_np(attr) == 0  # later threads' stacks
size = int(open("/proc/self/statm").read().split()[0]) * 4096
limit = size + {threads} * (stack + (1 << 20)) + (1 << 30)
resource.setrlimit(resource.RLIMIT_AS, (limit, limit))  # room for so many of them
got = ctx.download()
assert all(np.array_equal(got[k], want[k]) for k in want)
""")


def test_assignment_lists_hold_256_candidates(host_hip):
    """Repeated tokens put many centroids within a row's margin; up to 256 of
    them in one of its lists keep the row off the exact recomputation."""
    host_hip("""
ctx = context()
build(ctx, 20_000)
assert hip.host_hip_lane_cap() == 256
""")


def test_a_one_query_workspace_holds_the_visit_counts_it_can_use(host_hip):
    """Visit counts are held for the queries and for the parts that a small
    batch's visits are split into (16 of them on 256 CUs), not for more."""
    host_hip("""
capacity(1 << 40)
sizes = []
for batch in (8, 16):
    ctx = context(max_batch=batch)
    build(ctx, 10_000_000, doc_len=1, clusters=200_000)
    sizes.append(workspace())
    ctx.close()
assert sizes[0] < 0.56 * sizes[1], sizes
""")


def test_the_split_selection_holds_state_for_the_queries_that_take_it(host_hip):
    """At 2M documents that is 2 queries at most. Past k_refine 2048 its lists
    double (32 KB a query); nothing else grows by more than a word a query."""
    host_hip("""
capacity(1 << 40)
sizes = []
for k_refine in (2048, 2049):
    ctx = context(max_batch=1024, k_refine=k_refine)
    build(ctx, 2_000_000, doc_len=1, clusters=200_000)
    sizes.append(workspace())
    ctx.close()
assert 0 < sizes[1] - sizes[0] < 1 << 20, sizes
""")


def test_the_workspace_stays_within_its_budget(host_hip):
    """Per-query state, visit counts and split selection together take at most
    half of the free memory (and at least 1 GiB of budget)."""
    host_hip("""
capacity(4500 << 20)
for k_refine in (60, 4097):
    ctx = context(max_batch=1024, k_refine=k_refine)
    build(ctx, 7000, doc_len=300)
    batch_arrays = 1024 * (32 * (128 * 8 + 8 * 4 + 8) + 65536 + 3 * 4 * k_refine + 512)
    assert workspace() < (1 << 30) + batch_arrays + (64 << 10), (workspace(), batch_arrays)
    hip.host_hip_reset_launches()
    ctx.search(zeros(1024), 10)
    assert hip.host_hip_launches(b"cand_count") > 1  # the budget bounds the sub-batches
    ctx.close()
""")


# documents, k_refine, queries of the batch, split: on either side of every
# line of the rule (64 documents a group)
@pytest.mark.parametrize("docs,k_refine,nq,split", [
    (50_000, 1000, 160, True), (50_000, 1000, 161, False),    # the groups cannot prune: 8M documents of all queries
    (10_000, 1000, 256, True), (10_000, 1000, 257, False),    # and a query a CU
    (200_000, 2500, 20, True), (200_000, 2500, 21, False),    # more groups, lists past 4,096 keys: 4M
    (100_000, 1500, 10, True), (100_000, 1500, 11, False),    # shorter lists: 1M
    (100_000, 1024, 1, False), (20_000, 200, 1, False),       # short lists
    (5_000_000, 3000, 1, False)])
def test_calls_that_take_the_split_selection(host_hip, docs, k_refine, nq, split):
    host_hip(f"""
capacity(1 << 40)
ctx = context(max_batch=300, k_refine={k_refine})
build(ctx, {docs}, doc_len=1, clusters=4096)
hip.host_hip_reset_launches()
ctx.search(zeros({nq}), 10)
assert hip.host_hip_launches(b"select_refine") == 1
assert hip.host_hip_launches(b"select_collect") == {int(split)}
""")


@pytest.mark.parametrize("ex_bits,intervals", [(1, 256), (6, 256), (7, 512)])
def test_the_encoders_intervals(host_hip, ex_bits, intervals):
    host_hip(f"""
build(context(), 1000, ex_bits={ex_bits})
assert hip.host_hip_launches(b"encode_tokens_kernelILi{intervals}E") == 1
""")
