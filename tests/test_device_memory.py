"""The library's handling of device memory and of failing allocations, on the
CPU: the library runs on a model of the HIP runtime (tests/host_hip), whose
device memory has a set capacity and whose kernels do nothing. What is checked
is host code: what is allocated when, what a failure leaves behind and in which
order copies run."""
import pytest

from host_hip_child import host_hip  # noqa: F401


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
