"""Which kernels a call takes at the lines of the dispatch rules, on the CPU:
the library runs on a model of the HIP runtime (tests/host_hip) that counts
launches and runs no kernel. The kernels' results at these sizes are the GPU
tests' subject."""
import pytest

from host_hip_child import host_hip  # noqa: F401


def test_assignment_lists_hold_256_candidates(host_hip):
    """Repeated tokens put many centroids within a row's margin; up to 256 of
    them in one of its lists keep the row off the exact recomputation."""
    host_hip("""
ctx = context()
build(ctx, 20_000)
assert hip.host_hip_lane_cap() == 256
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


@pytest.mark.parametrize("nq,cands,waves", [(1, 1, 4), (8, 64, 4), (27, 19, 2), (2, 1024, 2), (3, 683, 0)])
def test_the_waves_of_a_small_rescoring_call(host_hip, nq, cands, waves):
    host_hip(f"""
ctx = context()
buf = C.c_void_p(4096)
capi.check(capi.lib().chimera_maxsim_rescore_device(
    ctx.handle, buf, buf, C.c_int64(60), buf, C.c_int32({nq}), buf, buf, C.c_int32({cands}), C.c_int32(0), buf,
    None, None, None))
assert hip.host_hip_threads(b"maxsim_rescore_small_kernel") == 64 * {waves}
assert hip.host_hip_launches(b"maxsim_rescore") == 1
""")


def probe_launches(host_hip, clusters, rows, *kernels):
    host_hip(f"""
ctx = context(max_batch=128, nprobe=128, k_refine=200)
build(ctx, 4000, doc_len=100, clusters={clusters})
hip.host_hip_reset_launches()
buf = C.c_void_p(4096)
capi.check(capi.lib().chimera_probe_device(ctx.handle, buf, {rows}, 128, buf))
for kernel in {kernels}:
    assert hip.host_hip_launches(kernel.encode()) == 1, kernel
""")


# sampled minima of a row: 128, 256, 257, 1,024, 1,559
@pytest.mark.parametrize("clusters,rows,kernel", [
    (4096, 32, "wave_kernelILi8E"), (8192, 32, "wave_kernelILi8E"), (8193, 384, "kernelEPKf"),
    (8193, 385, "wave_kernelILi8E"), (131_072, 384, "kernelEPKf"), (131_072, 385, "wave_kernelILi16E"),
    (399_000, 32, "kernelEPKf"), (399_000, 4096, "wave_kernelILi32E")])
def test_the_threshold_kernel(host_hip, clusters, rows, kernel):
    probe_launches(host_hip, clusters, rows, "probe_threshold_" + kernel)


# waves that share 64 rows, in the sampled and in the filtered pass; splits of
# one stage up to 8,192 centroids
@pytest.mark.parametrize("clusters,rows,sampled,filtered", [
    (8192, 32, 2, 2), (8192, 64, 2, 2), (8192, 65, 2, 1), (8192, 128, 2, 1), (8192, 129, 1, 1),
    (20_000, 64, 2, 8), (20_000, 65, 2, 2), (20_000, 128, 2, 2), (20_000, 129, 1, 1), (262_144, 32, 2, 8)])
def test_the_waves_that_share_probe_rows(host_hip, clusters, rows, sampled, filtered):
    probe_launches(host_hip, clusters, rows, f"probe_mfma_kernelILi0ELi1ELi{sampled}E",
                   f"probe_mfma_kernelILi1ELi4ELi{filtered}E")
