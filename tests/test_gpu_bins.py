"""The binned out-edge layout at every bin size its automatic rule picks: ranks
are bit-identical to those over explicit bins of 2^12 vertices (row sums are
integers) and within 1e-6 L1 of the FP64 oracle, and multi-source sweeps over
it give every lane its single-source levels."""
import time

import numpy as np
import pytest

import oracle
from conftest import gpu_case
from llama_amd.graph import DeviceGraph, GpuContext, HostGraph, SlcsrGraph, csr_of

pytestmark = pytest.mark.gpu


def skewed(V, per, seed):
    """per * V edges whose heads crowd the low IDs, a hub at V // 2, no self-loops."""
    rng = np.random.default_rng(seed)
    n = V * per
    src = rng.integers(0, V, n)
    dst = (V * rng.random(n) ** 3).astype(np.int64)
    dst[: n // 20] = V // 2
    keep = src != dst
    g = HostGraph(V)
    g.add_level(src[keep], dst[keep])
    return g


# vertices, edges per vertex: bins of 2^8 (one, two, fewer than a workgroup's
# waves, forty), then 2^9, 2^10, 2^11; chunks of a slot to thousands of slots
@pytest.mark.parametrize("V,per", [(2, 3), (256, 5), (257, 400), (3000, 20), (10007, 16),
                                   (20011, 8), (140001, 12), (600011, 16)])
def test_every_bin_size(ctx, V, per):
    gpu_case(f"bins V={V} per={per}")
    g = skewed(V, per, V)
    dg = DeviceGraph(ctx, g)
    r, diff = dg.pagerank(6)
    ctx.set_option("pr_bin_bits", 12)
    try:
        r12, diff12 = dg.pagerank(6)
    finally:
        ctx.set_option("pr_bin_bits", -1)
    assert np.array_equal(r, r12)
    # FP64 sums of the same FP32 differences in another order
    assert abs(diff - diff12) <= 1e-12 * max(abs(diff), 1e-30) + 1e-15
    if V <= 20011:
        ref, _ = oracle.OracleGraph.from_host(g).pagerank(6)
        assert float(np.abs(r - ref).sum() / np.abs(ref).sum()) <= 1e-6
    roots = np.random.default_rng(V).integers(0, V, 130)
    ctx.set_option("bfs_batch_bins", 1)
    try:
        for lanes in (16, 64, 128):
            gpu_case(f"bins V={V} lanes={lanes}")
            lv, reached, _ = dg.bfs_batch(roots, lane_width=lanes)
            for j in (0, 63, 129):
                one, n, _ = dg.bfs(int(roots[j]))
                assert np.array_equal(lv[j], one) and reached[j] == n
    finally:
        ctx.set_option("bfs_batch_bins", -1)


# one bin of any size holds every slot: from 40 edges on PageRank takes 2^8,
# below 2^14, whose 128-lane words do not fit a workgroup's LDS; those sweeps
# take 2^13 down to 32 edges, and none below
@pytest.mark.parametrize("E,lane_layout", [(31, False), (32, True), (39, True), (40, True)])
def test_wide_lanes_build_their_own_layout_alone(ctx, E, lane_layout):
    """A 128-lane sweep builds the one layout it reads, whatever PageRank's
    would be, and takes its levels from it."""
    V = 100
    rng = np.random.default_rng(E)
    pairs = rng.choice(V * (V - 1), E, replace=False)
    src, dst = pairs // (V - 1), pairs % (V - 1)
    dst = dst + (dst >= src)
    g = HostGraph(V)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    roots = np.concatenate([src, rng.integers(0, V, 128 - E)])
    gpu_case(f"lane layout E={E}")
    ctx.set_option("bfs_batch_bins", 1)
    ctx.profile(True)
    try:
        lv, reached, _ = dg.bfs_batch(roots, lane_width=128)
        builds, _ = ctx.kernel_time("pr_bins_build")
        sweeps, _ = ctx.kernel_time("k_msb_sweep")
    finally:
        ctx.profile(False)
        ctx.set_option("bfs_batch_bins", -1)
    assert (builds, sweeps > 0) == ((1, True) if lane_layout else (0, False))
    for j, root in enumerate(roots):
        one, n, _ = dg.bfs(int(root))
        assert np.array_equal(lv[j], one) and reached[j] == n


def test_autotuned_width_is_a_fast_one():
    """The width chosen on a new snapshot costs no more than the best explicit
    one (a fifth allowed; runs differ by 5%): what a width's trial finds
    unbuilt or unallocated is not held against it."""
    V, E, n = 1 << 22, 9_600_000, 512
    rng = np.random.default_rng(8)
    src, dst = np.zeros(E, np.int64), np.zeros(E, np.int64)
    for _ in range(22):  # R-MAT
        r = rng.random(E)
        src = 2 * src + (r >= 0.76)
        dst = 2 * dst + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    ids = rng.permutation(V)
    src, dst = ids[src], ids[dst]
    roots = src[rng.integers(0, E, n)]
    own = GpuContext(0)
    try:
        dg = SlcsrGraph(own, V, csr_of(V, src, dst), csr_of(V, dst, src))
        took = {}
        for w in (0, 16, 32, 64, 128):
            gpu_case(f"autotuned width, {w} lanes")
            for _ in range(4):
                t0 = time.perf_counter()
                dg.bfs_batch(roots, w, want_levels=False)
                took[w] = min(took.get(w, 1e9), time.perf_counter() - t0)
        assert took[0] <= 1.2 * min(took[w] for w in (16, 32, 64, 128)), took
    finally:
        own.close()
