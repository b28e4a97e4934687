"""Weighted searches where the one-launch rounds can go wrong: vertex counts
that are no multiple of four, rows around the bound of the shared ones (256)
and of their chunks (1024), more appends than a workgroup stages (2048), more
shared rows in one split than it stages (512), zero weights, equal distances.
Distances bit for bit against float32 Bellman-Ford."""
import numpy as np
import pytest

from conftest import gpu_case
from llama_amd.graph import DeviceGraph, HostGraph

pytestmark = pytest.mark.gpu

UNREACHED = np.float32(2147483646)


def bellman_ford(V, src, dst, w, root):
    d = np.full(V, UNREACHED, np.float32)
    d[root] = 0
    while True:
        n = d.copy()
        ok = d[src] < UNREACHED
        np.minimum.at(n, dst[ok], d[src[ok]] + w[ok])
        if np.array_equal(n, d):
            return d
        d = n


def check(ctx, V, src, dst, w, roots, name):
    g = HostGraph(V)
    g.add_level(src, dst, weights=w.astype(np.float32))
    dg = DeviceGraph(ctx, g)
    for root in roots:
        ref = bellman_ford(V, src, dst, w.astype(np.float32), root)
        for delta, mq in ((-1, -1), (0, -1), (1, 0), (400, 7)):
            gpu_case(f"sssp {name} V={V} root={root} delta={delta} min_queue={mq}")
            ctx.set_option("sssp_delta_milli", delta)
            ctx.set_option("sssp_min_queue", mq)
            try:
                d, n, mx, rounds = dg.sssp(root)
            finally:
                ctx.set_option("sssp_delta_milli", -1)
                ctx.set_option("sssp_min_queue", -1)
            assert np.array_equal(d, ref)
            reached = ref < UNREACHED
            assert n == int(reached.sum()) and mx == float(ref[reached].max()) and rounds > 0


@pytest.mark.parametrize("V", [1, 2, 3, 5, 67, 1001])
def test_small(ctx, V):
    rng = np.random.default_rng(V)
    n = 6 * V if V > 1 else 1
    s, d = rng.integers(0, V, n), rng.integers(0, V, n)
    check(ctx, V, s, d, rng.random(n), {0, V - 1}, "small")


@pytest.mark.parametrize("zero", [False, True])
def test_row_lengths(ctx, zero):
    """Rows of 1, 255..257, 1023..1025, 2048 and 5000 edges, some weights zero."""
    V = 6002
    rng = np.random.default_rng(9)
    src = np.concatenate([np.full(k, i) for i, k in enumerate(
        [5000, 255, 256, 257, 1023, 1024, 1025, 2048, 1])] + [np.arange(9, V)] * 3)
    dst = rng.integers(0, V, src.size)
    w = rng.random(src.size)
    if zero:
        w[rng.random(src.size) < 0.4] = 0
        w[(src < 9)] *= rng.random(int((src < 9).sum())) < 0.5
    check(ctx, V, src, dst, w, (0, 3, 7, 4000), f"rows zero={zero}")


def test_many_appends(ctx):
    """Every vertex of the third level queued in one round, 1500 rows of 2000."""
    mids, leaves = 1500, 2000
    V = 1 + mids + mids * leaves
    m = np.arange(1, 1 + mids)
    leaf = np.arange(1 + mids, V)
    src = np.concatenate([np.zeros(mids, np.int64), np.repeat(m, leaves), leaf])
    dst = np.concatenate([m, leaf, np.zeros(leaf.size, np.int64)])
    g = HostGraph(V)
    g.add_level(src, dst, weights=np.full(src.size, 0.25, np.float32))
    gpu_case("sssp many appends")
    d, n, mx, _ = DeviceGraph(ctx, g).sssp(0)
    assert n == V and mx == 0.5
    assert d[0] == 0 and np.all(d[m] == 0.25) and np.all(d[leaf] == 0.5)


def test_many_shared_rows_in_one_split(ctx):
    """8000 far vertices of 300 edges, all at one distance."""
    V, deg = 8003, 300
    rng = np.random.default_rng(4)
    rest = np.arange(1, V)
    src = np.concatenate([np.zeros(V - 1, np.int64), np.repeat(rest, deg)])
    dst = np.concatenate([rest, rng.integers(0, V, (V - 1) * deg)])
    w = np.concatenate([np.full(V - 1, 5.0), np.full((V - 1) * deg, 0.5)])
    check(ctx, V, src, dst, w, (0, 77), "one split")


@pytest.mark.parametrize("min_queue", [-1, 200_000])
def test_fixed_point_on_a_skewed_graph(ctx, min_queue):
    """Thousands of shared rows whose distances drop while their chunks wait,
    small queues rejoining the far pile: no edge is left that would lower its
    head, and every reached vertex has an edge that gives its distance."""
    V, E = 400_003, 6_000_000
    rng = np.random.default_rng(12)
    src = (V * rng.random(E) ** 3).astype(np.int64)
    dst = (V * rng.random(E) ** 2).astype(np.int64)
    w = rng.random(E).astype(np.float32)
    g = HostGraph(V)
    g.add_level(src, dst, weights=w)
    dg = DeviceGraph(ctx, g)
    ctx.set_option("sssp_min_queue", min_queue)
    try:
        for root in (0, 1, 200_000):
            gpu_case(f"sssp fixed point root={root} min_queue={min_queue}")
            d, n, _, _ = dg.sssp(root)
            ok = d[src] < UNREACHED
            best = np.full(V, UNREACHED, np.float32)
            np.minimum.at(best, dst[ok], d[src[ok]] + w[ok])
            best[root] = 0
            assert np.array_equal(best, d)
            assert n == int((d < UNREACHED).sum())
    finally:
        ctx.set_option("sssp_min_queue", -1)


@pytest.mark.parametrize("V,E", [(64, 400_000), (2000, 3_000_000)])
def test_few_vertices_many_edges(ctx, V, E):
    """The edges of few vertices are spread over the chip: a round moves at most
    12 bytes an edge (1 to 8 us at the rate of a large copy) and a launch takes
    about 10 us, so 100 us a launch is several times what it needs."""
    rng = np.random.default_rng(V)
    src, dst = rng.integers(0, V, E), rng.integers(0, V, E)
    w = rng.random(E).astype(np.float32)
    g = HostGraph(V)
    g.add_level(src, dst, weights=w)
    dg = DeviceGraph(ctx, g)
    gpu_case(f"sssp few vertices V={V} E={E}")
    assert np.array_equal(dg.sssp(0)[0], bellman_ford(V, src, dst, w, 0))
    ctx.profile(True)
    try:
        dg.sssp(0)
        n, ms = ctx.kernel_time("k_relax")
    finally:
        ctx.profile(False)
    assert n > 0 and ms / n < 0.1
