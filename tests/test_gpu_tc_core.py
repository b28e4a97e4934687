"""Triangle counts over the degree-numbered DAG: graphs within the core (32768
vertices), past it with hubs (most lists in the core), past it with even
degrees (many entries outside: the filter and its confirmation), and too even
for it (the form by vertex ID), against the CPU count; W and the arcs equal
the definition."""
import time

import numpy as np
import pytest

import oracle
from conftest import gpu_case
from llama_amd.graph import DIR_IN, DIR_OUT, DeviceGraph, HostGraph, SlcsrGraph, csr_of

pytestmark = pytest.mark.gpu


def dag_stats(V, src, dst):
    """Arcs and W = sum over arcs of d+(a) + d+(b), by the definition."""
    deg = np.bincount(src, minlength=V) + np.bincount(dst, minlength=V)
    k = src != dst
    s, d = src[k], dst[k]
    up = (deg[s] < deg[d]) | ((deg[s] == deg[d]) & (s < d))
    a, b = np.where(up, s, d), np.where(up, d, s)
    arcs = np.unique(a.astype(np.int64) * V + b)
    a, b = arcs // V, arcs % V
    dp = np.bincount(a, minlength=V)
    return arcs.size, int((dp[a] + dp[b]).sum())


def clustered(V, per, seed, skew):
    """Edges with closed wedges: random pairs, then ends of two-edge paths."""
    rng = np.random.default_rng(seed)
    n = V * per // 2
    s = (V * rng.random(n) ** skew).astype(np.int64)
    d = (V * rng.random(n) ** skew).astype(np.int64)
    near = (s + rng.integers(1, 40, n)) % V
    return np.concatenate([s, s]), np.concatenate([d, near])


@pytest.mark.parametrize("V,per,skew", [(3, 4, 1), (65, 30, 1), (2049, 40, 3), (32768, 10, 2),
                                        (32769, 12, 2), (70001, 16, 4), (100003, 12, 1),
                                        (220001, 8, 1), (250007, 10, 5)])
def test_counts(ctx, V, per, skew):
    gpu_case(f"tc core V={V} per={per} skew={skew}")
    src, dst = clustered(V, per, V, skew)
    g = HostGraph(V)
    g.add_level(src, dst)  # duplicates, both directions and self-loops included
    dg = DeviceGraph(ctx, g)
    n, arcs, work = dg.triangles(stats=True)
    assert n == oracle.OracleGraph.from_host(g).triangles()
    assert (arcs, work) == dag_stats(V, src, dst)
    assert dg.triangles() == n  # again, over the DAG already built
    assert dg.tc_i() >= n
    assert dg.triangles() == n


@pytest.mark.parametrize("outside", [0.60, 0.68, 0.74])
def test_hubs_beside_many_small_vertices(ctx, outside):
    """A core of hubs 16 times the mean degree or more with most edge ends
    outside it: on either side of, and between, the two limits of the share."""
    V, E, hubs = 2_200_000, 600_000, 32_768
    gpu_case(f"tc core hubs, {outside} of the ends outside")
    rng = np.random.default_rng(int(outside * 100))
    n = int(E * outside)
    top = rng.choice(V, hubs, replace=False)
    m = (E - n) // 2
    a, b = top[rng.integers(0, hubs, m)], top[(hubs * rng.random(m) ** 2).astype(np.int64)]
    s = rng.integers(0, V, n // 2)
    d = rng.integers(0, V, n // 2)
    src = np.concatenate([a, a, s, s])
    dst = np.concatenate([b, top[rng.integers(0, 300, m)], d, (s + 1) % V])
    g = HostGraph(V)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    n, arcs, work = dg.triangles(stats=True)
    assert n == oracle.OracleGraph.from_host(g).triangles()
    assert (arcs, work) == dag_stats(V, src, dst)


def test_rejected_graph_pays_no_sort(ctx):
    """Even degrees far past the core: the rule answers from a histogram and no
    vertex is numbered, so the first call is the DAG by vertex ID and a scan of
    the degrees (32 MB: 7 us at the copy rate; half a millisecond allowed)."""
    V = 4_000_000
    rng = np.random.default_rng(5)
    src, dst = rng.integers(0, V, 2 * V), rng.integers(0, V, 2 * V)
    dg = SlcsrGraph(ctx, V, csr_of(V, src, dst), csr_of(V, dst, src))

    def best(f):
        times = []
        for _ in range(6):
            dg.drop_snapshots()
            dg.degrees(DIR_OUT)
            dg.degrees(DIR_IN)
            dg.adjacency(DIR_OUT)
            t0 = time.perf_counter()
            f()
            times.append(time.perf_counter() - t0)
        return min(times)

    gpu_case("tc rejected graph")
    # tc_i builds the same DAG without the rule, and its count is the slower one
    assert best(dg.triangles) <= best(dg.tc_i) + 0.0005


def test_rows_of_one_arc(ctx):
    """A star: every row has one arc and closes nothing.  24 bytes a row are 12
    MB, 2.5 us at the copy rate; 25 times that is allowed."""
    V = 500_001
    leaf = np.arange(1, V)
    g = HostGraph(V)
    g.add_level(np.zeros(V - 1, np.int64), leaf)
    dg = DeviceGraph(ctx, g)
    gpu_case("tc star")
    n, arcs, work = dg.triangles(stats=True)
    # a leaf's row: its own d+ of 1 and the hub's of 0
    assert (n, arcs, work) == (0, V - 1, V - 1)
    ctx.profile(True)
    try:
        for _ in range(10):
            dg.triangles()
        k, ms = ctx.kernel_time("k_tc_core")
    finally:
        ctx.profile(False)
    assert k == 10 and ms / k < 0.0625, ms / k


def test_many_row_lengths(ctx):
    """Rows of no, one, two, 63..65 and more arcs beside each other, more rows
    than the waves' first 64, against the CPU count."""
    V = 300_000
    rng = np.random.default_rng(6)
    src = np.repeat(np.arange(V), rng.choice([0, 1, 1, 2, 3, 63, 64, 65], V,
                                             p=[.5, .2, .1, .1, .07, .01, .01, .01]))
    dst = (V * rng.random(src.size) ** 3).astype(np.int64)
    g = HostGraph(V)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    gpu_case("tc row lengths")
    n, arcs, work = dg.triangles(stats=True)
    assert n == oracle.OracleGraph.from_host(g).triangles()
    assert (arcs, work) == dag_stats(V, src, dst)
