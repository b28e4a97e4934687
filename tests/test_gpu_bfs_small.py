"""Searches on both sides of the one-workgroup form's limits (32768 vertices,
600000 edges) and the form each of them runs: shapes with one level per vertex,
a level past the in-LDS queue (4096), no out-edges, several components, rows
around the length that takes the whole workgroup (4096 out-edges), hubs whose
first level goes either way, and a search that returns to top-down, against a
plain queue search."""
from collections import deque

import numpy as np
import pytest

from conftest import gpu_case
from llama_amd.graph import UNREACHED, DeviceGraph, HostGraph

pytestmark = pytest.mark.gpu


def levels_of(V, src, dst, root):
    order = np.argsort(src, kind="stable")
    ofs = np.zeros(V + 1, np.int64)
    np.add.at(ofs, src + 1, 1)
    ofs = np.cumsum(ofs)
    adj = dst[order]
    lv = np.full(V, UNREACHED, np.int32)
    lv[root] = 0
    q = deque([root])
    while q:
        u = q.popleft()
        for v in adj[ofs[u]:ofs[u + 1]]:
            if lv[v] == UNREACHED:
                lv[v] = lv[u] + 1
                q.append(v)
    return lv


def shape(name, V, rng):
    ids = np.arange(V)
    if name == "path":
        return ids[:-1], ids[1:]
    if name == "star":  # out of the hub and back
        hub, rest = 1, np.delete(ids, 1)
        return (np.concatenate([np.full(V - 1, hub), rest[: V // 3]]),
                np.concatenate([rest, np.full(V // 3, hub)]))
    if name == "skewed":
        n = 14 * V
        s, d = rng.integers(0, V, n), (V * rng.random(n) ** 4).astype(np.int64)
        s[: n // 4] = (V * rng.random(n // 4) ** 4).astype(np.int64)
        k = s != d
        return s[k], d[k]
    # two-way random graph of one half, nothing in the other
    n, h = 3 * V, max(V // 2, 1)
    s, d = rng.integers(0, h, n), rng.integers(0, h, n)
    k = s != d
    return np.concatenate([s[k], d[k]]), np.concatenate([d[k], s[k]])


@pytest.mark.parametrize("name,V", [
    ("halves", 1), ("path", 2), ("halves", 63), ("halves", 64), ("skewed", 65), ("path", 3001),
    ("star", 4097), ("star", 4098), ("star", 4099), ("star", 32768), ("skewed", 32767),
    ("skewed", 32768), ("halves", 32769), ("star", 40000), ("path", 33000), ("skewed", 50001),
    ("skewed", 140001)])
def test_levels(ctx, name, V):
    if name == "path" and V > 32768:
        V = 32769  # past the limit: a host round trip per level
    rng = np.random.default_rng(V)
    src, dst = shape(name, V, rng)
    g = HostGraph(V)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    deg = np.bincount(src, minlength=V)
    roots = {0, V - 1, V // 2, int(np.argmax(deg)), int(np.argmin(deg)), min(1, V - 1)}
    if name == "path":
        roots = {0, V - 2}
    for root in sorted(roots):
        gpu_case(f"bfs {name} V={V} root={root}")
        ref = levels_of(V, src, dst, root)
        lv, reached, _ = dg.bfs(root)
        assert np.array_equal(lv, ref)
        assert reached == int((ref != UNREACHED).sum())
        assert dg.last_bfs_traversed == int(deg[ref != UNREACHED].sum())
        # the same without the reach set, and (past the limits) with the option
        # that lets a search return to top-down
        for opt, val in (("bfs_reach", 0), ("bfs_beta", 8)):
            ctx.set_option(opt, val)
            try:
                lv2, reached2, _ = dg.bfs(root)
            finally:
                ctx.set_option(opt, 1 if opt == "bfs_reach" else -1)
            assert np.array_equal(lv2, ref) and reached2 == reached


def forms(ctx, search):
    """The forms a search ran: launches of the one-workgroup search, of
    top-down levels past the first and of bottom-up levels."""
    ctx.profile(True)
    try:
        out = search()
        return out, [ctx.kernel_time(k)[0] for k in ("k_bfs_tiny", "k_td_expand", "k_bu_step")]
    finally:
        ctx.profile(False)


# 45400 edges among the others: 4540 are at most a tenth of them
@pytest.mark.parametrize("hub_edges,bottom_up", [(1, False), (4540, False), (4541, True),
                                                 (40000, True)])
def test_first_level_of_a_hub(ctx, hub_edges, bottom_up):
    """A root whose out-edges exceed the unexplored ones / alpha starts
    bottom-up, others top-down; the leaves lead nowhere, so level 1 is the
    last one."""
    V = 40001
    rng = np.random.default_rng(hub_edges)
    leaf = 1 + rng.choice(V - 1, hub_edges, replace=False)
    ring = np.arange(V, V + 100)  # edges the search never sees
    src = np.concatenate([np.zeros(hub_edges, np.int64), np.repeat(ring, 454)])
    dst = np.concatenate([leaf, np.tile(ring, 454)])
    g = HostGraph(V + 100)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    ctx.set_option("bfs_reach", 0)
    try:
        dg.bfs(0)
        gpu_case(f"bfs hub of {hub_edges} edges")
        (lv, reached, _), (tiny, _, bu) = forms(ctx, lambda: dg.bfs(0))
    finally:
        ctx.set_option("bfs_reach", 1)
    assert np.array_equal(lv, levels_of(V + 100, src, dst, 0)) and reached == 1 + hub_edges
    assert dg.last_bfs_traversed == hub_edges
    assert (tiny, bu > 0) == (0, bottom_up)


@pytest.mark.parametrize("V,E,one_workgroup", [
    (32768, 599_999, True), (32768, 600_000, True), (32768, 600_001, False), (1000, 600_001, False),
    (32769, 600_000, False), (32769, 1000, False), (32768, 1000, True)])
def test_form_limits(ctx, V, E, one_workgroup):
    rng = np.random.default_rng(E)
    src, dst = rng.integers(0, V, E), (V * rng.random(E) ** 2).astype(np.int64)
    g = HostGraph(V)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    root = int(src[0])
    dg.bfs(root)
    gpu_case(f"bfs limits V={V} E={E}")
    (lv, _, _), (tiny, td, bu) = forms(ctx, lambda: dg.bfs(root))
    assert np.array_equal(lv, levels_of(V, src, dst, root))
    assert tiny == (1 if one_workgroup else 0)
    assert not one_workgroup or td + bu == 0


def test_return_to_top_down(ctx):
    """A dense part, which goes bottom-up, and a tail of one vertex a level:
    with bfs_beta the search returns to top-down for the tail, without it
    stays bottom-up (the whole graph is the reach set)."""
    n, tail = 40_000, 60
    V = n + tail
    rng = np.random.default_rng(4)
    t = np.arange(n, V)
    src = np.concatenate([rng.integers(0, n, 8 * n), [0], t])
    dst = np.concatenate([rng.integers(0, n, 8 * n), [n], t[1:], [0]])
    g = HostGraph(V)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    ref = levels_of(V, src, dst, 1)
    dg.bfs(1)
    for beta, returns in ((8, True), (-1, False)):
        gpu_case(f"bfs return to top-down, beta {beta}")
        ctx.set_option("bfs_beta", beta)
        try:
            (lv, _, _), (_, td, bu) = forms(ctx, lambda: dg.bfs(1))
        finally:
            ctx.set_option("bfs_beta", -1)
        assert np.array_equal(lv, ref)
        assert bu > 0 and (td >= tail // 2) == returns  # the dense part ends within ten levels


@pytest.mark.parametrize("n", [4095, 4096, 4097, 25_000])
def test_long_rows_of_a_wide_level(ctx, n):
    """Twenty vertices queued together, three of them with n out-edges: at most
    a tenth of the edges, so their level goes top-down."""
    V = 32768
    rng = np.random.default_rng(n)
    mid = np.arange(1, 21)
    src = np.concatenate([np.zeros(20, np.int64), mid, np.repeat(mid[:3], n // 3 if n > 9000 else n),
                          rng.integers(21, V, 500_000)])
    dst = np.concatenate([mid, 21 + rng.integers(0, V - 21, src.size - 20)])
    g = HostGraph(V)
    g.add_level(src, dst)
    dg = DeviceGraph(ctx, g)
    dg.bfs(0)
    gpu_case(f"bfs long rows of {n}")
    (lv, _, _), (tiny, _, _) = forms(ctx, lambda: dg.bfs(0))
    assert tiny == 1 and np.array_equal(lv, levels_of(V, src, dst, 0))
