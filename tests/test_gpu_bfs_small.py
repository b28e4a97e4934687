"""Searches on both sides of the one-workgroup form's limits (32768 vertices,
600000 edges): shapes with one level per vertex, a level past the in-LDS
queue (4096), no out-edges, several components, rows of every length around
the long-row bound, against a plain queue search."""
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
        # the same without the reach set, and with a return to top-down
        for opt, val in (("bfs_reach", 0), ("bfs_beta", 8)):
            ctx.set_option(opt, val)
            try:
                lv2, reached2, _ = dg.bfs(root)
            finally:
                ctx.set_option(opt, 1 if opt == "bfs_reach" else -1)
            assert np.array_equal(lv2, ref) and reached2 == reached
