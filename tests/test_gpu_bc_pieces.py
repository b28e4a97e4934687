"""Betweenness around one hub whose in-edges and out-edges are split into
pieces of 1536 entries that one wave joins 64 at a time: the path counts and
the terms are whole numbers, so the expected values are exact.  And rows whose
starts lie around the words of 64 entries that name an entry's row."""
import numpy as np
import pytest

import oracle
from conftest import gpu_case
from llama_amd.graph import DeviceGraph, HostGraph

pytestmark = pytest.mark.gpu

PIECE = 1536


@pytest.mark.parametrize("mids,leaves", [
    (511, 512), (512, 511), (PIECE, PIECE + 1), (PIECE + 1, PIECE),
    (64 * PIECE, 64 * PIECE + 1), (64 * PIECE + 1, 3 * PIECE), (130 * PIECE - 7, 600),
])
def test_hub_split_into_pieces(ctx, mids, leaves):
    gpu_case(f"bc hub of {mids} in-edges and {leaves} out-edges")
    hub = 1 + mids
    V = hub + 1 + leaves
    mid = np.arange(1, 1 + mids, dtype=np.int64)
    leaf = np.arange(hub + 1, V, dtype=np.int64)
    g = HostGraph(V)
    g.add_level(np.concatenate([np.zeros(mids, np.int64), mid, np.full(leaves, hub, np.int64)]),
                np.concatenate([mid, np.full(mids, hub, np.int64), leaf]))
    b = DeviceGraph(ctx, g).bc([0])
    want = np.zeros(V, np.float32)
    want[hub] = leaves
    want[mid] = np.float32(1) / np.float32(mids) * (np.float32(1) + np.float32(leaves))
    assert np.array_equal(b, want)


@pytest.mark.parametrize("empty", [0, 1, 63, 200, 300])
def test_row_starts(ctx, empty):
    """Rows of 0, 1, 63, 64, 65, 127..129 and 511 entries in any order, with
    runs of empty rows between them, bit for bit as the oracle adds them."""
    gpu_case(f"bc row starts, runs of {empty} empty rows")
    rng = np.random.default_rng(empty)
    lengths = []
    for n in rng.permutation([0, 1, 2, 63, 64, 65, 127, 128, 129, 511] * 4):
        lengths += [n] + [0] * (empty if rng.random() < 0.2 else 0)
    V = max(len(lengths), 2000)
    rows = np.repeat(np.arange(len(lengths)), lengths)
    ends = rng.integers(0, V, rows.size)
    extra = rng.integers(0, V, (2, 3 * V))
    g = HostGraph(V)
    g.add_level(np.concatenate([rows, ends, extra[0]]), np.concatenate([ends, rows, extra[1]]))
    sources = rng.integers(0, V, 5)
    assert np.array_equal(DeviceGraph(ctx, g).bc(sources),
                          oracle.OracleGraph.from_host(g).bc(sources))
