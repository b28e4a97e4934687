"""Betweenness around one hub whose in-edges and out-edges are split into
pieces of 1536 entries that one wave joins 64 at a time: the path counts and
the terms are whole numbers, so the expected values are exact."""
import numpy as np
import pytest

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
