"""Batched personalised PageRank over rows of every length a wave meets: runs
of empty rows, rows ending inside, at and past a group of eight and a chunk of
64 entries, the longest row of a shared item, pieces of long rows and row
counts around 64 and 256."""
import numpy as np
import pytest

import oracle
from conftest import gpu_case
from llama_amd.graph import DeviceGraph, HostGraph

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 7, 8, 9, 0, 0, 63, 64, 65, 71, 72, 73, 126, 127, 128, 129, 191, 193, 1023, 1024,
           1025, 2047, 2049, 4101]


@pytest.mark.parametrize("width", [32, 64, 128])
@pytest.mark.parametrize("empty", [0, 63, 64, 257])
def test_row_lengths(ctx, width, empty):
    gpu_case(f"ppr rows width={width} empty={empty}")
    rng = np.random.default_rng(empty + 1)
    V = 6000
    lengths = np.concatenate([np.zeros(empty, np.int64), rng.permutation(LENGTHS),
                              rng.integers(0, 4, 700), rng.permutation(LENGTHS)])
    dst = np.repeat(np.arange(len(lengths)), lengths)
    src = np.concatenate([rng.choice(V, n, replace=False) for n in lengths])
    g = HostGraph(V)
    g.add_level(src, dst)
    seeds = rng.integers(0, V, width + 3)
    R, it = DeviceGraph(ctx, g).ppr_batch(seeds, iters=8, tol=0.0, batch_width=width)
    ref, it_ref = oracle.OracleGraph.from_host(g).ppr(seeds, 8)
    assert it == it_ref
    # per column: five FP32 roundings an iteration (1/outdeg, product, sum,
    # damping, teleport), at most 2^-24 of the value each
    err = np.abs(R.astype(np.float64) - ref).sum(axis=0) / np.abs(ref).sum(axis=0)
    assert err.max() <= 8 * 5 * 2.0 ** -24
