"""Results and uploads through the staging buffer, at the sizes where the path
changes: the read-back buffer (64 KiB), one piece (under 1 MiB), chunks of 2
MiB moved on in slices of 256 KiB, and more than the staging holds (64 MiB);
pinned destinations; what the copies cost the host."""
import ctypes
import os
import threading
import time

import numpy as np
import pytest
import torch

from conftest import gpu_case
from llama_amd.graph import DIR_IN, DIR_OUT, GpuContext, SlcsrGraph, csr_of

pytestmark = pytest.mark.gpu

MB = 1 << 20


def graph(ctx, V, E, seed):
    rng = np.random.default_rng(seed)
    begin = np.zeros(V + 1, np.int64)
    begin[1:-1] = np.sort(rng.integers(0, E + 1, V - 1))
    begin[-1] = E
    vals = rng.integers(0, V, E)
    return SlcsrGraph(ctx, V, (begin, vals), (begin, vals[::-1].copy())), begin, vals


# bytes of the neighbour array
@pytest.mark.parametrize("nbytes", [4, 65532, 65536, 65540, MB - 4, MB, MB + 4, 2 * MB - 4,
                                    2 * MB, 2 * MB + 4, 2 * MB + MB // 4 + 4, 8 * MB - 4,
                                    8 * MB + 4, 64 * MB, 64 * MB + 4, 133 * MB])
def test_round_trip(ctx, nbytes):
    gpu_case(f"host copy {nbytes} bytes")
    V, E = 1000, nbytes // 4
    dg, begin, vals = graph(ctx, V, E, nbytes)
    for d, ref in ((DIR_OUT, vals), (DIR_IN, vals[::-1])):
        ofs, adj = dg.adjacency(d)
        assert np.array_equal(ofs, begin.astype(np.uint64))
        assert np.array_equal(adj, ref.astype(np.uint32))
    assert np.array_equal(dg.degrees(DIR_OUT), np.diff(begin).astype(np.uint32))


def test_contexts_on_threads():
    """Two contexts, a host thread each, copy at the same time."""
    bad = []

    def work(seed):
        c = GpuContext(0)
        dg, _, vals = graph(c, 50_000, 3_000_000, seed)
        for _ in range(4):
            if not np.array_equal(dg.adjacency(DIR_OUT)[1], vals.astype(np.uint32)):
                bad.append(seed)
        dg.close()
        c.close()

    gpu_case("host copy, two contexts")
    ts = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_no_thread_spins_while_kernels_run(ctx):
    """A result whose kernels are still queued is awaited by the caller alone:
    push PageRank queues all its iterations and then copies 8 MiB.  One thread
    waiting costs at most the wall time; half as much again is left for the
    copy itself."""
    V = 1 << 20
    rng = np.random.default_rng(2)
    src, dst = rng.integers(0, V, 8 * V), rng.integers(0, V, 8 * V)
    dg = SlcsrGraph(ctx, V, csr_of(V, src, dst), csr_of(V, dst, src))
    dg.pagerank_push(2)
    gpu_case("push PageRank, CPU time")
    wall, cpu = time.perf_counter(), time.process_time()
    dg.pagerank_push(200)
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.05 and cpu <= 1.5 * wall, (wall, cpu)


def test_pinned_destination(ctx):
    """A caller's pinned array is filled by the device itself, at the rate of a
    plain copy into it (through the staging: 1.6 times as long)."""
    V, E = 1000, 48_000_000
    dg, _, vals = graph(ctx, V, E, 5)
    buf = torch.zeros(E, dtype=torch.int32, pin_memory=True)
    out = buf.numpy().view(np.uint32)
    ptr = out.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))
    dev = torch.ones(E, dtype=torch.int32, device="cuda")

    def best(f):
        times = []
        for _ in range(6):
            t0 = time.perf_counter()
            f()
            times.append(time.perf_counter() - t0)
        return min(times)

    gpu_case("pinned destination")
    plain = best(lambda: buf.copy_(dev))
    ours = best(lambda: ctx.check(
        dg.lib.ll_gpu_snapshot_adjacency(dg._h, -1, DIR_OUT, None, ptr)))
    assert np.array_equal(out, vals.astype(np.uint32))
    assert ours <= 1.25 * plain, (ours, plain)


def test_small_results_cost_one_round_trip(ctx):
    """80 KB of degrees and the snapshot's figures take one copy or launch and
    one wait each, as a copy into pinned memory does: half as much again is
    left for moving 80 KB on, twice as much for walking the degrees."""
    V = 20_000
    rng = np.random.default_rng(1)
    src, dst = rng.integers(0, V, 4 * V), rng.integers(0, V, 4 * V)
    dg = SlcsrGraph(ctx, V, csr_of(V, src, dst), csr_of(V, dst, src))
    out = np.empty(V, np.uint32)
    ptr = out.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))
    dev = torch.ones(V, dtype=torch.int32, device="cuda")
    pin = torch.empty(V, dtype=torch.int32, pin_memory=True)

    def best(f):
        times = []
        for _ in range(300):
            t0 = time.perf_counter()
            f()
            times.append(time.perf_counter() - t0)
        return sorted(times)[30]

    gpu_case("small results")
    plain = best(lambda: pin.copy_(dev))
    deg = best(lambda: ctx.check(dg.lib.ll_gpu_snapshot_degrees(dg._h, -1, DIR_OUT, ptr)))
    info = best(dg.snapshot_info)
    assert np.array_equal(out, np.bincount(src, minlength=V).astype(np.uint32))
    assert deg <= 1.5 * plain and info <= 2 * plain, (deg, info, plain)


def test_small_uploads_need_no_threads():
    """A context starts its copy threads for the first array of 1 MiB or more,
    up or down."""
    def threads():
        return len(os.listdir("/proc/self/task"))

    gpu_case("small uploads")
    c = GpuContext(0)
    try:
        dg, _, _ = graph(c, 1000, 100_000, 1)  # 800 KB of IDs
        dg.adjacency(DIR_OUT)
        before = threads()
        dg, _, vals = graph(c, 1000, 131_071, 2)  # 1 MiB less 8 bytes
        assert np.array_equal(dg.adjacency(DIR_OUT)[1], vals.astype(np.uint32))
        assert threads() == before
        dg, _, vals = graph(c, 1000, 131_072, 3)
        assert np.array_equal(dg.adjacency(DIR_OUT)[1], vals.astype(np.uint32))
        assert before < threads() <= before + 7
    finally:
        c.close()
