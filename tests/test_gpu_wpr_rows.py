"""Weighted PageRank sweeps at the edges of the sweep items: rows of 0, 1, 8,
32, 33, 255..257, 511..513, 767..769 and thousands of entries, over the
vertices' own numbers and, on both sides of the limits from which on it is
taken, over rows and columns by degree with the LDS table, against FP64."""
import time

import numpy as np
import pytest
import torch

from conftest import gpu_case
from llama_amd.autograd import weighted_pagerank
from llama_amd.graph import SlcsrGraph, csr_of

pytestmark = pytest.mark.gpu

DEGS = [0, 1, 7, 8, 9, 31, 32, 33, 64, 255, 256, 257, 511, 512, 513, 767, 768, 769, 1535, 1537, 9000]
D, K = 0.85, 12
# each sweep rounds the products, the sum and the result to FP32 (3 * 2^-24
# relative, every term positive), and the errors of earlier sweeps are damped
# by D per sweep: 3 * 2^-24 / (1 - D) = 1.2e-6; twice that allowed
TOL = 2.4e-6


def check(ctx, V, extra_src, extra_dst):
    rng = np.random.default_rng(V)
    src, dst = [extra_src], [extra_dst]
    for i, d in enumerate(DEGS * 3):
        if V < 2 or d >= 4 * V:
            continue
        v = int(rng.integers(0, V))
        other = rng.integers(0, V, d)
        (src if i % 2 else dst).append(np.full(d, v))
        (dst if i % 2 else src).append(other)
    src, dst = np.concatenate(src), np.concatenate(dst)
    ofs, adj = csr_of(V, src, dst)
    tail = np.repeat(np.arange(V), np.diff(ofs))
    E = adj.size
    dg = SlcsrGraph(ctx, V, (ofs, adj), csr_of(V, dst, src))
    outdeg = np.maximum(np.diff(ofs), 1)
    w = (rng.random(E) / outdeg[tail]).astype(np.float32)
    p = (rng.random(V) / V).astype(np.float32)
    grad = rng.random(V).astype(np.float32)
    wt = torch.tensor(w, device="cuda", requires_grad=True)
    pt = torch.tensor(p, device="cuda", requires_grad=True)
    r = weighted_pagerank(wt, pt, dg, K, D)
    r.backward(torch.tensor(grad, device="cuda"))
    w64, x, lam = w.astype(np.float64), p.astype(np.float64), grad.astype(np.float64)
    for _ in range(K):
        x = (1 - D) * p + D * np.bincount(adj, w64 * x[tail], V)
        lam = grad + D * np.bincount(tail, w64 * lam[adj], V)
    assert np.all(np.abs(r.detach().cpu().numpy() - x) <= TOL * x)
    assert np.all(np.abs(pt.grad.cpu().numpy() - (1 - D) * lam) <= TOL * lam)
    ref = D * x[tail] * lam[adj]
    assert np.all(np.abs(wt.grad.cpu().numpy() - ref) <= 2 * TOL * ref + 1e-30)
    again = weighted_pagerank(wt, pt, dg, K, D)
    assert torch.equal(again, r)  # the sums do not depend on the schedule


@pytest.mark.parametrize("V", [1, 70, 4001, 24576, 24577, 90001])
def test_rows_of_every_length(ctx, V):
    gpu_case(f"wpr rows V={V}")
    rng = np.random.default_rng(V)
    check(ctx, V, rng.integers(0, V, 3 * V), rng.integers(0, V, 3 * V))


# vertices, edges per vertex, power: the hottest 24576 columns hold 0.49 of the
# entries with power 3.4, 0.094 with 1; the table is taken in the second, third
# and last case
@pytest.mark.parametrize("V,per,power", [(262_143, 5, 3.4), (262_144, 5, 3.4), (262_145, 4, 3.4),
                                         (262_144, 3, 3.4), (262_144, 5, 1), (400_001, 6, 5)])
def test_table_form(ctx, V, per, power):
    gpu_case(f"wpr table form V={V} per={per} power={power}")
    rng = np.random.default_rng(per)
    ids = rng.permutation(V)
    s, d = (ids[(V * rng.random(per * V) ** power).astype(np.int64)] for _ in range(2))
    check(ctx, V, s, d)


@pytest.mark.parametrize("V", [24576, 24577, 262_143, 262_144])
def test_out_edges_alone(ctx, V):
    """A single-level CSR without its in-edges gives the same forward and
    adjoint, bit for bit; the last by degree, which it counts over the heads."""
    gpu_case(f"wpr out-edges alone V={V}")
    rng = np.random.default_rng(V)
    src = rng.integers(0, V, 6 * V)
    dst = (V * rng.random(6 * V) ** 3).astype(np.int64)
    w = (rng.random(src.size) / 8).astype(np.float32)
    p = (rng.random(V) / V).astype(np.float32)
    got = []
    for in_csr in (csr_of(V, dst, src), None):
        dg = SlcsrGraph(ctx, V, csr_of(V, src, dst), in_csr)
        wt = torch.tensor(w, device="cuda", requires_grad=True)
        pt = torch.tensor(p, device="cuda", requires_grad=True)
        r = weighted_pagerank(wt, pt, dg, K, D)
        r.backward(torch.ones(V, device="cuda"))
        got.append((r.detach(), wt.grad, pt.grad))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("V,n,m", [(1 << 22, 2000, 20_000), (1 << 20, 30_000, 2_200_000)])
def test_isolated_vertices_cost_little(ctx, V, n, m):
    """A few connected vertices among a million or four of isolated ones, by
    their own numbers and by degree, where the isolated ones come in one run:
    the first call on the snapshot writes 8 to 34 MB of row offsets per
    direction (10 us at the copy rate) and sorts 4.4 M entries at most (0.2 ms);
    20 ms are many times what it needs."""
    rng = np.random.default_rng(3)
    ids = rng.permutation(V)[:n]
    src, dst = ids[rng.integers(0, n, m)], ids[rng.integers(0, n, m)]
    src, dst = np.concatenate([src, dst]), np.concatenate([dst, src])
    ofs, adj = csr_of(V, src, dst)
    tail = np.repeat(np.arange(V), np.diff(ofs))
    dg = SlcsrGraph(ctx, V, (ofs, adj), csr_of(V, dst, src))
    w = (rng.random(adj.size) / 30).astype(np.float32)
    p = np.ones(V, np.float32)
    wt = torch.tensor(w, device="cuda", requires_grad=True)
    pt = torch.tensor(p, device="cuda", requires_grad=True)
    grad = torch.ones(V, device="cuda")
    gpu_case("wpr, isolated vertices")
    best = 1e9
    for _ in range(3):
        dg.drop_snapshots()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        r = weighted_pagerank(wt, pt, dg, K, D)
        r.backward(grad)
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t0)
    w64, x = w.astype(np.float64), p.astype(np.float64)
    for _ in range(K):
        x = (1 - D) * p + D * np.bincount(adj, w64 * x[tail], V)
    assert np.all(np.abs(r.detach().cpu().numpy() - x) <= TOL * x)
    assert best < 0.02, best
