"""GPU triangle counting parity: gg_tc counts must equal the reference's
exactly, on the graph as built and relabelled by degree (the reference's
Hybrid path), including hubs above the chunk threshold."""

import math

import numpy as np
import pytest

from conftest import cached_graph
from gapbs_amd import gpu
from gapbs_amd.graph import Graph
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tag,make", [("g10", lambda: Graph.kronecker(10)),
                                      ("g16", lambda: Graph.kronecker(16)),
                                      ("u12", lambda: Graph.uniform(12)),
                                      ("k18s", lambda: Graph.kronecker(18, seed=8675309))])
def test_tc_exact(golden, tag, make):
    print(f"[tc] {tag}", flush=True)
    g = cached_graph(tag, make)
    want = golden["tc"][tag]["triangles"] if tag in golden["tc"] else oracle.ordered_count(g)[0]
    assert gpu.OrderedCount(gpu.DeviceGraph(g)) == want
    assert gpu.OrderedCount(gpu.DeviceGraph(g.relabel_by_degree())) == want
    assert gpu.Hybrid(g) == want


def test_tc_closed_forms():
    print("[tc] closed forms", flush=True)
    iu, iv = np.triu_indices(300, 1)
    assert gpu.OrderedCount(gpu.DeviceGraph(Graph.from_edges(iu, iv))) == math.comb(300, 3)
    n = 6000  # wheel: hub n has n forward edges (> 4096-edge chunks)
    u = np.concatenate([np.arange(n), np.arange(n)])
    v = np.concatenate([(np.arange(n) + 1) % n, np.full(n, n)])
    assert gpu.OrderedCount(gpu.DeviceGraph(Graph.from_edges(u, v))) == n


def test_tc_rejects_directed():
    g = Graph.from_edges([0, 1], [1, 2], symmetrize=False)
    with pytest.raises(gpu.GpuError) as e:
        gpu.tc(gpu.DeviceGraph(g))
    assert e.value.code == -95


@pytest.mark.parametrize("lo", [98304 - 40, 98304, 131072 - 20, 262144])
def test_tc_high_ids(lo):
    # Long lists of ids that are all 2^16 or above (hash tables): a clique on
    # [lo, lo + 80), and 40 vertices 32768 higher, each joined to the clique's
    # upper half and to a neighbour.
    print(f"[tc] ids from {lo}", flush=True)
    iu, iv = np.triu_indices(80, 1)
    far = np.arange(40) + lo + 32768
    u = np.concatenate([iu + lo, np.repeat(far, 40), far[:-1]])
    v = np.concatenate([iv + lo, np.tile(np.arange(40, 80) + lo, 40), far[1:]])
    g = Graph.from_edges(u, v)
    # clique; far vertex + clique pair; far pair + clique vertex
    want = math.comb(80, 3) + 40 * math.comb(40, 2) + 39 * 40
    assert oracle.ordered_count(g)[0] == want
    assert gpu.OrderedCount(gpu.DeviceGraph(g)) == want


def _kernels_of(dg):
    dg.profile(True)
    gpu.tc(dg)
    return dg.profile_report()


@pytest.mark.parametrize("bits", [False, True])
@pytest.mark.parametrize("seed", range(4))
def test_tc_across_16_bit_ids(seed, bits):
    # Random pairs among ids on both sides of 2^16, where 16-bit ids end and
    # shared bits begin, and 32768 and 65536 higher, where the same shared bits
    # come again: lists with 0, 1 and more packed ids at even and odd places,
    # and probes that hit a bit set by another id.  Without and with a bipartite
    # filler of low ids, which decides whether the long lists are counted in
    # hash tables or bits.
    print(f"[tc] ids around 2^16, seed {seed}, bits {bits}", flush=True)
    rng = np.random.default_rng(seed)
    low = rng.choice(200, size=seed * seed * 4, replace=False)
    ids = np.concatenate([low, np.arange(65536 - 40 * (seed > 0), 65536 + 90), np.arange(98304 - 3, 98304 + 90),
                          np.arange(131072 - 60, 131072 + 60)])
    iu, iv = np.triu_indices(len(ids), 1)
    kept = rng.random(len(iu)) < 0.5
    u, v = ids[iu[kept]], ids[iv[kept]]
    if bits:
        u = np.concatenate([u, np.repeat(np.arange(1000, 1400), 600)])
        v = np.concatenate([v, np.tile(np.arange(2000, 2600), 400)])
    g = Graph.from_edges(u, v)
    dg = gpu.DeviceGraph(g)
    assert gpu.OrderedCount(dg) == oracle.ordered_count(g)[0]
    assert ("tc_narrow" in _kernels_of(dg)) == bits


@pytest.mark.parametrize("d", [2047, 2048, 2049, 4097])
def test_tc_hash_slices(d):
    # A wheel above 2^16 whose hub's list fills one table, one more or less,
    # and begins a third.
    print(f"[tc] hub of {d}", flush=True)
    rim = np.arange(d) + 70000
    g = Graph.from_edges(np.concatenate([rim, np.full(d, 90000)]), np.concatenate([np.roll(rim, 1), rim]))
    dg = gpu.DeviceGraph(g)
    assert gpu.OrderedCount(dg) == d
    assert "tc_narrow" not in _kernels_of(dg)
