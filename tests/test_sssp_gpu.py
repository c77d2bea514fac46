"""GPU SSSP parity: gg_sssp (through the C-ABI) against the CPU oracle.

Distances must be bit-exact (shortest distances are unique), for every
bucket width delta, on Kronecker, uniform, lattice and directed graphs.
"""

import numpy as np
import pytest

from conftest import cached_graph
from gapbs_amd import gpu
from gapbs_amd.graph import Graph
from oracle import oracle

pytestmark = pytest.mark.gpu
INF = (2**31 - 1) // 2
_DG = {}


def dev(tag, make):
    if tag not in _DG:
        _DG[tag] = gpu.DeviceGraph(cached_graph(tag, make))
    return _DG[tag]


def grid_graph(side, seed=7):
    return Graph.grid(side, seed=seed)


@pytest.mark.parametrize("tag,make", [("g10w", lambda: Graph.kronecker(10, weighted=True)),
                                      ("g16w", lambda: Graph.kronecker(16, weighted=True)),
                                      ("u12w", lambda: Graph.uniform(12, weighted=True))])
def test_sssp_matches_golden_roots(golden, tag, make):
    print(f"[sssp] {tag}", flush=True)
    g = cached_graph(tag, make)
    dg = dev(tag, make)
    for rec in golden["sssp"][tag]:
        res = gpu.sssp(dg, rec["root"], 2)
        want = oracle.dijkstra(g, rec["root"])
        assert np.array_equal(res.dist, want), rec["root"]
        assert res.stats["reached"] == rec["reached"]


@pytest.mark.parametrize("delta", [1, 3, 16, 255, 4096, 1 << 29])
def test_sssp_delta_sweep_kronecker(delta):
    print(f"[sssp] delta {delta}", flush=True)
    g = cached_graph("k16s", lambda: Graph.kronecker(16, seed=8675309, weighted=True))
    dg = dev("k16s", lambda: Graph.kronecker(16, seed=8675309, weighted=True))
    for r in g.strip_weights().pick_sources(3):
        assert np.array_equal(gpu.sssp(dg, int(r), delta).dist, oracle.dijkstra(g, int(r)))


@pytest.mark.parametrize("delta", [1, 100, 1000, 5000])
def test_sssp_grid_with_shortcuts(delta):
    print(f"[sssp] grid delta {delta}", flush=True)
    g = cached_graph("grid96", lambda: grid_graph(96))
    dg = dev("grid96", lambda: grid_graph(96))
    for r in (0, 4000, 9215):
        assert np.array_equal(gpu.sssp(dg, r, delta).dist, oracle.dijkstra(g, r))


def test_sssp_directed_and_unreachable():
    print("[sssp] directed", flush=True)
    rng = np.random.default_rng(11)
    n, m = 4000, 30000
    g = Graph.from_edges(rng.integers(0, n, m), rng.integers(0, n, m),
                         w=rng.integers(1, 1000, m), symmetrize=False)
    dg = gpu.DeviceGraph(g)
    for src in (0, 5, 77):
        for delta in (1, 50, 2000):
            assert np.array_equal(gpu.sssp(dg, src, delta).dist, oracle.dijkstra(g, src))
    iso = Graph.from_edges([0, 2], [1, 3], w=[5, 6])
    res = gpu.sssp(gpu.DeviceGraph(iso), 0, 1)
    assert res.dist.tolist() == [0, 5, INF, INF]


def test_sssp_hub_chunks():
    print("[sssp] hubs", flush=True)
    rng = np.random.default_rng(2)
    a = np.zeros(9000, np.int32)
    u = np.concatenate([a, np.full(5000, 1, np.int32), [0]])
    v = np.concatenate([np.arange(2, 9002), np.arange(9002, 14002), [1]])
    g = Graph.from_edges(u, v, w=rng.integers(1, 255, len(u)))
    dg = gpu.DeviceGraph(g)
    for src in (0, 5, 13000):
        for delta in (1, 64):
            assert np.array_equal(gpu.sssp(dg, src, delta).dist, oracle.dijkstra(g, src))


def test_sssp_errors():
    dg = dev("g10w", lambda: Graph.kronecker(10, weighted=True))
    with pytest.raises(gpu.GpuError) as e:
        gpu.sssp(dg, 0, 0)
    assert e.value.code == -22
    with pytest.raises(gpu.GpuError) as e:
        gpu.sssp(dg, -1, 2)
    assert e.value.code == -22
    ug = gpu.DeviceGraph(Graph.kronecker(8))
    with pytest.raises(gpu.GpuError) as e:
        gpu.sssp(ug, 0, 2)
    assert e.value.code == -95


@pytest.mark.parametrize("delta", [1, 64, 1024])
def test_sssp_and_bfs_list_lengths(delta):
    # Frontier vertices whose lists end around a step, a slice and a chunk of
    # the tile expansion, with empty and one-entry lists between them.
    print(f"[sssp] list lengths, delta {delta}", flush=True)
    rng = np.random.default_rng(9)
    lens = [0, 1, 2, 255, 256, 257, 1023, 1024, 1025, 4095, 4096, 4097, 5121, 8192, 8193] + [1, 3, 0] * 300
    first = 1 + len(lens)
    n = first + 9000
    u = np.concatenate([np.zeros(len(lens), int), np.repeat(np.arange(1, first), lens)])
    v = np.concatenate([np.arange(1, first)] + [rng.choice(np.arange(first, n), d, replace=False) for d in lens])
    w = rng.integers(1, 256, len(u))
    g = Graph.from_edges(u, v, w, symmetrize=False)
    assert np.array_equal(gpu.sssp(gpu.DeviceGraph(g), 0, delta).dist, oracle.dijkstra(g, 0))
    plain = g.strip_weights()
    assert np.array_equal(gpu.bfs(gpu.DeviceGraph(plain), 0, alpha=1).depth, oracle.bfs_depth(plain, 0))


@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("delta", [1, 7, 8, 9, 100])
def test_sssp_light_and_heavy_edges(delta, ordered):
    # Weights at and around the width that parts light from heavy edges, and
    # hubs whose chunks hold both kinds.
    print(f"[sssp] weights around 8, delta {delta}, ordered {ordered}", flush=True)
    rng = np.random.default_rng(delta)
    n = 6000
    u = np.concatenate([rng.integers(0, n, 20000), np.zeros(5000, int), np.ones(300, int)])
    v = np.concatenate([rng.integers(0, n, 20000), rng.choice(np.arange(2, n), 5000, replace=False),
                        rng.choice(np.arange(2, n), 300, replace=False)])
    g = Graph.from_edges(u, v, rng.choice([1, 7, 8, 9, 60], len(u)))
    dg = gpu.DeviceGraph(g, order_by_degree=ordered)
    for r in (0, 1, 77):
        assert np.array_equal(gpu.sssp(dg, r, delta).dist, oracle.dijkstra(g, r))


@pytest.mark.parametrize("width", [1, 300, 4096, 4097])
def test_lists_of_small_and_large_frontiers(width):
    # Frontiers of up to 4096 vertices spread lists of 256 entries, larger ones
    # lists of 512: lists around both, of single and batched searches and paths.
    print(f"[sssp] frontier of {width}", flush=True)
    rng = np.random.default_rng(width)
    lens = np.array([255, 256, 257, 400, 511, 512, 513, 1024, 1025] * 4)[:width]
    mids = np.arange(1, 1 + width)
    first, n = 1 + width, 1 + width + 6000
    u = np.concatenate([np.zeros(width, int), np.repeat(mids[:len(lens)], lens)])
    v = np.concatenate([mids] + [rng.choice(np.arange(first, n), d, replace=False) for d in lens])
    g = Graph.from_edges(u, v, rng.integers(1, 256, len(u)), symmetrize=False)
    dg = gpu.DeviceGraph(g)
    want = oracle.dijkstra(g, 0)
    for delta in (1, 64, 1024):
        assert np.array_equal(gpu.sssp(dg, 0, delta).dist, want)
    plain = g.strip_weights()
    dp = gpu.DeviceGraph(plain)
    assert np.array_equal(gpu.bfs(dp, 0, alpha=1).depth, oracle.bfs_depth(plain, 0))
    assert np.array_equal(gpu.bfs_batch(dp, [0, 1], alpha=1).depths[0], oracle.bfs_depth(plain, 0))
