"""GPU Brandes parity: gg_bc against the oracles.

FP32 mode reproduces the reference's float arithmetic: bit-identical to the
float oracle when path counts are exact integers (always at these sizes),
hence the reference's BCVerifier rule (|diff| <= FLT_EPSILON) holds.  The
Kahan mode stays within 2e-6 max-abs of the FP64 oracle and at least as
close to it as the reference's float result; FP64 mode within 1e-6
relative of the FP64 oracle (the output is float).
"""

import numpy as np
import pytest

from conftest import cached_graph
from gapbs_amd import gpu
from gapbs_amd.graph import Graph
from oracle import oracle

pytestmark = pytest.mark.gpu
_DG = {}


def dev(tag, make):
    if tag not in _DG:
        _DG[tag] = gpu.DeviceGraph(cached_graph(tag, make))
    return _DG[tag]


GRAPHS = [("g10", lambda: Graph.kronecker(10), 4), ("g16", lambda: Graph.kronecker(16), 4),
          ("u12", lambda: Graph.uniform(12), 8), ("k18s", lambda: Graph.kronecker(18, seed=8675309), 4)]


@pytest.mark.parametrize("tag,make,k", GRAPHS)
def test_bc_fp32_and_fp64(tag, make, k):
    print(f"[bc] {tag}", flush=True)
    g = cached_graph(tag, make)
    dg = dev(tag, make)
    roots = g.pick_sources(k)
    want = oracle.brandes(g, roots, fp64=True)
    ref32 = oracle.brandes(g, roots)
    r32 = gpu.bc(dg, roots)
    assert np.array_equal(r32.scores, ref32)
    if g.num_nodes <= 70000:
        assert g.verify_bc(roots, r32.scores)
    rk = gpu.bc(dg, roots, kahan=True)
    e_k = np.abs(rk.scores.astype(np.float64) - want)
    assert e_k.max() < 2e-6
    assert e_k.sum() <= np.abs(ref32.astype(np.float64) - want).sum() * 1.01
    r64 = gpu.bc(dg, roots, fp64=True)
    nz = want > 1e-3
    assert (np.abs(r64.scores - want)[nz] / want[nz]).max() < 1e-6
    assert np.abs(r64.scores - want).max() < 1e-7


def test_bc_closed_forms():
    print("[bc] closed forms", flush=True)
    n = 400
    path = Graph.from_edges(np.arange(n - 1), np.arange(1, n))
    s = gpu.bc(gpu.DeviceGraph(path), [0], fp64=True).scores
    want = (n - 1 - np.arange(n)) / (n - 1)
    np.testing.assert_allclose(s, want, rtol=1e-6)
    m = 3000  # star with a hub above the chunk threshold
    star = Graph.from_edges(np.zeros(m - 1, np.int32), np.arange(1, m))
    roots = np.arange(0, m, 37)
    got = gpu.bc(gpu.DeviceGraph(star), roots).scores
    assert np.array_equal(got, oracle.brandes(star, roots))


def test_bc_repeated_root_and_disconnected():
    g = Graph.from_edges([0, 1, 2, 5, 6], [1, 2, 3, 6, 7])
    dg = gpu.DeviceGraph(g)
    roots = [0, 0, 5]
    assert np.array_equal(gpu.bc(dg, roots).scores, oracle.brandes(g, roots))
    with pytest.raises(gpu.GpuError):
        gpu.bc(dg, [g.num_nodes])


def test_bc_hub_folds():
    # Vertices with 16384+ successors fold on a block (terms in parallel,
    # folded in edge order): two such hubs sharing neighbours, a partial
    # last round, roots around them; FP32 bit-exact with the reference's
    # float arithmetic, Kahan and FP64 within the stated tolerances.
    print("[bc] hub folds", flush=True)
    rng = np.random.default_rng(23)
    n = 40000
    u, v = [], []
    for h, d in ((0, 30000), (1, 16384)):
        u.append(np.full(d, h))
        v.append(rng.choice(np.arange(2, n), size=d, replace=False))
    u.append(rng.integers(2, n, 50000))
    v.append(rng.integers(2, n, 50000))
    g = Graph.from_edges(np.concatenate(u), np.concatenate(v))
    dg = gpu.DeviceGraph(g)
    roots = np.array([0, 1, 7, 123, 4567, 30001], dtype=np.int32)
    assert np.array_equal(gpu.bc(dg, roots).scores, oracle.brandes(g, roots))
    want = oracle.brandes(g, roots, fp64=True)
    assert np.abs(gpu.bc(dg, roots, fp64=True).scores - want).max() < 1e-6
    assert np.abs(gpu.bc(dg, roots, kahan=True).scores - want).max() < 1e-5
    dg.profile(True)
    gpu.bc(dg, roots[:1])
    assert "bc_delta_hub" in dg.profile_report()


def test_bc_deep_graph_uses_level_by_level_discovery():
    # More levels than the depth buckets hold (4096): discovery falls back to
    # the top-down level loop; results as the reference's.
    print("[bc] path of 5000", flush=True)
    g = Graph.from_edges(np.arange(4999), np.arange(1, 5000))
    dg = gpu.DeviceGraph(g)
    roots = np.array([0, 2500, 4999], dtype=np.int32)
    assert np.array_equal(gpu.bc(dg, roots).scores, oracle.brandes(g, roots))


@pytest.mark.parametrize("leaves", [70, 2500, 9000])
def test_bc_folds_ties_and_binades(leaves):
    # One vertex whose total passes many powers of two through terms of 1
    # and 2 (its leaves, some with a child of their own) interleaved with
    # terms of exactly 2^-10, which fall on rounding ties once the total is
    # 2^13: the fold must round each as the reference's one-by-one sum does,
    # on the thread, wavefront and block paths.
    print(f"[bc] ties, {leaves} leaves", flush=True)
    mids, apex = 1024, 200
    ids = np.random.default_rng(leaves).permutation(np.arange(1 + mids, 1 + mids + leaves + apex))
    leaf, top = ids[:leaves], ids[leaves:]
    child = np.arange(leaves // 2) + ids.max() + 1
    u = np.concatenate([np.zeros(mids, int), np.ones(leaves, int), np.repeat(np.arange(1, 1 + mids), apex),
                        leaf[:leaves // 2]])
    v = np.concatenate([np.arange(1, 1 + mids), leaf, np.tile(top, mids), child])
    g = Graph.from_edges(u, v)
    roots = np.array([0, 2, int(leaf[0])], dtype=np.int32)
    want = oracle.brandes(g, roots)
    dg = gpu.DeviceGraph(g)
    assert np.array_equal(gpu.bc(dg, roots).scores, want)
    assert np.array_equal(gpu.bc_batch(dg, roots).scores, want)


@pytest.mark.parametrize("n", [2, 31, 32, 33, 34, 65, 4097])
def test_bc_level_bitmaps_and_depths(n):
    # Paths of as many levels as the level bitmaps hold, and one more or less
    # (deeper traversals test depths), with lists around a wavefront's length
    # hanging off the middle.
    print(f"[bc] path of {n}", flush=True)
    u, v = list(range(n - 1)), list(range(1, n))
    at = n
    for d in (63, 64, 65, 1023, 1024, 1025):
        u += [min(d % 7, n - 1)] * d
        v += list(range(at, at + d))
        at += d
    g = Graph.from_edges(np.array(u), np.array(v))
    roots = np.array([0, n - 1, at - 1], dtype=np.int32)
    for order in (False, True):
        dg = gpu.DeviceGraph(g, order_by_degree=order)
        if not order:
            assert np.array_equal(gpu.bc(dg, roots).scores, oracle.brandes(g, roots))
        assert np.abs(gpu.bc(dg, roots, fp64=True).scores - oracle.brandes(g, roots, fp64=True)).max() < 1e-7


@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("n", [255, 256, 257, 512, 3840])
def test_bc_as_many_levels_as_vertices(n, directed):
    # A bare path from its end, and a directed cycle: the search's steps are
    # one more than the vertices (the last finds nothing), so at a multiple of
    # the block size one level count more than there are threads per vertex is
    # to be cleared.  A freed handle's counts come before, whose memory the new
    # handle may be given.
    print(f"[bc] {n} vertices in a row, directed {directed}", flush=True)
    before = gpu.DeviceGraph(Graph.from_edges(np.arange(4000), np.arange(1, 4001)))
    gpu.bc(before, [0])
    before.free()
    u = np.arange(n if directed else n - 1)
    g = Graph.from_edges(u, (u + 1) % n, symmetrize=not directed)
    roots = np.array([0, n - 1], dtype=np.int32)
    assert np.array_equal(gpu.bc(gpu.DeviceGraph(g), roots).scores, oracle.brandes(g, roots))


@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("length", [12, 40, 4000, 4200])
def test_bc_levels_with_and_without_long_lists(length, directed):
    # A path on which a few levels hold vertices for the wavefront and hub
    # kernels and the others none: fans of 63 to 5000 leaves, and joins of 64
    # and 300 in-neighbours (directed: long in-lists beside short out-lists);
    # levels bucketed with bitmaps, with depths, and found one by one.
    print(f"[bc] path of {length} with fans, directed {directed}", flush=True)
    u, v = list(range(length - 1)), list(range(1, length))
    at = length
    for k, d in enumerate((63, 64, 300, 4095, 4096, 5000)):
        u += [length // 2 + k % 4] * d
        v += list(range(at, at + d))
        at += d
    for k, d in enumerate((64, 300)):  # path vertex -> d vertices -> one vertex -> a leaf
        mids = list(range(at, at + d))
        u += [3 + k] * d + mids + [at + d]
        v += mids + [at + d] * d + [at + d + 1]
        at += d + 2
    g = Graph.from_edges(np.array(u), np.array(v), symmetrize=not directed)
    dg = gpu.DeviceGraph(g)
    roots = np.array([0, length - 1, at - 1], dtype=np.int32)
    assert np.array_equal(gpu.bc(dg, roots).scores, oracle.brandes(g, roots))
    want = oracle.brandes(g, roots, fp64=True)
    assert np.abs(gpu.bc(dg, roots, fp64=True).scores - want).max() < 1e-7
    assert np.abs(gpu.bc(dg, roots, kahan=True).scores - want).max() < 2e-6


@pytest.mark.parametrize("width", [2047, 2049, 70000])
def test_bc_delta_lists(width):
    # Levels of one and several list tiles, and one above the size from which
    # the three dependency kernels take three streams; every 50th vertex of
    # the level has a list for the wavefront kernel, one for the hub kernel.
    print(f"[bc] level of {width}", flush=True)
    mid = np.arange(1, 1 + width)
    par = np.concatenate([np.repeat(mid[::50], 70), np.full(5000, mid[7])])
    leaf = np.arange(len(par)) + 1 + width
    g = Graph.from_edges(np.concatenate([np.zeros(width, int), par]), np.concatenate([mid, leaf]))
    roots = np.array([0, int(mid[3]), int(leaf[-1])], dtype=np.int32)
    assert np.array_equal(gpu.bc(gpu.DeviceGraph(g), roots).scores, oracle.brandes(g, roots))
