"""Device relabelling by degree (gg_relabel_by_degree) against the host
restatement of BuilderBase::RelabelByDegree (src/builder.h:367-402): the
offsets and destinations must be byte-identical, on graphs whose rows
exercise every sort tier (<= 32 entries: one thread; <= 2048: a wavefront
in registers; longer: the (row, value) radix sort) and multi-tile radix
passes; and TC on the device-relabelled graph must give the reference's
count (its Hybrid path)."""

import numpy as np
import pytest

from conftest import cached_graph
from gapbs_amd import gpu
from gapbs_amd.graph import Graph

pytestmark = pytest.mark.gpu


def check(g):
    dg = gpu.DeviceGraph(g)
    dr, st = gpu.relabel_by_degree(dg)
    off, dst = dr.copy_out()
    h = g.relabel_by_degree()
    assert np.array_equal(off, h.out_offsets)
    assert np.array_equal(dst, h.out_neighbors)
    assert st["device_ms"] > 0
    return dr, h


@pytest.mark.parametrize("tag,make", [("g10", lambda: Graph.kronecker(10)),
                                      ("g16", lambda: Graph.kronecker(16)),
                                      ("u12", lambda: Graph.uniform(12)),
                                      ("k18s", lambda: Graph.kronecker(18, seed=8675309))])
def test_relabel_matches_host(golden, tag, make):
    print(f"[relabel] {tag}", flush=True)
    g = cached_graph(tag, make)
    dr, _ = check(g)
    if tag in golden["tc"]:
        assert gpu.OrderedCount(dr) == golden["tc"][tag]["triangles"]
        assert gpu.Hybrid(g) == golden["tc"][tag]["triangles"]


def test_relabel_hubs_and_ties():
    # Two hubs above 2048 entries, many equal degrees (ties go to the larger
    # old id first), isolated vertices and a 3000-vertex path.
    print("[relabel] hubs / ties", flush=True)
    a = np.zeros(9000, np.int32)
    b = np.full(3000, 1, np.int32)
    p = np.arange(20000, 22999)
    u = np.concatenate([a, b, [0], p])
    v = np.concatenate([np.arange(2, 9002), np.arange(9002, 12002), [1], p + 1])
    check(Graph.from_edges(u, v))


def test_relabel_scale_20():
    print("[relabel] kronecker s20", flush=True)
    check(Graph.kronecker(20, seed=3))


def test_relabel_rejects_directed_and_weighted():
    g = Graph.from_edges([0, 1], [1, 2], symmetrize=False)
    with pytest.raises(gpu.GpuError) as e:
        gpu.relabel_by_degree(gpu.DeviceGraph(g))
    assert e.value.code == -95
    with pytest.raises(gpu.GpuError) as e:
        gpu.relabel_by_degree(gpu.DeviceGraph(Graph.kronecker(8, weighted=True)))
    assert e.value.code == -95


def test_relabel_row_lengths():
    # Rows at and around every row-sorting tier's limit.
    print("[relabel] row lengths", flush=True)
    rng = np.random.default_rng(4)
    lens = [31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1024, 2047, 2048, 2049, 3000]
    hubs = np.arange(len(lens))
    u = np.repeat(hubs, lens)
    v = np.concatenate([rng.choice(np.arange(len(lens), 20000), d, replace=False) for d in lens])
    check(Graph.from_edges(u, v))


@pytest.mark.parametrize("n", [1, 2, 64, 65, 1024, 4095, 4096, 4097, 8193, 12289])
def test_relabel_sort_tiles(n):
    # One vertex to several 4096-key tiles, whole and ragged, with many equal
    # degrees and, from 2048 vertices, degrees of more than one digit.
    print(f"[relabel] {n} vertices", flush=True)
    i = np.arange(1, n, dtype=np.int32)
    hubs = i[: n // 2] if n > 2048 else i[:0]
    u = np.concatenate([i - 1, np.zeros(len(hubs), np.int32), [0] * (n == 1)]).astype(np.int32)
    v = np.concatenate([i, hubs, [0] * (n == 1)]).astype(np.int32)
    check(Graph.from_edges(u, v))


@pytest.mark.parametrize("mids", [120, 140])
def test_dense_graph_lists(mids):
    # 2000 vertices of about 126 and 146 entries on average, below and above
    # the density from which lists of 256 entries are spread over the grid in
    # relabelling and Shiloach-Vishkin (the sampled components leave them whole).
    print(f"[relabel] dense, {mids}", flush=True)
    rng = np.random.default_rng(mids)
    n = 2000
    deg = np.full(n, mids // 2)
    deg[:7] = [255, 256, 257, 511, 1023, 1024, 1500]
    u = np.repeat(np.arange(n), deg)
    v = np.concatenate([rng.choice(np.delete(np.arange(n), i), d, replace=False) for i, d in enumerate(deg)])
    g = Graph.from_edges(u, v)
    check(g)
    for rounds in (0, 2):
        assert np.array_equal(gpu.cc(gpu.DeviceGraph(g), rounds).comp, np.zeros(n, np.int32))
    assert np.array_equal(gpu.cc_sv(gpu.DeviceGraph(g)).comp, np.zeros(n, np.int32))
