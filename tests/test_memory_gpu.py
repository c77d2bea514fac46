"""Device memory of a call: buffers that only make a call faster are left out
where they do not fit (GAPGPU_MEM_CAP_BYTES stands for a full card), with the
same results, and make room for another call's buffers."""

import numpy as np
import pytest

from gapbs_amd import gpu
from gapbs_amd.graph import Graph

pytestmark = pytest.mark.gpu
MB = 1 << 20
ROOTS = [3, 5, 9, 11, 12, 13, 14, 15, 16]


def _fits(monkeypatch, call, mb):
    monkeypatch.setenv("GAPGPU_MEM_CAP_BYTES", str(mb * MB))
    try:
        return True, call()
    except gpu.GpuError as e:
        assert e.code == -12
        return False, None
    finally:
        monkeypatch.delenv("GAPGPU_MEM_CAP_BYTES")


def _least(monkeypatch, call, taken):
    for mb in range(taken, taken + 1024):
        ok, result = _fits(monkeypatch, call, mb)
        if ok:
            return mb, result
    raise AssertionError("does not fit")


def _allocated(monkeypatch):
    """The MB already taken (other handles' too), rounded up: the least at
    which two offsets more fit."""
    two = Graph.from_edges([0], [1])
    low, high = 0, 1 << 19  # does not fit, fits
    while high - low > 1:
        mid = (low + high) // 2
        if _fits(monkeypatch, lambda: gpu.DeviceGraph(two).free(), mid)[0]:
            high = mid
        else:
            low = mid
    return high


# What a call needed with no optional buffer, in MB beside the graph
# (Kronecker 18; every buffer is rounded up to 1 MB).
@pytest.mark.parametrize("name,need,call", [
    ("bc", 29, lambda g: gpu.bc(g, ROOTS[:2]).scores),
    ("bc fp64", 30, lambda g: gpu.bc(g, ROOTS[:2], fp64=True).scores),
    ("bc kahan", 29, lambda g: gpu.bc(g, ROOTS[:2], kahan=True).scores),
    ("tc", 7, lambda g: np.array([gpu.tc(g)[0]])),
    ("bfs batch", 54, lambda g: gpu.bfs_batch(g, ROOTS).depths),
])
def test_call_fits_without_optional_buffers(monkeypatch, name, need, call):
    print(f"[memory] {name}", flush=True)
    g, _ = gpu.generate_graph(0, 18, 16)
    if name == "tc":  # low ids, so with the optional 16-bit lists
        g, _ = gpu.relabel_by_degree(g)
    want = call(g)
    g.free()
    g, _ = gpu.generate_graph(0, 18, 16)
    if name == "tc":
        g, _ = gpu.relabel_by_degree(g)
    taken = _allocated(monkeypatch)
    least, got = _least(monkeypatch, lambda: call(g), taken)
    assert np.array_equal(got, want)
    assert least - taken <= need
    assert np.array_equal(call(g), want)  # and with them again


def test_spare_buffers_make_room(monkeypatch):
    # Nine roots' depths are read out through 8 MB that the next call may
    # take: components need 6 MB on this graph.
    print("[memory] spare buffers", flush=True)
    g, _ = gpu.generate_graph(0, 18, 16)
    depths = gpu.bfs_batch(g, ROOTS).depths
    taken = _allocated(monkeypatch)
    ok, comp = _fits(monkeypatch, lambda: gpu.cc(g).comp, taken)
    assert ok and np.array_equal(comp, gpu.cc(g).comp)
    assert np.array_equal(gpu.bfs_batch(g, ROOTS).depths, depths)
