"""A graph built where the device build and its working memory (54 bytes an
entry) do not fit and the host build (32 bytes an entry) does: the same graph.
Where neither fits the call fails and leaves no graph, and one that fits can be
built afterwards.  The device is filled with another library's buffers first."""

import numpy as np
import pytest
import torch

import distger
from distger import ffi

pytestmark = pytest.mark.gpu

MB = 1 << 20
V = 4_000_000
M = 4 * V  # each vertex to the next two, both ways


def fill(held, left):
    for size in (8192 * MB, 512 * MB, 64 * MB, 16 * MB):
        while torch.cuda.mem_get_info()[0] > left + size:
            held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
    print(f"[graph-no-room] {torch.cuda.mem_get_info()[0] // MB} MB left", flush=True)


def state(c):
    return [x.tobytes() for x in c.graph_csr()] + [c.graph_thresholds().tobytes()]


def test_graph_without_room():
    host_build, device_build = 32 * M + 14 * V, 54 * M + 14 * V
    left = (host_build + device_build) // 2 + 64 * MB
    assert host_build + 96 * MB < left < device_build
    edges = np.zeros(2 * V, distger.EDGE_DTYPE)
    ids = np.arange(V, dtype=np.uint32)
    edges["src"][:V] = edges["src"][V:] = ids
    edges["dst"][:V], edges["dst"][V:] = (ids + 1) % V, (ids + 2) % V
    with distger.Context(0) as c:
        c.graph_from_edges(V, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
        want = state(c)
        c.graph_from_edges(2, edges[:1], undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
        held = []
        try:
            fill(held, left)
            c.graph_from_edges(V, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
            # read back where there is room for what reading needs
            held.clear()
            torch.cuda.empty_cache()
            assert state(c) == want
            c.graph_from_edges(2, edges[:1], undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
            fill(held, host_build // 2)
            with pytest.raises(distger.DgError) as e:
                c.graph_from_edges(V, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
            assert e.value.code == -3  # DG_ERR_NOMEM
            for use in (c.graph_csr, lambda: c.walk_round(c.default_walk_params(V), 1, 0, 10)):
                with pytest.raises(distger.DgError):
                    use()
        finally:
            held.clear()
            torch.cuda.empty_cache()
        c.graph_from_edges(V, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
        assert state(c) == want
