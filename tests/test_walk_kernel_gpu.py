"""The walk and packing kernels at the edges of their layout, against the CPU
oracle (corpus and visit counts): rounds of fewer walks than a wavefront up to more than the resident lanes (the
queue's shards), walks around the 24 vertices a lane holds and the 32
tabulated lengths, rows whose degree does not fit an adjacency unit, and
vertices a walk cannot leave."""

import numpy as np
import pytest

import dgoracle
from distger import ffi

pytestmark = pytest.mark.gpu


def _compare(ctx, p, rnd, begin, n, threads=8):
    st = None
    try:
        st = ctx.walk_round(p, rnd, begin, n)
    except Exception as e:  # unvisited vertices: the round itself is complete
        assert getattr(e, "code", 0) == ffi.DG_ERR_RE_UNDEFINED, e
    g = dgoracle.OracleGraph.from_csr(*ctx.graph_csr())
    tok, off = g.walk_round(g.cfg(p.seed, p.min_length, p.max_length, p.mu), rnd, begin, n, threads=threads)
    dtok, doff = ctx.corpus()
    assert np.array_equal(doff, off)
    assert np.array_equal(dtok, tok)
    assert np.array_equal(ctx.vertex_freq(), np.bincount(tok, minlength=g.v_num))  # after a reset
    if st is not None:
        assert st.tokens == len(tok) and st.max_walk_len == int(np.diff(off).max())
    return tok, off


@pytest.mark.parametrize("n", [1, 65, 255, 257, 256 * 63 + 1, 256 * 64, 256 * 65 + 7, 300001])
def test_walkers_over_the_shards(ctx, c1_edges, n):
    print(f"[walk-kernel] {n} walks", flush=True)
    ctx.graph_from_edges(10000, c1_edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
    ctx.walk_reset()
    _compare(ctx, ctx.default_walk_params(seed=n), 1, 17, n)


@pytest.mark.parametrize("cap", [1, 2, 23, 24, 25, 31, 32, 33, 34, 70])
def test_walk_lengths(ctx, c1_edges, cap):
    print(f"[walk-kernel] walks of {cap} vertices", flush=True)
    ctx.graph_from_edges(10000, c1_edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
    ctx.walk_reset()
    # mu so low that most walks end at the cap
    _, off = _compare(ctx, ctx.default_walk_params(seed=cap, min_length=3, max_length=cap, mu=1e-6), 1, 0, 10000)
    assert np.diff(off).max() == cap


@pytest.mark.parametrize("leaves", [2 ** 23 - 2, 2 ** 23 - 1, 2 ** 23])
def test_degrees_past_the_packed_field(ctx, leaves):
    print(f"[walk-kernel] star of {leaves} leaves", flush=True)
    edges = np.zeros(leaves, ffi.EDGE_DTYPE)
    edges["dst"] = np.arange(1, leaves + 1)
    ctx.graph_from_edges(leaves + 1, edges, undirected=True, cn_mode=ffi.DG_CN_FROM_DATA)
    ctx.walk_reset()
    _compare(ctx, ctx.default_walk_params(seed=5, max_length=30), 1, 0, 2000)


def test_vertices_a_walk_cannot_leave(ctx):
    # directed rows: 0 -> {1, 2, 3}, 1 -> {1, 2} (stuck), 2 -> {} (no row), 3 -> {0, 3} (not first: not stuck)
    pairs = [(0, 1), (0, 2), (0, 3), (1, 1), (1, 2), (3, 0), (3, 3)]
    edges = np.zeros(len(pairs), ffi.EDGE_DTYPE)
    edges["src"], edges["dst"] = np.array(pairs).T
    ctx.graph_from_edges(4, edges, undirected=False, cn_mode=ffi.DG_CN_FROM_DATA)
    ctx.walk_reset()
    tok, off = _compare(ctx, ctx.default_walk_params(seed=9, min_length=5, max_length=50), 1, 0, 4000)
    assert len(np.unique(np.diff(off))) > 3


@pytest.mark.parametrize("v,n", [(15, 100), (2047, 262143), (2049, 262145), (40000, 300000), (2 ** 22, 3000),
                                 (2 ** 22 + 1, 3000)])
def test_counts_by_bins(ctx, v, n):
    """Bins of few and of the most counters, the first graph past them, and both tile sizes."""
    print(f"[walk-kernel] counts of {n} walks on {v} vertices", flush=True)
    edges = np.zeros(2 * v, ffi.EDGE_DTYPE)
    edges["src"] = np.tile(np.arange(v), 2)
    edges["dst"] = (edges["src"].astype(np.int64) + np.repeat([1, 5], v)) % v
    ctx.graph_from_edges(v, edges, undirected=True, cn_mode=ffi.DG_CN_FROM_DATA)
    ctx.walk_reset()
    _compare(ctx, ctx.default_walk_params(seed=v, max_length=40, mu=0.99, min_length=8), 1, v // 2, n)
