"""The CSR built on the device against the oracle's host build: the order of
every row, the counts (simple graphs, multigraphs, edge data, directed) and
the thresholds, at the edges of the sort's tiles (4,096 entries) and digits
(8 bits of the source), of the small rows (256 neighbours) and of the hot set
(4,096 vertices); a bad edge is refused and leaves the loaded graph."""

import numpy as np
import pytest

import dgoracle
import distger
from distger import ffi

pytestmark = pytest.mark.gpu


def _random_edges(v, e, seed, simple):
    rng = np.random.default_rng(seed)
    edges = np.zeros(e, ffi.EDGE_DTYPE)
    # a few hubs: half of the sources among the first vertices
    edges["src"] = np.where(rng.random(e) < 0.5, rng.integers(0, min(v, 3), e), rng.integers(0, v, e))
    edges["dst"] = rng.integers(0, v, e)
    if simple:
        lo, hi = np.minimum(edges["src"], edges["dst"]), np.maximum(edges["src"], edges["dst"])
        _, first = np.unique(lo.astype(np.uint64) << np.uint64(32) | hi, return_index=True)
        edges = edges[np.sort(first)]
        edges = edges[edges["src"] != edges["dst"]]
    edges["data"] = rng.integers(0, 50, len(edges))
    return edges


@pytest.mark.parametrize("v,e,simple,undirected,mode", [
    (2, 8, True, True, ffi.DG_CN_COMPUTE),
    (255, 2048, False, True, ffi.DG_CN_COMPUTE),
    (256, 2047, True, True, ffi.DG_CN_COMPUTE),
    (257, 2049, True, False, ffi.DG_CN_COMPUTE),
    (300, 4096, True, True, ffi.DG_CN_COMPUTE),
    (600, 4097, False, False, ffi.DG_CN_COMPUTE),
    (4096, 20000, True, True, ffi.DG_CN_COMPUTE),
    (4097, 20001, True, True, ffi.DG_CN_FROM_DATA),
    (65536, 60000, True, True, ffi.DG_CN_COMPUTE),
    (65537, 30000, False, True, ffi.DG_CN_FROM_DATA),
])
def test_device_build_matches_oracle(ctx, v, e, simple, undirected, mode):
    print(f"[graph-build] V={v} E={e} simple={simple} undirected={undirected} mode={mode}", flush=True)
    edges = _random_edges(v, e, v + e, simple)
    ctx.graph_from_edges(v, edges, undirected=undirected, cn_mode=mode)
    g = dgoracle.OracleGraph(v, edges, undirected=undirected, cn="data" if mode == ffi.DG_CN_FROM_DATA else None)
    rp, nbr, cn = ctx.graph_csr()
    assert np.array_equal(rp, g.row_ptr)
    assert np.array_equal(nbr, g.nbr[: g.m])
    assert np.array_equal(cn, g.cn[: g.m])
    # a threshold is the smallest 31-bit draw u with tanh(pa) <= u / (2^31 - 1)
    thr = ctx.graph_thresholds().astype(np.float64)
    deg = np.diff(rp.astype(np.int64)).astype(np.float64)
    du, dv = np.repeat(deg, deg.astype(np.int64)), deg[nbr]
    with np.errstate(divide="ignore", invalid="ignore"):
        pa = 1.0 / (du - cn) * np.maximum(du, dv) / np.minimum(du, dv)
        pn = np.tanh(pa)
    ok = np.isfinite(pn) & (pn > 0) & (pn < 1)
    M = 2.0 ** 31 - 1
    assert np.all(np.abs(thr[ok] - np.ceil(pn[ok] * M)) <= 1)  # numpy's tanh may differ in the last bit
    bad = edges.copy()
    bad["dst"][len(bad) // 2] = v
    with pytest.raises(distger.DgError) as err:
        ctx.graph_from_edges(v, bad, undirected=undirected, cn_mode=mode)
    assert err.value.code == ffi.DG_ERR_ARG and f"edge {len(bad) // 2} " in str(err.value)
    assert np.array_equal(ctx.graph_csr()[1], nbr)


@pytest.mark.parametrize("v", [4000, 4096, 4097, 9000])
def test_visit_counts_with_any_hot_set(ctx, v):
    """Rings with chords (every degree equal): no degree cut fits the hot slots."""
    edges = np.zeros(2 * v, ffi.EDGE_DTYPE)
    edges["src"] = np.tile(np.arange(v), 2)
    edges["dst"] = (edges["src"] + np.repeat([1, 7], v)) % v
    ctx.graph_from_edges(v, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
    ctx.walk_reset()
    ctx.walk_round(ctx.default_walk_params(seed=3, max_length=30), 1, 0, 2 * v)
    assert np.array_equal(ctx.vertex_freq(), np.bincount(ctx.corpus()[0], minlength=v))
