"""The round's tail at the edges of its chunks of 1,024 vertices: cumulative
visit counts (counted straight into the context's array) equal to the
corpora's, and the relative entropy the oracle's double, over two rounds; a
round that fails adds nothing."""

import numpy as np
import pytest

import dgoracle
import distger
from distger import ffi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v", [5, 1023, 1024, 1025, 2048, 5000])
def test_entropy_chunks_and_counts(ctx, v):
    rng = np.random.default_rng(v)
    edges = np.zeros(3 * v, ffi.EDGE_DTYPE)
    edges["src"] = np.tile(np.arange(v), 3)
    edges["dst"] = (edges["src"] + np.repeat(rng.choice(np.arange(1, v), 3, replace=False), v)) % v
    ctx.graph_from_edges(v, edges, undirected=True, cn_mode=ffi.DG_CN_COMPUTE)
    g = dgoracle.OracleGraph.from_csr(*ctx.graph_csr())
    p = ctx.default_walk_params(seed=v, max_length=30)
    ctx.walk_reset()
    freq = np.zeros(v, np.uint64)
    for rnd, n in ((1, 5 * v), (2, v)):
        print(f"[walk-entropy] V={v} round {rnd}", flush=True)
        st = ctx.walk_round(p, rnd, 0, n)
        freq += np.bincount(ctx.corpus()[0], minlength=v).astype(np.uint64)
        assert np.array_equal(ctx.vertex_freq(), freq)
        assert (st.re, 0) == g.relative_entropy(freq.astype(np.uint32))
    low = ctx.default_walk_params(seed=v, mu=1e-9, length_limit=40)  # walks that do not end
    with pytest.raises(distger.DgError) as e:
        ctx.walk_round(low, 3, 0, v)
    assert e.value.code == ffi.DG_ERR_WALK_TOO_LONG
    assert np.array_equal(ctx.vertex_freq(), freq)
