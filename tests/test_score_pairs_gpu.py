"""Pair scores against float64 at the edges of a wavefront's 16 pairs and of
the rows' 128-element steps, vertices without a rank, and bad ids."""

import numpy as np
import pytest

import distger
from distger import ffi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dim", [(1, 64), (3, 128), (15, 192), (16, 256), (17, 320), (63, 512), (1000, 128), (70001, 64)])
def test_scores(ctx, n, dim):
    print(f"[score] {n} pairs of dim {dim}", flush=True)
    rng = np.random.default_rng(n)
    rows = 701
    s0 = rng.normal(0, 0.3, (rows, dim)).astype(np.float32)
    ctx.sgns_tables_create(s0, np.zeros_like(s0))
    src, dst = (rng.integers(0, rows, n).astype(np.uint32) for _ in range(2))
    got = ctx.sgns_score_pairs(src, dst)
    x = s0.astype(np.float64)
    want = (x[src] * x[dst]).sum(1)
    # a dot of dim terms rounds at most dim times, each by 2^-24 of the sum of magnitudes
    bound = np.abs(x[src] * x[dst]).sum(1) * dim * 2.0 ** -24
    assert np.all(np.abs(got - want) <= bound)
    for k in {0, n // 2, n - 1}:
        bad = dst.copy()
        bad[k] = rows
        with pytest.raises(distger.DgError) as e:
            ctx.sgns_score_pairs(src, bad)
        assert e.value.code == ffi.DG_ERR_ARG and f"pair {k}:" in str(e.value)
    assert np.array_equal(ctx.sgns_score_pairs(src, dst), got)


def test_vertices_outside_the_vocabulary_score_zero(ctx):
    edges = np.zeros(4, ffi.EDGE_DTYPE)
    edges["src"], edges["dst"] = [0, 1, 2, 0], [1, 2, 0, 3]
    ctx.graph_from_edges(6, edges, undirected=True, cn_mode=ffi.DG_CN_FROM_DATA)
    sp = ctx.default_sgns_params(dim=64, table_size=1000, min_count=4)  # vertices 4, 5 have no edge, 3 one
    ctx.sgns_init(sp)
    got = ctx.sgns_score_pairs([0, 3, 4, 1], [1, 1, 5, 2])
    assert got[1] == 0.0 and got[2] == 0.0 and got[0] != 0.0 and got[3] != 0.0
