"""Whole runs on graphs whose vertex counts sit on the edges of the 2,048-item
tiles and 64-lane runs of the ordered selections and of the level plans,
bit-identical to the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 4095, 4097])
@pytest.mark.parametrize("algo,objective,mult", [("louvain", "Mod", 1.0), ("leiden+", "CPM", 0.4),
                                                 ("leiden", "WMod", 20.0)])
def test_runs_at_tile_edges(gpu_ctx, n, algo, objective, mult):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    if n < 3:
        g = graphs.from_edges(n, np.arange(n - 1), np.arange(1, n), np.ones(n - 1, np.int64))
    else:
        g = graphs.random_graph(n, 9, seed=n, weights=(1, 30))
    w = g.w if objective == "WMod" else None
    if g.nnz == 0 and objective != "CPM":
        return  # modularity of a graph without edges has no value
    print(f"n={n} {algo} {objective}", flush=True)
    q, part, info = C.cluster(C.DeviceGraph.from_csr(g, objective), algo, objective, mult, 1, seed=2)
    oq, op, oi = O.cluster(g.rp, g.col, w, g.vertex_weights(objective), objective, mult, algo, 1, seed=2)
    assert np.array_equal(part.cpu().numpy(), op)
    assert q == oq
    for key in ["labels", "uncut", "levels", "sweeps", "moves", "outer"]:
        assert info[key] == oi[key], key
