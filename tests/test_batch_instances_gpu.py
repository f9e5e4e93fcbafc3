"""Per-instance sums of a union batch with more instances than a 256-thread
block has threads, and instances that start inside a block."""
import numpy as np
import pytest

from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[2] * 600, [1, 3, 255, 2, 256, 1, 257, 5, 64] * 5])
def test_union_batch_of_tiny_instances(gpu_ctx, sizes):
    from oracle import oracle as O
    from pennsylvaniagpugraphclustering_amd import clustering as C
    hs = [graphs.random_graph(n, 4, seed=k) if n > 2 else
          graphs.from_edges(n, np.arange(n - 1), np.arange(1, n)) for k, n in enumerate(sizes)]
    print(f"union batch of {len(hs)} tiny graphs", flush=True)
    res = C.cluster_batch([C.DeviceGraph.from_csr(h, "CPM") for h in hs], "louvain", "CPM", 0.5, 0)
    for k, (h, (q, p, info)) in enumerate(zip(hs, res)):
        oq, op, oi = O.cluster(h.rp, h.col, None, h.vertex_weights("CPM"), "CPM", 0.5, "louvain", 0, seed=0)
        assert np.array_equal(p.cpu().numpy(), op), k
        assert q == oq and info["moves"] == oi["moves"] and info["sweeps"] == oi["sweeps"], k
