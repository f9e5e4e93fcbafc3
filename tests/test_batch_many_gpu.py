"""A union batch of thousands of tiny graphs: its per-instance arrays are larger
than the host staging area starts out, so that it wraps and grows.  Sampled
instances equal their single runs."""
import numpy as np
import pytest

from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [700, 9000])
def test_batch_of_thousands(gpu_ctx, count):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    distinct = [C.DeviceGraph.from_csr(graphs.random_graph(20 + 3 * k, 4, seed=k), "Mod") for k in range(12)]
    gs = [distinct[k % 12] for k in range(count)]
    print(f"batch of {count} graphs", flush=True)
    res = C.cluster_batch(gs, "louvain", "Mod", 1.0, 0, seeds=[0] * count)
    single = [C.cluster(g, "louvain", "Mod", 1.0, 0, seed=0) for g in distinct]
    for k in range(count):
        q, p, info = res[k]
        q1, p1, i1 = single[k % 12]
        assert q == q1 and info == i1, k
    for k in range(0, count, 97):
        assert np.array_equal(res[k][1].cpu().numpy(), single[k % 12][1].cpu().numpy()), k
