"""Hubs scored in chunks of 4,096 edges and slices of their clusters' hash
range: one sweep at the edges of the chunks and of the slices, with all their
neighbours in two clusters, in a few and in one each, with and without a
constraint, 32-bit and 64-bit sums, in one batch and in several, and hubs of more slices than a chunk has
buckets, bit-identical to the oracle; and scoring time that grows with the
degree, not with its square."""
import numpy as np
import pytest

from oracle import oracle as O
from pennsylvaniagpugraphclustering_amd import graphs

pytestmark = pytest.mark.gpu


def check_sweep(g, labels, L, constraint=None):
    from pennsylvaniagpugraphclustering_amd import clustering as C
    obj = "Mod" if g.w is None else "WMod"
    vw = g.vertex_weights(obj)
    part = labels.astype(np.int32)
    vol, _, _ = O.evaluate(g.rp, g.col, g.w, vw, part, L)
    dest = np.full(g.n, -1, np.int32)
    gain = np.zeros(g.n, np.float32)
    lam = 1.0 / float(vw.sum())
    mv, d2, g2, nc = C.sweep(C.DeviceGraph.from_csr(g, obj), part, vol, lam, 0.75, False, dest, gain, constraint)
    rmv, rd, rg, rnc = O.sweep(g.rp, g.col, g.w, vw, part, vol, lam, 0.75, False, dest, gain, constraint)
    assert nc == rnc
    assert np.array_equal(d2.cpu().numpy(), rd)
    assert np.array_equal(g2.cpu().numpy().view(np.int32), rg.view(np.int32))
    assert np.array_equal(mv.cpu().numpy(), rmv)


# chunks of 4,096 edges; slices of 8,192 edges with 32-bit sums, 5,461 with 64-bit ones
DEGREES = [8193, 10923, 12287, 12288, 12289, 16383, 16384, 16385, 20481, 65536, 98304, 98305]


@pytest.mark.parametrize("weights", [None, (1, 30), (1 << 29, (1 << 30) - 1)])
@pytest.mark.parametrize("labels", [2, 60, 0])
@pytest.mark.parametrize("constrained", [False, True])
@pytest.mark.parametrize("batched", [False, True])
def test_hubs_at_chunk_edges(gpu_ctx, weights, labels, constrained, batched):
    rng = np.random.default_rng(5)
    m = len(DEGREES)
    n = 110000
    src = [np.full(d, k) for k, d in enumerate(DEGREES)] + [rng.integers(m, n, 60000)]
    dst = [m + rng.permutation(n - m)[:d] for d in DEGREES] + [rng.integers(m, n, 60000)]
    src, dst = np.concatenate(src), np.concatenate(dst)
    w = None if weights is None else rng.integers(weights[0], weights[1] + 1, len(src))
    g = graphs.from_edges(n, src, dst, w)
    assert list(g.degrees()[:m]) == DEGREES
    L = labels or n
    part = rng.integers(0, L, n) if labels else rng.permutation(n)
    if labels:
        part[:L] = np.arange(L)
    cons = rng.integers(0, 2, L).astype(np.int32) if constrained else None
    print(f"hub sweep labels={labels} weights={weights} constrained={constrained} batched={batched}", flush=True)
    try:
        if batched:  # every 8 hubs a batch of their own
            gpu_ctx.set_knob("contract_batch", 1)
        check_sweep(g, part, L, cons)
    finally:
        gpu_ctx.set_knob("contract_batch", 1 << 30)


@pytest.mark.parametrize("weights,degree", [(None, 8500000), ((1 << 29, (1 << 30) - 1), 5700000)])
def test_more_slices_than_buckets(gpu_ctx, weights, degree):
    """1,038 slices with 32-bit sums, 1,044 with 64-bit ones: two to a bucket."""
    rng = np.random.default_rng(6)
    n = degree + 1
    leaves = np.arange(1, n, dtype=np.int32)
    # a star in CSR form: the hub's row, then one entry per leaf
    rp = np.concatenate([[0], degree + np.arange(n, dtype=np.int64)])
    col = np.concatenate([leaves, np.zeros(degree, np.int32)])
    w = None
    if weights:
        half = rng.integers(weights[0], weights[1] + 1, degree)
        w = np.concatenate([half, half]).astype(np.int32)
    g = graphs.CSR(n, rp, col, w)
    part = rng.permutation(n)
    print(f"hub of {degree} edges weights={weights}", flush=True)
    check_sweep(g, part, n)


def test_time_grows_with_the_degree(gpu_ctx):
    """Scoring a hub of 2^23 edges against one of 2^20: 8 times the work, and
    64 times where every slice reads all of the hub's edges (120 was measured)."""
    import torch
    from pennsylvaniagpugraphclustering_amd import clustering as C
    ms = []
    for scale in (20, 23):
        d = 1 << scale
        src = torch.zeros(d, dtype=torch.int32, device="cuda")
        dst = torch.arange(1, d + 1, dtype=torch.int32, device="cuda")
        rp, col, _ = graphs.from_edges_device(d + 1, src, dst)
        dg = C.DeviceGraph(rp, col, None, None, objective="Mod")
        part = torch.arange(d + 1, dtype=torch.int32, device="cuda")
        dest = torch.full((d + 1,), -1, dtype=torch.int32, device="cuda")
        gain = torch.zeros(d + 1, device="cuda")
        print(f"hub of {d} edges", flush=True)
        best = []
        try:
            for _ in range(4):
                gpu_ctx.set_timing(True)
                C.sweep(dg, part, dg.vtx_w, 1.0 / (2 * d), 0.75, False, dest, gain)
                launches, t, _ = gpu_ctx.kernel_stats()["score_hub"]
                assert launches == 1
                best.append(t)
        finally:
            gpu_ctx.set_timing(False)
        ms.append(min(best))
    print(f"hub scoring {ms[0]:.3f} ms, {ms[1]:.3f} ms", flush=True)
    assert ms[1] < 24 * ms[0]
