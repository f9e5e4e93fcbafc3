// Leiden refinement (src/leidenR.cpp): gamma-well-connected flags, seeded
// neighbour choice, pointer-chasing forests, gamma-connectivity splitting
// inside each tree (radix-sorted by (tree, order, id)), contiguous relabel.
#include <algorithm>

#include "device.h"
#include "leiden.h"

namespace pggc {

// :281-287.  A vertex's record: its cluster, -1 when it is not well connected,
// and in the high word its weight as a float, so that the test of a neighbour
// is one gather.
__global__ void k_well(const i64* vw, const i32* louv, const i64* vol, const i64* pv, i64 n, float gamma,
                       u64* well) {
    const i64 i = thread_item();
    if (i >= n) return;
    const i64 wd = vw[i];
    const i32 ci = louv[i];
    const bool ok = (float)pv[i] >= gamma * (float)wd * (float)(vol[ci] - wd);
    well[i] = ((u64)__float_as_uint((float)wd) << 32) | (u32)(ok ? ci : -1);
}
__device__ __forceinline__ i32 well_cluster(u64 r) { return (i32)(u32)r; }
__device__ __forceinline__ float well_weight(u64 r) { return __uint_as_float((u32)(r >> 32)); }

// :296-393 (unit weights): first satisfactory neighbour cyclically from a
// hashed start; 1/1000 of the vertices keep themselves.
// list: the vertices of degree < 128 (order1 prefix); larger degrees take
// k_hn_uniform_wave
__global__ void k_hn_uniform(const i64* rp, const i32* col, const u64* well, const i32* list, i64 m, float gamma,
                             i32 seed, i32* hn) {
    const i64 x = thread_item();
    if (x >= m) return;
    const i32 i = list[x];
    const i64 s = rp[i], e = rp[i + 1], width = e - s;
    const u64 me = well[i];
    const i32 ci = well_cluster(me);
    const float multi = gamma * well_weight(me);
    const u32 h = murmur3_i32((i32)((u32)seed + (u32)i));
    const i32 jx32 = (i32)h;
    i32 pick = i;
    if (jx32 % 1000 != 0 && ci >= 0) {
        const i64 off = width ? (i64)(h % (u32)width) : 0;
        for (i64 t = 0; t < width; t++) {
            const i32 v = col[s + (off + t < width ? off + t : off + t - width)];
            const u64 o = well[v];
            if (well_cluster(o) == ci && 1.0f >= multi * well_weight(o)) {
                pick = v;
                break;
            }
        }
    }
    hn[i] = pick;
}

// the same choice with one wave per vertex: the lanes test 64 consecutive
// positions of the cyclic scan from the hashed start at a time, and the
// first passing position (lowest lane of the first chunk with one) is the
// serial scan's pick
__global__ void __launch_bounds__(256) k_hn_uniform_wave(const i64* rp, const i32* col, const u64* well,
                                                         const i32* list, i64 m, float gamma, i32 seed, i32* hn) {
    const int lane = threadIdx.x & 63;
    const i64 x = block_id() * 4 + (threadIdx.x >> 6);
    if (x >= m) return;
    const i32 i = list[x];
    const i64 s = rp[i], e = rp[i + 1], width = e - s;
    const u64 me = well[i];
    const i32 ci = well_cluster(me);
    const float multi = gamma * well_weight(me);
    const u32 h = murmur3_i32((i32)((u32)seed + (u32)i));
    const i32 jx32 = (i32)h;
    if (jx32 % 1000 == 0 || ci < 0 || width == 0) {
        if (lane == 0) hn[i] = (i32)i;
        return;
    }
    const i64 off = (i64)(h % (u32)width);
    for (i64 base = 0; base < width; base += 64) {  // wave-uniform loop control
        const i64 t = base + lane;
        i32 ok = 0;
        i32 v = -1;
        if (t < width) {
            const i64 q = off + t;
            v = col[s + (q < width ? q : q - width)];
            const u64 o = well[v];
            ok = well_cluster(o) == ci && 1.0f >= multi * well_weight(o);
        }
        xlane_fence(ok);  // the values below cross lanes
        xlane_fence(v);
        const u64 bal = __ballot(ok != 0);
        if (bal) {
            const int first = __ffsll((unsigned long long)bal) - 1;
            const i32 pick = __shfl(v, first);
            if (lane == 0) hn[i] = pick;
            return;
        }
    }
    if (lane == 0) hn[i] = (i32)i;
}

// :395-474 (weighted): argmax over neighbours of rand * (w - gamma w_i w_v)^4
// with (.)^4 evaluated as ((double)val^2)^2.  Degree < 128 keeps the last
// maximum (serial path); larger degrees keep the first (MaxFirstLoc).  A sample
// is never negative, so its key is never 0.
//
// The gathers of the neighbours' records bound it: G lanes share a vertex and
// have HN_U edges each in flight (a thread per vertex took 5.1 ms on the LFR
// graph of 8.4M vertices' top level, loading its own row edge by edge; 2.35
// now), and the vertices of MASSIVE_CUTOFF edges and more take HN_B blocks, whose
// maxima meet in `best` (with one wave on each, a level of R-MAT scale 22 took 4.3
// ms; 0.7 now).
constexpr int HN_U = 4, HN_G = 8, HN_B = 16;
template <bool LAST, class WT>
__device__ __forceinline__ u64 hn_best(const i32* __restrict__ col, WT W, const u64* __restrict__ well, i64 s, i64 e,
                                       i64 first, i64 step, i32 ci, float multi, i32 seed) {
    u64 best = 0;
    for (i64 jb = s + first; __any(jb < e); jb += step * HN_U) {  // wave-uniform loop control
        i32 v[HN_U];
        u64 o[HN_U];
#pragma unroll
        for (int u = 0; u < HN_U; u++) {
            const i64 j = jb + u * step;
            v[u] = j < e ? col[j] : -1;
        }
#pragma unroll
        for (int u = 0; u < HN_U; u++) o[u] = v[u] >= 0 ? well[v[u]] : 0;
#pragma unroll
        for (int u = 0; u < HN_U; u++) {
            if (v[u] < 0 || well_cluster(o[u]) != ci) continue;
            const i64 j = jb + u * step;
            const float val = fmaf(-multi, well_weight(o[u]), (float)W(j));
            if (!(val >= 0.0f)) continue;
            const float r = (float)murmur3_i32((i32)((u32)seed + (u32)j)) / (float)ORD_MAX;
            const double v2 = (double)val * (double)val;
            const float smp = (float)((double)r * (v2 * v2));
            const u32 at = (u32)(j - s);
            const u64 k = ((u64)ord_f32(smp) << 32) | (LAST ? at : 0xFFFFFFFFu - at);
            best = k > best ? k : best;
        }
    }
    return best;
}
__device__ __forceinline__ bool hn_skips(i32 seed, i32 i, i32 ci) {
    return murmur3_i32((i32)((u32)seed + (u32)i)) % 10000u == 0 || ci < 0;
}

// G lanes per vertex: HN_G for degrees below LARGE_CUTOFF, a wave above
template <int G, class WT>
__global__ void __launch_bounds__(256) k_hn_weighted(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                     const u64* __restrict__ well, const i32* __restrict__ list,
                                                     i64 m, float gamma, i32 seed, i32* __restrict__ hn) {
    constexpr bool LAST = G == HN_G;
    const int lane = threadIdx.x & (G - 1);
    const i64 x = block_id() * (256 / G) + threadIdx.x / G;
    i32 i = -1, ci = -1;
    i64 s = 0, e = 0;
    float multi = 0.0f;
    if (x < m) {
        i = list[x];
        s = e = rp[i];
        const u64 me = well[i];
        ci = well_cluster(me);
        multi = gamma * well_weight(me);
        if (!hn_skips(seed, i, ci)) e = rp[i + 1];
    }
    u64 best = hn_best<LAST>(col, W, well, s, e, lane, G, ci, multi, seed);
    xlane_fence(best);
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        const u64 b = __shfl_xor(best, o, G);
        best = b > best ? b : best;
    }
    if (i >= 0 && lane == 0)
        hn[i] = best ? col[s + (i64)(LAST ? (u32)best : 0xFFFFFFFFu - (u32)best)] : i;
}
// HN_B blocks per vertex, and the picks from their maxima
template <class WT>
__global__ void __launch_bounds__(256) k_hn_massive(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                    const u64* __restrict__ well, const i32* __restrict__ list, i64 m,
                                                    float gamma, i32 seed, u64* best) {
    const i64 b = block_id();
    if (b >= m * HN_B) return;
    const i32 i = list[b / HN_B];
    const u64 me = well[i];
    const i32 ci = well_cluster(me);
    if (hn_skips(seed, i, ci)) return;  // block-uniform
    u64 k = hn_best<false>(col, W, well, rp[i], rp[i + 1], (b % HN_B) * 256 + threadIdx.x, 256 * HN_B, ci,
                           gamma * well_weight(me), seed);
    k = block_max_u64<256>(k);
    if (threadIdx.x == 0 && k) atomicMax((unsigned long long*)&best[b / HN_B], (unsigned long long)k);
}
__global__ void k_hn_pick(const i64* rp, const i32* col, const i32* list, i64 m, const u64* best, i32* hn) {
    const i64 x = thread_item();
    if (x >= m) return;
    const i32 i = list[x];
    const u64 k = best[x];
    hn[i] = k ? col[rp[i] + (i64)(0xFFFFFFFFu - (u32)k)] : i;
}

// :482-494
__global__ void k_order(i64 n, i32 seed, i32* order) {
    const i64 i = thread_item();
    if (i >= n) return;
    i32 o = (i32)murmur3_i32((i32)((u32)i + (u32)seed));
    i32 r = o % SPLIT;
    order[i] = r < 0 ? -r : r;
}
__global__ void k_unselect(i64 n, const i32* order, i32* hn) {
    const i64 i = thread_item();
    if (i >= n) return;
    if (order[i] == order[hn[i]]) hn[i] = (i32)i;
}

// find_trees (:212-260)
__global__ void k_trees1(i64 n, const i32* hn, const i32* order, i32* vcmap) {
    const i64 i = thread_item();
    if (i >= n) return;
    i32 now = (i32)i, then = hn[i];
    if (now == then) {
        vcmap[i] = (i32)i;
        return;
    }
    while (order[now] > order[then]) {
        now = then;
        then = hn[then];
    }
    if (now != i) {
        vcmap[i] = now;
        vcmap[now] = now;
    }
}
__global__ void k_trees_flip(i64 n, const i32* vcmap, i32* order) {
    const i64 i = thread_item();
    if (i >= n) return;
    if (vcmap[i] == ORD_MAX) order[i] = 2 * SPLIT - order[i];
}
__global__ void k_trees2(i64 n, const i32* hn, const i32* order, i32* vcmap) {
    const i64 i = thread_item();
    if (i >= n) return;
    if (vcmap[i] != ORD_MAX) return;
    i32 now = (i32)i, then = hn[i];
    while (__hip_atomic_load(&vcmap[now], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == ORD_MAX &&
           order[now] > order[then]) {
        now = then;
        then = hn[then];
    }
    vcmap[i] = __hip_atomic_load(&vcmap[now], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ensure_gamma_connectivity (:41-187)
__global__ void k_gkeys(i64 n, const i32* vcmap, const i32* order, u64* key, u64* tree, i32* val) {
    const i64 i = thread_item();
    if (i >= n) return;
    key[i] = tree[i] = ((u64)(u32)vcmap[i] << 31) | (u64)(u32)order[i];
    val[i] = (i32)i;
}
__global__ void k_gstarts(i64 n, const i32* ids, const i32* vcmap, i64* cbeg, const i64* vw, i64* wsorted) {
    const i64 x = thread_item();
    if (x >= n) return;
    i32 i = ids[x];
    i32 c = vcmap[i];
    if (x == 0 || vcmap[ids[x - 1]] != c) cbeg[c] = x;
    wsorted[x] = vw[i];
}

// inner[i] = weight of i's edges to earlier members (by order) of its
// refined cluster: keys of the same tree with a smaller order
struct EarlierInTree {
    __device__ __forceinline__ bool operator()(u64 mine, u64 other) const {
        return other < mine && (other >> 31) == (mine >> 31);
    }
};

__global__ void k_outer_vals(i64 n, const i32* ids, const i64* pv, const i64* inner, i64* ov) {
    const i64 x = thread_item();
    if (x >= n) return;
    i32 i = ids[x];
    ov[x] = pv[i] - 2 * inner[i];
}

__global__ void k_breaks(i64 n, const i32* ids, const i32* vcmap, const i32* louv, const i64* cbeg, const i64* tsz,
                         const i64* osc, const i64* inner, const i64* vw, const i64* vol, float gamma,
                         long long* breakers) {
    const i64 x = thread_item();
    if (x >= n) return;
    i32 i = ids[x];
    i32 c = vcmap[i];
    i64 cb = cbeg[c];
    i64 prev = tsz[x] - tsz[cb];
    if ((float)inner[i] < gamma * (float)vw[i] * (float)prev) atomicMin(&breakers[c], (long long)x);
    i64 cur = tsz[x] + vw[i] - tsz[cb];
    i64 other = vol[louv[i]] - cur;
    i64 out = osc[x + 1] - osc[cb];
    if ((float)out < gamma * (float)cur * (float)other) atomicMin(&breakers[c], (long long)(x + 1));
}

__global__ void k_break_apply(i64 n, const i32* ids, const long long* breakers, i32* vcmap) {
    const i64 x = thread_item();
    if (x >= n) return;
    i32 i = ids[x];
    i32 c = vcmap[i];
    if (x >= breakers[c]) vcmap[i] = i;
}

// contigitize_clusters (:189-210)
__global__ void k_root_flags(i64 n, const i32* vcmap, i32* f) {
    const i64 u = thread_item();
    if (u >= n) return;
    f[u] = vcmap[u] == u ? 1 : 0;
}
__global__ void k_root_relabel(i64 n, const i64* rank, const i32* in, i32* out) {
    const i64 u = thread_item();
    if (u >= n) return;
    out[u] = (i32)rank[in[u]];
}

static int bitsfor(i64 v) {
    int b = 0;
    while (b < 62 && ((i64)1 << b) <= v) b++;
    return b;
}

i64 leiden_refine(Ctx& c, const DGraph& g, const Orders& ord, const i32* louv, const i64* vol, double lambda,
                  const i64* pv, bool uniform, i32* vcmap_out) {
    const i64 n = g.n;
    const float gamma = (float)lambda;
    const dim3 G = grid_items(n, 256);
    // algorithmic bytes: two adjacency passes (neighbour choice: column,
    // weight and the neighbour's record; inner weights: column, weight and the
    // neighbour's tree and order) and about 40
    // int32/int64 vertex arrays read or written by the flag, order, forest,
    // sort, scan, break and relabel steps
    const int wb = g.wk == W_UNIT ? 0 : g.wk == W_I32 ? 4 : 8;
    const int tk = c.kt_begin(KS_LEIDEN);
    Buf<u64> well(c, n + 1);
    Buf<i32> hn(c, n + 1), order(c, n + 1), vcmap(c, n + 1);
    k_well<<<G, 256, 0, c.stream>>>(g.vw, louv, vol, pv, n, gamma, well);
    PGGC_LAUNCH_CHECK();
    const i32 hseed = (i32)c.next_draw();
    const i64 big = ord.off_large, huge = ord.off_large2;  // order1: degree < LARGE_CUTOFF, then < MASSIVE_CUTOFF
    if (uniform) {
        if (big > 0)
            k_hn_uniform<<<grid_items(big, 256), 256, 0, c.stream>>>(g.rp, g.col, well, ord.o1, big, gamma, hseed, hn);
        if (n > big)
            k_hn_uniform_wave<<<grid_items(n - big, 4), 256, 0, c.stream>>>(g.rp, g.col, well, ord.o1.p + big, n - big,
                                                                            gamma, hseed, hn);
        PGGC_LAUNCH_CHECK();
    } else {
        PGGC_WDISPATCH(g, {
            if (big > 0)
                k_hn_weighted<HN_G><<<grid_items(big, 256 / HN_G), 256, 0, c.stream>>>(g.rp, g.col, W, well, ord.o1,
                                                                                       big, gamma, hseed, hn);
            if (huge > big)
                k_hn_weighted<64><<<grid_items(huge - big, 4), 256, 0, c.stream>>>(
                    g.rp, g.col, W, well, ord.o1.p + big, huge - big, gamma, hseed, hn);
        });
        PGGC_LAUNCH_CHECK();
        const i64 m = n - huge;
        if (m > 0) {
            const i32* list = ord.o1.p + huge;
            Buf<u64> best(c, m);
            fill_i64(c, (i64*)best.p, m, 0);
            PGGC_WDISPATCH(g, (k_hn_massive<<<grid_blocks(m * HN_B), 256, 0, c.stream>>>(g.rp, g.col, W, well, list, m,
                                                                                       gamma, hseed, best)));
            PGGC_LAUNCH_CHECK();
            k_hn_pick<<<grid_items(m, 256), 256, 0, c.stream>>>(g.rp, g.col, list, m, best, hn);
            PGGC_LAUNCH_CHECK();
        }
    }
    {
        const i32 seed = (i32)c.next_draw();
        k_order<<<G, 256, 0, c.stream>>>(n, seed, order);
        PGGC_LAUNCH_CHECK();
    }
    k_unselect<<<G, 256, 0, c.stream>>>(n, order, hn);
    fill_i32(c, vcmap, n, ORD_MAX);
    k_trees1<<<G, 256, 0, c.stream>>>(n, hn, order, vcmap);
    k_trees_flip<<<G, 256, 0, c.stream>>>(n, vcmap, order);
    k_trees2<<<G, 256, 0, c.stream>>>(n, hn, order, vcmap);
    PGGC_LAUNCH_CHECK();
    // sort vertices by (tree, order, id)
    Buf<u64> key(c, n);
    Buf<i32> ids(c, n);
    u64* tree = well.p;  // (the records are read no more)
    k_gkeys<<<G, 256, 0, c.stream>>>(n, vcmap, order, key, tree, ids);
    PGGC_LAUNCH_CHECK();
    radix_sort_pairs(c, key, ids, n, 31 + bitsfor(n));
    Buf<i64> cbeg(c, n + 1), wsorted(c, n + 1), tsz(c, n + 1), inner(c, n + 1), ov(c, n + 1), osc(c, n + 1);
    k_gstarts<<<G, 256, 0, c.stream>>>(n, ids, vcmap, cbeg, g.vw, wsorted);
    PGGC_LAUNCH_CHECK();
    scan_i64(c, wsorted, tsz, n);
    fill_i64(c, inner, n, 0);
    if (g.nnz > 0) {
        PGGC_WDISPATCH(g, (k_row_sums<EarlierInTree><<<(int)ceil_div(g.nnz, RS_E), 256, 0, c.stream>>>(
                              g.rp, g.col, W, (const u64*)tree, n, g.nnz, inner)));
        PGGC_LAUNCH_CHECK();
    }
    k_outer_vals<<<G, 256, 0, c.stream>>>(n, ids, pv, inner, ov);
    PGGC_LAUNCH_CHECK();
    scan_i64(c, ov, osc, n);
    Buf<i64> breakers(c, n + 1);
    fill_i64(c, breakers, n, n);
    k_breaks<<<G, 256, 0, c.stream>>>(n, ids, vcmap, louv, cbeg, tsz, osc, inner, g.vw, vol, gamma,
                                     (long long*)breakers.p);
    PGGC_LAUNCH_CHECK();
    k_break_apply<<<G, 256, 0, c.stream>>>(n, ids, (const long long*)breakers.p, vcmap);
    PGGC_LAUNCH_CHECK();
    // contiguous ids by root order
    k_root_flags<<<G, 256, 0, c.stream>>>(n, vcmap, hn);
    PGGC_LAUNCH_CHECK();
    scan_i32_to_i64(c, hn, tsz, n);
    k_root_relabel<<<G, 256, 0, c.stream>>>(n, tsz, vcmap, vcmap_out);
    PGGC_LAUNCH_CHECK();
    c.kt_end(tk, 2.0 * 8.0 * (n + 1) + (double)g.nnz * (24 + 2 * wb) + 250.0 * n);
    return c.read1(tsz.p + n);
}

}  // namespace pggc
