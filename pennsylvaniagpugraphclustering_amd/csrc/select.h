// Ordered selection: the items x in [0, n) that pass a test, in order, with
// their count (and a few others) left in the context's pinned host slots.
#pragma once
#include "ctx.h"
#include "device.h"

namespace pggc {

// A selection functor F has
//   bool test(i64 x)             whether item x is selected;
//   void emit(i64 pos, i64 x)    item x is the pos-th selected one;
//   static constexpr bool extra; when set, bool first(i64 x, bool sel) and bool
//                                second(i64 x, bool sel) count two more
//                                properties of the items.
//
// Tiles of SEL_TILE items, consecutive lanes on consecutive items; an item's
// place is its tile's offset, plus the selected items of the (step, wave) runs
// before its own, plus its rank in the ballot of its wave.  Bound by reads of
// what the tests look at, on small inputs by launches: two kernels (one for a
// single tile) do what took six (flags, tile sums, a scan of one to three
// kernels, write, read-back).  The write kernel adds up the counts of the tiles
// before its own itself for up to SEL_INLINE tiles; above, a scan does.
constexpr int SEL_T = 256, SEL_I = 8, SEL_TILE = SEL_T * SEL_I, SEL_W = SEL_T / 64;
constexpr i64 SEL_INLINE = 4096;

// The results go to coherent host memory, which the end of the kernel makes
// visible to a host that waits for the stream:
// host[0] selected items, host[1], host[2] those before bounds b0 and b1,
// host[3], host[4] the extra counts
struct SelBounds {
    i64 b0, b1;
};

template <class F>
__device__ __forceinline__ void sel_extra(const F& f, i64 x, bool in, bool sel, int& e0, int& e1) {
    e0 += __popcll(__ballot(in && f.first(x, sel)));
    e1 += __popcll(__ballot(in && f.second(x, sel)));
}

template <class F>
__global__ void __launch_bounds__(SEL_T) k_sel_count(F f, i64 n, i32* __restrict__ tile, i64* extra) {
    __shared__ int cnt[SEL_W][3];
    const i64 base = block_id() * SEL_TILE;
    if (base >= n) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int c = 0, e0 = 0, e1 = 0;  // wave-uniform
#pragma unroll
    for (int k = 0; k < SEL_I; k++) {
        const i64 x = base + k * SEL_T + threadIdx.x;
        const bool in = x < n;
        const bool sel = in && f.test(x);
        c += __popcll(__ballot(sel));
        if constexpr (F::extra) sel_extra(f, x, in, sel, e0, e1);
    }
    if (lane == 0) {
        cnt[wv][0] = c;
        cnt[wv][1] = e0;
        cnt[wv][2] = e1;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        int s = 0;
        for (int w = 0; w < SEL_W; w++) s += cnt[w][threadIdx.x];
        if (threadIdx.x == 0) tile[block_id()] = s;
        else if (F::extra && s) atomicAdd((unsigned long long*)&extra[threadIdx.x - 1], (unsigned long long)s);
    }
}

// toff: tile offsets (nb + 1) when there are more than SEL_INLINE tiles
template <class F>
__global__ void __launch_bounds__(SEL_T) k_sel_write(F f, i64 n, i64 nb, const i32* __restrict__ tile,
                                                     const i64* __restrict__ toff, SelBounds sb, i64* extra,
                                                     i64* host) {
    __shared__ int cnt[SEL_I * SEL_W];
    __shared__ int ex[SEL_W][2];
    const i64 b = block_id();
    if (b >= nb) return;
    const i64 base = b * SEL_TILE;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    u64 bal[SEL_I];
    int e0 = 0, e1 = 0;
#pragma unroll
    for (int k = 0; k < SEL_I; k++) {
        const i64 x = base + k * SEL_T + threadIdx.x;
        const bool in = x < n;
        const bool sel = in && f.test(x);
        bal[k] = __ballot(sel);
        if (lane == 0) cnt[k * SEL_W + wv] = __popcll(bal[k]);
        if constexpr (F::extra) {
            if (nb == 1) sel_extra(f, x, in, sel, e0, e1);
        }
    }
    if (F::extra && lane == 0) {
        ex[wv][0] = e0;
        ex[wv][1] = e1;
    }
    i64 b0 = 0;
    if (toff) {
        b0 = toff[b];
    } else if (b > 0) {
        i64 s = 0;
        for (i64 q = threadIdx.x; q < b; q += SEL_T) s += tile[q];
        b0 = block_sum_i64<SEL_T>(s);
    }
    __syncthreads();
    i64 run = b0;  // selected items before run (k, wave)
#pragma unroll
    for (int k = 0; k < SEL_I; k++) {
        i64 before = run;
#pragma unroll
        for (int w = 0; w < SEL_W; w++) {
            const int c = cnt[k * SEL_W + w];
            before += w < wv ? c : 0;
            run += c;
        }
        const i64 x = base + k * SEL_T + threadIdx.x;
        const i64 pos = before + __popcll(bal[k] & (((u64)1 << lane) - 1));
        if ((bal[k] >> lane) & 1) f.emit(pos, x);
        if (x == sb.b0) host[1] = pos;
        if (x == sb.b1) host[2] = pos;
    }
    if (b == nb - 1 && threadIdx.x == 0) {
        host[0] = run;
        if (sb.b0 >= n) host[1] = run;
        if (sb.b1 >= n) host[2] = run;
    }
    if (F::extra && b == 0 && threadIdx.x < 2) {
        if (nb == 1) {
            i64 s = 0;
            for (int w = 0; w < SEL_W; w++) s += ex[w][threadIdx.x];
            host[3 + threadIdx.x] = s;
        } else {  // summed by k_sel_count; zero for the next selection
            host[3 + threadIdx.x] = extra[threadIdx.x];
            extra[threadIdx.x] = 0;
        }
    }
}

// Runs the selection and waits; the result is in c.pinned[0..4].  extra: two
// device words that are zero (F::extra only).  n = 0 gives zeros.
template <class F>
const i64* select_items(Ctx& c, const F& f, i64 n, SelBounds sb = {0, 0}, i64* extra = nullptr) {
    if (n <= 0) {
        for (int k = 0; k < 5; k++) c.pinned[k] = 0;
        return c.pinned;
    }
    const i64 nb = ceil_div(n, SEL_TILE);
    Buf<i32> tile;
    Buf<i64> toff;
    if (nb > 1) {
        tile = Buf<i32>(c, nb);
        k_sel_count<<<grid_blocks(nb), SEL_T, 0, c.stream>>>(f, n, tile.p, extra);
        PGGC_LAUNCH_CHECK();
        if (nb > SEL_INLINE) {
            toff = Buf<i64>(c, nb + 1);
            scan_i32_to_i64(c, tile, toff, nb);
        }
    }
    k_sel_write<<<grid_blocks(nb), SEL_T, 0, c.stream>>>(f, n, nb, tile.p, toff.p, sb, extra, c.pinned_dev);
    PGGC_LAUNCH_CHECK();
    c.sync();
    return c.pinned;
}

// indices x (or src[x]) of nonzero flags
struct SelFlags {
    static constexpr bool extra = false;
    const i32* flag;
    const i32* src;
    i32* out;
    __device__ __forceinline__ bool test(i64 x) const { return flag[x] != 0; }
    __device__ __forceinline__ void emit(i64 pos, i64 x) const { out[pos] = src ? src[x] : (i32)x; }
};
// Ordered compaction of the indices x in [0, n) with flag[x] != 0, writing
// src ? src[x] : x; returns the count.
inline i64 compact_flags(Ctx& c, const i32* flag, const i32* src, i64 n, i32* out) {
    return select_items(c, SelFlags{flag, src, out}, n)[0];
}

// Stable partition of [0, n) by class: out receives the items grouped by
// f(x) in [0, K) (K <= 15), and starts[0..K] the class boundaries (waits).
// Tiles and runs as in the selections; an item's rank among the lanes of its
// class comes from a ballot per class bit.
constexpr int CLS_MAX = 15;
// lanes of the wave whose 4-bit class equals this lane's
__device__ __forceinline__ u64 same_class(int cls) {
    u64 m = ~(u64)0;
#pragma unroll
    for (int bit = 0; bit < 4; bit++) {
        const u64 s = __ballot((cls >> bit) & 1);
        m &= ((cls >> bit) & 1) ? s : ~s;
    }
    return m;
}
template <class F>
__global__ void __launch_bounds__(SEL_T) k_cls_count(F f, i64 n, i64 nb, int K, i64* counts) {
    __shared__ int cnt[CLS_MAX];
    const i64 b = block_id();
    if (b >= nb) return;
    if (threadIdx.x < CLS_MAX) cnt[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SEL_I; k++) {
        const i64 x = b * SEL_TILE + k * SEL_T + threadIdx.x;
        if (x < n) atomicAdd(&cnt[f(x)], 1);
    }
    __syncthreads();
    if ((int)threadIdx.x < K) counts[(i64)threadIdx.x * nb + b] = cnt[threadIdx.x];
}
template <class F>
__global__ void __launch_bounds__(SEL_T) k_cls_write(F f, i64 n, i64 nb, int K, const i64* __restrict__ offs,
                                                     i32* __restrict__ out, i64* host) {
    __shared__ int cnt[SEL_I * SEL_W][CLS_MAX + 1];  // class counts of the runs, then their prefix
    const i64 b = block_id();
    if (b >= nb) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int q = threadIdx.x; q < SEL_I * SEL_W * (CLS_MAX + 1); q += SEL_T) cnt[q / (CLS_MAX + 1)][q % (CLS_MAX + 1)] = 0;
    __syncthreads();
    int cl[SEL_I], rk[SEL_I];
#pragma unroll
    for (int k = 0; k < SEL_I; k++) {
        const i64 x = b * SEL_TILE + k * SEL_T + threadIdx.x;
        cl[k] = x < n ? f(x) : CLS_MAX;
        const u64 m = same_class(cl[k]);
        rk[k] = __popcll(m & (((u64)1 << lane) - 1));
        if (rk[k] == 0) cnt[k * SEL_W + wv][cl[k]] = __popcll(m);
    }
    __syncthreads();
    if ((int)threadIdx.x < K) {
        int run = 0;
        for (int q = 0; q < SEL_I * SEL_W; q++) {
            const int v = cnt[q][threadIdx.x];
            cnt[q][threadIdx.x] = run;
            run += v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SEL_I; k++) {
        const i64 x = b * SEL_TILE + k * SEL_T + threadIdx.x;
        if (x < n) out[offs[(i64)cl[k] * nb + b] + cnt[k * SEL_W + wv][cl[k]] + rk[k]] = (i32)x;
    }
    if (b == 0 && (int)threadIdx.x <= K) host[threadIdx.x] = offs[(i64)threadIdx.x * nb];
}
template <class F>
void class_partition(Ctx& c, const F& f, i64 n, int K, i32* out, i64* starts) {
    if (K > CLS_MAX) throw Error(-5, "class_partition: too many classes");
    const i64 nb = ceil_div(n > 0 ? n : 1, SEL_TILE);
    Buf<i64> counts(c, K * nb + 1);
    k_cls_count<<<grid_blocks(nb), SEL_T, 0, c.stream>>>(f, n, nb, K, counts);
    PGGC_LAUNCH_CHECK();
    scan_i64(c, counts, counts, K * nb);
    k_cls_write<<<grid_blocks(nb), SEL_T, 0, c.stream>>>(f, n, nb, K, counts, out, c.pinned_dev);
    PGGC_LAUNCH_CHECK();
    c.sync();
    for (int k = 0; k <= K; k++) starts[k] = c.pinned[k];
}

}  // namespace pggc
