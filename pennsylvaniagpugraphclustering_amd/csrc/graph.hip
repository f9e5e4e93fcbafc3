// Degree ordering, evaluator, own-cluster weights and contraction kernels.
#include <algorithm>
#include <vector>

#include "batching.h"
#include "device.h"
#include "graph.h"
#include "hash.h"
#include "select.h"
#include "widths.h"

namespace pggc {

// ------------------------------------------------------------------ orderings
struct Order1 {
    const i64* rp;
    __device__ __forceinline__ int operator()(i64 i) const { return order_class(rp[i + 1] - rp[i]); }
};
struct Order2 {
    const i64* rp;
    __device__ __forceinline__ int operator()(i64 i) const {
        const i64 d = rp[i + 1] - rp[i];
        return d < MID_CUTOFF ? 0 : (d < MASSIVE_CUTOFF ? 1 : 2);
    }
};

void make_orders(Ctx& c, const DGraph& g, Orders& o) {
    i64 n = g.n;
    // per partition the row bounds read twice and the ids written
    const int tk = c.kt_begin(KS_ORDER);
    if (o.o1.n < (size_t)n || !o.o2.p) {
        o.o1 = Buf<i32>(c, std::max<i64>(n, 1));
        o.o2 = Buf<i32>(c, std::max<i64>(n, 1));
    }
    i64 s1[4], s2[4];
    class_partition(c, Order1{g.rp}, n, 3, o.o1, s1);
    class_partition(c, Order2{g.rp}, n, 3, o.o2, s2);
    o.off_large = s1[1];
    o.off_large2 = s1[2];
    o.off_mid = s2[1];
    o.off_mid2 = s2[2];
    c.kt_end(tk, 2.0 * (16.0 * (n + 1) + 4.0 * n));
}

// ------------------------------------------------- edge-chunk row reductions
// (ChunkRows / chunk_rows in device.h)

template <class WT>
__global__ void __launch_bounds__(EB) k_eval_uncut(const i64* rp, const i32* col, WT W, const i32* lab, i64 n,
                                                    i64 nnz, i64* uncut) {
    ChunkRows cr;
    chunk_rows(rp, n, nnz, cr);
    i64 j0 = cr.eb + (i64)threadIdx.x * EPT;
    i64 acc = 0;
    if (j0 < cr.ee) {
        i64 r = upper_row(rp, cr.rlo, cr.rhi, j0);
        i64 nxt = rp[r + 1];
        i32 lr = lab[r];
        for (int k = 0; k < EPT; k++) {
            i64 j = j0 + k;
            if (j >= cr.ee) break;
            if (j >= nxt) {
                r = advance_row(rp, r, cr.rhi, j, nxt);
                lr = lab[r];
            }
            if (lab[col[j]] == lr) acc += W(j);
        }
    }
    acc = block_sum_i64<EB>(acc);
    if (threadIdx.x == 0 && acc) atomicAdd((unsigned long long*)uncut, (unsigned long long)acc);
}

__global__ void k_eval_vol(const i32* lab, const i64* vw, i64 n, i64* vol) {
    const i64 i = thread_item();
    if (i >= n) return;
    atomicAdd((unsigned long long*)&vol[lab[i]], (unsigned long long)vw[i]);
}

void evaluate(Ctx& c, const DGraph& g, const i32* labels, i64 L, i64* vol, i64* dev_uncut) {
    fill_i64(c, vol, L, 0);
    fill_i64(c, dev_uncut, 1, 0);
    if (g.nnz > 0) {
        // algorithmic bytes: row offsets, columns, labels of both ends, weights
        const double wb = g.wk == W_UNIT ? 0.0 : (g.wk == W_I32 ? 4.0 : 8.0);
        const double bytes = 8.0 * (g.n + 1) + 4.0 * g.n + (8.0 + wb) * g.nnz;
        const int tk = c.kt_begin(KS_EVAL);
        PGGC_WDISPATCH(g, (k_eval_uncut<<<(int)ceil_div(g.nnz, EC), EB, 0, c.stream>>>(g.rp, g.col, W, labels, g.n,
                                                                                       g.nnz, dev_uncut)));
        c.kt_end(tk, bytes);
        PGGC_LAUNCH_CHECK();
    }
    if (g.n > 0) {
        k_eval_vol<<<grid_items(g.n, 256), 256, 0, c.stream>>>(labels, g.vw, g.n, vol);
        PGGC_LAUNCH_CHECK();
    }
}

struct SameLabel {
    __device__ __forceinline__ bool operator()(i32 mine, i32 other) const { return mine == other; }
};
void own_weight(Ctx& c, const DGraph& g, const i32* labels, i64* out) {
    fill_i64(c, out, g.n, 0);
    if (g.nnz == 0) return;
    PGGC_WDISPATCH(g, (k_row_sums<SameLabel><<<(int)ceil_div(g.nnz, RS_E), 256, 0, c.stream>>>(g.rp, g.col, W, labels,
                                                                                              g.n, g.nnz, out)));
    PGGC_LAUNCH_CHECK();
}

__global__ void k_coarsen_vw(const i32* map, const i64* vw, i64 n, i64* out) {
    const i64 i = thread_item();
    if (i >= n) return;
    atomicAdd((unsigned long long*)&out[map[i]], (unsigned long long)vw[i]);
}

void coarsen_vertex_weights(Ctx& c, const DGraph& g, const i32* map, i64 nc, i64* out) {
    fill_i64(c, out, nc, 0);
    if (g.n == 0) return;
    k_coarsen_vw<<<grid_items(g.n, 256), 256, 0, c.stream>>>(map, g.vw, g.n, out);
    PGGC_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- contraction
// members and summed degrees per coarse vertex; a block's 256 vertices are
// merged per coarse id in LDS first (large clusters take many members of
// every block), then each distinct id gets one pair of HBM atomics
constexpr int CC_SLOTS = 512;
__global__ void __launch_bounds__(256) k_ccount(const i64* rp, const i32* vcmap, i64 n, i64* cnt, i64* bound) {
    __shared__ i32 lk[CC_SLOTS];
    __shared__ i64 lc[CC_SLOTS], lb[CC_SLOTS];
    for (int q = threadIdx.x; q < CC_SLOTS; q += 256) {
        lk[q] = EMPTY_KEY;
        lc[q] = 0;
        lb[q] = 0;
    }
    __syncthreads();
    const i64 i = thread_item();
    if (i < n) {
        const i32 u = vcmap[i];
        const i64 d = rp[i + 1] - rp[i];
        u32 h = slot_hash(u, CC_SLOTS - 1);
        while (true) {  // at most 256 keys in 512 slots: an empty slot is always found
            const i32 old = atomicCAS(&lk[h], EMPTY_KEY, u);
            if (old == EMPTY_KEY || old == u) break;
            h = (h + 1) & (CC_SLOTS - 1);
        }
        atomicAdd((unsigned long long*)&lc[h], 1ull);
        atomicAdd((unsigned long long*)&lb[h], (unsigned long long)d);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < CC_SLOTS; q += 256) {
        const i32 u = lk[q];
        if (u == EMPTY_KEY) continue;
        atomicAdd((unsigned long long*)&cnt[u], (unsigned long long)lc[q]);
        atomicAdd((unsigned long long*)&bound[u], (unsigned long long)lb[q]);
    }
}

// member lists: a block's vertices take ranks per coarse id in LDS, each
// distinct id reserves its run of the list with one HBM atomic (left counts the
// members not placed yet down from the member counts), and every vertex writes
// at run start + rank (the order inside a list is free: the merges that read it
// are order-independent)
__global__ void __launch_bounds__(256) k_cscatter(const i32* vcmap, i64 n, const i64* __restrict__ mstart, i64* left,
                                                  i32* members) {
    __shared__ i32 lk[CC_SLOTS], lc[CC_SLOTS];
    __shared__ i64 lb[CC_SLOTS];
    for (int q = threadIdx.x; q < CC_SLOTS; q += 256) {
        lk[q] = EMPTY_KEY;
        lc[q] = 0;
    }
    __syncthreads();
    const i64 i = thread_item();
    u32 h = 0;
    i32 r = 0;
    if (i < n) {
        const i32 u = vcmap[i];
        h = slot_hash(u, CC_SLOTS - 1);
        while (true) {  // at most 256 keys in 512 slots
            const i32 old = atomicCAS(&lk[h], EMPTY_KEY, u);
            if (old == EMPTY_KEY || old == u) break;
            h = (h + 1) & (CC_SLOTS - 1);
        }
        r = atomicAdd(&lc[h], 1);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < CC_SLOTS; q += 256)
        if (lk[q] != EMPTY_KEY)
            lb[q] = mstart[lk[q]] +
                    (i64)atomicAdd((unsigned long long*)&left[lk[q]], (unsigned long long)-(i64)lc[q]) - lc[q];
    __syncthreads();
    if (i < n) members[lb[h] + r] = (i32)i;
}

// Merge classes by bound (the summed degrees of a row's members): LDS tables
// for bounds up to C_BOUND[q], then big rows and empty ones.
constexpr int C_BIG = 5, C_EMPTY = 6, C_CLS = 7;
struct MergeClass {
    const i64* bound;
    __device__ __forceinline__ int operator()(i64 u) const {
        const i64 b = bound[u];
        return b == 0 ? C_EMPTY : b <= 256 ? 0 : b <= 1024 ? 1 : b <= 2048 ? 2 : b <= 4096 ? 3 : b <= C_TOP ? 4 : C_BIG;
    }
};

__host__ __device__ __forceinline__ i64 table_slots(i64 bound, i64 nc) {
    i64 cap = bound < nc ? bound : nc;
    i64 s = 2;
    while (s < 2 * cap) s <<= 1;
    return s;
}

__global__ void k_goff_sizes(const i32* list, i64 m, const i64* bound, i64 nc, i64* sz) {
    const i64 x = thread_item();
    if (x >= m) return;
    sz[x] = table_slots(bound[list[x]], nc);
}

// the wave's smallest lo and largest hi, in every lane
__device__ __forceinline__ void wave_min_max(i32& lo, i32& hi) {
    xlane_fence(lo);
    xlane_fence(hi);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const i32 a = __shfl_xor(lo, o), b = __shfl_xor(hi, o);
        lo = a < lo ? a : lo;
        hi = b > hi ? b : hi;
    }
}
// ascending bitonic sort of the first n keys in LDS (room for the next power
// of two); every thread of the block calls it
template <int BS>
__device__ __forceinline__ void lds_sort_keys(i32* k, int n) {
    int P = 2;
    while (P < n) P <<= 1;
    for (int q = n + threadIdx.x; q < P; q += BS) k[q] = 0x7fffffff;
    __syncthreads();
    for (int len = 2; len <= P; len <<= 1)
        for (int o = len >> 1; o > 0; o >>= 1) {
            for (int q = threadIdx.x; q < P / 2; q += BS) {
                const int i = (q / o) * 2 * o + (q % o), j = i + o;
                const bool up = (i & len) == 0;
                const i32 a = k[i], b = k[j];
                if ((a > b) == up) {
                    k[i] = b;
                    k[j] = a;
                }
            }
            __syncthreads();
        }
}
constexpr i32 C_FAT = 96;  // largest bucket that is ranked by comparing every pair of its keys

// One block per coarse vertex of bound at most D: hash-merge the members' edges
// by coarse neighbour in LDS, then write the distinct (neighbour, weight) pairs,
// sorted by neighbour, to the temporary row at toff[u].
//
// The gathers of the neighbours' coarse ids bound the merge, so each thread has
// CR edges in flight; the member that holds an edge is a binary search over the
// members' degree prefix in LDS.  AT: u32 when every row sum of bound C_TOP fits
// 32 bits, else i64 (the same sums).  The sort: the distinct keys are counted
// into D buckets of equal id ranges between their smallest and largest, moved to
// their bucket, and ranked among the keys of their bucket (one or two on
// average; a row with a bucket of more than C_FAT keys, ids that bunch within
// their range, is sorted instead, and the ranks are searched).  R-MAT scale 22
// into 65,536 random clusters: rows of bounds up to 2048 took 4.2 ms with one
// gather in flight, 64-bit sums and a bitonic sort of the whole table (66
// barriers for 2,048 slots); rows up to 8192 take 2.05 ms now, and the rows
// above, which alone are merged in HBM and sorted there, 1.5 + 1.6 ms (from 4.6
// + 3.5, and 14.8 -> 6.6 ms for the whole call).
template <int BS, int D, int SLOTS, class AT, class TT, class WT>
__global__ void __launch_bounds__(BS) k_cagg(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                              const i32* __restrict__ vcmap, i64 nc, const i32* __restrict__ list,
                                              i64 nlist, const i64* __restrict__ mstart,
                                              const i32* __restrict__ members, const i64* __restrict__ bound,
                                              const i64* __restrict__ toff, i32* __restrict__ tcol,
                                              TT* __restrict__ tw, i64* __restrict__ ccnt) {
    static_assert(SLOTS > D, "the table holds every key and the bucket starts");
    __shared__ i32 keys[SLOTS];  // the table's keys, then the keys in bucket order
    __shared__ AT vals[SLOTS];   // the table's sums, then the bucket starts
    __shared__ i32 pre[BS];
    __shared__ i64 rs[BS];
    __shared__ i32 s_min, s_max, s_fat;
    const int t = threadIdx.x;
    const i64 li = block_id();
    if (li >= nlist) return;
    if (t == 0) {
        s_min = 0x7fffffff;
        s_max = -1;
        s_fat = 0;
    }
    const i32 u = list[li];
    const i64 cap = bound[u] < nc ? bound[u] : nc;
    int S = 2;
    while (S < 2 * cap) S <<= 1;
    S = S < SLOTS ? S : SLOTS;
    for (int s = t; s < S; s += BS) {
        keys[s] = EMPTY_KEY;
        vals[s] = 0;
    }
    __syncthreads();
    const i64 m0 = mstart[u], m1 = mstart[u + 1];
    for (i64 mb = m0; mb < m1; mb += BS) {
        const i64 mi = mb + t;
        i64 d = 0, st = 0;
        if (mi < m1) {
            const i32 v = members[mi];
            st = rp[v];
            d = rp[v + 1] - st;
        }
        i64 tot;
        const i64 ex = block_excl_scan_i64(d, &tot);
        pre[t] = (i32)ex;
        rs[t] = st;
        __syncthreads();
        const int nm = (int)(m1 - mb < BS ? m1 - mb : BS);
        constexpr int CR = 4;
        for (i64 eb = 0; eb < tot; eb += (i64)BS * CR) {  // block-uniform loop control
            i32 cv[CR];
            i64 j[CR];
#pragma unroll
            for (int r = 0; r < CR; r++) {
                const i32 e = (i32)eb + r * BS + t;
                j[r] = -1;
                if (e < tot) {
                    int lo = 0, hi = nm;
                    while (hi - lo > 1) {
                        const int md = (lo + hi) >> 1;
                        if (pre[md] <= e) lo = md;
                        else hi = md;
                    }
                    j[r] = rs[lo] + (e - pre[lo]);
                }
            }
#pragma unroll
            for (int r = 0; r < CR; r++) cv[r] = j[r] >= 0 ? col[j[r]] : -1;
#pragma unroll
            for (int r = 0; r < CR; r++) cv[r] = cv[r] >= 0 ? vcmap[cv[r]] : u;
#pragma unroll
            for (int r = 0; r < CR; r++) {
                if (cv[r] == u) continue;  // inside the cluster, or no entry
                const AT w = (AT)W(j[r]);
                u32 h = __umulhi((u32)cv[r] * 0x9E3779B1u, (u32)S);
                while (true) {  // fewer keys than slots: an empty slot is always found
                    const i32 old = atomicCAS(&keys[h], EMPTY_KEY, cv[r]);
                    if (old == EMPTY_KEY || old == cv[r]) break;
                    h = h + 1 < (u32)S ? h + 1 : 0;
                }
                if (sizeof(AT) == 4) atomicAdd((u32*)&vals[h], (u32)w);
                else atomicAdd((unsigned long long*)&vals[h], (unsigned long long)w);
            }
        }
        __syncthreads();
    }
    // the distinct entries in registers, their smallest and largest key
    constexpr int R = (SLOTS + BS - 1) / BS;
    i32 ek[R];
    AT ev[R];
    i32 kmin = 0x7fffffff, kmax = -1;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int q = t + r * BS;
        ek[r] = q < S ? keys[q] : EMPTY_KEY;
        ev[r] = q < S ? vals[q] : 0;
        if (ek[r] != EMPTY_KEY) {
            kmin = ek[r] < kmin ? ek[r] : kmin;
            kmax = ek[r] > kmax ? ek[r] : kmax;
        }
    }
    wave_min_max(kmin, kmax);
    if ((t & 63) == 0) {
        atomicMin(&s_min, kmin);
        atomicMax(&s_max, kmax);
    }
    __syncthreads();
    kmin = s_min;
    kmax = s_max;
    if (kmax < 0) {  // no coarse neighbour (block-uniform)
        if (t == 0) ccnt[u] = 0;
        return;
    }
    u32* hist = (u32*)vals;
    for (int q = t; q < D; q += BS) hist[q] = 0;
    __syncthreads();
    // bucket of key k: (k - kmin) * scale >> 32, below D and monotone in k
    const u64 scale = ((u64)D << 32) / (u64)((i64)kmax - kmin + 1);
    u32 eb_[R], ep[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        eb_[r] = ep[r] = 0;
        if (ek[r] == EMPTY_KEY) continue;
        eb_[r] = (u32)(((u64)(u32)(ek[r] - kmin) * scale) >> 32);
        ep[r] = atomicAdd(&hist[eb_[r]], 1u);
    }
    __syncthreads();
    // exclusive scan of the bucket counts, D / BS consecutive ones per thread
    constexpr int HB = D / BS;
    u32 hc[HB];
    i64 mine = 0;
    i32 none = 0, fat = 0;
#pragma unroll
    for (int q = 0; q < HB; q++) {
        hc[q] = hist[t * HB + q];
        mine += hc[q];
        fat = (i32)hc[q] > fat ? (i32)hc[q] : fat;
    }
    wave_min_max(none, fat);
    if ((t & 63) == 0) atomicMax(&s_fat, fat);
    i64 c;
    u32 run = (u32)block_excl_scan_i64(mine, &c);
#pragma unroll
    for (int q = 0; q < HB; q++) {
        hist[t * HB + q] = run;
        run += hc[q];
    }
    if (t == 0) hist[D] = (u32)c;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++)
        if (ek[r] != EMPTY_KEY) keys[hist[eb_[r]] + ep[r]] = ek[r];
    __syncthreads();
    const bool crowded = s_fat > C_FAT;  // block-uniform
    if (crowded) lds_sort_keys<BS>(keys, (int)c);
    const i64 base = toff[u];
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (ek[r] == EMPTY_KEY) continue;
        const u32 b0 = hist[eb_[r]], b1 = hist[eb_[r] + 1];
        u32 rank = b0;
        if (crowded) {
            u32 hi = b1;
            while (hi - rank > 1) {
                const u32 md = (rank + hi) >> 1;
                if (keys[md] <= ek[r]) rank = md;
                else hi = md;
            }
        } else {
            for (u32 q = b0; q < b1; q++) rank += keys[q] < ek[r] ? 1 : 0;
        }
        tcol[base + rank] = ek[r];
        tw[base + rank] = (TT)ev[r];
    }
    if (t == 0) ccnt[u] = c;
}

// Big coarse rows (bound > C_TOP): the flattened member-edge range of each
// such row is split into work items of BCH_E edges, each item a block that
// merges its edges in LDS and then inserts the distinct pairs into the row's
// HBM hash table; a second pass splits each table into slot items of BCH_S
// slots and compacts the occupied slots.
constexpr int BCH_E = 2048;      // member edges per insert item (8 per thread)
constexpr int BCH_S = 4096;      // table slots per extract item (16 per thread)
constexpr int BLDS = 2 * BCH_E;  // LDS pre-aggregation slots
__global__ void k_member_degs(const i32* members, const i64* rp, i64 n, i64* mdp) {
    const i64 k = thread_item();
    if (k >= n) return;
    i32 v = members[k];
    mdp[k] = rp[v + 1] - rp[v];
}
__global__ void k_items(const i32* list, i64 m, const i64* bound, const i64* goff, i64 nc, int slots, i64* items) {
    const i64 x = thread_item();
    if (x >= m) return;
    i64 len = slots ? goff[x + 1] - goff[x] : bound[list[x]];
    const i64 per = slots ? BCH_S : BCH_E;
    items[x] = (len + per - 1) / per;
}

// row of every work item of the big rows: a block per row
__global__ void __launch_bounds__(256) k_item_rows(const i64* __restrict__ items, i64 m, i32* __restrict__ row) {
    const i64 x = block_id();
    if (x >= m) return;
    for (i64 b = items[x] + threadIdx.x; b < items[x + 1]; b += 256) row[b] = (i32)x;
}

// An item's threads take EPI consecutive edges each: the member that holds the
// first one is searched between the members of the item's first and last edge,
// and columns and coarse ids are gathered EPI at a time.  AT as in k_cagg for
// the sums of an item.  The gathers and the inserts bound it: 6.2 ms for the
// rows above 8192 of R-MAT scale 24's first level (13.1 ms for those above 2048
// with the member searched in the whole list by every thread, one gather in
// flight and 1024-edge items).
template <class AT, class WT>
__global__ void __launch_bounds__(256) k_cbig_insert(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                      const i32* __restrict__ vcmap, const i32* __restrict__ members,
                                                      const i64* __restrict__ mstart, const i64* __restrict__ mdp,
                                                      const i32* __restrict__ big, i64 r0, i64 nbig,
                                                      const i32* __restrict__ row, const i64* __restrict__ items,
                                                      const i64* __restrict__ goff, i32* gkeys, i64* gvals, u64* gtab) {
    // a batch of rows, from row r0 on: big, items and goff point at its first
    // row, items[0] and goff[0] are its first work item and first table slot
    __shared__ i32 lk[BLDS];
    __shared__ AT lv[BLDS];
    __shared__ i64 s_k[2];
    const i64 b = block_id() + items[0];
    if (b >= items[nbig]) return;
    const int t = threadIdx.x;
    const i64 ui = (i64)row[b] - r0;
    const i32 u = big[ui];
    const i64 m0 = mstart[u], m1 = mstart[u + 1];
    const i64 e_lo = mdp[m0] + (b - items[ui]) * BCH_E;
    const i64 e_end = mdp[m1];
    const i64 e_hi = e_lo + BCH_E < e_end ? e_lo + BCH_E : e_end;
    for (int q = t; q < BLDS; q += 256) {
        lk[q] = EMPTY_KEY;
        lv[q] = 0;
    }
    if (t < 2) s_k[t] = upper_row(mdp, m0, m1, t == 0 ? e_lo : e_hi - 1);
    __syncthreads();
    constexpr int EPI = BCH_E / 256;
    const i64 e0 = e_lo + (i64)t * EPI;
    if (e0 < e_hi) {
        i64 k = upper_row(mdp, s_k[0], s_k[1] + 1, e0);
        i64 nxt = mdp[k + 1];
        i64 shift = rp[members[k]] - mdp[k];
        i64 j[EPI];
        i32 cv[EPI];
#pragma unroll
        for (int q = 0; q < EPI; q++) {
            const i64 e = e0 + q;
            j[q] = -1;
            if (e < e_hi) {
                if (e >= nxt) {
                    k = advance_row(mdp, k, s_k[1] + 1, e, nxt);
                    shift = rp[members[k]] - mdp[k];
                }
                j[q] = shift + e;
            }
        }
#pragma unroll
        for (int q = 0; q < EPI; q++) cv[q] = j[q] >= 0 ? col[j[q]] : -1;
#pragma unroll
        for (int q = 0; q < EPI; q++) cv[q] = cv[q] >= 0 ? vcmap[cv[q]] : u;
#pragma unroll
        for (int q = 0; q < EPI; q++) {
            if (cv[q] == u) continue;
            const AT w = (AT)W(j[q]);
            u32 h = slot_hash(cv[q], BLDS - 1);
            while (true) {  // at most BLDS / 2 keys
                const i32 old = atomicCAS(&lk[h], EMPTY_KEY, cv[q]);
                if (old == EMPTY_KEY || old == cv[q]) break;
                h = (h + 1) & (BLDS - 1);
            }
            if (sizeof(AT) == 4) atomicAdd((u32*)&lv[h], (u32)w);
            else atomicAdd((unsigned long long*)&lv[h], (unsigned long long)w);
        }
    }
    const u32 gmask = (u32)(goff[ui + 1] - goff[ui] - 1);
    const i64 t0 = goff[ui] - goff[0];
    if (gtab) lds_agg_flush_packed<256, BLDS>(lk, lv, gtab + t0, gmask);  // kernel-uniform
    else lds_agg_flush<256, BLDS>(lk, lv, gkeys + t0, gvals + t0, gmask);
}

// gtab non-null: packed tables (key << 32 | weight), else gkeys / gvals
template <class TT>
__global__ void __launch_bounds__(256) k_cbig_extract(const i32* big, i64 nbig, const i64* items, const i64* goff,
                                                       const i32* gkeys, const i64* gvals, const u64* gtab,
                                                       const i64* toff, i32* tcol, TT* tw, i64* ccnt) {
    __shared__ int s_cnt;
    __shared__ i64 s_base;
    // a batch of rows, as in k_cbig_insert; slot sl lives at sl - g0
    const i64 b = block_id() + items[0];
    if (b >= items[nbig]) return;
    const i64 g0 = goff[0];
    const i64 ui = upper_row(items, 0, nbig, b);
    const i32 u = big[ui];
    const i64 s_lo = goff[ui] + (b - items[ui]) * BCH_S;
    const i64 s_end = goff[ui + 1];
    const i64 s_hi = s_lo + BCH_S < s_end ? s_lo + BCH_S : s_end;
    if (threadIdx.x == 0) s_cnt = 0;
    __syncthreads();
    i32 kk[16];
    int pos[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const i64 sl = s_lo + threadIdx.x + (i64)q * 256;
        if (gtab) {
            const u64 e = sl < s_hi ? gtab[sl - g0] : PEMPTY;
            kk[q] = e == PEMPTY ? EMPTY_KEY : (i32)(e >> 32);
        } else {
            kk[q] = sl < s_hi ? gkeys[sl - g0] : EMPTY_KEY;
        }
        pos[q] = kk[q] != EMPTY_KEY ? atomicAdd(&s_cnt, 1) : -1;
    }
    __syncthreads();
    if (threadIdx.x == 0) s_base = (i64)atomicAdd((unsigned long long*)&ccnt[u], (unsigned long long)s_cnt);
    __syncthreads();
    const i64 base = toff[u] + s_base;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        if (pos[q] >= 0) {
            const i64 sl = s_lo + threadIdx.x + (i64)q * 256;
            tcol[base + pos[q]] = kk[q];
            tw[base + pos[q]] = (TT)(gtab ? (i64)(gtab[sl - g0] & 0xffffffffull) : gvals[sl - g0]);
        }
    }
}

// Copy temporary rows into the compact coarse CSR.  Consecutive lanes copy
// consecutive output entries (EPT steps of EB entries per block), so each
// wave-wide load and store covers whole cache lines.  The row of an entry is
// a binary search over the chunk's row starts, staged in LDS as offsets from
// the chunk start clamped to [0, EC]; a chunk spanning more than EC rows (runs
// of empty rows) searches the row pointers in global memory instead.  The
// search interval carries over between steps since entries only move right.
template <class TT, class OT>
__global__ void __launch_bounds__(EB) k_crow_copy(const i64* crp, i64 nc, i64 nnzc, const i64* toff, const i32* tcol,
                                                   const TT* tw, i32* ocol, OT* ow) {
    __shared__ i32 s_st[EC + 1];
    ChunkRows cr;
    chunk_rows(crp, nc, nnzc, cr);
    const i64 nr = cr.rhi - cr.rlo;
    const bool staged = nr <= EC;
    if (staged) {
        for (int i = threadIdx.x; i <= (int)nr; i += EB) {
            const i64 v = crp[cr.rlo + i] - cr.eb;
            s_st[i] = (i32)(v < 0 ? 0 : (v > EC ? EC : v));
        }
    }
    __syncthreads();
    int lo = 0;
    i64 r = cr.rlo;
    for (int k = 0; k < EPT; k++) {
        const i64 j = cr.eb + (i64)k * EB + threadIdx.x;
        if (j >= cr.ee) break;
        if (staged) {
            // s_st[lo] <= o < s_st[hi]: s_st[0] = 0 and s_st[nr] >= ee - eb
            const int o = (int)(j - cr.eb);
            int hi = (int)nr;
            while (hi - lo > 1) {
                const int m = (lo + hi) >> 1;
                if (s_st[m] <= o) lo = m;
                else hi = m;
            }
            r = cr.rlo + lo;
        } else {
            r = upper_row(crp, r, cr.rhi, j);
        }
        const i64 src = toff[r] + (j - crp[r]);
        ocol[j] = tcol[src];
        ow[j] = (OT)tw[src];
    }
}

// Sorting of rows merged in global tables: flatten, radix sort by
// (row rank, column), scatter back.
__global__ void k_big_count(const i32* list, i64 m, const i64* crp, i64* cnt) {
    const i64 x = thread_item();
    if (x >= m) return;
    i32 u = list[x];
    cnt[x] = crp[u + 1] - crp[u];
}
// key = (big row index in the batch << cb) | column (columns < 2^cb), so the
// radix sort needs only cb + bits(rows in the batch) bits
template <class OT>
__global__ void k_big_flatten(const i32* list, i64 m, const i64* crp, const i64* boff, const i32* ocol,
                              const OT* ow, int cb, u64* key, OT* val, i64* target) {
    const i64 x = block_id();
    if (x >= m) return;
    {
        i32 u = list[x];
        i64 s = crp[u], e = crp[u + 1], b = boff[x] - boff[0];  // within the batch
        for (i64 j = s + threadIdx.x; j < e; j += blockDim.x) {
            i64 f = b + (j - s);
            key[f] = ((u64)x << cb) | (u32)ocol[j];
            val[f] = ow[j];  // the weight travels with its key through the sort
            target[f] = j;
        }
    }
}
// the f-th smallest key of the batch goes to the f-th position of its rows
// in row order (rows keep their order and their lengths through the sort)
template <class OT>
__global__ void k_big_scatter(const u64* key, const i64* target, i64 E, const OT* wsorted, int cb, i32* ocol,
                              OT* ow) {
    const u64 mask = ((u64)1 << cb) - 1;
    for (i64 f = (i64)blockIdx.x * blockDim.x + threadIdx.x; f < E; f += (i64)gridDim.x * blockDim.x) {
        i64 j = target[f];
        ocol[j] = (i32)(key[f] & mask);
        ow[j] = wsorted[f];
    }
}

// Algorithmic bytes of the coarse-row merge (timing runs only, counted after
// it ran): per coarse row its list entry, member range and output count; per
// member its id and row bounds; per member edge the column, weight and the
// neighbour's coarse id; per distinct coarse neighbour the column and int64
// weight written.
__global__ void __launch_bounds__(256) k_contract_bytes(const i32* __restrict__ list, i64 m,
                                                        const i64* __restrict__ mstart, const i64* __restrict__ bound,
                                                        const i64* __restrict__ ccnt, int wb, i64* acc) {
    const i64 x = thread_item();
    i64 b = 0;
    if (x < m) {
        const i32 u = list[x];
        b = 28 + 20 * (mstart[u + 1] - mstart[u]) + bound[u] * (8 + wb) + 12 * ccnt[u];
    }
    b = block_sum_i64<256>(b);
    if (threadIdx.x == 0 && b) atomicAdd((unsigned long long*)acc, (unsigned long long)b);
}
static void contract_bytes(Ctx& c, int tk, const i32* list, i64 m, const i64* mstart, const i64* bound,
                           const i64* ccnt, int wb) {
    if (tk < 0 || m <= 0) return;
    Buf<i64> acc(c, 1);
    fill_i64(c, acc, 1, 0);
    k_contract_bytes<<<grid_items(m, 256), 256, 0, c.stream>>>(list, m, mstart, bound, ccnt, wb, acc);
    PGGC_LAUNCH_CHECK();
    acct_add(c, c.kt_counter(tk), acc);
}


static int bits_for(i64 v) {
    int b = 0;
    while (b < 62 && ((i64)1 << b) <= v) b++;
    return b;
}

template <class T>
__global__ void __launch_bounds__(256) k_max(const T* __restrict__ in, i64 n, u64* out) {
    u64 m = 0;
    // block-uniform loop control (the reduction below is cross-lane)
    for (i64 base = (i64)blockIdx.x * blockDim.x; base < n; base += (i64)gridDim.x * blockDim.x) {
        const i64 x = base + threadIdx.x;
        if (x < n) m = (u64)in[x] > m ? (u64)in[x] : m;
    }
    m = block_max_u64<256>(m);
    if (threadIdx.x == 0 && m) atomicMax((unsigned long long*)out, (unsigned long long)m);
}
__global__ void k_narrow(const i64* __restrict__ in, i64 n, i32* __restrict__ out) {
    for (i64 x = (i64)blockIdx.x * blockDim.x + threadIdx.x; x < n; x += (i64)gridDim.x * blockDim.x)
        out[x] = (i32)in[x];
}

u64 max_weight(Ctx& c, const DGraph& g) {
    if (g.wk == W_UNIT) return 1;
    Buf<u64> mx(c, 1);
    fill_i64(c, (i64*)mx.p, 1, 0);
    const int grid = grid_for(g.nnz, 256 * 8, 8192);
    if (g.wk == W_I32) k_max<i32><<<grid, 256, 0, c.stream>>>((const i32*)g.w, g.nnz, mx);
    else k_max<i64><<<grid, 256, 0, c.stream>>>((const i64*)g.w, g.nnz, mx);
    PGGC_LAUNCH_CHECK();
    return (u64)c.read1((const i64*)mx.p);
}

// int64 coarse weights replaced by int32 ones when every one fits
static void narrow_weights(Ctx& c, OwnedGraph& g) {
    if (g.nnz == 0) return;
    g.wmax = max_weight(c, g.view());
    if (g.wmax > 0x7fffffffull) return;
    g.w32 = Buf<i32>(c, g.nnz);
    k_narrow<<<grid_for(g.nnz, 256 * 8, 8192), 256, 0, c.stream>>>(g.w, g.nnz, g.w32);
    PGGC_LAUNCH_CHECK();
    g.w.reset();
}

// AT: sums of rows merged in LDS; TT: staged weights; OT: weights written to
// `ow` (out.w or out.w32, allocated here), or int64 ones to the caller's arrays;
// packed: the big rows' tables have one word per slot (one CAS per new key)
template <class AT, class TT, class OT>
static void contract_t(Ctx& c, const DGraph& g, const i32* vcmap, i64 nc, bool packed, OwnedGraph& out, Buf<OT>& ow,
                       const ContractTo* to) {
    const i64 n = g.n;
    // member counts, bounds and coarse degrees, zeroed by one launch
    Buf<i64> zero(c, 3 * (nc + 1)), mstart(c, nc + 1), toff(c, nc + 1);
    i64 *cnt = zero.p, *bound = cnt + nc + 1, *ccnt = bound + nc + 1;
    Buf<i32> members(c, std::max<i64>(n, 1));
    fill_i64(c, zero, 3 * (nc + 1), 0);
    k_ccount<<<grid_items(n, 256), 256, 0, c.stream>>>(g.rp, vcmap, n, cnt, bound);
    PGGC_LAUNCH_CHECK();
    scan_i64(c, cnt, mstart, nc);
    scan_i64(c, bound, toff, nc);
    k_cscatter<<<grid_items(n, 256), 256, 0, c.stream>>>(vcmap, n, mstart, cnt, members);
    PGGC_LAUNCH_CHECK();
    c.mem_note("contract: before row staging");
    Buf<i32> tcol(c, std::max<i64>(g.nnz, 1));  // (the bounds add up to nnz)
    Buf<TT> tw(c, std::max<i64>(g.nnz, 1));
    Buf<i32> list(c, std::max<i64>(nc, 1));
    i64 st[C_CLS + 1];
    class_partition(c, MergeClass{bound}, nc, C_CLS, list, st);
    int tk = c.kt_begin(KS_CONTRACT_AGG);
#define PGGC_CAGG(q, BS, D, SLOTS)                                                                                    \
    if (st[q + 1] > st[q])                                                                                            \
    k_cagg<BS, D, SLOTS, AT, TT><<<grid_blocks(st[q + 1] - st[q]), BS, 0, c.stream>>>(                                \
        g.rp, g.col, W, vcmap, nc, list.p + st[q], st[q + 1] - st[q], mstart, members, bound, toff, tcol, tw, ccnt)
    PGGC_WDISPATCH(g, {
        PGGC_CAGG(0, 64, 256, 512);
        PGGC_CAGG(1, 256, 1024, 2048);
        PGGC_CAGG(2, 256, 2048, 4096);
        PGGC_CAGG(3, 512, 4096, 8192);
        PGGC_CAGG(4, 1024, 8192, 9600);
    });
#undef PGGC_CAGG
    c.kt_end(tk, 0.0);
    PGGC_LAUNCH_CHECK();
    const int wb = g.wk == W_UNIT ? 0 : g.wk == W_I32 ? 4 : 8;
    contract_bytes(c, tk, list.p, st[C_BIG], mstart, bound, ccnt, wb);
    const i64 n2 = st[C_BIG + 1] - st[C_BIG];
    const i32* big = list.p + st[C_BIG];
    if (n2 > 0) {
        Buf<i64> goff(c, n2 + 1), items(c, n2 + 1), items2(c, n2 + 1), mdp(c, n + 1);
        k_goff_sizes<<<grid_items(n2, 256), 256, 0, c.stream>>>(big, n2, bound, nc, goff);
        PGGC_LAUNCH_CHECK();
        scan_i64(c, goff, goff, n2);
        k_member_degs<<<grid_items(n, 256), 256, 0, c.stream>>>(members, g.rp, n, mdp);
        PGGC_LAUNCH_CHECK();
        scan_i64(c, mdp, mdp, n);
        k_items<<<grid_items(n2, 256), 256, 0, c.stream>>>(big, n2, bound, goff, nc, 0, items);
        PGGC_LAUNCH_CHECK();
        scan_i64(c, items, items, n2);
        k_items<<<grid_items(n2, 256), 256, 0, c.stream>>>(big, n2, bound, goff, nc, 1, items2);
        PGGC_LAUNCH_CHECK();
        scan_i64(c, items2, items2, n2);
        // rows in batches whose tables hold at most c.contract_batch slots
        // together (a larger row is a batch of its own), so the tables'
        // memory stays bounded on graphs of billions of edges
        const i64 slot_cap = std::max<i64>(c.contract_batch, 1);
        std::vector<i64> hg, hi, hi2;
        const Fetch f[3] = {fetch(hg, goff.p, n2 + 1), fetch(hi, items.p, n2 + 1), fetch(hi2, items2.p, n2 + 1)};
        copy_d2h(c, f, 3);
        Buf<i32> row(c, std::max<i64>(hi[n2], 1));
        k_item_rows<<<grid_blocks(n2), 256, 0, c.stream>>>(items, n2, row);
        PGGC_LAUNCH_CHECK();
        i64 gmax = 0;
        const std::vector<i64> cuts = batch_cuts(hg, slot_cap, &gmax);
        Buf<i32> gkeys(c, packed ? 1 : gmax);
        Buf<i64> gvals(c, packed ? 1 : gmax);
        Buf<u64> gtab(c, packed ? gmax : 1);
        u64* gt = packed ? gtab.p : nullptr;
        c.mem_note("contract: big-row tables");
        tk = c.kt_begin(KS_CONTRACT_BIG);
        for (size_t q = 0; q + 1 < cuts.size(); q++) {
            const i64 r0 = cuts[q], r1 = cuts[q + 1], gsb = hg[r1] - hg[r0];
            if (packed) {
                fill_i64(c, (i64*)gtab.p, gsb, (i64)PEMPTY);
            } else {
                fill_i32(c, gkeys, gsb, EMPTY_KEY);
                fill_i64(c, gvals, gsb, 0);
            }
            const i64 I = hi[r1] - hi[r0];
            if (I > 0) {
                PGGC_WDISPATCH(g, (k_cbig_insert<AT><<<grid_blocks(I), 256, 0, c.stream>>>(
                                      g.rp, g.col, W, vcmap, members, mstart, mdp, big + r0, r0, r1 - r0, row,
                                      items.p + r0, goff.p + r0, gkeys, gvals, gt)));
                PGGC_LAUNCH_CHECK();
            }
            const i64 I2 = hi2[r1] - hi2[r0];
            if (I2 > 0) {
                k_cbig_extract<<<grid_blocks(I2), 256, 0, c.stream>>>(big + r0, r1 - r0, items2.p + r0, goff.p + r0,
                                                                      gkeys, gvals, gt, toff, tcol, tw.p, ccnt);
                PGGC_LAUNCH_CHECK();
            }
        }
        c.kt_end(tk, 0.0);
        contract_bytes(c, tk, big, n2, mstart, bound, ccnt, wb);
    }
    out.n = nc;
    // (a coarse graph's weights sum to at most the finer level's)
    out.wsmall = sizeof(TT) == 4;
    out.rp = Buf<i64>(c, nc + 1);
    scan_i64(c, ccnt, out.rp, nc);
    out.nnz = c.read1(out.rp.p + nc);
    i32* ocol;
    OT* owt;
    if (to) {
        if (out.nnz > to->cap) return;
        ocol = to->col;
        owt = (OT*)(void*)to->w;  // (OT is i64)
    } else {
        out.col = Buf<i32>(c, std::max<i64>(out.nnz, 1));
        ow = Buf<OT>(c, std::max<i64>(out.nnz, 1));
        ocol = out.col;
        owt = ow;
    }
    if (out.nnz > 0) {
        // algorithmic bytes: coarse offsets, row starts in the temporary rows,
        // (column, weight) read and written once
        const double bytes = 16.0 * (nc + 1) + (8.0 + sizeof(TT) + sizeof(OT)) * out.nnz;
        const int tkc = c.kt_begin(KS_CONTRACT_COPY);
        k_crow_copy<<<(int)ceil_div(out.nnz, EC), EB, 0, c.stream>>>(out.rp, nc, out.nnz, toff, tcol, tw.p, ocol,
                                                                   owt);
        c.kt_end(tkc, bytes);
        PGGC_LAUNCH_CHECK();
    }
    tcol.reset();  // the staged rows are copied out
    tw.reset();
    if (n2 > 0) {
        // the rows merged in HBM tables come out unsorted: sort each by
        // column, in batches of at most c.contract_batch / 4 entries (a
        // larger row is a batch of its own)
        const i64 sort_cap = std::max<i64>(c.contract_batch / 4, 1);
        Buf<i64> boff(c, n2 + 1);
        k_big_count<<<grid_items(n2, 256), 256, 0, c.stream>>>(big, n2, out.rp, boff);
        PGGC_LAUNCH_CHECK();
        scan_i64(c, boff, boff, n2);
        std::vector<i64> hb;
        const Fetch f = fetch(hb, boff.p, n2 + 1);
        copy_d2h(c, &f, 1);
        i64 emax = 0;
        const std::vector<i64> cuts = batch_cuts(hb, sort_cap, &emax);
        if (emax > 0) {
            Buf<u64> key(c, emax);
            Buf<OT> val(c, emax);
            Buf<i64> target(c, emax);
            const int cb = bits_for(nc - 1);
            for (size_t q = 0; q + 1 < cuts.size(); q++) {
                const i64 r0 = cuts[q], r1 = cuts[q + 1], E = hb[r1] - hb[r0];
                if (E == 0) continue;
                k_big_flatten<<<grid_blocks(r1 - r0), 256, 0, c.stream>>>(big + r0, r1 - r0, out.rp, boff.p + r0,
                                                                          ocol, owt, cb, key, val.p, target);
                PGGC_LAUNCH_CHECK();
                radix_sort_pairs(c, key, val.p, E, cb + bits_for(r1 - r0));
                k_big_scatter<<<grid_for(E, 256 * 4, 8192), 256, 0, c.stream>>>(key, target, E, val.p, cb, ocol,
                                                                                owt);
                PGGC_LAUNCH_CHECK();
            }
        }
    }
}

void know_max_weight(Ctx& c, DGraph& g) {
    if (g.wk != W_UNIT && g.nnz > 0 && g.wmax == 0) g.wmax = max_weight(c, g);
}

void contract(Ctx& c, const DGraph& g, const i32* vcmap, i64 nc, OwnedGraph& out, const ContractTo* to) {
    DGraph f = g;
    if (nc <= 1) f.wsmall = true;  // no coarse edges
    if (!f.wsmall) know_max_weight(c, f);
    const ContractWidths w = contract_widths(f.nnz, f.wk == W_UNIT ? 1 : f.wmax, f.wsmall);
    if (w.small && !to) {
        contract_t<u32, i32>(c, g, vcmap, nc, true, out, out.w32, nullptr);
        return;
    }
    if (w.small) {
        contract_t<u32, i32>(c, g, vcmap, nc, true, out, out.w, to);
        return;
    }
    if (w.sum32) contract_t<u32, i64>(c, g, vcmap, nc, w.packed, out, out.w, to);
    else contract_t<i64, i64>(c, g, vcmap, nc, w.packed, out, out.w, to);
    if (!to) narrow_weights(c, out);
}

}  // namespace pggc
