// Internal degree order of a level for its local mover.
#include "renum.h"

#include "device.h"

namespace pggc {

// Where the copy pays.  Below RN_MIN_NNZ nonzeros the records of all vertices
// fit the caches anyway (weighted pLeiden+ on R-MAT scale 17, levels of 3M
// nonzeros: 51.3 ms with copies, 50.7 without).  Above it the copy pays when few
// vertices take most of the gathers, that is when the first sixteenth of the
// vertices (by degree) holds at least RN_HOT of the edges: R-MAT levels hold
// 73-100% there (scale 24, two passes: 651 ms with copies of the coarse levels,
// 690 without; pLeiden+ on scale 22: 217 and 231 ms; scale 20 to stable: 552 and
// 561 ms), an LFR graph 33% (165 ms with copies, 153 without).
constexpr i64 RN_MIN_NNZ = (i64)1 << 23;
constexpr double RN_HOT = 0.5;

// 8-bit sort key of vertex v: descending degree in steps of an eighth of a
// power of two (one digit pass; the radix sort is stable, so vertices of one
// step keep their order)
__device__ __forceinline__ u32 degree_step(i64 d) {
    if (d < 8) return (u32)d;
    const int l = 63 - __clzll((unsigned long long)d);  // >= 3
    const u32 q = (u32)(l - 2) * 8 + (u32)((d >> (l - 3)) & 7);
    return q < 255 ? q : 255;
}
__global__ void k_renum_keys(const i64* __restrict__ rp, i64 n, u64* __restrict__ key, i32* __restrict__ id) {
    const i64 v = thread_item();
    if (v >= n) return;
    key[v] = (u64)(255 - degree_step(rp[v + 1] - rp[v]));
    id[v] = (i32)v;
}
// out[0] = first x with deg[x] == 0 (deg[n] when none), out[1] = rp[hot]
__global__ void k_renum_shape(const i64* __restrict__ deg, const i64* __restrict__ rp, i64 n, i64 hot, i64* out) {
    if (threadIdx.x != 0) return;
    i64 lo = 0, hi = n;
    while (lo < hi) {
        const i64 mid = (lo + hi) >> 1;
        if (deg[mid] == 0) hi = mid;
        else lo = mid + 1;
    }
    out[0] = lo;
    out[1] = rp[hot];
}

// inv[ids[i']] = i'; deg[i'] = degree of ids[i']; vw' = vw[ids]
__global__ void k_renum_index(const i64* __restrict__ rp, const i32* __restrict__ ids, const i64* __restrict__ vw,
                              i64 n, i32* __restrict__ inv, i64* __restrict__ deg, i64* __restrict__ nvw) {
    const i64 x = thread_item();
    if (x >= n) return;
    const i32 v = ids[x];
    inv[v] = (i32)x;
    deg[x] = rp[v + 1] - rp[v];
    nvw[x] = vw[v];
}

// Row i' of the renumbered graph is row ids[i'] with its columns mapped
// through inv, entries in their original order.  Consecutive lanes copy
// consecutive entries (EPT steps of EB entries per block), so a wave reads and
// writes whole lines but for the gather of inv; the row of an entry is a binary
// search over the chunk's row starts in LDS, as in the contraction's copy, and a
// chunk of more than EC rows searches the row offsets instead.  With 8
// consecutive entries per thread 505M weighted nonzeros took 13.3 ms, now 4.8.
template <class T>
__global__ void __launch_bounds__(EB) k_renum_rows(const i64* __restrict__ rp, const i32* __restrict__ col,
                                                   const T* __restrict__ w, const i64* __restrict__ nrp,
                                                   const i32* __restrict__ ids, const i32* __restrict__ inv, i64 n,
                                                   i64 nnz, i32* __restrict__ ncol, T* __restrict__ nw) {
    __shared__ i32 s_st[EC + 1];
    ChunkRows cr;
    chunk_rows(nrp, n, nnz, cr);
    const i64 nr = cr.rhi - cr.rlo;
    const bool staged = nr <= EC;
    if (staged) {
        for (int i = threadIdx.x; i <= (int)nr; i += EB) {
            const i64 v = nrp[cr.rlo + i] - cr.eb;
            s_st[i] = (i32)(v < 0 ? 0 : (v > EC ? EC : v));
        }
    }
    __syncthreads();
    constexpr int U = 4;  // entries in flight per thread
    int lo = 0;
    for (int k0 = 0; k0 < EPT; k0 += U) {
        i64 j[U], src[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            j[u] = cr.eb + (i64)(k0 + u) * EB + threadIdx.x;
            src[u] = -1;
            if (j[u] >= cr.ee) continue;
            i64 r;
            if (staged) {
                // s_st[lo] <= o < s_st[hi]: s_st[0] = 0 and s_st[nr] >= ee - eb
                const int o = (int)(j[u] - cr.eb);
                int hi = (int)nr;
                while (hi - lo > 1) {
                    const int m = (lo + hi) >> 1;
                    if (s_st[m] <= o) lo = m;
                    else hi = m;
                }
                r = cr.rlo + lo;
            } else {
                r = upper_row(nrp, cr.rlo, cr.rhi, j[u]);
            }
            src[u] = rp[ids[r]] + (j[u] - nrp[r]);
        }
        i32 c[U];
#pragma unroll
        for (int u = 0; u < U; u++) c[u] = src[u] >= 0 ? col[src[u]] : -1;
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (src[u] < 0) continue;
            ncol[j[u]] = inv[c[u]];
            if (w) nw[j[u]] = w[src[u]];
        }
    }
}

__global__ void k_renum_gather(i64 n, const i32* __restrict__ ids, const i32* __restrict__ part,
                               i32* __restrict__ out) {
    const i64 x = thread_item();
    if (x >= n) return;
    out[x] = part[ids[x]];
}
__global__ void k_renum_scatter(i64 n, const i32* __restrict__ ids, const i32* __restrict__ in,
                                i32* __restrict__ part) {
    const i64 x = thread_item();
    if (x >= n) return;
    part[ids[x]] = in[x];
}

bool renum_build(Ctx& c, const DGraph& top, Renum& r, bool force) {
    if (r.built_for(top)) return r.copied;
    const i64 n = top.n, nnz = top.nnz;
    r.key = top.rp;
    r.n = n;
    r.copied = false;
    if (!force && nnz < RN_MIN_NNZ) return false;
    r.plan = LevelPlan();
    r.ord_built = false;
    r.ids = Buf<i32>(c, std::max<i64>(n, 1));
    r.rp = Buf<i64>(c, n + 1);
    r.vw = Buf<i64>(c, std::max<i64>(n, 1));
    r.w32 = Buf<i32>();
    r.w64 = Buf<i64>();
    Buf<i32> inv(c, std::max<i64>(n, 1));
    Buf<i64> deg(c, std::max<i64>(n, 1)), shape(c, 2);
    if (n > 0) {
        Buf<u64> key(c, n);
        k_renum_keys<<<grid_items(n, 256), 256, 0, c.stream>>>(top.rp, n, key, r.ids);
        PGGC_LAUNCH_CHECK();
        radix_sort_pairs(c, key, r.ids, n, 8);
        k_renum_index<<<grid_items(n, 256), 256, 0, c.stream>>>(top.rp, r.ids, top.vw, n, inv, deg, r.vw);
        PGGC_LAUNCH_CHECK();
    }
    scan_i64(c, deg, r.rp, n);
    const i64 hot = n / 16;
    k_renum_shape<<<1, 64, 0, c.stream>>>(deg, r.rp, n, hot, shape);
    PGGC_LAUNCH_CHECK();
    const i64* h = c.read(shape, 2);
    r.ncore = h[0];
    if (!force && (double)h[1] < RN_HOT * (double)nnz) {
        r.ids.reset();
        r.rp.reset();
        r.vw.reset();
        return false;
    }
    r.copied = true;
    r.part = Buf<i32>(c, std::max<i64>(n, 1));
    r.col = Buf<i32>(c, std::max<i64>(nnz, 1));
    DGraph g;
    g.n = n;
    g.nnz = nnz;
    g.rp = r.rp;
    g.col = r.col;
    g.wk = top.wk;
    g.vw = r.vw;
    g.wsmall = top.wsmall;
    g.wmax = top.wmax;
    if (nnz > 0) {
        const int grid = (int)ceil_div(nnz, EC);
        if (top.wk == W_I32) {
            r.w32 = Buf<i32>(c, nnz);
            k_renum_rows<i32><<<grid, EB, 0, c.stream>>>(top.rp, top.col, (const i32*)top.w, r.rp, r.ids, inv, n,
                                                          nnz, r.col, r.w32);
            g.w = r.w32.p;
        } else if (top.wk == W_I64) {
            r.w64 = Buf<i64>(c, nnz);
            k_renum_rows<i64><<<grid, EB, 0, c.stream>>>(top.rp, top.col, (const i64*)top.w, r.rp, r.ids, inv, n,
                                                          nnz, r.col, r.w64);
            g.w = r.w64.p;
        } else {
            k_renum_rows<i32><<<grid, EB, 0, c.stream>>>(top.rp, top.col, nullptr, r.rp, r.ids, inv, n, nnz, r.col,
                                                          nullptr);
        }
        PGGC_LAUNCH_CHECK();
    }
    r.g = g;
    return true;
}

// Whether every vertex without neighbours is inert: alone (among vertices of
// nonzero weight) in a cluster that no vertex with neighbours belongs to, so
// its gain stays that of staying (its p_conn is 0) and nobody joins it.
__global__ void k_mark_core(i64 ncore, const i32* __restrict__ part, i32* __restrict__ used) {
    const i64 x = thread_item();
    if (x >= ncore) return;
    used[part[x]] = 1;
}
__global__ void __launch_bounds__(256) k_check_isolated(i64 ncore, i64 n, const i32* __restrict__ part,
                                                        const i32* __restrict__ used, const i64* __restrict__ vol,
                                                        const i64* __restrict__ vw, i64* bad) {
    const i64 x = ncore + thread_item();
    if (x >= n) return;
    const i32 p = part[x];
    if (used[p] || vol[p] != vw[x]) *bad = 1;
}
static bool isolated_inert(Ctx& c, MoveScratch& s, const Renum& r, const RefineData& best) {
    if (r.ncore == r.n) return true;
    s.ensure(c, std::max<i64>(r.n, best.label_count));
    Buf<i64> bad(c, 1);
    fill_i64(c, bad, 1, 0);
    fill_i32(c, s.flag, best.label_count, 0);
    if (r.ncore > 0) k_mark_core<<<grid_items(r.ncore, 256), 256, 0, c.stream>>>(r.ncore, r.part, s.flag);
    k_check_isolated<<<grid_items(r.n - r.ncore, 256), 256, 0, c.stream>>>(r.ncore, r.n, r.part, s.flag, best.vol,
                                                                           r.vw, bad);
    PGGC_LAUNCH_CHECK();
    return c.read1(bad) == 0;
}

void renum_gather(Ctx& c, const Renum& r, const i32* in, i32* out) {
    if (r.n == 0) return;
    k_renum_gather<<<grid_items(r.n, 256), 256, 0, c.stream>>>(r.n, r.ids, in, out);
    PGGC_LAUNCH_CHECK();
}

void local_move_renum(Ctx& c, MoveScratch& s, Renum& r, i32* part, RefineData& best, bool is_initial,
                      bool constrained, i32* cons, bool SA, MoveStats* st) {
    const i64 n = r.n;
    renum_gather(c, r, part, r.part);
    DGraph g = r.g;
    if (isolated_inert(c, s, r, best)) g.n = r.ncore;
    local_move(c, s, r.plan, g, r.part, best, is_initial, constrained, cons, SA, st, r.ids, n);
    if (n > 0) {
        k_renum_scatter<<<grid_items(n, 256), 256, 0, c.stream>>>(n, r.ids, r.part, part);
        PGGC_LAUNCH_CHECK();
    }
}

}  // namespace pggc
