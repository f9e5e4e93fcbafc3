// Local mover: degree-classed neighbour-cluster aggregation with gain argmax,
// the afterburner conflict filter, move application with exact uncut deltas,
// the strict prefix filter, relabelling, and the local_move drivers.
//
// Determinism (shared with the CPU oracle):
//  * destination = max gain, ties -> smallest label; NEW_PART (-4) competes
//    with j_conn 0 when p_conn < 0 (team-path rule, src/local_mover.cpp:553-561)
//  * afterburner FP32 sums: degree < 128 sequential in adjacency order,
//    128..14999 64 strided partials + halving tree, >= 15000 1024 strided
//    partials + halving tree
//  * uncut is updated by the exact integer delta of the moved vertices
#include <algorithm>
#include <cfloat>
#include <cstdio>
#include <chrono>
#include <type_traits>

#include "batching.h"
#include "device.h"
#include "gnn.h"
#include "hash.h"
#include "localmove.h"
#include "select.h"

namespace pggc {

// ------------------------------------------------------------- objective
double objective_value(i64 uncut, double lambda, u64 sq_hi, u64 sq_lo) {
    unsigned __int128 sq = ((unsigned __int128)sq_hi << 64) | (unsigned __int128)sq_lo;
    double m = (double)uncut;
    m -= lambda * (double)sq;
    return m;
}

void update_objective(Ctx& c, RefineData& rd) {
    Buf<i64> sq(c, 2);
    sum_sq_u128(c, rd.vol, rd.label_count, sq);
    const i64* h = c.read(sq, 2);
    rd.obj = objective_value(rd.uncut, rd.lambda, (u64)h[0], (u64)h[1]);
}

// ------------------------------------------------------------- scratch
// Scalars of a sweep in MoveScratch::scal, zero at the start of a call and
// between sweeps: SC_EXTRA the two words of select_items, SC_NEW the movers that
// need a new cluster (direct sweeps), SC_TICKET k_finish's blocks (at most
// FIN_BLOCKS), then MV_SLOTS words each over which the uncut change, and in
// direct sweeps the movers and the candidates, are summed.
constexpr int SC_EXTRA = 0, SC_NEW = 2, SC_TICKET = 4, MV_SLOTS = 64, SC_SLOTS = 16, SC_KM = SC_SLOTS + MV_SLOTS,
              SC_CAND = SC_KM + MV_SLOTS, SC_COUNT = SC_CAND + MV_SLOTS;
constexpr int FIN_BLOCKS = 256;
void MoveScratch::ensure(Ctx& c, i64 n) {
    if (cap >= n) return;
    cap = std::max<i64>(n, 1);
    part = Buf<i32>(c, cap);
    dest = Buf<i32>(c, cap);
    cand = Buf<i32>(c, cap);
    moves = Buf<i32>(c, cap);
    flag = Buf<i32>(c, cap);
    tmp = Buf<i32>(c, cap);
    tmp2 = Buf<i32>(c, cap + 1);
    gain = Buf<float>(c, cap);
    abi = Buf<AbInfo>(c, cap);
    mvp = Buf<u64>(c, cap);
    rec = Buf<u64>(c, cap);
    rec16.reset();
    prio = Buf<i64>(c, cap + 1);
    scal = Buf<i64>(c, SC_COUNT);
    sqpart = Buf<u64>(c, 2 * FIN_BLOCKS);
}

// ------------------------------------------------------------- level plan
__host__ __device__ __forceinline__ int score_class(i64 d) {
    return d <= 4 ? 0 : d <= 8 ? 1 : d <= 16 ? 2 : d <= 32 ? 3 : d <= 64 ? 4 : d <= 128 ? 5 : d <= 256 ? 6
         : d <= 512 ? 7 : d <= 1024 ? 8 : d <= 2048 ? 9 : 10;
}
// small levels, bound by launches (direct_sweep)
constexpr i64 DIRECT_MAX = (i64)1 << 18, DIRECT_NNZ = (i64)1 << 22;
// Level of at most this many rows of degree 65 to 2048: one launch for their
// five classes (its 256-thread blocks take 33 KB of LDS each with 32-bit sums, so a
// CU holds 4 of them and the chip 1,024 at once; a class of its own takes 5 to 9
// us of a launch's latency however few its rows).
// At 2,048 rows, and only without longer ones, a CPM run of 30,011 vertices took 2.94
// ms, 2.70 now, weighted pLeiden+ on R-MAT scale 17 28.7, 27.3 now; at the 12,000 to
// 200,000 rows of R-MAT scale 22's levels the classes' own widths are better.
constexpr i64 TABLE_ONE_LAUNCH = 8192;
// LDS table of a vertex of degree d: the power of two >= spe * d slots, at most
// `most`
__host__ __device__ __forceinline__ int tslots(i64 d, int spe, int most) {
    int s = 2;
    while (s < spe * d) s <<= 1;
    return s < most ? s : most;
}
// Vertices of the hub class scored from one LDS table each: degree at most
// HUB_HALF from 8,192 slots (two blocks per CU with 32-bit sums), at most
// HUB_LDS_BOUND from 10,112 slots, which is the most that still lets two
// 1,024-thread blocks share a CU's LDS (at most 81% full)
constexpr i64 HUB_HALF = 4096, HUB_LDS_BOUND = 8192;
constexpr int HUB_LDS_SLOTS = 10112;
// Larger hubs (k_hub_score): slots of the LDS table of one slice, 12 bytes each
// with 32-bit sums, 16 with 64-bit ones (144 and 128 KB of LDS), and the
// slices of a hub: 1.5 slots per edge, so a slice is at most 2/3 full on average
constexpr int HUB_SLOTS32 = 12288, HUB_SLOTS64 = 8192;
__host__ __device__ __forceinline__ i64 hub_slices(i64 d, int slots) { return (3 * d + 2 * slots - 1) / (2 * slots); }
// Their edges are gathered in chunks of HUB_E, merged in an LDS table of HUB_GS
// slots (2/3 full at most; two blocks per CU with 32-bit sums) and left grouped
// by bucket: a slice, or several slices of a hub that has more than HUB_BUCKETS
constexpr int HUB_E = 4096, HUB_GS = 6144, HUB_BUCKETS = 1024;
__host__ __device__ __forceinline__ i64 hub_chunks(i64 d) { return (d + HUB_E - 1) / HUB_E; }
__host__ __device__ __forceinline__ i64 hub_per(i64 ns) { return (ns + HUB_BUCKETS - 1) / HUB_BUCKETS; }
__host__ __device__ __forceinline__ i64 hub_nb(i64 ns) { return (ns + hub_per(ns) - 1) / hub_per(ns); }

// Both partitions of a plan in one pass each of counting and writing: the
// order1 classes (src/header/ordering.h:17-19; ORD_CLS) and the scoring classes,
// each stable by id.  Classes 0 .. ORD_CLS - 1 are the former, the others the
// latter; counts[class * nb + tile].  Consecutive lanes take consecutive
// vertices, and a vertex's place within its tile is the count of its class in
// the (step, wave) runs before its own plus its rank among the lanes of its
// class, found with a ballot per class bit.  As two partitions of three and
// four kernels each over class arrays, 8 consecutive vertices per thread and a
// block scan per class, a plan took 16 launches and 3 waits, now 3 and 1.
constexpr int ORD_CLS = 3, PL_CLS = ORD_CLS + NCLS, PL_T = 256, PL_I = 8, PL_TILE = PL_T * PL_I, PL_W = PL_T / 64;
__global__ void __launch_bounds__(PL_T) k_plan_count(const i64* __restrict__ rp, i64 n, i64 nb, i64* counts) {
    __shared__ int cnt[PL_CLS];
    const i64 b = block_id();
    if (b >= nb) return;
    if (threadIdx.x < PL_CLS) cnt[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PL_I; k++) {
        const i64 i = b * PL_TILE + k * PL_T + threadIdx.x;
        if (i < n) {
            const i64 d = rp[i + 1] - rp[i];
            atomicAdd(&cnt[order_class(d)], 1);
            atomicAdd(&cnt[ORD_CLS + score_class(d)], 1);
        }
    }
    __syncthreads();
    if (threadIdx.x < PL_CLS) counts[(i64)threadIdx.x * nb + b] = cnt[threadIdx.x];
}
// offs: exclusive scan of counts; host[0..PL_CLS] = class starts (the scoring
// classes' from n on)
__global__ void __launch_bounds__(PL_T) k_plan_write(const i64* __restrict__ rp, i64 n, i64 nb,
                                                     const i64* __restrict__ offs, i32* __restrict__ o1,
                                                     i32* __restrict__ list, i64* host) {
    __shared__ int cnt[PL_I * PL_W][PL_CLS];  // class counts of the runs, then their prefix
    const i64 b = block_id();
    if (b >= nb) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int q = threadIdx.x; q < PL_I * PL_W * PL_CLS; q += PL_T) cnt[q / PL_CLS][q % PL_CLS] = 0;
    __syncthreads();
    int c1[PL_I], c2[PL_I], r1[PL_I], r2[PL_I];
    const u64 below = ((u64)1 << lane) - 1;
#pragma unroll
    for (int k = 0; k < PL_I; k++) {
        const i64 i = b * PL_TILE + k * PL_T + threadIdx.x;
        const bool in = i < n;
        const i64 d = in ? rp[i + 1] - rp[i] : 0;
        c1[k] = in ? order_class(d) : 15;
        c2[k] = in ? score_class(d) : 15;
        const u64 m1 = same_class(c1[k]), m2 = same_class(c2[k]);
        r1[k] = __popcll(m1 & below);
        r2[k] = __popcll(m2 & below);
        if (in && r1[k] == 0) cnt[k * PL_W + wv][c1[k]] = __popcll(m1);
        if (in && r2[k] == 0) cnt[k * PL_W + wv][ORD_CLS + c2[k]] = __popcll(m2);
    }
    __syncthreads();
    if (threadIdx.x < PL_CLS) {
        int run = 0;
        for (int q = 0; q < PL_I * PL_W; q++) {
            const int v = cnt[q][threadIdx.x];
            cnt[q][threadIdx.x] = run;
            run += v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PL_I; k++) {
        const i64 i = b * PL_TILE + k * PL_T + threadIdx.x;
        if (i >= n) continue;
        o1[offs[(i64)c1[k] * nb + b] + cnt[k * PL_W + wv][c1[k]] + r1[k]] = (i32)i;
        list[offs[(i64)(ORD_CLS + c2[k]) * nb + b] - n + cnt[k * PL_W + wv][ORD_CLS + c2[k]] + r2[k]] = (i32)i;
    }
    if (b == 0 && threadIdx.x <= PL_CLS) host[threadIdx.x] = offs[(i64)threadIdx.x * nb];
}

// Work of the large hubs: groups of NXCD consecutive hubs (sorted by degree, so
// of similar size), each hub with as many blocks as the group's largest hub
// has slices.  Block ids go round-robin over the XCDs, so with the blocks of a
// group interleaved all slices of one hub run on one XCD and read the hub's
// edges and records through its L2.
constexpr int NXCD = 8;
// sizes whose exclusive scan is LevelPlan::hub_pre: per hub its edges, its
// chunks and the bucket starts of its chunks, and the slices per group of hubs
__global__ void k_hub_sizes(const i64* rp, const i32* hubs, i64 m, int slots, i64* sz) {
    const i64 x = thread_item();
    const i64 ng = (m + NXCD - 1) / NXCD;
    if (x < m) {
        const i64 d = rp[hubs[x] + 1] - rp[hubs[x]];
        sz[x] = d;
        sz[m + x] = hub_chunks(d);
        sz[2 * m + x] = hub_chunks(d) * (hub_nb(hub_slices(d, slots)) + 1);
    }
    if (x < ng) {
        const i64 last = (x + 1) * NXCD < m ? (x + 1) * NXCD - 1 : m - 1;
        const i32 i = hubs[last];
        sz[3 * m + x] = hub_slices(rp[i + 1] - rp[i], slots);
    }
}
// A batch of m hubs: its rows of the scanned sizes, each relative to the batch's
// first entry.
struct HubView {
    const i32* hubs;
    const i64 *edges, *chunks, *starts, *groups;
    i64 m, ng, nblk;
    __device__ __forceinline__ i64 edge0(i64 h) const { return edges[h] - edges[0]; }
    __device__ __forceinline__ i64 chunk0(i64 h) const { return chunks[h] - chunks[0]; }
    __device__ __forceinline__ i64 start0(i64 h) const { return starts[h] - starts[0]; }
    // block -> hub and slice; false for padding.  The largest hubs come first.
    __device__ __forceinline__ bool slice(i64 bid, i64& h, i64& sl) const {
        if (bid >= nblk) return false;
        const i64 b = nblk - 1 - bid;
        const i64 q = b / NXCD + groups[0];
        const i64 g = upper_row(groups, 0, ng, q);
        h = g * NXCD + b % NXCD;
        sl = q - groups[g];
        return h < m;
    }
};
// the hubs [h0, h1) of a level's, h0 a multiple of NXCD
static HubView hub_view(const LevelPlan& p, i64 h0, i64 h1, i64 blocks) {
    const i64* pre = p.hub_pre.p + h0;
    return HubView{p.sc_list.p + p.hub0 + h0, pre, pre + p.nhub, pre + 2 * p.nhub,
                   p.hub_pre.p + 3 * p.nhub + h0 / NXCD, h1 - h0, ceil_div(h1 - h0, NXCD), blocks};
}
// Batches of hubs hold at most this share of the device's memory (a larger group
// of hubs is a batch of its own): scratch for all hub edges at once, up to 20 GB
// on R-MAT scale 27, made the allocator give blocks back and take them again, and
// a pLeiden+ pass took 21.4 s, with batches 18.2.
constexpr double HUB_MEM = 1.0 / 64;
static size_t hub_scratch(const LevelPlan::HubBatch& b, bool sum32) {
    return (size_t)(b.edges + (sum32 ? ceil_div(b.edges, 2) : b.edges) + ceil_div(b.starts, 4));
}

__global__ void k_hub_deg_keys(const i64* rp, const i32* list, i64 m, u64* keys, i32* vals) {
    const i64 x = thread_item();
    if (x >= m) return;
    const i32 i = list[x];
    keys[x] = (u64)(rp[i + 1] - rp[i]);
    vals[x] = i;
}
// of a list sorted by degree: out[0] and out[1] = first x with degree(list[x]) >
// HUB_HALF and HUB_LDS_BOUND, out[2] = the largest degree
__global__ void k_hub_shape(const i64* rp, const i32* list, i64 m, i64* out) {
    if (threadIdx.x >= 2) return;
    const i64 bound = threadIdx.x == 0 ? HUB_HALF : HUB_LDS_BOUND;
    i64 lo = 0, hi = m;
    while (lo < hi) {
        const i64 mid = (lo + hi) >> 1;
        const i32 i = list[mid];
        if (rp[i + 1] - rp[i] > bound) hi = mid;
        else lo = mid + 1;
    }
    out[threadIdx.x] = lo;
    out[2] = rp[list[m - 1] + 1] - rp[list[m - 1]];
}

void plan_level(Ctx& c, const DGraph& g, LevelPlan& p) {
    if (p.key == (const void*)g.rp && p.n == g.n) return;
    p.key = g.rp;
    p.n = g.n;
    {
        const int tk = c.kt_begin(KS_ORDER);
        const i64 n = g.n, nb = ceil_div(std::max<i64>(n, 1), PL_TILE);
        if (p.ord.o1.n < (size_t)n) p.ord.o1 = Buf<i32>(c, std::max<i64>(n, 1));
        p.sc_list = Buf<i32>(c, std::max<i64>(n, 1));
        Buf<i64> counts(c, PL_CLS * nb + 1);
        k_plan_count<<<grid_blocks(nb), PL_T, 0, c.stream>>>(g.rp, n, nb, counts);
        PGGC_LAUNCH_CHECK();
        scan_i64(c, counts, counts, PL_CLS * nb);
        k_plan_write<<<grid_blocks(nb), PL_T, 0, c.stream>>>(g.rp, n, nb, counts, p.ord.o1, p.sc_list,
                                                             c.pinned_dev);
        PGGC_LAUNCH_CHECK();
        // row bounds read twice, ids written twice
        c.kt_end(tk, 16.0 * (n + 1) + 8.0 * n);
        c.sync();
        p.ord.off_large = c.pinned[1];
        p.ord.off_large2 = c.pinned[2];
        for (int k = 0; k <= NCLS; k++) p.sc_start[k] = c.pinned[ORD_CLS + k] - n;
    }
    // hub class by degree (stable: ties by id), so that the hubs scored in
    // LDS form a prefix; every hub is scored on its own, so the order within
    // the class does not change results
    const i64 nh = p.sc_start[CL_HUB + 1] - p.sc_start[CL_HUB];
    p.nlds = p.nhalf = 0;
    p.max_deg = 0;
    if (nh > 0) {
        i32* hl = p.sc_list.p + p.sc_start[CL_HUB];
        Buf<u64> hk(c, nh);
        Buf<i64> f(c, 3);
        k_hub_deg_keys<<<grid_items(nh, 256), 256, 0, c.stream>>>(g.rp, hl, nh, hk, hl);
        PGGC_LAUNCH_CHECK();
        radix_sort_pairs(c, hk, hl, nh, 40);
        k_hub_shape<<<1, 64, 0, c.stream>>>(g.rp, hl, nh, f);
        PGGC_LAUNCH_CHECK();
        const i64* h = c.read(f, 3);
        p.nhalf = h[0];
        p.nlds = h[1];
        p.max_deg = h[2];
    }
    // 32-bit sums for the rows scored in registers and LDS (degree at most
    // HUB_LDS_BOUND) and for the larger hubs: unit weights, a level whose
    // weights sum to less than 2^32 (contracted from a unit-weight graph), or
    // weights small enough for the degrees
    p.agg32 = p.hub32 = g.wk == W_UNIT || g.wsmall;
    if (!p.agg32 && g.nnz > 0) {
        const u64 mx = g.wmax ? g.wmax : max_weight(c, g);
        p.agg32 = mx <= 0xffffffffull / HUB_LDS_BOUND;
        p.hub32 = mx <= 0xffffffffull / (u64)std::max(p.max_deg, HUB_LDS_BOUND);
    }
    p.hub0 = p.sc_start[CL_HUB] + p.nlds;
    p.nhub = nh - p.nlds;
    p.hub_blocks = 0;
    if (p.nhub > 0) {
        const i64 m = p.nhub, ng = ceil_div(m, NXCD), np = 3 * m + ng;
        p.hub_pre = Buf<i64>(c, np + 1);
        p.hub_pv = Buf<i64>(c, m);
        p.hub_best = Buf<u64>(c, m);
        k_hub_sizes<<<grid_items(m, 256), 256, 0, c.stream>>>(g.rp, p.sc_list.p + p.hub0, m,
                                                              p.hub32 ? HUB_SLOTS32 : HUB_SLOTS64, p.hub_pre);
        PGGC_LAUNCH_CHECK();
        scan_i64(c, p.hub_pre, p.hub_pre, np);
        fill_i64(c, (i64*)p.hub_best.p, m, 0);  // zero between sweeps (k_hub_decide)
        fill_i64(c, p.hub_pv, m, 0);
        i64 e[4];
        const i64 at[4] = {m, 2 * m, 3 * m, np};
        Fetch f[4];
        for (int k = 0; k < 4; k++) f[k] = Fetch{&e[k], p.hub_pre.p + at[k], sizeof(i64)};
        copy_d2h(c, f, 4);
        p.hub_blocks = (e[3] - e[2]) * NXCD;
        p.hub_batches.assign(1, LevelPlan::HubBatch{0, m, e[0], e[1] - e[0], e[2] - e[1], p.hub_blocks});
        const i64 cap = std::min<i64>(c.contract_batch, (i64)(HUB_MEM * (double)c.mem_total) / (p.hub32 ? 12 : 16));
        if (e[0] > cap) {
            std::vector<i64> pre, ge(ng + 1);
            const Fetch all = fetch(pre, p.hub_pre.p, (size_t)np + 1);
            copy_d2h(c, &all, 1);
            for (i64 k = 0; k <= ng; k++) ge[k] = pre[std::min(k * NXCD, m)];
            const std::vector<i64> cuts = batch_cuts(ge, cap, nullptr);
            p.hub_batches.clear();
            for (size_t q = 0; q + 1 < cuts.size(); q++) {
                const i64 h0 = cuts[q] * NXCD, h1 = std::min(cuts[q + 1] * NXCD, m);
                p.hub_batches.push_back({h0, h1, pre[h1] - pre[h0], pre[m + h1] - pre[m + h0],
                                         pre[2 * m + h1] - pre[2 * m + h0],
                                         (pre[3 * m + cuts[q + 1]] - pre[3 * m + cuts[q]]) * NXCD});
            }
        }
        p.hub_words = 0;
        for (const LevelPlan::HubBatch& b : p.hub_batches) p.hub_words = std::max(p.hub_words, hub_scratch(b, p.hub32));
    }
}

// a mover's word in MoveScratch::mvp
__device__ __forceinline__ u64 mvp_moved(i32 from, i32 to) {
    return (u64)((u32)from | 0x80000000u) | ((u64)(u32)to << 32);
}

// ------------------------------------------------------------- scoring
__device__ __forceinline__ u64 pack_cand(float jc, i32 key) {
    return ((u64)ord_f32(jc) << 32) | (u64)(0xFFFFFFFFu - (u32)(key + 4));
}

// What scoring writes per scored vertex: the cached destination, the gain
// (when some caller reads the array) and the afterburner's record.  A vertex
// that is not scored keeps its record: it is NO_MOVE, and its cluster cannot
// have changed since that was decided.
struct ScoreOut {
    i32* dest;
    float* gain;   // nullable
    AbInfo* info;  // nullable: k_ab_pack builds the records from the arrays
};

__device__ __forceinline__ void decide(i32 i, float p_conn, u64 bk, i32 p, i64 wv, const ScoreOut& o) {
    bool have = bk != 0;
    float bj = have ? unord_f32((u32)(bk >> 32)) : 0.0f;
    i32 bc = have ? (i32)(0xFFFFFFFFu - (u32)(bk & 0xffffffffull)) - 4 : 0;
    AbInfo a;
    a.part = p;
    a.vwf = (float)wv;
    if (p_conn < 0.0f && (!have || !(bj > 0.0f))) {
        a.gain = 0.0f - p_conn;
        a.dest = NEW_PART;
    } else if (have) {
        a.gain = bj - p_conn;
        a.dest = bc;
    } else {
        a.gain = -FLT_MAX;
        a.dest = NO_MOVE;
    }
    o.dest[i] = a.dest;
    if (o.gain) o.gain[i] = a.gain;
    if (o.info) o.info[i] = a;
}

// lambda of a vertex's objective and the sweep's filter ratio: one value
// each for a single graph, per-vertex tables for a batch of graphs held as
// one disjoint union (each vertex carries its instance's values), whose
// instances can be at different sweeps of their ratio schedules.  The batch
// tables are filled per sweep by k_vertex_lam rather than looked up as
// lam[inst[v]] inside the scoring kernels: that two-step lookup there gave
// wrong values in about 1% of the lanes on gfx950, run to run different,
// while the same lookup in its own kernel and the per-vertex tables were
// exact.
struct LamOne {
    float v;
    __device__ __forceinline__ float operator()(i64) const { return v; }
    __device__ __forceinline__ float rt(i64, float r) const { return r; }
};
struct LamVert {
    const float* lam;    // lambda of vertex i's instance
    const float* ratio;  // filter ratio of vertex i's instance this sweep
    __device__ __forceinline__ float operator()(i64 i) const { return lam[i]; }
    __device__ __forceinline__ float rt(i64 i, float) const { return ratio[i]; }
};
// afterburner priority hash of a vertex (src/local_mover.cpp:319): xorshift32
// of its id, or of its id within its instance for a batch held as one union
// (loc[v] = v - first vertex of v's instance)
struct PrioOne {
    __device__ __forceinline__ i32 operator()(i32 v) const { return (i32)xorshift32((u32)v); }
};
struct PrioInst {
    const i32* loc;
    __device__ __forceinline__ i32 operator()(i32 v) const { return (i32)xorshift32((u32)loc[v]); }
};

// p_conn and the filter threshold (src/local_mover.cpp:481-487)
__device__ __forceinline__ void own_terms(i64 pv, i64 volp, i64 wv, float lam, float ratio, float& multi,
                                          float& p_conn, float& b) {
    multi = (float)wv * lam;
    p_conn = fmaf(-(float)(volp - wv), multi, (float)pv);
    b = (float)((double)p_conn * (1.0 - (double)ratio));
    if (p_conn < 0.0f) b = 0.0f;
}

// What scoring reads of a neighbour, packed per vertex once per sweep
// (k_rec_pack): its cluster and that cluster's volume as the fp32 value the
// gain arithmetic uses, in 8 bytes; with a constraint also the cluster's
// constraint value, in 16.  The gathers at random neighbour ids bound the
// scoring kernels, so an edge costs one of them instead of one for the cluster
// and another, at a random label, for each distinct cluster's volume (and a
// third for its constraint).
struct RecView {
    const u64* r8;
    const uint4* r16;  // set (instead of r8) when there is a constraint
};
struct NbRec {
    i32 part;
    float volf;
    i32 cons;
};
__device__ __forceinline__ NbRec load_rec(const RecView& rv, i32 v) {
    NbRec r;
    if (rv.r16) {  // kernel-uniform
        const uint4 q = rv.r16[v];
        r.part = (i32)q.x;
        r.volf = __uint_as_float(q.y);
        r.cons = (i32)q.z;
    } else {
        const u64 q = rv.r8[v];
        r.part = (i32)(u32)q;
        r.volf = __uint_as_float((u32)(q >> 32));
        r.cons = 0;
    }
    return r;
}
__device__ __forceinline__ void rec_pack(i64 i, const i32* part, const i64* vol, const i32* cons, u64* r8,
                                         uint4* r16) {
    const i32 p = part[i];
    const u32 vf = __float_as_uint((float)vol[p]);
    if (r16) {
        r16[i] = make_uint4((u32)p, vf, (u32)cons[p], 0u);
    } else {
        r8[i] = (u64)(u32)p | ((u64)vf << 32);
    }
}
__global__ void __launch_bounds__(256) k_rec_pack(i64 n, const i32* __restrict__ part, const i64* __restrict__ vol,
                                                  const i32* __restrict__ cons, u64* __restrict__ r8,
                                                  uint4* __restrict__ r16) {
    const i64 i = thread_item();
    if (i < n) rec_pack(i, part, vol, cons, r8, r16);
}

// Lane exchange inside groups of G consecutive lanes.  DPP moves cover 16
// lanes (quad permutes, half-row and row mirrors, row rotations); shuffles
// reach the other 16-lane rows.
template <int CTRL>
__device__ __forceinline__ i32 dpp(i32 v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ u32 dpp(u32 v) {
    return (u32)dpp<CTRL>((i32)v);
}
template <int CTRL>
__device__ __forceinline__ i64 dpp(i64 v) {
    const u32 lo = dpp<CTRL>((u32)(u64)v), hi = dpp<CTRL>((u32)((u64)v >> 32));
    return (i64)(((u64)hi << 32) | lo);
}
template <int CTRL>
__device__ __forceinline__ u64 dpp(u64 v) {
    return (u64)dpp<CTRL>((i64)v);
}
constexpr int DPP_X1 = 0xB1, DPP_X2 = 0x4E, DPP_X3 = 0x1B, DPP_HMIRROR = 0x141, DPP_MIRROR = 0x140;

// reduction over the group with `op` (commutative); every lane gets the result
template <int G, class T, class Op>
__device__ __forceinline__ T group_reduce(T v, Op op) {
    xlane_fence(v);
    v = op(v, dpp<DPP_X1>(v));
    v = op(v, dpp<DPP_X2>(v));
    if (G >= 8) v = op(v, dpp<DPP_HMIRROR>(v));
    if (G >= 16) v = op(v, dpp<DPP_MIRROR>(v));
    if (G >= 32) v = op(v, (T)__shfl_xor(v, 16));
    if (G >= 64) v = op(v, (T)__shfl_xor(v, 32));
    return v;
}
template <int G, class T>
__device__ __forceinline__ T group_max(T v) {
    return group_reduce<G>(v, [](T a, T b) { return a > b ? a : b; });
}
// over the block; every thread gets the result
template <int BS, class T, class Op>
__device__ __forceinline__ T block_reduce(T v, Op op) {
    v = group_reduce<64>(v, op);
    if (BS > 64) {
        __shared__ T sh[BS / 64];
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
        __syncthreads();
        v = sh[0];
#pragma unroll
        for (int w = 1; w < BS / 64; w++) v = op(v, sh[w]);
        __syncthreads();
    }
    return v;
}

// agg += w of the lanes of the 16-lane row (or 4 / 8 lane group) whose key
// equals `key`, given this lane's partner values (kk, ww) of one offset
template <bool UNIT, class AT>
__device__ __forceinline__ void merge_one(i32 kk, AT ww, i32 key, AT& agg) {
    agg += kk == key ? (UNIT ? (AT)1 : ww) : (AT)0;
}
template <bool UNIT, class AT, int C>
__device__ __forceinline__ void merge_dpp(i32 k, AT w, i32 key, AT& agg) {
    merge_one<UNIT>(dpp<C>(k), UNIT ? (AT)0 : dpp<C>(w), key, agg);
}
// rotations 1..15 of a 16-lane row
template <bool UNIT, class AT>
__device__ __forceinline__ void merge_row(i32 k, AT w, i32 key, AT& agg) {
    merge_dpp<UNIT, AT, 0x121>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x122>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x123>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x124>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x125>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x126>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x127>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x128>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x129>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x12A>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x12B>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x12C>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x12D>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x12E>(k, w, key, agg);
    merge_dpp<UNIT, AT, 0x12F>(k, w, key, agg);
}
// sum of the weights of the group's lanes that hold this lane's key
template <int G, bool UNIT, class AT>
__device__ __forceinline__ AT merge_group(i32 key, AT w) {
    xlane_fence(key);
    xlane_fence(w);
    AT agg = w;
    if (G == 4 || G == 8) {
        merge_dpp<UNIT, AT, DPP_X1>(key, w, key, agg);
        merge_dpp<UNIT, AT, DPP_X2>(key, w, key, agg);
        merge_dpp<UNIT, AT, DPP_X3>(key, w, key, agg);
        if (G == 8) {  // the mirrored half row is offset 7, its quad permutes 6, 5, 4
            const i32 k7 = dpp<DPP_HMIRROR>(key);
            const AT w7 = UNIT ? (AT)0 : dpp<DPP_HMIRROR>(w);
            merge_one<UNIT>(k7, w7, key, agg);
            merge_dpp<UNIT, AT, DPP_X1>(k7, w7, key, agg);
            merge_dpp<UNIT, AT, DPP_X2>(k7, w7, key, agg);
            merge_dpp<UNIT, AT, DPP_X3>(k7, w7, key, agg);
        }
        return agg;
    }
    merge_row<UNIT>(key, w, key, agg);
#pragma unroll
    for (int r = 16; r < G; r += 16) {  // the other rows of the group
        const i32 kr = __shfl_xor(key, r);
        const AT wr = UNIT ? (AT)0 : (AT)__shfl_xor(w, r);
        merge_one<UNIT>(kr, wr, key, agg);
        merge_row<UNIT>(kr, wr, key, agg);
    }
    return agg;
}

template <class WT>
struct IsUnit {
    static constexpr bool v = false;
};
template <>
struct IsUnit<WUnit> {
    static constexpr bool v = true;
};

// G lanes per vertex, one edge per lane (degree <= G): duplicate clusters are
// merged in registers.  AT: u32 when every row sum of the level's small
// degrees fits 32 bits (LevelPlan::agg32), else i64; the sums are the same
// integers.  raw rows have distinct columns and no own-cluster edge.  Merging
// by DPP moves in 32 bits instead of three shuffles per partner lane took the
// five classes from 50.4 to 31.5 ms (R-MAT scale 24, two passes), 84 to 33 ms
// on scale 20, where the 64-lane class was instruction bound.
template <int G, class AT, class WT, class LT>
__device__ __forceinline__ void score_group(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                            const i64* __restrict__ vw, const i32* __restrict__ list, i64 x0, i64 x1,
                                            i64 blk, const i32* __restrict__ part, const i64* __restrict__ vol,
                                            const RecView& rv, const i32* __restrict__ cons, int raw, LT lam,
                                            float ratio, const ScoreOut& out) {
    const int gl = threadIdx.x & (G - 1);
    const i64 gi = x0 + blk * (256 / G) + threadIdx.x / G;
    if (gi >= x1) return;
    const i32 i = list[gi];
    if (out.dest[i] == NO_MOVE) return;
    const i64 s = rp[i];
    const int d = (int)(rp[i + 1] - s);
    const i32 p = part[i];
    const i64 wv = vw[i];
    const i32 cp = cons ? cons[p] : 0;
    NbRec r;
    r.part = -5;
    r.volf = 0.0f;
    r.cons = 0;
    AT wt = 0;
    const bool has = gl < d;
    if (has) {
        r = load_rec(rv, col[s + gl]);
        wt = (AT)W(s + gl);
    }
    const i32 key = r.part;
    AT agg = wt;
    bool own = false;
    AT pv = 0;
    if (!raw) {
        agg = merge_group<G, IsUnit<WT>::v>(key, wt);
        own = has && key == p;
        pv = group_max<G>(own ? agg : (AT)0);
    }
    float multi, p_conn, b;
    own_terms((i64)pv, vol[p], wv, lam(i), lam.rt(i, ratio), multi, p_conn, b);
    u64 bk = 0;
    if (has && !own && agg > 0 && (float)agg >= b && r.cons == cp) {
        const float jc = fmaf(-r.volf, multi, (float)agg);
        if (jc >= b) bk = pack_cand(jc, key);
    }
    bk = group_max<G>(bk);
    if (gl == 0) decide(i, p_conn, bk, p, wv, out);
}

// the five group classes in one launch: blocks [blk[q], blk[q + 1]) score the
// list entries [s[q], s[q + 1]) with 4 << q lanes each
struct GroupRanges {
    i64 s[CL_TABLE + 1], blk[CL_TABLE + 1];
};
template <class AT, class WT, class LT>
__global__ void __launch_bounds__(256) k_score_groups(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                      const i64* __restrict__ vw, const i32* __restrict__ list,
                                                      GroupRanges gr, const i32* __restrict__ part,
                                                      const i64* __restrict__ vol, RecView rv,
                                                      const i32* __restrict__ cons, int raw, LT lam, float ratio,
                                                      ScoreOut out) {
    const i64 b = block_id();
#define PGGC_GROUP(q, G)                                                                                              \
    score_group<G, AT>(rp, col, W, vw, list, gr.s[q], gr.s[q + 1], b - gr.blk[q], part, vol, rv, cons, raw, lam, ratio, \
                       out)
    if (b < gr.blk[1]) PGGC_GROUP(0, 4);
    else if (b < gr.blk[2]) PGGC_GROUP(1, 8);
    else if (b < gr.blk[3]) PGGC_GROUP(2, 16);
    else if (b < gr.blk[4]) PGGC_GROUP(3, 32);
    else if (b < gr.blk[5]) PGGC_GROUP(4, 64);
#undef PGGC_GROUP
}

// One block per vertex with a hash table in LDS, for degrees up to D: the power
// of two >= SPE * degree slots, at most SLOTS (> D).
// A thread gathers the records of all its (at most R) edges first, so the
// gathers are in flight together, inserts them, and after the barrier looks
// each edge's slot up again: its record still holds the cluster's volume, so
// the arg-max needs neither a scan of the table nor another gather (a cluster
// met by several edges is evaluated by each; the packed maximum is the same).
// AT as in score_group: with u32 sums a slot takes 8 bytes of LDS.  The
// 65..2048 classes went from 148 to 93 ms on R-MAT scale 24 (two passes) and
// from 147 to 78 ms on scale 20.
template <class AT>
__device__ __forceinline__ u32 table_add_slot(i32* keys, AT* vals, u32 S, i32 key, AT w) {
    u32 h = __umulhi((u32)key * 0x9E3779B1u, S);
    while (true) {  // fewer keys than slots: an empty slot is always found
        const i32 old = atomicCAS(&keys[h], EMPTY_KEY, key);
        if (old == EMPTY_KEY || old == key) break;
        h = h + 1 < S ? h + 1 : 0;
    }
    if (sizeof(AT) == 4) atomicAdd((u32*)&vals[h], (u32)w);
    else atomicAdd((unsigned long long*)&vals[h], (unsigned long long)w);
    return h;
}
template <int BS, int D, int SLOTS, int SPE, class AT, class WT, class LT>
__global__ void __launch_bounds__(BS) k_score_table(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                    const i64* __restrict__ vw, const i32* __restrict__ list, i64 m,
                                                    const i32* __restrict__ part, const i64* __restrict__ vol,
                                                    RecView rv, const i32* __restrict__ cons, LT lam, float ratio,
                                                    ScoreOut out) {
    __shared__ i32 keys[SLOTS];
    __shared__ AT vals[SLOTS];
    constexpr int R = (D + BS - 1) / BS;
    const int t = threadIdx.x;
    const i64 li = block_id();
    if (li >= m) return;
    const i32 i = list[li];
    if (out.dest[i] == NO_MOVE) return;
    const i64 s = rp[i];
    const int d = (int)(rp[i + 1] - s);
    const int S = tslots(d, SPE, SLOTS);
    const i32 p = part[i];
    const i64 wi = vw[i];
    NbRec r[R];
    AT w[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int e = q * BS + t;
        r[q].part = EMPTY_KEY;
        w[q] = 0;
        if (e < d) {
            r[q] = load_rec(rv, col[s + e]);
            w[q] = (AT)W(s + e);
        }
    }
    for (int q = t; q < S; q += BS) {
        keys[q] = EMPTY_KEY;
        vals[q] = 0;
    }
    AT pv = 0;  // (summed before the inserts: probing ends lane by lane)
#pragma unroll
    for (int q = 0; q < R; q++) pv += r[q].part == p ? w[q] : (AT)0;
    pv = block_reduce<BS>(pv, [](AT a, AT b) { return a + b; });
    __syncthreads();
    u32 h[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
        h[q] = 0;
        if (r[q].part == EMPTY_KEY || r[q].part == p) continue;
        h[q] = table_add_slot(keys, vals, (u32)S, r[q].part, w[q]);
    }
    __syncthreads();
    float multi, p_conn, b;
    own_terms((i64)pv, vol[p], wi, lam(i), lam.rt(i, ratio), multi, p_conn, b);
    const i32 cp = cons ? cons[p] : 0;
    u64 bk = 0;
#pragma unroll
    for (int q = 0; q < R; q++) {
        if (r[q].part == EMPTY_KEY || r[q].part == p) continue;
        const AT agg = vals[h[q]];
        if (agg > 0 && (float)agg >= b && r[q].cons == cp) {
            const float jc = fmaf(-r[q].volf, multi, (float)agg);
            if (jc >= b) {
                const u64 k2 = pack_cand(jc, r[q].part);
                bk = k2 > bk ? k2 : bk;
            }
        }
    }
    bk = block_reduce<BS>(bk, [](u64 a, u64 b2) { return a > b2 ? a : b2; });
    if (t == 0) decide(i, p_conn, bk, p, wi, out);
}

// Raw sweep (first sweep of an initial local_move, src/local_mover.cpp:1391-1395):
// every neighbour is its own cluster with weight w_ij (rows carry no duplicate
// columns and no self loop), so the own-cluster weight is 0 and the best
// candidate is a streaming arg-max over the adjacency, with the same packed
// (gain, smallest label) order as the table path.
template <class WT>
__device__ __forceinline__ u64 raw_cand(const i32* __restrict__ col, WT W, const RecView& rv, i32 cp, i64 j,
                                        float multi, float b) {
    const NbRec r = load_rec(rv, col[j]);
    const i64 agg = W(j);
    if (agg > 0 && (float)agg >= b && r.cons == cp) {
        const float jc = fmaf(-r.volf, multi, (float)agg);
        if (jc >= b) return pack_cand(jc, r.part);
    }
    return 0;
}
// arg-max over the edges [jlo, jhi) by a block
template <int BS, class WT>
__device__ __forceinline__ u64 raw_best(const i32* __restrict__ col, WT W, const RecView& rv, i32 cp, i64 jlo, i64 jhi,
                                        float multi, float b) {
    u64 bk = 0;
    for (i64 jb = jlo; jb < jhi; jb += 4 * BS) {  // block-uniform loop control
#pragma unroll
        for (int u = 0; u < 4; u++) {  // independent gathers in flight
            const i64 j = jb + u * BS + threadIdx.x;
            if (j < jhi) {
                const u64 k2 = raw_cand(col, W, rv, cp, j, multi, b);
                bk = k2 > bk ? k2 : bk;
            }
        }
    }
    return block_max_u64<BS>(bk);
}

// one block per vertex (64 < degree <= 2048)
template <int BS, class WT, class LT>
__global__ void __launch_bounds__(BS) k_score_raw(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                  const i64* __restrict__ vw, const i32* __restrict__ list, i64 m,
                                                  const i32* __restrict__ part, const i64* __restrict__ vol,
                                                  RecView rv, const i32* __restrict__ cons, LT lam, float ratio,
                                                  ScoreOut out) {
    const i64 li = block_id();
    if (li >= m) return;
    const i32 i = list[li];
    if (out.dest[i] == NO_MOVE) return;
    const i32 p = part[i];
    const i32 cp = cons ? cons[p] : 0;
    float multi, p_conn, b;
    const i64 wi = vw[i];
    own_terms(0, vol[p], wi, lam(i), lam.rt(i, ratio), multi, p_conn, b);
    const u64 bk = raw_best<BS>(col, W, rv, cp, rp[i], rp[i + 1], multi, b);
    if (threadIdx.x == 0) decide(i, p_conn, bk, p, wi, out);
}

// Hubs of degree above HUB_LDS_BOUND.
//
// k_hub_gather takes a chunk of HUB_E edges per block: it gathers the neighbours'
// records, so that each edge costs one random access, sums the own-cluster
// weights, which the candidates' threshold needs, merges the others by cluster in
// LDS, and writes the distinct (cluster, volume, weight) entries grouped by the
// bucket of their cluster's hash, with the buckets' starts.  k_hub_score takes a
// slice of a hub's hash range per block: it reads its bucket's run of every
// chunk (the slices of one hub share an XCD's L2), adds the weights per cluster
// in an LDS table and takes the best candidate from it.  Nothing but the best
// candidate leaves the chip.  Each entry is read once, or once per slice of its
// bucket, and a cluster that most of the edges lead to is merged by the chunks
// that meet it, so the work grows with the degree.
// The random record gathers and the LDS atomics bound them.  R-MAT scale 24 (two
// passes, 64M hub edges): 0.59 + 0.47 ms a sweep, 47 ms in all; with records left
// in edge order, so that every slice of a hub read all of them (5.7 times each),
// 0.6 + 1.2 ms and 78 ms, and time that grew with the square of the degree: one
// hub of 2^20, 2^22 or 2^24 edges took 0.28, 2.8 or 33.8 ms a sweep, now 0.042,
// 0.087 and 0.30.  Each slice gathering at random: 3.0 ms at scale 24.
//
// The hash is a bijection of the 32-bit id, split by range: a slice whose keys
// do not fit (never seen with 1.5 slots per edge) is done again in 2, 4, ...
// parts, which ends at the latest when a part covers fewer ids than slots.
__device__ __forceinline__ u32 mix32(u32 x) {  // the finalizer of MurmurHash3
    x ^= x >> 16;
    x *= 0x85ebca6bu;
    x ^= x >> 13;
    x *= 0xc2b2ae35u;
    x ^= x >> 16;
    return x;
}
constexpr int HUB_GT = 512;
template <int SL, class AT, class WT>
__global__ void __launch_bounds__(HUB_GT) k_hub_gather(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                       HubView hv, const i32* __restrict__ part, RecView rv,
                                                       const i32* __restrict__ cons, const i32* __restrict__ dest,
                                                       u64* __restrict__ kv, AT* __restrict__ kw,
                                                       unsigned short* __restrict__ starts, i64* hub_pv) {
    __shared__ i32 lk[HUB_GS];
    __shared__ AT lv[HUB_GS];
    __shared__ float lf[HUB_GS];
    __shared__ u32 hist[HUB_BUCKETS];
    const i64 b = block_id();
    if (b >= hv.chunk0(hv.m)) return;
    const i64 h = upper_row(hv.chunks, 0, hv.m, b + hv.chunks[0]);
    const i32 i = hv.hubs[h];
    if (dest[i] == NO_MOVE) return;
    const int t = threadIdx.x;
    const i64 s = rp[i], d = rp[i + 1] - s, c = b - hv.chunk0(h);
    const i64 j0 = s + c * HUB_E;
    const int n = (int)(d - c * HUB_E < HUB_E ? d - c * HUB_E : HUB_E);
    const i64 ns = hub_slices(d, SL);
    const u32 per = (u32)hub_per(ns);
    const int nb = (int)hub_nb(ns);
    const i32 p = part[i];
    const i32 cp = cons ? cons[p] : 0;
    constexpr int U = HUB_E / HUB_GT;  // edges in flight per thread
    i32 v[U];
    NbRec r[U];
    AT w[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = u * HUB_GT + t < n ? col[j0 + u * HUB_GT + t] : -1;
#pragma unroll
    for (int u = 0; u < U; u++) {
        w[u] = 0;
        r[u].part = p;
        if (v[u] >= 0) {
            r[u] = load_rec(rv, v[u]);
            w[u] = (AT)W(j0 + u * HUB_GT + t);
        }
    }
    for (int q = t; q < HUB_GS; q += HUB_GT) {
        lk[q] = EMPTY_KEY;
        lv[q] = 0;
    }
    for (int q = t; q < HUB_BUCKETS; q += HUB_GT) hist[q] = 0;
    AT own = 0;
#pragma unroll
    for (int u = 0; u < U; u++) own += r[u].part == p ? w[u] : (AT)0;
    own = block_reduce<HUB_GT>(own, [](AT x, AT y) { return x + y; });
    if (t == 0 && own) atomicAdd((unsigned long long*)&hub_pv[h], (unsigned long long)own);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (r[u].part == p || r[u].cons != cp) continue;
        const u32 q = table_add_slot(lk, lv, (u32)HUB_GS, r[u].part, w[u]);
        lf[q] = r[u].volf;  // (the same value whoever stores it)
    }
    __syncthreads();
    constexpr int R = HUB_GS / HUB_GT;
    u32 bu[R], rk[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
        const i32 key = lk[t + q * HUB_GT];
        bu[q] = ~0u;
        rk[q] = 0;
        if (key == EMPTY_KEY) continue;
        const u32 sl = (u32)(((u64)mix32((u32)key) * (u64)ns) >> 32);
        bu[q] = per == 1 ? sl : sl / per;
        rk[q] = atomicAdd(&hist[bu[q]], 1u);
    }
    __syncthreads();
    constexpr int HB = HUB_BUCKETS / HUB_GT;
    u32 hc[HB];
    i64 mine = 0, total;
#pragma unroll
    for (int q = 0; q < HB; q++) {
        hc[q] = hist[t * HB + q];
        mine += hc[q];
    }
    u32 run = (u32)block_excl_scan_i64(mine, &total);
    unsigned short* st = starts + hv.start0(h) + c * (nb + 1);
#pragma unroll
    for (int q = 0; q < HB; q++) {
        hist[t * HB + q] = run;
        if (t * HB + q < nb) st[t * HB + q] = (unsigned short)run;
        run += hc[q];
    }
    if (t == 0) st[nb] = (unsigned short)total;
    __syncthreads();
    const i64 o = hv.edge0(h) + c * HUB_E;
#pragma unroll
    for (int q = 0; q < R; q++) {
        if (bu[q] == ~0u) continue;
        const int sl = t + q * HUB_GT;
        const i64 x = o + hist[bu[q]] + rk[q];
        kv[x] = (u64)(u32)lk[sl] | ((u64)__float_as_uint(lf[sl]) << 32);
        kw[x] = lv[sl];
    }
}

template <int SL, int BS, class AT, class LT>
__global__ void __launch_bounds__(BS) k_hub_score(const i64* __restrict__ rp, const i64* __restrict__ vw, HubView hv,
                                                  const i32* __restrict__ part, const i64* __restrict__ vol, LT lam,
                                                  float ratio, const i32* __restrict__ dest,
                                                  const u64* __restrict__ kv, const AT* __restrict__ kw,
                                                  const unsigned short* __restrict__ starts,
                                                  const i64* __restrict__ hub_pv, u64* hub_best) {
    __shared__ i32 lk[SL];
    __shared__ AT lv[SL];
    __shared__ float lf[SL];
    __shared__ int full;
    i64 h, sl;
    if (!hv.slice(block_id(), h, sl)) return;
    const i32 i = hv.hubs[h];
    if (dest[i] == NO_MOVE) return;
    const i64 d = rp[i + 1] - rp[i];
    const i64 ns = hub_slices(d, SL);
    if (sl >= ns) return;
    const int t = threadIdx.x;
    const i64 nch = hub_chunks(d), per = hub_per(ns), nb = hub_nb(ns);
    const unsigned short* st = starts + hv.start0(h) + sl / per;
    const u64* in = kv + hv.edge0(h);
    const AT* iw = kw + hv.edge0(h);
    // as many lanes per chunk as its run is long on average
    int lg = 2;
    while (lg < 10 && ((i64)2 << lg) * nb <= HUB_E) lg++;
    const int lane = t & ((1 << lg) - 1), G = 1 << lg;
    float multi, p_conn, b;
    own_terms(hub_pv[h], vol[part[i]], vw[i], lam(i), lam.rt(i, ratio), multi, p_conn, b);
    u64 bk = 0;
    for (u64 parts = 1;; parts *= 2) {  // block-uniform
        bool over = false;
        bk = 0;
        for (u64 part_no = 0; part_no < parts; part_no++) {
            const u64 total = (u64)ns * parts, want = (u64)sl * parts + part_no;
            for (int q = t; q < SL; q += BS) {
                lk[q] = EMPTY_KEY;
                lv[q] = 0;
            }
            if (t == 0) full = 0;
            __syncthreads();
            bool ok = true;
            auto add = [&](u64 rec, AT w) {
                const i32 key = (i32)(u32)rec;
                const u64 y = (u64)mix32((u32)key) * total;
                if ((y >> 32) != want) return;  // of another slice of the bucket, or part
                u32 q = __umulhi((u32)y, (u32)SL);
                int probe = 0;
                for (; probe < SL; probe++) {
                    const i32 old = atomicCAS(&lk[q], EMPTY_KEY, key);
                    if (old == EMPTY_KEY) lf[q] = __uint_as_float((u32)(rec >> 32));
                    if (old == EMPTY_KEY || old == key) {
                        if (sizeof(AT) == 4) atomicAdd((u32*)&lv[q], (u32)w);
                        else atomicAdd((unsigned long long*)&lv[q], (unsigned long long)w);
                        break;
                    }
                    q = q + 1 < (u32)SL ? q + 1 : 0;
                }
                ok = ok && probe < SL;
            };
            constexpr int U = 4;  // chunks in flight per lane group
            const i64 step = BS >> lg;
            for (i64 cb = 0; cb < nch; cb += step * U) {  // block-uniform loop control
                i64 x[U], e[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const i64 c = cb + u * step + (t >> lg);
                    x[u] = e[u] = 0;
                    if (c < nch) {
                        const unsigned short* q = st + c * (nb + 1);
                        x[u] = c * HUB_E + q[0] + lane;
                        e[u] = c * HUB_E + q[1];
                    }
                }
                u64 r[U];
                AT w[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    r[u] = (u64)(u32)EMPTY_KEY;
                    w[u] = 0;
                    if (x[u] < e[u]) {
                        r[u] = in[x[u]];
                        w[u] = iw[x[u]];
                    }
                }
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (x[u] < e[u]) add(r[u], w[u]);
#pragma unroll
                for (int u = 0; u < U; u++)
                    for (i64 y = x[u] + G; y < e[u]; y += G) add(in[y], iw[y]);
            }
            if (!ok) full = 1;
            __syncthreads();
            if (full) {  // block-uniform
                over = true;
                break;
            }
            for (int q = t; q < SL; q += BS) {
                const i32 key = lk[q];
                if (key == EMPTY_KEY) continue;
                const AT agg = lv[q];
                if (agg > 0 && (float)agg >= b) {
                    const float jc = fmaf(-lf[q], multi, (float)agg);
                    if (jc >= b) {
                        const u64 k2 = pack_cand(jc, key);
                        bk = k2 > bk ? k2 : bk;
                    }
                }
            }
            __syncthreads();  // the next part clears the table
        }
        if (!over) break;
        __syncthreads();
    }
    bk = block_reduce<BS>(bk, [](u64 x, u64 y) { return x > y ? x : y; });
    if (t == 0 && bk) atomicMax((unsigned long long*)&hub_best[h], (unsigned long long)bk);
}

// raw sweep: a block per slice again, each with an equal share of the hub's edges
template <int SL, class WT, class LT>
__global__ void __launch_bounds__(256) k_hub_raw(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                 const i64* __restrict__ vw, HubView hv,
                                                 const i32* __restrict__ part, const i64* __restrict__ vol,
                                                 RecView rv, const i32* __restrict__ cons, LT lam, float ratio,
                                                 const i32* __restrict__ dest, u64* hub_best) {
    i64 h, sl;
    if (!hv.slice(block_id(), h, sl)) return;
    const i32 i = hv.hubs[h];
    if (dest[i] == NO_MOVE) return;
    const i64 s = rp[i], e = rp[i + 1];
    const i64 ns = hub_slices(e - s, SL);
    if (sl >= ns) return;
    const i64 share = (e - s + ns - 1) / ns;
    const i64 j_lo = s + sl * share, j_hi = j_lo + share < e ? j_lo + share : e;
    const i32 p = part[i];
    const i32 cp = cons ? cons[p] : 0;
    float multi, p_conn, bth;
    own_terms(0, vol[p], vw[i], lam(i), lam.rt(i, ratio), multi, p_conn, bth);
    const u64 bk = raw_best<256>(col, W, rv, cp, j_lo, j_hi, multi, bth);
    if (threadIdx.x == 0 && bk) atomicMax((unsigned long long*)&hub_best[h], (unsigned long long)bk);
}

template <class LT>
__global__ void k_hub_decide(const i32* hubs, i64 m, const i32* part, const i64* vw, const i64* vol, LT lam,
                             float ratio, i64* hub_pv, u64* hub_best, ScoreOut out) {
    const i64 hi = thread_item();
    if (hi >= m) return;
    const i32 i = hubs[hi];
    if (out.dest[i] == NO_MOVE) return;
    const u64 bk = hub_best[hi];
    const i64 pv = hub_pv[hi];
    hub_best[hi] = 0;  // for the next sweep
    hub_pv[hi] = 0;
    const i32 p = part[i];
    const i64 wi = vw[i];
    float multi, p_conn, bth;
    own_terms(pv, vol[p], wi, lam(i), lam.rt(i, ratio), multi, p_conn, bth);
    decide(i, p_conn, bk, p, wi, out);
}


// Algorithmic bytes of one scoring sweep, counted (on timing runs only)
// before it runs, since dest decides which vertices it scores.  A scored
// vertex reads its row bounds, destination, cluster, vertex weight and its
// cluster's volume, every edge's column (and weight) and the neighbour's
// record, and writes its destination, gain and record: 48 + d (4 + weight
// bytes + 8) bytes.  Every listed vertex also costs its list entry
// and destination read.  acc3[0..2] = group, table and hub classes.
struct ScoreBounds {
    i64 s[NCLS + 1];
    i64 hub0;  // first hub of k_hub_score
};
template <int WB>
__global__ void __launch_bounds__(256) k_score_bytes(const i64* __restrict__ rp, const i32* __restrict__ list,
                                                     ScoreBounds sb, const i32* __restrict__ dest, i64* acc3) {
    const i64 x = thread_item();
    i64 b0 = 0, b1 = 0, b2 = 0;
    if (x < sb.s[NCLS]) {
        const i32 i = list[x];
        const int grp = x < sb.s[CL_TABLE] ? 0 : (x < sb.hub0 ? 1 : 2);
        i64 by = 8;
        if (dest[i] != NO_MOVE) by += 48 + (rp[i + 1] - rp[i]) * (4 + WB + 8);
        if (grp == 0) b0 = by;
        else if (grp == 1) b1 = by;
        else b2 = by;
    }
    b0 = block_sum_i64<256>(b0);
    b1 = block_sum_i64<256>(b1);
    b2 = block_sum_i64<256>(b2);
    if (threadIdx.x == 0) {
        if (b0) atomicAdd((unsigned long long*)&acc3[0], (unsigned long long)b0);
        if (b1) atomicAdd((unsigned long long*)&acc3[1], (unsigned long long)b1);
        if (b2) atomicAdd((unsigned long long*)&acc3[2], (unsigned long long)b2);
    }
}

// alpha + beta * degree bytes per listed vertex (per candidate of the
// afterburner, per mover of perform_moves) that is not NO_MOVE in dest and is
// marked in mvp (when given), plus `extra` once
__global__ void __launch_bounds__(256) k_list_bytes(const i64* __restrict__ rp, const i32* __restrict__ list,
                                                    const i32* __restrict__ dest, const u64* __restrict__ mvp, i64 k,
                                                    i64 alpha, i64 beta, i64 extra, i64* acc) {
    const i64 x = thread_item();
    i64 b = 0;
    if (x < k) {
        const i32 i = list[x];
        if ((!dest || dest[i] != NO_MOVE) && (!mvp || ((u32)mvp[i] >> 31))) b = alpha + beta * (rp[i + 1] - rp[i]);
    }
    if (x == 0) b += extra;
    b = block_sum_i64<256>(b);
    if (threadIdx.x == 0 && b) atomicAdd((unsigned long long*)acc, (unsigned long long)b);
}

// What the scoring launches share.
template <class LT>
struct ScoreArgs {
    const i32* L;
    const i32* part;
    const i64* vol;
    RecView rv;
    const i32* cons;
    LT lam;
    float ratio;
    ScoreOut out;
};
// LDS-table scoring of the list entries [x0, x1) (one block per vertex):
// degrees up to D, BS threads, SPE slots per edge, at most SLOTS.
template <class AT, int BS, int D, int SLOTS, int SPE, class WT, class LT>
static void launch_table(Ctx& c, const DGraph& g, WT W, const ScoreArgs<LT>& a, i64 x0, i64 x1) {
    const i64 m = x1 - x0;
    if (m <= 0) return;
    k_score_table<BS, D, SLOTS, SPE, AT><<<grid_blocks(m), BS, 0, c.stream>>>(
        g.rp, g.col, W, g.vw, a.L + x0, m, a.part, a.vol, a.rv, a.cons, a.lam, a.ratio, a.out);
}
// class with degree bound D (128, 256, 512): threads per vertex and slots per
// edge from the knobs
template <class AT, int D, class WT, class LT>
static void launch_table_class(Ctx& c, const DGraph& g, WT W, const ScoreArgs<LT>& a, i64 x0, i64 x1) {
    const int bs = c.table_threads, spe = c.table_spe;
    if (bs == 64 && spe == 2) launch_table<AT, 64, D, 2 * D, 2>(c, g, W, a, x0, x1);
    else if (bs == 64) launch_table<AT, 64, D, 4 * D, 4>(c, g, W, a, x0, x1);
    else if (bs == 128 && spe == 2) launch_table<AT, 128, D, 2 * D, 2>(c, g, W, a, x0, x1);
    else if (bs == 128) launch_table<AT, 128, D, 4 * D, 4>(c, g, W, a, x0, x1);
    else if (spe == 2) launch_table<AT, 256, D, 2 * D, 2>(c, g, W, a, x0, x1);
    else launch_table<AT, 256, D, 4 * D, 4>(c, g, W, a, x0, x1);
}
template <class AT, class WT, class LT>
static void launch_groups(Ctx& c, const DGraph& g, WT W, const ScoreArgs<LT>& a, const i64* st, int raw) {
    GroupRanges gr;
    i64 nb = 0;
    for (int q = 0; q <= CL_TABLE; q++) {
        gr.s[q] = st[q];
        gr.blk[q] = nb;
        if (q < CL_TABLE) nb += ceil_div(st[q + 1] - st[q], 256 / (4 << q));
    }
    if (nb == 0) return;
    k_score_groups<AT><<<grid_blocks(nb), 256, 0, c.stream>>>(g.rp, g.col, W, g.vw, a.L, gr, a.part, a.vol, a.rv,
                                                              a.cons, raw, a.lam, a.ratio, a.out);
}
template <class AT, class WT, class LT>
static void launch_tables(Ctx& c, const LevelPlan& lp, const DGraph& g, WT W, const ScoreArgs<LT>& a) {
    const i64* st = lp.sc_start;
    const bool one = st[CL_HUB] - st[CL_TABLE] <= TABLE_ONE_LAUNCH;
    if (one) launch_table<AT, 256, 2048, 4096, 2>(c, g, W, a, st[CL_TABLE], st[CL_HUB]);
    launch_table<AT, 1024, HUB_HALF, 8192, 2>(c, g, W, a, st[CL_HUB], st[CL_HUB] + lp.nhalf);
    launch_table<AT, 1024, HUB_LDS_BOUND, HUB_LDS_SLOTS, 2>(c, g, W, a, st[CL_HUB] + lp.nhalf, lp.hub0);
    if (one) return;
    // LDS tables sized for the class, so the many low-degree rows keep more
    // waves resident per CU; threads per vertex and slots per edge are knobs
    launch_table_class<AT, 128>(c, g, W, a, st[5], st[6]);
    launch_table_class<AT, 256>(c, g, W, a, st[6], st[7]);
    launch_table_class<AT, 512>(c, g, W, a, st[7], st[8]);
    if (c.table_spe == 2) {
        launch_table<AT, 256, 1024, 2048, 2>(c, g, W, a, st[8], st[9]);
        launch_table<AT, 512, 2048, 4096, 2>(c, g, W, a, st[9], st[10]);
    } else {
        launch_table<AT, 256, 1024, 4096, 4>(c, g, W, a, st[8], st[9]);
        launch_table<AT, 512, 2048, 8192, 4>(c, g, W, a, st[9], st[10]);
    }
}

template <class LT>
static void score_all(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, const i32* part, const i64* vol,
                      const i32* cons, int raw, LT lam, float ratio, const ScoreOut& out, bool packed = false) {
    i32* dest = out.dest;
    // raw: every vertex a cluster of its own; 0: any clustering
    const i64* st = lp.sc_start;
    const i32* L = lp.sc_list.p;
    Buf<i64> acct;
    if (c.kt.on && g.n > 0) {  // timing runs only
        acct = Buf<i64>(c, 3);
        fill_i64(c, acct, 3, 0);
        ScoreBounds sb;
        for (int k = 0; k <= NCLS; k++) sb.s[k] = st[k];
        sb.hub0 = lp.hub0;
        PGGC_WDISPATCH(g, (k_score_bytes<decltype(W)::bytes><<<grid_items(g.n, 256), 256, 0, c.stream>>>(
                              g.rp, L, sb, dest, acct)));
        PGGC_LAUNCH_CHECK();
    }
    if (g.n > 0 && !packed) {
        if (cons && s.rec16.n < (size_t)g.n) s.rec16 = Buf<uint4>(c, s.cap);
        k_rec_pack<<<grid_items(g.n, 256), 256, 0, c.stream>>>(g.n, part, vol, cons, s.rec, cons ? s.rec16.p : nullptr);
        PGGC_LAUNCH_CHECK();
    }
#define PGGC_HUB_RAW(SL)                                                                                             \
    k_hub_raw<SL><<<grid_blocks(lp.hub_blocks), 256, 0, c.stream>>>(g.rp, g.col, W, g.vw, hv, part, vol, a.rv, cons, \
                                                                    lam, ratio, dest, lp.hub_best)
#define PGGC_HUB(SL, AT)                                                                                             \
    for (const LevelPlan::HubBatch& hb : lp.hub_batches) {                                                           \
        const HubView bv = hub_view(lp, hb.h0, hb.h1, hb.blocks);                                                    \
        u64* kv = s.hub_buf;                                                                                         \
        AT* kw = (AT*)(void*)(kv + hb.edges);                                                                        \
        unsigned short* hs = (unsigned short*)(void*)(kv + hub_scratch(hb, sizeof(AT) == 4) - ceil_div(hb.starts, 4)); \
        k_hub_gather<SL, AT><<<grid_blocks(hb.chunks), HUB_GT, 0, c.stream>>>(                                       \
            g.rp, g.col, W, bv, part, a.rv, cons, dest, kv, kw, hs, lp.hub_pv.p + hb.h0);                            \
        k_hub_score<SL, 1024, AT><<<grid_blocks(hb.blocks), 1024, 0, c.stream>>>(                                    \
            g.rp, g.vw, bv, part, vol, lam, ratio, dest, kv, kw, hs, lp.hub_pv.p + hb.h0, lp.hub_best.p + hb.h0);    \
    }
    const ScoreArgs<LT> a{L, part, vol, RecView{s.rec.p, cons ? s.rec16.p : nullptr}, cons, lam, ratio, out};
    PGGC_WDISPATCH(g, {
        using WT = decltype(W);
        constexpr bool unit = IsUnit<WT>::v;  // (agg32 and hub32 hold)
        i64 m;
        int tk = c.kt_begin(KS_SCORE_GROUP);
        if (lp.agg32) launch_groups<u32>(c, g, W, a, st, raw);
        else if constexpr (!unit) launch_groups<i64>(c, g, W, a, st, raw);
        c.kt_end(tk, 0.0);
        if (tk >= 0) acct_add(c, c.kt_counter(tk), acct.p);
        tk = c.kt_begin(KS_SCORE_TABLE);
        if (raw) {
            if ((m = st[CL_BIG] - st[CL_TABLE]) > 0)
                k_score_raw<64><<<grid_blocks(m), 64, 0, c.stream>>>(g.rp, g.col, W, g.vw, L + st[CL_TABLE], m,
                                                                     part, vol, a.rv, cons, lam, ratio, out);
            if ((m = lp.hub0 - st[CL_BIG]) > 0)  // big rows and the LDS-scored hubs
                k_score_raw<256><<<grid_blocks(m), 256, 0, c.stream>>>(g.rp, g.col, W, g.vw, L + st[CL_BIG], m,
                                                                       part, vol, a.rv, cons, lam, ratio, out);
        } else if (lp.agg32) {
            launch_tables<u32>(c, lp, g, W, a);
        } else if constexpr (!unit) {
            launch_tables<i64>(c, lp, g, W, a);
        }
        c.kt_end(tk, 0.0);
        if (tk >= 0) acct_add(c, c.kt_counter(tk), acct.p + 1);
        if ((m = lp.nhub) > 0) {
            const HubView hv = hub_view(lp, 0, m, lp.hub_blocks);
            if (!raw && s.hub_buf.n < lp.hub_words) {
                s.hub_buf.reset();
                s.hub_buf = Buf<u64>(c, lp.hub_words);
            }
            tk = c.kt_begin(KS_SCORE_HUB);
            if (lp.hub32) {
                if (raw) PGGC_HUB_RAW(HUB_SLOTS32);
                else PGGC_HUB(HUB_SLOTS32, u32)
            } else if constexpr (!unit) {
                if (raw) PGGC_HUB_RAW(HUB_SLOTS64);
                else PGGC_HUB(HUB_SLOTS64, i64)
            }
            k_hub_decide<<<grid_items(m, 256), 256, 0, c.stream>>>(hv.hubs, m, part, g.vw, vol, lam, ratio, lp.hub_pv,
                                                                       lp.hub_best, out);
            c.kt_end(tk, 0.0);
            if (tk >= 0) acct_add(c, c.kt_counter(tk), acct.p + 2);
        }
    });
#undef PGGC_HUB
#undef PGGC_HUB_RAW
    PGGC_LAUNCH_CHECK();
}

// ------------------------------------------------------------- candidates
struct SelCands {
    static constexpr bool extra = false;
    const i32* o1;
    const i32* dest;
    i32* out;
    __device__ __forceinline__ bool test(i64 x) const { return dest[o1[x]] != NO_MOVE; }
    __device__ __forceinline__ void emit(i64 pos, i64 x) const { out[pos] = o1[x]; }
};
// candidates in order1 order; returns the count, b[0]/b[1] = class boundaries
static i64 gather_candidates(Ctx& c, const LevelPlan& lp, const DGraph& g, const i32* dest, i32* out, i64* b) {
    const i64* h = select_items(c, SelCands{lp.ord.o1, dest, out}, g.n, SelBounds{lp.ord.off_large, lp.ord.off_large2});
    b[0] = h[1];
    b[1] = h[2];
    return h[0];
}

// ------------------------------------------------------------- afterburner
// afterburner_filter (src/local_mover.cpp:374-433): the change in the
// candidate's gain if every neighbour with a larger gain (ties broken by the
// xorshift hash) also makes its move.  An edge gives two FP32 terms, added in
// this order: what the neighbour's destination means for the candidate's own
// and best cluster, then what its leaving its cluster means.  (At most one
// comparison of each pair holds, as the best cluster is never the own one;
// an edge without effect adds zeros.)  The kernels take a list of candidates,
// or all vertices in order1 order and skip those whose record says NO_MOVE.
struct AbSelf {
    i32 p, best, hi;
    float multi, igain;
};
template <class LT, class PT>
__device__ __forceinline__ AbSelf ab_self(const AbInfo* info, i32 i, LT lam, PT prio) {
    const AbInfo me = info[i];
    return AbSelf{me.part, me.dest, prio(i), me.vwf * lam(i), me.gain};
}
template <class PT>
__device__ __forceinline__ float2 ab_terms(const AbInfo& q4, i32 v, i64 w, const AbSelf& m, PT prio) {
    float2 t = make_float2(0.0f, 0.0f);
    const float vg = q4.gain;
    if ((vg - m.igain) >= AFTERBURNER_EPS || (fabsf(vg - m.igain) < AFTERBURNER_EPS && prio(v) < m.hi)) {
        const float q = fmaf(-m.multi, q4.vwf, (float)w);
        t.x = q4.dest == m.p ? -q : ((q4.dest == m.best && m.best != NEW_PART) ? q : 0.0f);
        t.y = q4.part == m.p ? q : (q4.part == m.best ? -q : 0.0f);
    }
    return t;
}

// Direct sweeps (find_movers): a kept vertex is marked as a mover right away.
struct AbMark {
    u64* mvp;   // null: not marked here
    i64* knew;  // counts the movers that need a new cluster
    __device__ __forceinline__ void operator()(i32 i, const AbSelf& m) const {
        if (!mvp) return;
        mvp[i] = mvp_moved(m.p, m.best);
        if (m.best == NEW_PART) atomicAdd((unsigned long long*)knew, 1ull);
    }
};

// Degree below LARGE_CUTOFF: the terms are added in adjacency order.  The
// gathers of the neighbours' records bound it, so AB_G lanes gather a
// candidate's edges (AB_U in flight per lane) and leave the terms in LDS, and
// one lane adds them in order.  With one thread per candidate, which also
// gathered in order, a sweep of R-MAT scale 20 took 137 us here on the top
// level (unit weights), now 53 us; on scale 24 1804 -> 1007 us.  16 lanes: most
// candidates have at most a few dozen edges.
constexpr int AB_G = 16, AB_U = 4, AB_PB = 256 / AB_G;
template <class WT, class LT, class PT>
__device__ __forceinline__ void ab_small(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                         const AbInfo* __restrict__ info, const i32* __restrict__ cand, i64 blk, i64 k,
                                         LT lam, PT prio, i32* __restrict__ keep, const AbMark& mark) {
    __shared__ float2 term[AB_PB][LARGE_CUTOFF + 1];
    const int lane = threadIdx.x & (AB_G - 1), grp = threadIdx.x / AB_G;
    const i64 x = blk * AB_PB + grp;
    int d = 0;
    i32 i = 0;
    AbSelf m = {0, 0, 0, 0.0f, 0.0f};
    if (x < k) {
        i = cand[x];
        m = ab_self(info, i, lam, prio);
        const i64 s = rp[i];
        d = m.best == NO_MOVE ? -1 : (int)(rp[i + 1] - s);
        for (int jb = lane; jb < d; jb += AB_G * AB_U) {
            i32 v[AB_U];
            AbInfo q[AB_U];
#pragma unroll
            for (int u = 0; u < AB_U; u++) v[u] = jb + u * AB_G < d ? col[s + jb + u * AB_G] : -1;
#pragma unroll
            for (int u = 0; u < AB_U; u++)
                if (v[u] >= 0) q[u] = info[v[u]];
#pragma unroll
            for (int u = 0; u < AB_U; u++)
                if (v[u] >= 0) term[grp][jb + u * AB_G] = ab_terms(q[u], v[u], W(s + jb + u * AB_G), m, prio);
        }
    }
    __syncthreads();
    if (lane == 0 && x < k) {
        float acc = 0.0f;
#pragma unroll 8
        for (int e = 0; e < d; e++) {
            const float2 t = term[grp][e];
            acc = acc + t.x;
            acc = acc + t.y;
        }
        const bool kept = d >= 0 && m.igain + acc >= 0.0f;
        keep[x] = kept ? 1 : 0;
        if (kept) mark(i, m);
    }
}

// One wave per candidate: 64 strided partials and a halving tree.
template <class WT, class LT, class PT>
__device__ __forceinline__ void ab_wave(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                        const AbInfo* __restrict__ info, const i32* __restrict__ cand, i64 x, i64 k1,
                                        LT lam, PT prio, i32* __restrict__ keep, const AbMark& mark) {
    const int lane = threadIdx.x & 63;
    if (x >= k1) return;
    const i32 i = cand[x];
    const AbSelf m = ab_self(info, i, lam, prio);
    if (m.best == NO_MOVE) {  // wave-uniform
        if (lane == 0) keep[x] = 0;
        return;
    }
    float acc = 0.0f;
    const i64 e = rp[i + 1];
    constexpr int U = 4;
    for (i64 base = rp[i]; base < e; base += 64 * U) {  // wave-uniform loop control
        i32 v[U];
        AbInfo q[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = base + u * 64 + lane < e ? col[base + u * 64 + lane] : -1;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (v[u] >= 0) q[u] = info[v[u]];
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (v[u] < 0) continue;
            const float2 t = ab_terms(q[u], v[u], W(base + u * 64 + lane), m, prio);
            acc = acc + t.x;
            acc = acc + t.y;
        }
    }
    xlane_fence(acc);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc = acc + __shfl_down(acc, off);
    if (lane == 0) {
        const bool kept = m.igain + acc >= 0.0f;
        keep[x] = kept ? 1 : 0;
        if (kept) mark(i, m);
    }
}

// both classes in one launch: list entries [0, k0) in the first b0 blocks
// (AB_PB each), [k0, k1) in the others (a wave each)
template <class WT, class LT, class PT>
__global__ void __launch_bounds__(256) k_ab_lanes(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                  const AbInfo* __restrict__ info, const i32* __restrict__ cand,
                                                  i64 k0, i64 k1, i64 b0, LT lam, PT prio, i32* __restrict__ keep,
                                                  AbMark mark) {
    const i64 b = block_id();
    if (b < b0) ab_small(rp, col, W, info, cand, b, k0, lam, prio, keep, mark);
    else ab_wave(rp, col, W, info, cand, k0 + (b - b0) * 4 + (threadIdx.x >> 6), k1, lam, prio, keep, mark);
}

// A 1024-thread block per candidate: 1024 strided partials and a halving tree.
template <class WT, class LT, class PT>
__global__ void __launch_bounds__(1024) k_ab_block(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                   const AbInfo* __restrict__ info, const i32* __restrict__ cand,
                                                   i64 k0, i64 k1, LT lam, PT prio, i32* __restrict__ keep,
                                                   AbMark mark) {
    __shared__ float sh[1024];
    const int t = threadIdx.x;
    const i64 x = k0 + block_id();
    if (x >= k1) return;
    const i32 i = cand[x];
    const AbSelf m = ab_self(info, i, lam, prio);
    if (m.best == NO_MOVE) {  // block-uniform
        if (t == 0) keep[x] = 0;
        return;
    }
    float acc = 0.0f;
    const i64 e = rp[i + 1];
    constexpr int U = 4;
    for (i64 base = rp[i]; base < e; base += 1024 * U) {  // block-uniform loop control
        i32 v[U];
        AbInfo q[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = base + u * 1024 + t < e ? col[base + u * 1024 + t] : -1;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (v[u] >= 0) q[u] = info[v[u]];
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (v[u] < 0) continue;
            const float2 tt = ab_terms(q[u], v[u], W(base + u * 1024 + t), m, prio);
            acc = acc + tt.x;
            acc = acc + tt.y;
        }
    }
    sh[t] = acc;
    __syncthreads();
    for (int off = 512; off >= 64; off >>= 1) {
        if (t < off) sh[t] = sh[t] + sh[t + off];
        __syncthreads();
    }
    if (t < 64) {
        acc = sh[t];
        xlane_fence(acc);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) acc = acc + __shfl_down(acc, off);
        if (t == 0) {
            const bool kept = m.igain + acc >= 0.0f;
            keep[x] = kept ? 1 : 0;
            if (kept) mark(i, m);
        }
    }
}

__global__ void __launch_bounds__(256) k_ab_pack(i64 n, const float* __restrict__ gain, const i32* __restrict__ dest,
                                                 const i32* __restrict__ part, const i64* __restrict__ vw,
                                                 AbInfo* __restrict__ info) {
    const i64 i = thread_item();
    if (i >= n) return;
    AbInfo a;
    a.gain = gain[i];
    a.dest = dest[i];
    a.part = part[i];
    a.vwf = (float)vw[i];
    info[i] = a;
}

// The kept candidates become the sweep's movers, in order1 order, and are
// marked in mvp.  first counts the movers that take a new cluster, second the
// candidates.
struct SelMoves {
    static constexpr bool extra = true;
    const i32* cand;
    const i32* keep;
    const i32* dest;
    const i32* part;
    i32* moves;
    u64* mvp;
    __device__ __forceinline__ bool test(i64 x) const { return keep[x] != 0; }
    __device__ __forceinline__ bool first(i64 x, bool sel) const { return sel && dest[cand[x]] == NEW_PART; }
    __device__ __forceinline__ bool second(i64 x, bool) const { return dest[cand[x]] != NO_MOVE; }
    __device__ __forceinline__ void emit(i64 pos, i64 x) const {
        const i32 i = cand[x];
        moves[pos] = i;
        mvp[i] = mvp_moved(part[i], dest[i]);
    }
};
struct Movers {
    i64 k;      // movers
    i64 knew;   // of them with destination NEW_PART
    i64 cands;  // candidates
};

// The filter over cand (k candidates, or every vertex, in order1 order; b: class
// boundaries): s.flag[x] = keep.
template <class LT, class PT>
static void afterburner(Ctx& c, MoveScratch& s, const DGraph& g, const i32* cand, i64 k, const i64* b, LT lam,
                        PT prio, bool pack, AbMark mark = {nullptr, nullptr}) {
    const int tk = c.kt_begin(KS_AFTERBURNER);
    if (pack) {
        k_ab_pack<<<grid_items(g.n, 256), 256, 0, c.stream>>>(g.n, s.gain, s.dest, s.part, g.vw, s.abi);
        PGGC_LAUNCH_CHECK();
    }
    const i64 nb0 = ceil_div(b[0], AB_PB), nb1 = ceil_div(b[1] - b[0], 4);
    PGGC_WDISPATCH(g, {
        if (nb0 + nb1 > 0)
            k_ab_lanes<<<grid_blocks(nb0 + nb1), 256, 0, c.stream>>>(g.rp, g.col, W, s.abi, cand, b[0], b[1], nb0, lam,
                                                                     prio, s.flag, mark);
        if (k > b[1])
            k_ab_block<<<grid_blocks(k - b[1]), 1024, 0, c.stream>>>(g.rp, g.col, W, s.abi, cand, b[1], k, lam,
                                                                     prio, s.flag, mark);
    });
    c.kt_end(tk, 0.0);
    PGGC_LAUNCH_CHECK();
    if (tk >= 0) {  // timing runs only: count the bytes outside the timed region
        // per candidate edge the column, weight and the neighbour's record,
        // per candidate its id, record, row bounds and keep flag; a pack reads
        // gain, dest, part and vertex weight and writes a record per vertex
        Buf<i64> acc(c, 1);
        fill_i64(c, acc, 1, 0);
        k_list_bytes<<<grid_items(std::max<i64>(k, 1), 256), 256, 0, c.stream>>>(
            g.rp, cand, s.dest, nullptr, k, 40, 20 + (g.wk == W_UNIT ? 0 : g.wk == W_I32 ? 4 : 8), pack ? 36 * g.n : 0, acc);
        PGGC_LAUNCH_CHECK();
        acct_add(c, c.kt_counter(tk), acc);
    }
}

// the kept ones of cand, marked in mvp
static Movers select_movers(Ctx& c, MoveScratch& s, const i32* cand, i64 k, i32* moves) {
    const i64* h = select_items(c, SelMoves{cand, s.flag, s.dest, s.part, moves, s.mvp}, k, SelBounds{0, 0},
                                s.scal.p + SC_EXTRA);
    return Movers{h[0], h[3], h[4]};
}

// ------------------------------------------------------------- new labels
__global__ void k_new_flags(const i32* moves, i64 k, const i32* dest, i32* flag) {
    const i64 x = thread_item();
    if (x >= k) return;
    flag[x] = dest[moves[x]] == NEW_PART ? 1 : 0;
}
__global__ void k_mark_used(const i32* part, i64 n, i32* used) {
    const i64 i = thread_item();
    if (i >= n) return;
    used[part[i]] = 1;
}
__global__ void k_unused_flags(const i32* used, i64 L, i32* flag) {
    const i64 l = thread_item();
    if (l >= L) return;
    flag[l] = used[l] == 0 ? 1 : 0;
}
__global__ void k_assign_new(const i32* newv, i64 K, const i32* avail, i64 A, i32 curr, i32* dest, i32* cons,
                             const i32* part) {
    const i64 x = thread_item();
    if (x >= K) return;
    i32 i = newv[x];
    i32 l = x < A ? avail[x] : (i32)(x - A) + curr;
    dest[i] = l;
    if (cons) cons[l] = cons[part[i]];
}

// key of a NEW_PART mover in the caller's move order: order class
// (src/header/ordering.h:17-19), then the caller's id
__global__ void k_newid_keys(const i32* newv, i64 K, const i64* rp, const i32* ids, u64* key) {
    const i64 x = thread_item();
    if (x >= K) return;
    const i32 i = newv[x];
    const i64 d = rp[i + 1] - rp[i];
    const u64 cls = d < LARGE_CUTOFF ? 0 : (d < MASSIVE_CUTOFF ? 1 : 2);
    key[x] = cls << 32 | (u32)ids[i];
}

// set_new_cluster_ids (src/local_mover.cpp:215-274).  ids non-null: the
// graph is renumbered and ids[i] is vertex i's id in the caller's order; the
// movers are then taken in the caller's move order.
static void set_new_cluster_ids(Ctx& c, MoveScratch& s, const DGraph& g, RefineData& rd, const i32* moves, i64 k,
                                i32* cons, const i32* ids, i64 nfull) {
    k_new_flags<<<grid_items(k, 256), 256, 0, c.stream>>>(moves, k, s.dest, s.flag);
    PGGC_LAUNCH_CHECK();
    i64 K = compact_flags(c, s.flag, moves, k, s.tmp);
    if (K == 0) return;
    if (ids && K > 1) {
        Buf<u64> key(c, K);
        k_newid_keys<<<grid_items(K, 256), 256, 0, c.stream>>>(s.tmp, K, g.rp, ids, key);
        PGGC_LAUNCH_CHECK();
        radix_sort_pairs(c, key, s.tmp.p, K, 34);
    }
    const i32 curr = rd.label_count;
    fill_i32(c, s.flag, curr, 0);
    k_mark_used<<<grid_items(nfull, 256), 256, 0, c.stream>>>(s.part, nfull, s.flag);
    PGGC_LAUNCH_CHECK();
    Buf<i32> uf(c, std::max<i64>(curr, 1));
    k_unused_flags<<<grid_items(curr, 256), 256, 0, c.stream>>>(s.flag, curr, uf);
    PGGC_LAUNCH_CHECK();
    i64 A = compact_flags(c, uf, nullptr, curr, s.tmp2);
    if (K > A) {
        i64 need = K - A;
        if (curr + need > rd.cap) throw Error(-4, "label capacity exceeded while assigning new clusters");
        fill_i64(c, rd.vol + curr, need, 0);
        rd.label_count = (i32)(curr + need);
    }
    k_assign_new<<<grid_items(K, 256), 256, 0, c.stream>>>(s.tmp, K, s.tmp2, A, curr, s.dest, cons, s.part);
    PGGC_LAUNCH_CHECK();
}

// ------------------------------------------------------------- perform moves
// mvp[v]: low word the cluster of v | moved << 31 (cluster ids are >= 0), high
// word the cluster after this sweep's moves.  Between sweeps both words are
// v's cluster (k_mvp_init at the start of a call); a sweep marks its movers
// (SelMoves, or k_mvp_moves once new cluster ids are known) and k_apply_moves settles them, so a sweep touches the movers'
// words only, and an edge's uncut change reads one 8-byte word.
__device__ __forceinline__ u64 mvp_settled(i32 p) { return (u64)(u32)p | ((u64)(u32)p << 32); }
__global__ void __launch_bounds__(256) k_mvp_init(i64 n, const i32* __restrict__ part, u64* __restrict__ mvp,
                                                  i64* scal) {
    const i64 i = thread_item();
    if (i < SC_COUNT) scal[i] = 0;
    if (i < n) mvp[i] = mvp_settled(part[i]);
}
// The start of a local move: volumes and clusters copied, the vertices' words
// settled, every vertex active, the scalars zero.
__global__ void __launch_bounds__(256) k_move_begin(const i64* __restrict__ bvol, i64 L, i64* __restrict__ vol,
                                                    const i32* __restrict__ bpart, i64 nfull, i32* __restrict__ part,
                                                    i64 n, u64* __restrict__ mvp, i32* __restrict__ dest, i64* scal) {
    const i64 x = thread_item();
    if (x < SC_COUNT) scal[x] = 0;
    if (x < L) vol[x] = bvol[x];
    if (x < nfull) {
        const i32 p = bpart[x];
        part[x] = p;
        if (x < n) {
            mvp[x] = mvp_settled(p);
            dest[x] = NULL_PART;
        }
    }
}
__global__ void __launch_bounds__(256) k_mvp_moves(const i32* __restrict__ moves, i64 k, const i32* __restrict__ part,
                                                   const i32* __restrict__ dest, u64* __restrict__ mvp) {
    const i64 x = thread_item();
    if (x >= k) return;
    const i32 i = moves[x];
    mvp[i] = mvp_moved(part[i], dest[i]);
}

// Where the uncut changes of the movers are added: AccOne spreads one sum over
// MV_SLOTS words (summed by k_finish), AccInst adds per instance of a union
// batch, merged per block in LDS.
constexpr int IC_SLOTS = 512;  // LDS slots for at most 256 distinct instances per block
struct AccOne {
    i64* slots;
    template <int BS>
    __device__ __forceinline__ void add(i32, i64 acc) const {
        acc = block_sum_i64<BS>(acc);
        if (threadIdx.x == 0 && acc)
            atomicAdd((unsigned long long*)&slots[block_id() & (MV_SLOTS - 1)], (unsigned long long)acc);
    }
};
struct AccInst {
    const i32* inst;
    i64* sums;
    template <int BS>
    __device__ __forceinline__ void add(i32 i, i64 acc) const {
        __shared__ i32 lk[IC_SLOTS];
        __shared__ i64 lv[IC_SLOTS];
        lds_agg_clear<BS, IC_SLOTS>(lk, lv);
        if (i >= 0 && acc) table_add_lds(lk, lv, IC_SLOTS - 1, inst[i], acc);
        __syncthreads();
        for (int q = threadIdx.x; q < IC_SLOTS; q += BS)
            if (lk[q] != EMPTY_KEY && lv[q] != 0)
                atomicAdd((unsigned long long*)&sums[lk[q]], (unsigned long long)lv[q]);
    }
};

// One pass over the movers' edges (src/local_mover.cpp:1274-1277, 717, 798):
//  - the exact uncut change, per edge w * ([new_i == new_v] - [old_i ==
//    old_v]), counted once for mover pairs and twice for neighbours that stay
//    (the reference computes the same quantity from pvals);
//  - the neighbour's cached destination becomes NULL_PART (but RS_NONE).
// What bounds it is latency: each edge is a chain of dependent loads (column,
// neighbour word).  So a mover of degree below LARGE_CUTOFF takes MV_G lanes, one
// below MASSIVE_CUTOFF a 128-thread half block, the rest chunks of MV_CHUNK edges
// per block, and each thread has MV_U edges in flight.  As one thread per small
// mover and one wave per mid-size one, in a kernel each for the two jobs, they
// took 86 ms on R-MAT scale 20 (to stable), now 39 ms.
// The list holds the movers, or in direct sweeps every vertex, in order1 order
// (knew set: nothing is done when it counts any): those of degree >=
// LARGE_CUTOFF are a suffix of at most nw entries, those >= MASSIVE_CUTOFF one of at most nb.
constexpr int MV_G = 16, MV_U = 4;
constexpr i64 MV_CHUNK = 8192;
// RS_STORE resets with a store per edge.  Where a vertex is met by many movers'
// edges those stores meet on the same lines from every XCD and take most of the
// pass, and RS_TEST reads the destination first: when the movers have RS_TEST_DEG
// edges per vertex of the level or more, taken at its average degree (k * nnz / n
// >= RS_TEST_DEG * n).
// On a coarse level of R-MAT scale 24 (1.4M vertices with neighbours, about 280
// edges each) the first such sweep took 6.98 ms with stores, 4.75 with tests; on
// levels of 20 to 60 edges per vertex the tests cost 1 to 6% of a run.
enum ResetMode { RS_NONE, RS_STORE, RS_TEST };
constexpr double RS_TEST_DEG = 64.0;
template <int RESET, class WT, class AT>
__global__ void __launch_bounds__(256) k_move_edges(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                    const i32* __restrict__ moves, i64 k, i64 b1, i64 b2, i64 nw,
                                                    i64 nb, i64 cpm, const u64* __restrict__ mvp,
                                                    i32* __restrict__ dest, AT at, const i64* __restrict__ knew) {
    if (knew && *knew != 0) return;  // kernel-uniform: the host takes the movers from here
    const i64 b = block_id();
    i64 x;         // list entry
    int lane, gs;  // this thread among the gs threads of the entry
    i64 lo = 0, hi = 0, c0 = 0, cl = (i64)1 << 62;
    if (b < b1) {
        x = b * (256 / MV_G) + threadIdx.x / MV_G;
        lane = threadIdx.x & (MV_G - 1);
        gs = MV_G;
        hi = LARGE_CUTOFF;
        if (x >= k) x = -1;
    } else if (b < b1 + b2) {
        const i64 w = (b - b1) * 2 + (threadIdx.x >> 7);
        x = w < nw ? k - 1 - w : -1;
        lane = threadIdx.x & 127;
        gs = 128;
        lo = LARGE_CUTOFF;
        hi = MASSIVE_CUTOFF;
    } else {
        const i64 w = (b - b1 - b2) / cpm;
        x = w < nb ? k - 1 - w : -1;
        lane = threadIdx.x;
        gs = 256;
        lo = MASSIVE_CUTOFF;
        hi = (i64)1 << 62;
        c0 = ((b - b1 - b2) % cpm) * MV_CHUNK;
        cl = MV_CHUNK;
    }
    i64 acc = 0;
    i32 i = -1;
    if (x >= 0) {
        i = moves[x];
        const i64 s0 = rp[i], d = rp[i + 1] - s0;
        const u64 me = mvp[i];
        const i32 oi = (i32)((u32)me & 0x7fffffffu), ni = (i32)(u32)(me >> 32);
        const bool moved = ((u32)me >> 31) != 0;
        if (moved && d >= lo && d < hi && c0 < d) {
            const i64 e = s0 + (d < c0 + cl ? d : c0 + cl);
            for (i64 jb = s0 + c0 + lane; jb < e; jb += (i64)gs * MV_U) {
                i32 v[MV_U];
                u64 q[MV_U];
#pragma unroll
                for (int u = 0; u < MV_U; u++) {
                    const i64 j = jb + (i64)u * gs;
                    v[u] = j < e ? col[j] : -1;
                }
#pragma unroll
                for (int u = 0; u < MV_U; u++) q[u] = v[u] >= 0 ? mvp[v[u]] : 0;
                i32 dv[MV_U];
                if (RESET == RS_TEST) {
#pragma unroll
                    for (int u = 0; u < MV_U; u++) dv[u] = v[u] >= 0 ? dest[v[u]] : NULL_PART;
                }
#pragma unroll
                for (int u = 0; u < MV_U; u++) {
                    if (v[u] < 0) continue;
                    if (RESET == RS_STORE || (RESET == RS_TEST && dv[u] != NULL_PART)) dest[v[u]] = NULL_PART;
                    const i64 w = W(jb + (i64)u * gs);
                    const u32 ql = (u32)q[u];
                    const i32 ov = (i32)(ql & 0x7fffffffu), nv = (i32)(u32)(q[u] >> 32);
                    const i64 dd = (i64)(ni == nv) - (i64)(oi == ov);
                    acc += dd * w * ((ql >> 31) ? 1 : 2);
                }
            }
        }
    }
    at.template add<256>(i, acc);
}

// The volume changes of a block's 256 movers are merged per cluster in an
// LDS table first (many movers of a sweep leave or join the same clusters),
// then each distinct cluster gets one HBM atomic; the sums are exact
// integers, so the order does not matter.  The movers' words and cached
// destinations are settled for the next sweep.
// In direct sweeps (info set) every vertex is looked at, k of them, and the
// movers and candidates are counted.
constexpr int AM_SLOTS = 1024;  // >= 2 keys per mover of a 256-thread block, at most half full
__global__ void __launch_bounds__(256) k_apply_moves(const i32* __restrict__ moves, i64 k,
                                                     const i64* __restrict__ vw, u64* __restrict__ mvp,
                                                     i32* __restrict__ part, i32* __restrict__ dest, i64* vol,
                                                     const AbInfo* __restrict__ info, i64* scal) {
    __shared__ i32 lk[AM_SLOTS];
    __shared__ i64 lv[AM_SLOTS];
    if (info && scal[SC_NEW] != 0) return;  // kernel-uniform
    const i64 x = thread_item();
    i32 i = -1;
    u64 q = 0;
    if (x < k) {
        i = moves ? moves[x] : (i32)x;
        q = mvp[i];
        if (((u32)q >> 31) == 0) i = -1;
    }
    if (info) {
        const int km = __syncthreads_count(i >= 0);
        const int kc = __syncthreads_count(x < k && info[x < k ? x : 0].dest != NO_MOVE);
        if (threadIdx.x == 0) {
            const i64 w = block_id() & (MV_SLOTS - 1);
            if (km) atomicAdd((unsigned long long*)&scal[SC_KM + w], (unsigned long long)km);
            if (kc) atomicAdd((unsigned long long*)&scal[SC_CAND + w], (unsigned long long)kc);
        }
        if (km == 0) return;  // block-uniform
    }
    lds_agg_clear<256, AM_SLOTS>(lk, lv);
    if (i >= 0) {
        const i32 p = (i32)((u32)q & 0x7fffffffu);
        i32 b = (i32)(u32)(q >> 32);
        if (b >= 0) {  // unresolved NEW_PART cannot reach here (p_conn is 0 for singletons)
            const i64 w = vw[i];
            table_add_lds(lk, lv, AM_SLOTS - 1, p, -w);
            table_add_lds(lk, lv, AM_SLOTS - 1, b, w);
            part[i] = b;
        } else {
            b = p;
        }
        mvp[i] = mvp_settled(b);
        dest[i] = NULL_PART;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < AM_SLOTS; q += 256) {
        const i32 key = lk[q];
        const i64 v = lv[q];
        if (key != EMPTY_KEY && v != 0) atomicAdd((unsigned long long*)&vol[key], (unsigned long long)v);
    }
}

// End of a sweep: the exact 128-bit sum of squared volumes and the sums over
// the slots, stored to the host slots by the last block to finish: host[0] =
// uncut change, host[1..2] = sum of squares high and low, and in direct sweeps
// host[3] = movers, host[4] = candidates, host[5] = movers that need a new
// cluster.  rec / rec16 set: the vertices' records for the next sweep too.  One
// launch instead of seven (fills, two reductions of two kernels each,
// read-back): on small levels the sweep is bound by launches.
struct Sq128 {
    u64 hi, lo;
};
__device__ __forceinline__ Sq128 add_sq(Sq128 a, Sq128 b) {
    const u64 lo = a.lo + b.lo;
    return Sq128{a.hi + b.hi + (lo < a.lo ? 1 : 0), lo};
}
// over the block's 256 threads; thread 0 gets the result
__device__ __forceinline__ Sq128 block_sq(Sq128 v) {
    __shared__ Sq128 sh[4];
    xlane_fence(v.hi);
    xlane_fence(v.lo);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = add_sq(v, Sq128{(u64)__shfl_xor(v.hi, o), (u64)__shfl_xor(v.lo, o)});
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < 4; w++) v = add_sq(v, sh[w]);
    __syncthreads();
    return v;
}
__global__ void __launch_bounds__(256) k_finish(const i64* __restrict__ vol, i64 L, u64* part, i64* scal, i64* host,
                                                i64 n, const i32* __restrict__ label, const i32* __restrict__ cons,
                                                u64* __restrict__ rec, uint4* __restrict__ rec16) {
    const int t = threadIdx.x;
    for (i64 x = (i64)blockIdx.x * 256 + t; x < n; x += (i64)gridDim.x * 256)
        rec_pack(x, label, vol, cons, rec, rec16);
    Sq128 sq{0, 0};
    for (i64 xb = (i64)blockIdx.x * 256; xb < L; xb += (i64)gridDim.x * 256) {  // block-uniform loop control
        const i64 x = xb + t;
        const i64 v = x < L ? vol[x] : 0;
        const u64 a = (u64)(v < 0 ? -v : v);
        sq = add_sq(sq, Sq128{__umul64hi(a, a), a * a});
    }
    sq = block_sq(sq);
    if (gridDim.x > 1) {
        __shared__ int last;
        if (t == 0) {
            // agent-scope stores and loads: the blocks run on different XCDs
            __hip_atomic_store(&part[2 * blockIdx.x], sq.hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&part[2 * blockIdx.x + 1], sq.lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __threadfence();
            last = atomicAdd((unsigned long long*)&scal[SC_TICKET], 1ull) == gridDim.x - 1;
        }
        __syncthreads();
        if (!last) return;  // block-uniform
        __threadfence();
        sq = Sq128{0, 0};
        if (t < (int)gridDim.x)  // gridDim.x <= FIN_BLOCKS
            sq = Sq128{__hip_atomic_load(&part[2 * t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                       __hip_atomic_load(&part[2 * t + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
        sq = block_sq(sq);
    }
    static_assert(MV_SLOTS == 64, "a wave sums each group of slots");
    if (t < 64) {  // the first wave sums the slots and reports
        i64 du = scal[SC_SLOTS + t], km = scal[SC_KM + t], kc = scal[SC_CAND + t];
        scal[SC_SLOTS + t] = scal[SC_KM + t] = scal[SC_CAND + t] = 0;
        const auto sum = [](i64 a, i64 b) { return a + b; };
        du = group_reduce<64>(du, sum);
        km = group_reduce<64>(km, sum);
        kc = group_reduce<64>(kc, sum);
        if (t == 0) {  // (the end of the kernel makes them visible to the host)
            host[0] = du;
            host[1] = (i64)sq.hi;
            host[2] = (i64)sq.lo;
            host[3] = km;
            host[4] = kc;
            host[5] = scal[SC_NEW];
            scal[SC_NEW] = 0;
            scal[SC_TICKET] = 0;
        }
    }
}

// perform_moves (src/local_mover.cpp:1241-1279).  moves is in order1 order;
// n_large / n_massive = vertices of the level with degree >= LARGE_CUTOFF /
// MASSIVE_CUTOFF, which bound the movers of the last two classes.  The uncut
// change goes to `at`.
// reset: the movers' neighbours are scored again in the next sweep.  marked:
// the movers' words are in mvp already.  direct: moves lists every vertex.
template <class AT>
static void apply_moves_core(Ctx& c, MoveScratch& s, const LevelPlan& lp, const DGraph& g, i64* vol, const i32* moves,
                             i64 k, bool marked, i64 n_large, i64 n_massive, bool reset, AT at,
                             bool direct = false) {
    const i64 nw = std::min(k, n_large);
    const i64 nb = std::min(k, n_massive);
    if (!marked) {
        k_mvp_moves<<<grid_items(k, 256), 256, 0, c.stream>>>(moves, k, s.part, s.dest, s.mvp);
        PGGC_LAUNCH_CHECK();
    }
    Buf<i64> acct;
    if (c.kt.on) {  // timing runs only
        // per mover its word (written, read, settled), row bounds, cluster,
        // destination, vertex weight and two volume updates; per mover edge
        // the column, weight, the neighbour's word and its destination reset
        const int wb = g.wk == W_UNIT ? 0 : g.wk == W_I32 ? 4 : 8;
        acct = Buf<i64>(c, 1);
        fill_i64(c, acct, 1, 0);
        k_list_bytes<<<grid_items(std::max<i64>(k, 1), 256), 256, 0, c.stream>>>(
            g.rp, moves, nullptr, s.mvp, k, 84, 12 + wb + (reset ? 4 : 0), 0, acct);
        PGGC_LAUNCH_CHECK();
    }
    const int tk = c.kt_begin(KS_MOVES);
    const i64 cpm = nb > 0 ? ceil_div(lp.max_deg, MV_CHUNK) : 1;
    const i64* knew = direct ? s.scal.p + SC_NEW : nullptr;
    const i64 b1 = ceil_div(k, 256 / MV_G), b2 = ceil_div(nw, 2), b3 = nb * cpm;
#define PGGC_MOVE_EDGES(RS)                                                                                          \
    k_move_edges<RS><<<grid_blocks(b1 + b2 + b3), 256, 0, c.stream>>>(g.rp, g.col, W, moves, k, b1, b2, nw, nb, cpm,  \
                                                                      s.mvp, s.dest, at, knew)
    const bool test = (double)k * (double)g.nnz >= RS_TEST_DEG * (double)g.n * (double)g.n;
    PGGC_WDISPATCH(g, {
        if (!reset) PGGC_MOVE_EDGES(RS_NONE);
        else if (test) PGGC_MOVE_EDGES(RS_TEST);
        else PGGC_MOVE_EDGES(RS_STORE);
    });
#undef PGGC_MOVE_EDGES
    PGGC_LAUNCH_CHECK();
    k_apply_moves<<<grid_items(k, 256), 256, 0, c.stream>>>(direct ? nullptr : moves, k, g.vw, s.mvp, s.part, s.dest, vol,
                                                            direct ? s.abi.p : nullptr, s.scal);
    c.kt_end(tk, 0.0);
    PGGC_LAUNCH_CHECK();
    if (tk >= 0) acct_add(c, c.kt_counter(tk), acct);
}

// k_finish, and its results; the first n vertices' records when n > 0
static const i64* finish_sweep(Ctx& c, MoveScratch& s, const RefineData& curr, i64 n, const i32* cons) {
    const i64 L = curr.label_count;
    if (n > 0 && cons && s.rec16.n < (size_t)n) s.rec16 = Buf<uint4>(c, s.cap);
    k_finish<<<grid_for(std::max<i64>(std::max(L, n), 1), 256 * 4, FIN_BLOCKS), 256, 0, c.stream>>>(
        curr.vol, L, s.sqpart, s.scal, c.pinned_dev, n, s.part, cons, s.rec, cons ? s.rec16.p : nullptr);
    PGGC_LAUNCH_CHECK();
    c.sync();
    return c.pinned;
}

static void init_mvp(Ctx& c, MoveScratch& s, i64 n) {
    if (n <= 0) return;
    k_mvp_init<<<grid_items(n, 256), 256, 0, c.stream>>>(n, s.part, s.mvp, s.scal);
    PGGC_LAUNCH_CHECK();
}

static void perform_moves(Ctx& c, MoveScratch& s, const LevelPlan& lp, const DGraph& g, RefineData& curr,
                          const i32* moves, i64 k, bool marked, i64 n_large, i64 n_massive, bool& tables) {
    apply_moves_core(c, s, lp, g, curr.vol, moves, k, marked, n_large, n_massive, tables, AccOne{s.scal.p + SC_SLOTS});
    if (!tables) {
        tables = true;
        fill_i32(c, s.dest, g.n, NULL_PART);
    }
    const i64* h = finish_sweep(c, s, curr, 0, nullptr);
    curr.uncut += h[0];
    curr.obj = objective_value(curr.uncut, curr.lambda, (u64)h[1], (u64)h[2]);
}

// ------------------------------------------------------------- relabel
// the pos-th used label becomes label pos
struct SelLabels {
    static constexpr bool extra = false;
    const i32* used;
    const i64* vol;
    i64* nvol;
    i32* map;
    __device__ __forceinline__ bool test(i64 l) const { return used[l] != 0; }
    __device__ __forceinline__ void emit(i64 pos, i64 l) const {
        nvol[pos] = vol[l];
        map[l] = (i32)pos;
    }
};
__global__ void k_relabel_part(const i32* map, i64 n, i32* part) {
    const i64 i = thread_item();
    if (i >= n) return;
    part[i] = map[part[i]];
}

// relabel_contiguously (src/local_mover.cpp:100-129)
static void relabel(Ctx& c, MoveScratch& s, i64 n, i32* labels, RefineData& rd) {
    const i64 L = rd.label_count;
    fill_i32(c, s.flag, L, 0);
    k_mark_used<<<grid_items(n, 256), 256, 0, c.stream>>>(labels, n, s.flag);
    PGGC_LAUNCH_CHECK();
    Buf<i32> map(c, std::max<i64>(L, 1));
    Buf<i64> nvol(c, std::max<i64>(L, 1));
    const i64 t = select_items(c, SelLabels{s.flag, rd.vol, nvol, map}, L)[0];
    copy_dev(c, rd.vol, nvol, t * sizeof(i64));
    k_relabel_part<<<grid_items(n, 256), 256, 0, c.stream>>>(map, n, labels);
    PGGC_LAUNCH_CHECK();
    rd.label_count = (i32)t;
}

static void copy_state(Ctx& c, RefineData& dst, const RefineData& src) {
    if (src.label_count > dst.cap) throw Error(-4, "label capacity exceeded");
    copy_dev(c, dst.vol, src.vol, (size_t)src.label_count * sizeof(i64));
    dst.top_nnz = src.top_nnz;
    dst.uncut = src.uncut;
    dst.obj = src.obj;
    dst.label_count = src.label_count;
    dst.lambda = src.lambda;
}

// the best state so far: volumes and clusters, on small levels in one launch
__global__ void __launch_bounds__(256) k_copy_best(const i64* __restrict__ vol, i64 L, i64* __restrict__ bvol,
                                                   const i32* __restrict__ part, i64 n, i32* __restrict__ bpart) {
    const i64 x = thread_item();
    if (x < L) bvol[x] = vol[x];
    if (x < n) bpart[x] = part[x];
}
static void copy_best(Ctx& c, RefineData& best, const RefineData& curr, i32* best_part, const i32* part, i64 n) {
    const i64 L = curr.label_count;
    if (std::max(n, L) > DIRECT_MAX) {  // 16-byte words
        copy_state(c, best, curr);
        copy_dev(c, best_part, part, n * sizeof(i32));
        return;
    }
    if (L > best.cap) throw Error(-4, "label capacity exceeded");
    k_copy_best<<<grid_items(std::max(n, L), 256), 256, 0, c.stream>>>(curr.vol, L, best.vol, part, n, best_part);
    PGGC_LAUNCH_CHECK();
    i64* vol = best.vol;
    const i64 cap = best.cap;
    const double scale = best.scale, offset = best.offset;
    best = curr;
    best.vol = vol;
    best.cap = cap;
    best.scale = scale;
    best.offset = offset;
}

// ------------------------------------------------------------- drivers

// ------------------------------------------------------------ sweep trace
__global__ void __launch_bounds__(256) k_count_active(const i32* dest, i64 n, i64* out) {
    const i64 i = thread_item();
    const i64 a = (i < n && dest[i] != NO_MOVE) ? 1 : 0;
    const i64 s = block_sum_i64<256>(a);
    if (threadIdx.x == 0 && s) atomicAdd((unsigned long long*)out, (unsigned long long)s);
}

// Host side of the per-sweep trace: begin() counts the vertices the sweep
// will score and starts the clock, end() reports the record.  Both are
// no-ops unless a trace callback is set.
struct SweepTrace {
    Ctx& c;
    const DGraph& g;
    i64 phase, sweep = 0, active = 0;
    i64 n;      // vertices of the level
    i64 inert;  // of them left out of g, and counted while every vertex is active
    std::chrono::steady_clock::time_point t0;
    SweepTrace(Ctx& cc, const DGraph& gg, i64 ph, i64 nfull) : c(cc), g(gg), phase(ph), n(nfull), inert(nfull - gg.n) {}
    void begin(const i32* dest, bool all, bool fresh = false) {
        if (!c.sweep_trace) return;
        if (all) {
            active = n;
        } else {
            Buf<i64> cnt(c, 1);
            fill_i64(c, cnt, 1, 0);
            if (g.n > 0) {
                k_count_active<<<grid_items(g.n, 256), 256, 0, c.stream>>>(dest, g.n, cnt);
                PGGC_LAUNCH_CHECK();
            }
            active = c.read1(cnt) + (fresh ? inert : 0);
        }
        c.sync();
        t0 = std::chrono::steady_clock::now();
    }
    void end(i64 cands, i64 moves) {
        if (!c.sweep_trace) return;
        c.sync();
        const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
        const int64_t rec[8] = {n, g.nnz, phase, sweep++, active, cands, moves, (int64_t)us};
        c.sweep_trace(c.sweep_user, rec, 8);
    }
};

static RefineData begin_curr(Ctx& c, const RefineData& best, Buf<i64>& cv, i64 n) {
    i64 cap = std::max<i64>(best.cap, n);
    cv = Buf<i64>(c, cap + 1);
    RefineData curr = best;
    curr.vol = cv;
    curr.cap = cap;
    return curr;
}
static void move_begin(Ctx& c, MoveScratch& s, const RefineData& best, RefineData& curr, const i32* best_part, i64 n,
                       i64 nfull) {
    const i64 L = best.label_count;
    if (L > curr.cap) throw Error(-4, "label capacity exceeded");
    k_move_begin<<<grid_items(std::max<i64>(std::max(L, nfull), SC_COUNT), 256), 256, 0, c.stream>>>(
        best.vol, L, curr.vol, best_part, nfull, s.part, n, s.mvp, s.dest, s.scal);
    PGGC_LAUNCH_CHECK();
}

// the sweep's movers from its scored vertices
template <class LT, class PT>
static Movers find_movers(Ctx& c, MoveScratch& s, const LevelPlan& lp, const DGraph& g, LT lam, PT prio, bool pack) {
    i64 b[2];
    const i64 k = gather_candidates(c, lp, g, s.dest, s.cand, b);
    if (k == 0) return Movers{0, 0, 0};
    afterburner(c, s, g, s.cand, k, b, lam, prio, pack);
    return select_movers(c, s, s.cand, k, s.moves);
}

// Filter and moves of a small level's sweep without lists and with one
// read-back: the afterburner runs over all vertices and marks the movers, the
// move kernels look at every vertex's mark, and the end of the sweep reports
// the counts and packs the next sweep's records.  Levels of at most DIRECT_MAX
// vertices and DIRECT_NNZ nonzeros: they are bound by launches and waits (a
// sweep takes 7 launches and 1 wait; with lists 10 and 2, at first 34 and 5 or
// 6).  Larger levels would spend lanes on the vertices that are no candidates
// or do not move: the coarse level of R-MAT scale 20 (108,000 vertices, 30M
// nonzeros) took 55 us per sweep in k_move_edges that way, with lists 36.
// When movers need new cluster ids the move kernels leave everything as it is,
// and the movers are selected, numbered and moved as on large levels.
template <class LT, class PT>
static Movers direct_sweep(Ctx& c, MoveScratch& s, const LevelPlan& lp, const DGraph& g, RefineData& curr, LT lam,
                           PT prio, bool first, i32* cons, const i32* ids, i64 nfull, bool& tables, bool& fresh,
                           bool& packed) {
    const i64 n = g.n, n_large = n - lp.ord.off_large, n_massive = n - lp.ord.off_large2;
    const i64 b[2] = {lp.ord.off_large, lp.ord.off_large2};
    const i32* o1 = lp.ord.o1;
    afterburner(c, s, g, o1, n, b, lam, prio, false, AbMark{s.mvp, s.scal.p + SC_NEW});
    apply_moves_core(c, s, lp, g, curr.vol, o1, n, true, n_large, n_massive, tables, AccOne{s.scal.p + SC_SLOTS}, true);
    const i64* h = finish_sweep(c, s, curr, n, cons);
    Movers mv{h[3], h[5], h[4]};
    if (mv.knew > 0) {
        mv = select_movers(c, s, o1, n, s.moves);
        // (the first sweep of an initial call gives no new ids)
        if (!first) set_new_cluster_ids(c, s, g, curr, s.moves, mv.k, cons, ids, nfull);
        fresh = !tables;
        perform_moves(c, s, lp, g, curr, s.moves, mv.k, false, n_large, n_massive, tables);
        return mv;
    }
    packed = true;
    if (mv.k == 0) return mv;
    curr.uncut += h[0];
    curr.obj = objective_value(curr.uncut, curr.lambda, (u64)h[1], (u64)h[2]);
    fresh = !tables;
    if (!tables) {
        tables = true;
        fill_i32(c, s.dest, n, NULL_PART);
    }
    return mv;
}

static void sweep_note(const Ctx& c, i64 n, int iter, const Movers& mv, const RefineData& curr) {
    if (c.verbose < 3) return;
    fprintf(stderr, "sweep n=%lld it=%d cands=%lld moves=%lld labels=%d uncut=%lld obj=%.17g\n", (long long)n, iter,
            (long long)mv.cands, (long long)mv.k, curr.label_count, (long long)curr.uncut, curr.obj);
}

template <class PT>
static void local_move_t(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, i32* best_part, RefineData& best,
                         bool is_initial, bool constrained, i32* cons, bool SA, MoveStats* stats, PT prio,
                         const i32* ids, i64 nfull);

void local_move(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, i32* best_part, RefineData& best,
                bool is_initial, bool constrained, i32* cons, bool SA, MoveStats* stats, const i32* ids, i64 nfull) {
    if (nfull < 0) nfull = g.n;
    if (ids) {
        local_move_t(c, s, lp, g, best_part, best, is_initial, constrained, cons, SA, stats, PrioInst{ids}, ids,
                     nfull);
    } else {
        local_move_t(c, s, lp, g, best_part, best, is_initial, constrained, cons, SA, stats, PrioOne{}, nullptr,
                     nfull);
    }
}

template <class PT>
static void local_move_t(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, i32* best_part, RefineData& best,
                         bool is_initial, bool constrained, i32* cons, bool SA, MoveStats* stats, PT prio,
                         const i32* ids, i64 nfull) {
    const i64 n = g.n;
    s.ensure(c, nfull);
    plan_level(c, g, lp);
    c.mem_note("local move: plan ready");
    Buf<i64> cv;
    RefineData curr = begin_curr(c, best, cv, nfull);
    move_begin(c, s, best, curr, best_part, n, nfull);
    bool tables = !is_initial;
    const float ratios[2] = {0.75f, 0.25f};
    const int limits[2] = {4, 2};
    int iter = 0;
    const i32* ccons = constrained ? cons : nullptr;
    const int raw_mode = c.raw_sweeps ? 1 : 0;
    SweepTrace tr(c, g, is_initial ? 0 : 1, nfull);
    // active-set predictor: on levels of at least min_nnz nonzeros, from the
    // second sweep of a call that starts at singletons (whose first sweep
    // moves most vertices), from the first sweep otherwise, and only while
    // the previous sweep left at least n/16 candidates (below that the
    // active set is mostly the movers' neighbourhood and little is to gain)
    Gnn* G = (s.gnn && s.gnn->cfg.mode != GNN_OFF && g.nnz >= s.gnn->cfg.min_nnz) ? s.gnn : nullptr;
    const bool train = G && G->cfg.mode == GNN_TRAIN;
    // pruned vertices are not scored, so with the predictor on the records
    // are packed from the arrays
    const ScoreOut so = G ? ScoreOut{s.dest, s.gain, nullptr} : ScoreOut{s.dest, nullptr, s.abi};
    if (G) gnn_begin(c, *G, n, train);
    i64 kprev = n;
    i64 npred = 0;  // predicted sweeps in this call
    bool fresh = false;   // every vertex was made active by the last sweep
    bool packed = false;  // the last sweep packed this one's records
    for (int x = 0; x < 2; x++) {
        const float fr = SA ? ratios[x] : 0.0f;
        for (int cnt = 0; cnt < limits[x]; cnt++) {
            iter++;
            const LamOne lam{(float)curr.lambda};
            const bool use = G && !(is_initial && iter == 1) && kprev * 16 >= n &&
                             (c.gnn_max_sweeps <= 0 || npred < c.gnn_max_sweeps);
            const bool full = use && G->cfg.full_every > 0 && iter % G->cfg.full_every == 0;
            if (full) gnn_restore(c, *G, n, s.dest);
            if (use && !full) {
                gnn_predict(c, *G, lp, g, s.part, s.dest, s.gain, curr.vol, iter, iter == 1,
                            G->cfg.mode == GNN_PRUNE, train);
                npred++;
            }
            tr.begin(s.dest, iter == 1 && !use, fresh);
            fresh = false;
            score_all(c, s, lp, g, s.part, curr.vol, ccons, tables ? 0 : raw_mode, lam, fr, so, packed);
            packed = false;
            if (n <= DIRECT_MAX && g.nnz <= DIRECT_NNZ && !G && n > 0) {
                const Movers mv = direct_sweep(c, s, lp, g, curr, lam, prio, is_initial && iter == 1,
                                               constrained ? cons : nullptr, ids, nfull, tables, fresh, packed);
                if (stats) {
                    stats->sweeps++;
                    stats->cands += mv.cands;
                    stats->moves += mv.k;
                }
                sweep_note(c, nfull, iter, mv, curr);
                if (mv.k > 0 && curr.obj > best.obj) copy_best(c, best, curr, best_part, s.part, n);
                tr.end(mv.cands, mv.k);
                if (mv.k == 0) break;
                continue;
            }
            Movers mv = find_movers(c, s, lp, g, lam, prio, so.info == nullptr);
            if (mv.k == 0 && G && gnn_restore(c, *G, n, s.dest)) {
                // nothing to move among the vertices let through: score the
                // pruned ones too, so the call ends as the plain method does
                score_all(c, s, lp, g, s.part, curr.vol, ccons, tables ? 0 : raw_mode, lam, fr, so);
                mv = find_movers(c, s, lp, g, lam, prio, so.info == nullptr);
            }
            const i64 k = mv.cands, km = mv.k;
            if (stats) {
                stats->sweeps++;
                stats->cands += k;
            }
            kprev = k;
            if (G) gnn_stamp(c, *G, s.moves, km, iter);
            if (train && use && !full) gnn_backward(c, *G, lp, g, nullptr, iter, true);
            if (k == 0) {
                tr.end(0, 0);
                break;
            }
            if (km == 0) {
                tr.end(k, 0);
                break;
            }
            // (the first sweep of an initial call has no NEW_PART movers)
            const bool fresh_ids = mv.knew > 0 && (iter > 1 || !is_initial);
            if (fresh_ids)
                set_new_cluster_ids(c, s, g, curr, s.moves, km, constrained ? cons : nullptr, ids, nfull);
            fresh = !tables;
            perform_moves(c, s, lp, g, curr, s.moves, km, !fresh_ids, g.n - lp.ord.off_large, g.n - lp.ord.off_large2, tables);
            if (stats) stats->moves += km;
            sweep_note(c, nfull, iter, mv, curr);
            if (curr.obj > best.obj) copy_best(c, best, curr, best_part, s.part, n);
            tr.end(k, km);
        }
    }
    relabel(c, s, nfull, best_part, best);
    s.hub_buf.reset();
}

// afterburner_filter_strict (src/local_mover.cpp:131-213): exact sequential
// FP32 evaluation of each move given all earlier moves in list order.
__global__ void k_prio(const i32* moves, i64 k, i64* prio) {
    const i64 x = thread_item();
    if (x >= k) return;
    prio[moves[x]] = x;
}

template <class WT>
__global__ void __launch_bounds__(256) k_strict_gain(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                     const i64* __restrict__ vw, const i32* __restrict__ moves,
                                                     i64 k, const i64* __restrict__ prio,
                                                     const i32* __restrict__ part, const i32* __restrict__ dest,
                                                     const float* __restrict__ gain, float lam, float* sg) {
    const i64 x = thread_item();
    if (x >= k) return;
    const i32 i = moves[x];
    const i32 best = dest[i], p = part[i];
    const float multi = (float)vw[i] * lam;
    float oc = gain[i];
    const i64 pi = prio[i];
    for (i64 j = rp[i]; j < rp[i + 1]; j++) {
        const i32 v = col[j];
        const i64 wgt = W(j);
        if (prio[v] < pi) {
            i32 vp = dest[v];
            oc = oc - (float)((vp == p) ? wgt : 0);
            oc = oc + (float)((vp == best && best != NEW_PART) ? wgt : 0);
            vp = part[v];
            oc = oc + (float)((vp == p) ? wgt : 0);
            oc = oc - (float)((vp == best) ? wgt : 0);
        }
    }
    for (i64 jx = 0; jx < x; jx++) {
        const i32 v = moves[jx];
        i32 vp = dest[v];
        const float wg = -multi * (float)vw[v];
        oc = oc - ((vp == p) ? wg : 0.0f);
        oc = oc + ((vp == best && best != NEW_PART) ? wg : 0.0f);
        vp = part[v];
        oc = oc + ((vp == p) ? wg : 0.0f);
        oc = oc - ((vp == best) ? wg : 0.0f);
    }
    sg[x] = oc;
}

// sequential inclusive FP32 prefix sum and first arg-max (one thread)
__global__ void k_strict_scan(const i32* moves, i64 k, float* sg, float* gain, i64* out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    float run = 0.0f, bv = -1.0f;
    i64 bl = -1;
    for (i64 x = 0; x < k; x++) {
        run = run + sg[x];
        sg[x] = run;
        gain[moves[x]] = run;
        if (run > bv) {
            bv = run;
            bl = x;
        }
    }
    out[0] = (bl >= 0 && bv > 0.0f) ? bl + 1 : 0;
}

void local_move_strict(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, i32* best_part, RefineData& best,
                       bool is_initial, bool constrained, i32* cons, MoveStats* stats) {
    const i64 n = g.n;
    s.ensure(c, n);
    plan_level(c, g, lp);
    Buf<i64> cv;
    RefineData curr = begin_curr(c, best, cv, n);
    move_begin(c, s, best, curr, best_part, n, n);
    bool tables = !is_initial;
    const i32* ccons = constrained ? cons : nullptr;
    Buf<float> sg(c, std::max<i64>(n, 1));
    SweepTrace trc(c, g, 2, n);
    for (int it = 0; it < 6; it++) {
        const float lam = (float)curr.lambda;
        trc.begin(s.dest, true);
        score_all(c, s, lp, g, s.part, curr.vol, ccons, !tables && c.raw_sweeps, LamOne{lam}, 0.0f,
                  ScoreOut{s.dest, s.gain, nullptr});
        i64 b[2];
        i64 k = gather_candidates(c, lp, g, s.dest, s.moves, b);
        if (stats) {
            stats->sweeps++;
            stats->cands += k;
        }
        if (k == 0) {
            trc.end(0, 0);
            break;
        }
        if (it > 0 || !is_initial) set_new_cluster_ids(c, s, g, curr, s.moves, k, constrained ? cons : nullptr, nullptr, n);
        fill_i64(c, s.prio, n, n + 1);
        k_prio<<<grid_items(k, 256), 256, 0, c.stream>>>(s.moves, k, s.prio);
        PGGC_LAUNCH_CHECK();
        PGGC_WDISPATCH(g, (k_strict_gain<<<grid_items(k, 256), 256, 0, c.stream>>>(
                              g.rp, g.col, W, g.vw, s.moves, k, s.prio, s.part, s.dest, s.gain, lam, sg)));
        PGGC_LAUNCH_CHECK();
        k_strict_scan<<<1, 64, 0, c.stream>>>(s.moves, k, sg, s.gain, s.scal);
        PGGC_LAUNCH_CHECK();
        i64 tr = c.read1(s.scal);
        if (tr == 0) {
            trc.end(k, 0);
            break;
        }
        perform_moves(c, s, lp, g, curr, s.moves, tr, false, g.n - lp.ord.off_large, g.n - lp.ord.off_large2, tables);
        if (stats) stats->moves += tr;
        if (curr.obj > best.obj) copy_best(c, best, curr, best_part, s.part, n);
        fill_i32(c, s.dest, n, NULL_PART);
        trc.end(k, tr);
    }
    relabel(c, s, n, best_part, best);
    s.hub_buf.reset();
}

i64 sweep_once(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, const i32* part, const i64* vol, i64 L,
               double lambda, float ratio, bool raw, const i32* cons, i32* dest, float* gain, i32* moves_out,
               i64* ncand) {
    const i64 n = g.n;
    (void)L;
    s.ensure(c, n);
    plan_level(c, g, lp);
    copy_dev(c, s.part, part, n * sizeof(i32));
    copy_dev(c, s.dest, dest, n * sizeof(i32));
    copy_dev(c, s.gain, gain, n * sizeof(float));
    init_mvp(c, s, n);
    const float lam = (float)lambda;
    score_all(c, s, lp, g, s.part, vol, cons, raw, LamOne{lam}, ratio,
              ScoreOut{s.dest, s.gain, nullptr});
    i64 b[2];
    i64 k = gather_candidates(c, lp, g, s.dest, s.cand, b);
    *ncand = k;
    i64 km = 0;
    if (k > 0) {
        afterburner(c, s, g, s.cand, k, b, LamOne{lam}, PrioOne{}, true);
        km = select_movers(c, s, s.cand, k, moves_out).k;
    }
    copy_dev(c, dest, s.dest, n * sizeof(i32));
    copy_dev(c, gain, s.gain, n * sizeof(float));
    c.sync();
    s.hub_buf.reset();
    return km;
}


// ================================================================ batches
// A batch of graphs as one disjoint union (see BatchLevel): the sweep
// kernels run once over the union with per-instance lambda, ratio and
// priority ids; the control flow of local_move runs per instance on the host
// from per-instance counts read back once per sweep.
__global__ void k_batch_ids(i64 n, const i64* __restrict__ voff, i64 K, i32* __restrict__ inst,
                            i32* __restrict__ loc) {
    const i64 v = thread_item();
    if (v >= n) return;
    const i64 k = upper_row(voff, 0, K, v);  // last instance starting at or before v (skips empty ones)
    inst[v] = (i32)k;
    loc[v] = (i32)(v - voff[k]);
}

void BatchLevel::build(Ctx& c, const std::vector<i64>& offsets) {
    voff = offsets;
    K = (i64)voff.size() - 1;
    const i64 n = voff[K];
    dvoff = Buf<i64>(c, K + 1);
    copy_h2d(c, dvoff.p, voff.data(), (K + 1) * sizeof(i64));
    inst = Buf<i32>(c, std::max<i64>(n, 1));
    loc = Buf<i32>(c, std::max<i64>(n, 1));
    if (n > 0) {
        k_batch_ids<<<grid_items(n, 256), 256, 0, c.stream>>>(n, dvoff, K, inst, loc);
        PGGC_LAUNCH_CHECK();
    }
    c.sync();
}

template <class T>
static void upload(Ctx& c, T* dst, const std::vector<T>& src) {
    copy_h2d(c, dst, src.data(), src.size() * sizeof(T));
}
template <class T>
static void download(Ctx& c, std::vector<T>& dst, const T* src, size_t count) {
    const Fetch f = fetch(dst, src, count);
    copy_d2h(c, &f, 1);
}

// Per-instance sums.  A list holds long runs of one instance (instances own
// contiguous id ranges), so a block merges its 256 entries per instance in
// LDS and adds each distinct instance once: one HBM atomic per block instead
// of one per entry.  Per-entry atomics on a few dozen counters ran at the
// rate of one address: 241 us per launch on average over 48 instances
// (2.8M vertices), 6.4 ms for the largest list; merged 4-6 us.
__global__ void __launch_bounds__(256) k_inst_count(const i32* __restrict__ list, i64 k,
                                                    const i32* __restrict__ owner, i64* cnt) {
    __shared__ i32 lk[IC_SLOTS];
    __shared__ i64 lv[IC_SLOTS];
    lds_agg_clear<256, IC_SLOTS>(lk, lv);
    const i64 x = thread_item();
    if (x < k) table_add_lds(lk, lv, IC_SLOTS - 1, owner[list[x]], 1);
    __syncthreads();
    for (int q = threadIdx.x; q < IC_SLOTS; q += 256)
        if (lk[q] != EMPTY_KEY) atomicAdd((unsigned long long*)&cnt[lk[q]], (unsigned long long)lv[q]);
}
// vertices of instances outside this sweep are never scored
__global__ void k_inst_gate(i64 n, const i32* __restrict__ inst, const i32* __restrict__ on, i32* dest) {
    const i64 v = thread_item();
    if (v >= n) return;
    if (!on[inst[v]]) dest[v] = NO_MOVE;
}
__global__ void k_inst_fill(i64 n, const i32* __restrict__ inst, const i32* __restrict__ mask, i32* a, i32 val) {
    const i64 v = thread_item();
    if (v >= n) return;
    if (mask[inst[v]]) a[v] = val;
}
// exact 128-bit sum of squared volumes over each masked instance's labels
// [loff[k], loff[k] + L[k]); one block per instance, out[2k] = high word
__global__ void __launch_bounds__(256) k_inst_sumsq(const i64* __restrict__ vol, const i64* __restrict__ loff,
                                                    const i64* __restrict__ L, const i32* __restrict__ mask, i64 K,
                                                    u64* out) {
    const i64 k = block_id();
    if (k >= K) return;
    u64 lo = 0, hi = 0;
    if (mask[k]) {
        const i64 e = loff[k] + L[k];
        for (i64 l = loff[k] + threadIdx.x; l < e; l += 256) {
            const i64 v = vol[l];
            const u64 a = (u64)(v < 0 ? -v : v);
            const u64 plo = a * a, phi = __umul64hi(a, a);
            lo += plo;
            hi += phi + (lo < plo ? 1 : 0);
        }
    }
    __shared__ u64 slo[256], shi[256];
    slo[threadIdx.x] = lo;
    shi[threadIdx.x] = hi;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            const u64 a = slo[threadIdx.x], b = slo[threadIdx.x + o];
            slo[threadIdx.x] = a + b;
            shi[threadIdx.x] = shi[threadIdx.x] + shi[threadIdx.x + o] + (a + b < a ? 1 : 0);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[2 * k] = shi[0];
        out[2 * k + 1] = slo[0];
    }
}
__global__ void k_inst_copy_v(i64 n, const i32* __restrict__ inst, const i32* __restrict__ mask,
                              const i32* __restrict__ src, i32* dst) {
    const i64 v = thread_item();
    if (v >= n) return;
    if (mask[inst[v]]) dst[v] = src[v];
}
// labels l < loff[k] + L[k] of masked instances
__global__ void k_inst_copy_l(i64 nl, const i32* __restrict__ linst, const i64* __restrict__ loff,
                              const i64* __restrict__ L, const i32* __restrict__ mask, const i64* __restrict__ src,
                              i64* dst) {
    const i64 l = thread_item();
    if (l >= nl) return;
    const i32 k = linst[l];
    if (mask[k] && l - loff[k] < L[k]) dst[l] = src[l];
}
__global__ void k_unused_inst(i64 nl, const i32* __restrict__ used, const i32* __restrict__ linst,
                              const i64* __restrict__ loff, const i64* __restrict__ L, i32* flag) {
    const i64 l = thread_item();
    if (l >= nl) return;
    const i32 k = linst[l];
    flag[l] = (used[l] == 0 && l - loff[k] < L[k]) ? 1 : 0;
}
__global__ void k_inst_keys(const i32* __restrict__ list, i64 k, const i32* __restrict__ inst, u64* keys) {
    const i64 x = thread_item();
    if (x >= k) return;
    keys[x] = (u64)(u32)inst[list[x]];
}
// x-th NEW_PART mover of instance q (movers grouped by instance, in move
// order) takes the instance's x-th unused label, then labels appended after
// its label count (src/local_mover.cpp:215-274)
__global__ void k_assign_new_batch(const i32* __restrict__ np, i64 K_, const i32* __restrict__ inst,
                                   const i64* __restrict__ npstart, const i64* __restrict__ ustart,
                                   const i64* __restrict__ acnt, const i32* __restrict__ unused,
                                   const i64* __restrict__ loff, const i64* __restrict__ L, i32* dest) {
    const i64 x = thread_item();
    if (x >= K_) return;
    const i32 v = np[x];
    const i32 q = inst[v];
    const i64 r = x - npstart[q];
    dest[v] = r < acnt[q] ? unused[ustart[q] + r] : (i32)(loff[q] + L[q] + (r - acnt[q]));
}
__global__ void k_mark_used_inst(const i32* __restrict__ part, i64 n, const i32* __restrict__ inst,
                                 const i32* __restrict__ mask, i32* used) {
    const i64 v = thread_item();
    if (v >= n) return;
    if (mask[inst[v]]) used[part[v]] = 1;
}
__global__ void k_relabel_vol_inst(i64 nl, const i32* __restrict__ used, const i64* __restrict__ pos,
                                   const i32* __restrict__ linst, const i64* __restrict__ loff,
                                   const i64* __restrict__ vol, i64* nvol) {
    const i64 l = thread_item();
    if (l >= nl) return;
    if (!used[l]) return;
    const i32 k = linst[l];
    nvol[loff[k] + pos[l] - pos[loff[k]]] = vol[l];
}
__global__ void k_relabel_part_inst(i64 n, const i32* __restrict__ inst, const i32* __restrict__ mask,
                                    const i64* __restrict__ pos, const i64* __restrict__ loff, i32* part) {
    const i64 v = thread_item();
    if (v >= n) return;
    const i32 k = inst[v];
    if (mask[k]) part[v] = (i32)(loff[k] + pos[part[v]] - pos[loff[k]]);
}
__global__ void k_inst_newcount(i64 K, const i64* __restrict__ pos, const i64* __restrict__ loff,
                                const i64* __restrict__ L, i64* out) {
    const i64 k = thread_item();
    if (k >= K) return;
    out[k] = pos[loff[k] + L[k]] - pos[loff[k]];
}

static std::vector<i64> label_counts(const std::vector<RefineData>& rd) {
    std::vector<i64> L(rd.size());
    for (size_t k = 0; k < rd.size(); k++) L[k] = rd[k].label_count;
    return L;
}

// set_new_cluster_ids per instance over the batch's move list
static void set_new_cluster_ids_batch(Ctx& c, MoveScratch& s, const DGraph& g, const BatchLevel& bl,
                                      const BatchState& st, std::vector<RefineData>& cur, i64* vol,
                                      const i32* moves, i64 k) {
    const i64 K = bl.K, NL = st.loff[K];
    k_new_flags<<<grid_items(k, 256), 256, 0, c.stream>>>(moves, k, s.dest, s.flag);
    PGGC_LAUNCH_CHECK();
    const i64 KN = compact_flags(c, s.flag, moves, k, s.tmp);
    if (KN == 0) return;
    Buf<i64> Ld(c, K);
    upload(c, Ld.p, label_counts(cur));
    fill_i32(c, s.flag, NL, 0);
    k_mark_used<<<grid_items(g.n, 256), 256, 0, c.stream>>>(s.part, g.n, s.flag);
    Buf<i32> uf(c, std::max<i64>(NL, 1));
    k_unused_inst<<<grid_items(NL, 256), 256, 0, c.stream>>>(NL, s.flag, st.linst, st.dloff, Ld, uf);
    PGGC_LAUNCH_CHECK();
    const i64 A = compact_flags(c, uf, nullptr, NL, s.tmp2);
    Buf<i64> acnt(c, K), kcnt(c, K);
    fill_i64(c, acnt, K, 0);
    fill_i64(c, kcnt, K, 0);
    if (A > 0) k_inst_count<<<grid_items(A, 256), 256, 0, c.stream>>>(s.tmp2, A, st.linst, acnt);
    k_inst_count<<<grid_items(KN, 256), 256, 0, c.stream>>>(s.tmp, KN, bl.inst, kcnt);
    PGGC_LAUNCH_CHECK();
    {  // group the NEW_PART movers by instance, keeping move order inside each
        Buf<u64> keys(c, KN);
        k_inst_keys<<<grid_items(KN, 256), 256, 0, c.stream>>>(s.tmp, KN, bl.inst, keys);
        PGGC_LAUNCH_CHECK();
        int bits = 1;
        while (((i64)1 << bits) < K) bits++;
        radix_sort_pairs(c, keys, s.tmp.p, KN, bits);
    }
    std::vector<i64> ha, hk;
    const Fetch f[2] = {fetch(ha, acnt.p, K), fetch(hk, kcnt.p, K)};
    copy_d2h(c, f, 2);
    std::vector<i64> us(K), ns(K);
    i64 u0 = 0, n0 = 0;
    for (i64 q = 0; q < K; q++) {
        us[q] = u0;
        ns[q] = n0;
        u0 += ha[q];
        n0 += hk[q];
    }
    Buf<i64> dus(c, K), dns(c, K);
    upload(c, dus.p, us);
    upload(c, dns.p, ns);
    k_assign_new_batch<<<grid_items(KN, 256), 256, 0, c.stream>>>(s.tmp, KN, bl.inst, dns, dus, acnt, s.tmp2,
                                                                  st.dloff, Ld, s.dest);
    PGGC_LAUNCH_CHECK();
    for (i64 q = 0; q < K; q++) {
        const i64 need = hk[q] - ha[q];
        if (need <= 0) continue;
        const i64 L = cur[q].label_count;
        if (L + need > st.loff[q + 1] - st.loff[q]) throw Error(-4, "label capacity exceeded while assigning new clusters");
        fill_i64(c, vol + st.loff[q] + L, need, 0);
        cur[q].label_count = (i32)(L + need);
    }
}

// relabel_contiguously (src/local_mover.cpp:100-129) of every active instance
static void relabel_batch(Ctx& c, MoveScratch& s, const BatchLevel& bl, i32* labels, BatchState& st,
                          const std::vector<char>& active) {
    const i64 K = bl.K, NL = st.loff[K], n = bl.voff[K];
    std::vector<i32> ha(K);
    for (i64 q = 0; q < K; q++) ha[q] = active[q] ? 1 : 0;
    Buf<i32> act(c, K);
    upload(c, act.p, ha);
    Buf<i64> Ld(c, K);
    upload(c, Ld.p, label_counts(st.rd));
    fill_i32(c, s.flag, NL, 0);
    if (n > 0) k_mark_used_inst<<<grid_items(n, 256), 256, 0, c.stream>>>(labels, n, bl.inst, act, s.flag);
    PGGC_LAUNCH_CHECK();
    Buf<i64> pos(c, NL + 1), nvol(c, std::max<i64>(NL, 1)), nl(c, K);
    scan_i32_to_i64(c, s.flag, pos, NL);
    k_relabel_vol_inst<<<grid_items(NL, 256), 256, 0, c.stream>>>(NL, s.flag, pos, st.linst, st.dloff, st.vol, nvol);
    k_inst_newcount<<<grid_items(K, 256), 256, 0, c.stream>>>(K, pos, st.dloff, Ld, nl);
    k_inst_copy_l<<<grid_items(NL, 256), 256, 0, c.stream>>>(NL, st.linst, st.dloff, nl, act, nvol, st.vol);
    if (n > 0) k_relabel_part_inst<<<grid_items(n, 256), 256, 0, c.stream>>>(n, bl.inst, act, pos, st.dloff, labels);
    PGGC_LAUNCH_CHECK();
    std::vector<i64> hn;
    download(c, hn, nl.p, K);
    for (i64 q = 0; q < K; q++)
        if (active[q]) st.rd[q].label_count = (i32)hn[q];
}

// per-vertex lambda and filter ratio of a batch sweep (LamVert's tables)
__global__ void k_vertex_lam(i64 n, const i32* __restrict__ inst, const float* __restrict__ lam,
                             const float* __restrict__ ratio, float* __restrict__ vlam, float* __restrict__ vrat) {
    const i64 v = thread_item();
    if (v >= n) return;
    const i32 k = inst[v];
    vlam[v] = lam[k];
    vrat[v] = ratio[k];
}

void local_move_batch(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, const BatchLevel& bl,
                      i32* best_part, BatchState& best, bool is_initial, const std::vector<char>& active,
                      std::vector<MoveStats>& stats) {
    const i64 n = g.n, K = bl.K, NL = best.loff[K];
    s.ensure(c, std::max(n, NL));
    plan_level(c, g, lp);
    Buf<i64> cvol(c, std::max<i64>(NL, 1));
    copy_dev(c, cvol, best.vol, NL * sizeof(i64));
    std::vector<RefineData> cur = best.rd;
    copy_dev(c, s.part, best_part, n * sizeof(i32));
    init_mvp(c, s, n);
    fill_i32(c, s.dest, n, NULL_PART);
    Buf<i32> on(c, K), full(c, K), imp(c, K);
    Buf<float> rat(c, K);
    Buf<i64> cnt2(c, 2 * K), acc(c, K), Ld(c, K);
    Buf<u64> sq(c, 2 * K);
    const float ratios[2] = {0.75f, 0.25f};
    const int limits[2] = {4, 2};
    std::vector<int> phase(K, 0), cnt(K, 0), iter(K, 0);
    std::vector<char> tables(K, is_initial ? 0 : 1), done(K);
    for (i64 q = 0; q < K; q++) done[q] = !active[q];
    Buf<float> vlam(c, std::max<i64>(n, 1)), vrat(c, std::max<i64>(n, 1));
    const LamVert lam{vlam.p, vrat.p};
    const PrioInst prio{bl.loc.p};
    const i64 n_large = g.n - lp.ord.off_large, n_massive = g.n - lp.ord.off_large2;
    std::vector<i32> hon(K), hfull(K), himp(K);
    std::vector<float> hrat(K);
    std::vector<i64> hc, hacc;
    std::vector<u64> hsq;
    while (true) {
        bool any = false;
        for (i64 q = 0; q < K; q++) {
            hon[q] = done[q] ? 0 : 1;
            any = any || !done[q];
            hrat[q] = ratios[std::min(phase[q], 1)];
        }
        if (!any) break;
        upload(c, on.p, hon);
        upload(c, rat.p, hrat);
        if (n > 0) {
            k_inst_gate<<<grid_items(n, 256), 256, 0, c.stream>>>(n, bl.inst, on, s.dest);
            k_vertex_lam<<<grid_items(n, 256), 256, 0, c.stream>>>(n, bl.inst, best.dlam, rat, vlam, vrat);
            PGGC_LAUNCH_CHECK();
        }
        // table scoring throughout: on a singleton clustering it gives what
        // the raw first sweep gives (every neighbour its own cluster)
        score_all(c, s, lp, g, s.part, cvol, nullptr, false, lam, 0.0f, ScoreOut{s.dest, nullptr, s.abi});
        i64 b[2];
        const i64 kc = gather_candidates(c, lp, g, s.dest, s.cand, b);
        Movers mv{0, 0, 0};
        if (kc > 0) {
            afterburner(c, s, g, s.cand, kc, b, lam, prio, false);
            mv = select_movers(c, s, s.cand, kc, s.moves);
        }
        const i64 km = mv.k;
        fill_i64(c, cnt2, 2 * K, 0);
        if (kc > 0) k_inst_count<<<grid_items(kc, 256), 256, 0, c.stream>>>(s.cand, kc, bl.inst, cnt2);
        if (km > 0) k_inst_count<<<grid_items(km, 256), 256, 0, c.stream>>>(s.moves, km, bl.inst, cnt2.p + K);
        PGGC_LAUNCH_CHECK();
        download(c, hc, cnt2.p, 2 * K);
        for (i64 q = 0; q < K; q++) {
            if (!hon[q]) continue;
            iter[q]++;
            stats[q].sweeps++;
            stats[q].cands += hc[q];
        }
        if (km > 0) {
            if (mv.knew > 0) set_new_cluster_ids_batch(c, s, g, bl, best, cur, cvol, s.moves, km);
            fill_i64(c, acc, K, 0);
            // resets the movers and their neighbours; every vertex of an
            // instance whose first moves these are follows below
            apply_moves_core(c, s, lp, g, cvol, s.moves, km, mv.knew == 0, n_large, n_massive, true, AccInst{bl.inst, acc});
            bool anyfull = false;
            for (i64 q = 0; q < K; q++) {
                const bool moved = hc[K + q] > 0;
                hfull[q] = (moved && !tables[q]) ? 1 : 0;
                anyfull = anyfull || hfull[q];
                if (moved) tables[q] = 1;
                himp[q] = moved ? 1 : 0;  // instances whose objective changes
            }
            if (anyfull) {
                upload(c, full.p, hfull);
                k_inst_fill<<<grid_items(n, 256), 256, 0, c.stream>>>(n, bl.inst, full, s.dest, NULL_PART);
                PGGC_LAUNCH_CHECK();
            }
            upload(c, Ld.p, label_counts(cur));
            upload(c, imp.p, himp);
            k_inst_sumsq<<<grid_blocks(K), 256, 0, c.stream>>>(cvol, best.dloff, Ld, imp, K, sq);
            PGGC_LAUNCH_CHECK();
            const Fetch f[2] = {fetch(hacc, acc.p, K), fetch(hsq, sq.p, 2 * K)};
            copy_d2h(c, f, 2);
            bool anyimp = false;
            for (i64 q = 0; q < K; q++) {
                const bool moved = himp[q] != 0;
                himp[q] = 0;
                if (!moved) continue;
                stats[q].moves += hc[K + q];
                cur[q].uncut += hacc[q];
                cur[q].obj = objective_value(cur[q].uncut, cur[q].lambda, hsq[2 * q], hsq[2 * q + 1]);
                if (c.verbose >= 3)
                    fprintf(stderr, "sweep n=%lld it=%d cands=%lld moves=%lld labels=%d uncut=%lld obj=%.17g inst=%lld\n",
                            (long long)(bl.voff[q + 1] - bl.voff[q]), iter[q], (long long)hc[q],
                            (long long)hc[K + q], cur[q].label_count, (long long)cur[q].uncut, cur[q].obj,
                            (long long)q);
                if (cur[q].obj > best.rd[q].obj) {
                    best.rd[q] = cur[q];
                    himp[q] = 1;
                    anyimp = true;
                }
            }
            if (anyimp) {  // best state of the improved instances (copy_state)
                upload(c, imp.p, himp);
                k_inst_copy_v<<<grid_items(n, 256), 256, 0, c.stream>>>(n, bl.inst, imp, s.part, best_part);
                k_inst_copy_l<<<grid_items(NL, 256), 256, 0, c.stream>>>(NL, best.linst, best.dloff, Ld, imp, cvol,
                                                                        best.vol);
                PGGC_LAUNCH_CHECK();
            }
        }
        for (i64 q = 0; q < K; q++) {  // ratio schedule: 0.75 x4, then 0.25 x2; a sweep without moves ends a phase
            if (!hon[q]) continue;
            if (hc[q] == 0 || hc[K + q] == 0) {
                phase[q]++;
                cnt[q] = 0;
            } else if (++cnt[q] == limits[phase[q]]) {
                phase[q]++;
                cnt[q] = 0;
            }
            if (phase[q] >= 2) done[q] = 1;
        }
    }
    relabel_batch(c, s, bl, best_part, best, active);
    s.hub_buf.reset();
}

}  // namespace pggc
