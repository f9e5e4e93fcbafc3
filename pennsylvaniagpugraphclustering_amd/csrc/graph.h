// Level-graph operations: degree ordering, evaluator, own-cluster weights,
// contraction, and the device-resident coarse graph type.
#pragma once
#include "ctx.h"
#include "device.h"

namespace pggc {

// A graph level that owns its device arrays (coarse levels).
struct OwnedGraph {
    Buf<i64> rp;
    Buf<i32> col;
    Buf<i64> w;    // int64 coarse weights, or
    Buf<i32> w32;  // the same weights in 32 bits when every one fits (narrow_weights)
    Buf<i64> vw;
    i64 n = 0, nnz = 0;
    bool wsmall = false;  // DGraph::wsmall
    u64 wmax = 0;         // DGraph::wmax
    DGraph view() const {
        DGraph g;
        g.n = n;
        g.nnz = nnz;
        g.rp = rp.p;
        g.col = col.p;
        if (w32.p) {
            g.w = w32.p;
            g.wk = W_I32;
        } else {
            g.w = w.p;
            g.wk = W_I64;
        }
        g.vw = vw.p;
        g.wsmall = wsmall;
        g.wmax = wmax;
        return g;
    }
};

// out[r] += the weights of row r's edges whose neighbour passes Pass()(key[r],
// key[neighbour]); out is zeroed by the caller, sums are exact integers.
//
// A block takes RS_E consecutive edges.  The gathers of the neighbours' keys
// bound it: columns, weights and keys are loaded by consecutive lanes, RS_T of
// each in flight per thread, and staged in LDS; every thread then walks RS_T
// consecutive edges with a row pointer.  Row sums meet in LDS, where a row that lies
// within the chunk is written with a plain store (rows cut by the chunk's ends,
// and chunks of more than RS_R rows, add with atomics).  With each thread
// loading its own consecutive edges and one atomic per thread and row, the weights of
// the own clusters of an LFR graph (8.4M vertices, 160M nonzeros) took 4.6 ms;
// 2.65 now.
constexpr int RS_T = 8, RS_E = 256 * RS_T, RS_R = 1024;
template <class Pass, class KT, class WT>
__global__ void __launch_bounds__(256) k_row_sums(const i64* __restrict__ rp, const i32* __restrict__ col, WT W,
                                                  const KT* __restrict__ key, i64 n, i64 nnz, i64* out) {
    __shared__ KT sk[RS_E + RS_E / RS_T];  // one pad per thread: its entries start in a bank of their own
    __shared__ typename WT::value sw[RS_E + RS_E / RS_T];
    __shared__ i64 acc[RS_R];
    ChunkRows cr;
    chunk_rows<RS_E>(rp, n, nnz, cr);
    const int t = threadIdx.x;
    const i64 nr = cr.rhi - cr.rlo;
    const bool local = nr <= RS_R;
    i32 v[RS_T];
#pragma unroll
    for (int q = 0; q < RS_T; q++) {
        const i64 j = cr.eb + q * 256 + t;
        v[q] = j < cr.ee ? col[j] : 0;
    }
#pragma unroll
    for (int q = 0; q < RS_T; q++) {
        const int o = q * 256 + t;
        const i64 j = cr.eb + o;
        sk[o + o / RS_T] = key[v[q]];
        if (WT::bytes) sw[o + o / RS_T] = j < cr.ee ? (typename WT::value)W(j) : 0;
    }
    for (int q = t; q < (local ? (int)nr : 0); q += 256) acc[q] = 0;
    __syncthreads();
    const i64 j0 = cr.eb + (i64)t * RS_T;
    if (j0 < cr.ee) {
        i64 r = upper_row(rp, cr.rlo, cr.rhi, j0);
        i64 nxt = rp[r + 1];
        KT mine = key[r];
        i64 a = 0;
#pragma unroll
        for (int q = 0; q < RS_T; q++) {
            const i64 j = j0 + q;
            if (j >= cr.ee) break;
            if (j >= nxt) {
                if (a) atomicAdd((unsigned long long*)(local ? &acc[r - cr.rlo] : &out[r]), (unsigned long long)a);
                a = 0;
                r = advance_row(rp, r, cr.rhi, j, nxt);
                mine = key[r];
            }
            const int o = t * (RS_T + 1) + q;
            if (Pass()(mine, sk[o])) a += WT::bytes ? (i64)sw[o] : 1;
        }
        if (a) atomicAdd((unsigned long long*)(local ? &acc[r - cr.rlo] : &out[r]), (unsigned long long)a);
    }
    if (!local) return;  // block-uniform
    __syncthreads();
    for (int q = t; q < (int)nr; q += 256) {
        const i64 a = acc[q];
        if (a == 0) continue;
        // only the first and the last row can reach beyond the chunk
        if (q == 0 || q == (int)nr - 1) atomicAdd((unsigned long long*)&out[cr.rlo + q], (unsigned long long)a);
        else out[cr.rlo + q] = a;
    }
}

__device__ __forceinline__ int order_class(i64 d) { return d < LARGE_CUTOFF ? 0 : (d < MASSIVE_CUTOFF ? 1 : 2); }
// Stable degree bucketing (src/ordering.cpp:131-164).
struct Orders {
    Buf<i32> o1, o2;
    i64 off_large = 0, off_large2 = 0, off_mid = 0, off_mid2 = 0;
};
void make_orders(Ctx& c, const DGraph& g, Orders& o);

// Evaluator (app/verify_objective.cpp:64-89): vol[l] += vw[i], uncut.
// vol must hold L entries; result scalars are left in dev_out[0] (uncut).
void evaluate(Ctx& c, const DGraph& g, const i32* labels, i64 L, i64* vol, i64* dev_uncut);

// out[i] = sum of w(i,j) over neighbours j with labels[j] == labels[i].
void own_weight(Ctx& c, const DGraph& g, const i32* labels, i64* out);

// Contraction (src/contract.cpp:234-336) with sorted coarse rows.  The coarse
// weights are int32 when every one fits (the values, and so every result, are
// the same; the sweeps read 4 instead of 8 weight bytes per edge and the level
// holds 8 instead of 12 bytes per nonzero) and int64 otherwise, or always with
// `to`: when the finer level's weights sum to less than 2^31 they are written
// as int32 at once, else after a max reduction (contract_widths).
// With `to` the columns and int64 weights go to the caller's arrays instead of
// out's (nothing is written there when they do not fit cap); the copy from out's
// took 0.4 of 7.0 ms for 100M coarse nonzeros.
struct ContractTo {
    i32* col;
    i64* w;
    i64 cap;
};
void contract(Ctx& c, const DGraph& g, const i32* vcmap, i64 nc, OwnedGraph& out, const ContractTo* to = nullptr);

// largest weight of g as an unsigned value (a negative weight is huge); g.nnz > 0
u64 max_weight(Ctx& c, const DGraph& g);
// g.wmax of a weighted graph, read once by the calls whose plans and contractions
// ask for it
void know_max_weight(Ctx& c, DGraph& g);

// next.vw[map[i]] += g.vw[i]  (src/clustering_methods.cpp:33-38)
void coarsen_vertex_weights(Ctx& c, const DGraph& g, const i32* map, i64 nc, i64* out);

}  // namespace pggc
