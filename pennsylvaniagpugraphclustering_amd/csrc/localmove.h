// Local mover (src/local_mover.cpp) on one level graph.
#pragma once
#include <vector>

#include "graph.h"

namespace pggc {

// Objective state: the cluster_data mirror (interface/cluster_data.hpp:18-88).
struct RefineData {
    i64* vol = nullptr;   // total_deg, device, capacity `cap` labels
    i64 cap = 0;
    i64 uncut = 0;
    i64 top_nnz = 0;
    double obj = -1.0;
    i32 label_count = 0;
    double lambda = 1.0;
    double scale = 1.0;   // get_objective() = obj * scale + offset
    double offset = 0.0;
    double objective() const { return obj * scale + offset; }
};

// obj = uncut - lambda * sum(vol^2) with the exact 128-bit sum of squares
// given as (hi, lo) words (interface/cluster_data.hpp:76-87).
double objective_value(i64 uncut, double lambda, u64 sq_hi, u64 sq_lo);
// recompute rd.obj from the device volumes
void update_objective(Ctx& c, RefineData& rd);

struct MoveStats {
    i64 sweeps = 0, moves = 0, cands = 0;
};

// Scoring classes by degree: 0..4 lane groups (d <= 4, 8, 16, 32, 64),
// CL_TABLE..CL_BIG-1 one wave per vertex with an LDS table sized for the class
// (d <= 128, 256, 512), CL_BIG..CL_HUB-1 one block per vertex (256 threads for
// d <= 1024, 512 for d <= 2048), CL_HUB hubs.
constexpr int NCLS = 11;
constexpr int CL_TABLE = 5, CL_BIG = 8, CL_HUB = 10;

// Per-level cached work partitioning (reused by every local_move on a level).
struct LevelPlan {
    const void* key = nullptr;  // graph identity (row offsets pointer)
    i64 n = -1;
    Orders ord;                 // order1 only
    Buf<i32> sc_list;           // vertices grouped by scoring class
    i64 sc_start[NCLS + 1] = {0};
    // hubs (the class above 2048, sorted by degree): the first nlds of them
    // (degree <= 8192; the first nhalf <= 4096) are scored from LDS tables like
    // the smaller classes, the others (from list entry hub0 on) in chunks of
    // their edges and slices of their clusters' hash range: hub_pre holds the
    // prefixes of their edges, chunks and bucket starts and of the slices of
    // groups of 8 hubs (k_hub_sizes).  hub_pv and hub_best are zero between
    // sweeps.  They are scored in batches of whole groups, [h0, h1) with the
    // batch's sizes, normally one.
    Buf<i64> hub_pre, hub_pv;
    Buf<u64> hub_best;
    struct HubBatch {
        i64 h0, h1, edges, chunks, starts, blocks;
    };
    std::vector<HubBatch> hub_batches;
    i64 hub_blocks = 0;     // of all hubs
    size_t hub_words = 0;   // 8-byte words of scratch for the largest batch
    i64 nhalf = 0;
    bool hub32 = false;   // their row sums fit 32 bits
    i64 nlds = 0, hub0 = 0, nhub = 0;
    bool agg32 = false;  // sums of rows of degree <= 8192 fit 32 bits
    i64 max_deg = 0;  // of the hub class (0 without hubs)
};

// Device scratch sized for the top level, shared by every level.
struct Gnn;

// What the afterburner reads of a neighbour, in one 16-byte load: its gain,
// destination and cluster of this sweep and its vertex weight as the fp32
// value the gain arithmetic uses.
struct __align__(16) AbInfo {
    float gain;
    i32 dest;
    i32 part;
    float vwf;
};

struct MoveScratch {
    i64 cap = 0;
    Gnn* gnn = nullptr;  // active-set predictor (null or mode off: plain sweeps)
    Buf<AbInfo> abi;
    Buf<u64> mvp;  // per vertex: cluster | moved << 31, and the cluster after this sweep's moves
    Buf<u64> rec;     // per vertex: cluster and its volume as fp32 (scoring)
    Buf<uint4> rec16; // the same with the cluster's constraint value, when there is one
    // the gathered entries of a batch of large hubs, while a local move runs:
    // cluster and volume, then the weights (32 or 64 bits), then the bucket
    // starts of every chunk
    Buf<u64> hub_buf;
    Buf<u64> sqpart;  // partial sums of k_finish
    Buf<i32> part, dest, cand, moves, flag, tmp, tmp2;
    Buf<float> gain;
    Buf<i64> prio, scal;
    void ensure(Ctx& c, i64 n);
};

void plan_level(Ctx& c, const DGraph& g, LevelPlan& p);

// local_move<constrained> (src/local_mover.cpp:1360-1417) and
// local_move_strict (:1419-1483).  best_part and cons are device arrays.
// ids (optional, device, n): g is a renumbering of the caller's graph and
// ids[i] is vertex i's caller id, which then stands in for i wherever the
// result depends on vertex ids (afterburner priorities, new cluster ids).
// nfull (optional, >= g.n): best_part has nfull entries, the ones from g.n on
// those of inert vertices without neighbours, which keep their clusters.
void local_move(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, i32* best_part, RefineData& best,
                bool is_initial, bool constrained, i32* cons, bool SA, MoveStats* st, const i32* ids = nullptr,
                i64 nfull = -1);
void local_move_strict(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, i32* best_part, RefineData& best,
                       bool is_initial, bool constrained, i32* cons, MoveStats* st);

// ---------------------------------------------------------------- batches
// Many independent graphs held as one disjoint union graph: instance k owns
// the contiguous vertex range [voff[k], voff[k+1]) of every level, and the
// label range [loff[k], loff[k] + n0[k]) at every level (n0 = its top-level
// vertex count), so its labels are its single-run labels plus loff[k].
// Kernels run once over the union; every per-instance decision of the
// reference's control flow (sweep phases, early stops, best-state tracking,
// new cluster ids, relabelling) is taken per instance, so each instance
// ends exactly as it would alone.
struct BatchLevel {
    i64 K = 0;
    std::vector<i64> voff;  // K+1 vertex offsets at this level (host)
    Buf<i64> dvoff;
    Buf<i32> inst;  // instance of every vertex
    Buf<i32> loc;   // vertex id within its instance
    void build(Ctx& c, const std::vector<i64>& offsets);
};
struct BatchState {
    i64 K = 0;
    std::vector<i64> loff;  // K+1 label offsets (host)
    Buf<i64> dloff;
    Buf<i32> linst;          // instance owning every label
    Buf<float> dlam;         // float lambda per instance
    Buf<i64> vol;            // volumes over the whole label space
    std::vector<RefineData> rd;  // per-instance objective state (rd[k].vol unused)
};

// local_move (src/local_mover.cpp:1360-1417, SA on, unconstrained) of every
// instance k with active[k] at once; best_part holds labels (label space).
void local_move_batch(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, const BatchLevel& bl,
                      i32* best_part, BatchState& best, bool is_initial, const std::vector<char>& active,
                      std::vector<MoveStats>& stats);

// One scoring + afterburner sweep from a fixed state (parity entry point).
// Returns the number of accepted moves written to moves_out (order1 order).
i64 sweep_once(Ctx& c, MoveScratch& s, LevelPlan& lp, const DGraph& g, const i32* part, const i64* vol, i64 L,
               double lambda, float ratio, bool raw, const i32* cons, i32* dest, float* gain, i32* moves_out,
               i64* ncand);

}  // namespace pggc
