// Device context: stream, caching allocator, pinned readback slots, and the
// primitive operations (scan, compaction, radix sort, reductions) shared by
// the hot-path kernels.
#pragma once
#include <map>
#include <string>
#include <unordered_map>
#include <vector>

#include "common.h"

namespace pggc {

// Kernel timing slots: HIP events recorded on the context stream around the
// launches of the kernels named here, with the algorithmic bytes each launch
// moves (measurement hooks; off unless enabled).
enum KSlot {
    KS_SCORE_GROUP = 0,  // k_score_groups
    KS_SCORE_TABLE,      // k_score_table / k_score_raw (LDS tables, block arg-max)
    KS_SCORE_HUB,        // hub scoring: k_hub_gather, k_hub_score (k_hub_raw), k_hub_decide
    KS_AFTERBURNER,      // k_ab_lanes, k_ab_block (k_ab_pack)
    KS_MOVES,            // k_mvp_moves + k_move_edges + k_apply_moves
    KS_CONTRACT_AGG,     // k_cagg (LDS merge of coarse rows)
    KS_CONTRACT_BIG,     // k_cbig_insert + k_cbig_extract
    KS_CONTRACT_COPY,    // k_crow_copy
    KS_EVAL,             // k_eval_uncut
    KS_LEIDEN,           // leidenR refinement (all its kernels)
    KS_ORDER,            // ordering pass (two stable partitions by class)
    KS_COUNT
};

struct KTimer {
    struct Pending {
        int slot;
        hipEvent_t a, b;
        double bytes;
        bool stopped;
    };
    bool on = false;
    int open = 0;  // regions started and not yet stopped
    std::vector<Pending> pend;
    u64* dcnt = nullptr;  // per-region device byte counters (kernels add to dcnt[token])
    std::vector<hipEvent_t> pool;
    i64 launches[KS_COUNT] = {0};
    double ms[KS_COUNT] = {0};
    double bytes[KS_COUNT] = {0};
};

struct Ctx {
    hipStream_t stream = nullptr;
    int device = 0;
    std::string last_error;
    // caching allocator: blocks are kept for reuse until the context ends
    std::multimap<size_t, void*> free_blocks;
    std::unordered_map<void*, size_t> live;
    size_t bytes_live = 0, bytes_cached = 0;
    i64* pinned = nullptr;      // 64 pinned int64 readback slots
    i64* pinned_dev = nullptr;  // the same slots as seen from the device
    // pinned coherent staging area for small copies between host and device: a
    // copy takes the next bytes of it and needs no wait of its own; a wait for the
    // stream frees all of it
    char* stage = nullptr;
    char* stage_dev = nullptr;  // the same bytes as seen from the device
    size_t stage_cap = 0, stage_off = 0;
    u64 seed = 0;           // leidenR seed stream
    u64 draws = 0;
    int verbose = 0;        // >0: per-iteration progress lines on stderr; >=2: memory by stage
    // per-outer-iteration callback (iteration, seconds, cut, objective, labels)
    void (*progress)(void*, int64_t, double, int64_t, double, int32_t) = nullptr;
    void* progress_user = nullptr;
    // per-sweep trace of the local mover (level n, nnz, phase, sweep, active,
    // candidates, moves, microseconds); synchronises per sweep when set
    void (*sweep_trace)(void*, const int64_t*, int) = nullptr;
    void* sweep_user = nullptr;
    double last_contract_s = 0.0, last_refine_s = 0.0;  // of the last clustering call
    // tuning knobs (pggc_ctx_set_knob); the execution shape of the scoring
    // kernels does not change results, pggc_autotune picks it by timing:
    //   table_threads: threads per vertex of the LDS-table classes with
    //     64 < degree <= 512 (64, 128 or 256);
    //   table_spe: LDS hash-table slots per edge of a class's degree bound
    //     (2 or 4), classes 64 < degree <= 2048;
    //   the hub knobs are kept for callers that set them and have no effect
    i64 hub_update_div = 32;
    int table_threads = 64;
    int table_spe = 2;
    i64 hub_lds_max = 2048;
    i64 hub_edges_item = 1024;
    i64 hub_slots_item = 4096;
    // the first sweep of a call from singletons scores the raw adjacency
    // (every neighbour its own cluster); 0 scores it with the tables
    int raw_sweeps = 1;
    int hub_build = 0;
    // levels' local movers run on a copy renumbered by degree: 0 never, 1
    // always, 2 where it pays
    int renumber = 2;
    // big-row contraction batches: table slots per batch (sort entries per
    // batch: a quarter of it); edges per batch of large hubs
    i64 contract_batch = (i64)1 << 30;
    // the active-set predictor runs on at most this many sweeps of a
    // local-move call (0: on every eligible sweep)
    i64 gnn_max_sweeps = 0;
    KTimer kt;

    void* alloc(size_t bytes);
    // verbose >= 2: a line on stderr with the bytes this context holds
    void mem_note(const char* where) const;
    void release(void* p);
    void trim();
    // Gives the cached blocks back when they hold more than cache_keep bytes
    // (1/32 of the device's memory), as after building a graph of hundreds of
    // millions of edges.  Below that the blocks serve the next call: freeing
    // and allocating them again took 18 of the 25 ms of a 16M-edge build.
    size_t cache_keep = 0;
    size_t mem_total = 0;  // of the device
    void trim_large();
    void sync() {
        PGGC_HIP(hipStreamSynchronize(stream));
        stage_off = 0;
    }
    // `bytes` of the staging area (waits when it is full)
    char* stage_take(size_t bytes, char** dev);
    // copy `count` int64 device values to the pinned slots and wait
    const i64* read(const i64* dev, int count);
    i64 read1(const i64* dev) { return read(dev, 1)[0]; }
    u32 next_draw() { return seed_draw(seed, draws++); }
    // kernel timing: kt_start/kt_stop bracket launches on `stream`;
    // kt_resolve waits for the stream and folds the pending pairs into the
    // per-slot totals.
    hipEvent_t kt_event();
    int kt_start(int slot);
    void kt_stop(int token, double bytes);
    void kt_resolve();
    void kt_free();
    // timed region on `stream`: token (or -1 when timing is off) ...
    int kt_begin(int slot) { return kt.on ? kt_start(slot) : -1; }
    // ... closed with the algorithmic bytes it moved (added to what the
    // kernels counted in kt_counter(tok))
    void kt_end(int tok, double bytes) {
        if (tok >= 0) kt_stop(tok, bytes);
    }
    u64* kt_counter(int tok) { return tok >= 0 ? kt.dcnt + tok : nullptr; }
};

// RAII device buffer from the context's caching allocator.
template <class T>
struct Buf {
    Ctx* c = nullptr;
    T* p = nullptr;
    size_t n = 0;
    Buf() = default;
    Buf(Ctx& ctx, size_t count) : c(&ctx), n(count) { p = (T*)ctx.alloc(count * sizeof(T) + 16); }
    Buf(const Buf&) = delete;
    Buf& operator=(const Buf&) = delete;
    Buf(Buf&& o) noexcept : c(o.c), p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
    Buf& operator=(Buf&& o) noexcept {
        if (this != &o) {
            reset();
            c = o.c; p = o.p; n = o.n;
            o.p = nullptr; o.n = 0;
        }
        return *this;
    }
    ~Buf() { reset(); }
    void reset() {
        if (p && c) c->release(p);
        p = nullptr;
        n = 0;
    }
    T* get() const { return p; }
    operator T*() const { return p; }
};

// ---- primitives (prims.hip) ----
void fill_i32(Ctx& c, i32* p, i64 n, i32 v);
void fill_i64(Ctx& c, i64* p, i64 n, i64 v);
void iota_i32(Ctx& c, i32* p, i64 n);
void copy_dev(Ctx& c, void* dst, const void* src, size_t bytes);  // on c.stream
// Host to device in stream order; src may be changed at once.  The bytes go
// through the pinned coherent staging area and a copy kernel on the stream, so
// later kernels read them through the same cache path as data written by kernels.
void copy_h2d(Ctx& c, void* dst, const void* src, size_t bytes);
// Device to host, for several arrays with one wait.
struct Fetch {
    void* dst;
    const void* src;
    size_t bytes;
};
void copy_d2h(Ctx& c, const Fetch* f, int nf);
template <class T>
inline Fetch fetch(std::vector<T>& dst, const T* src, size_t count) {
    dst.resize(count);
    return Fetch{dst.data(), src, count * sizeof(T)};
}
// out[0..n] = exclusive scan of in[0..n); out[n] = total.  in may alias out.
void scan_i64(Ctx& c, const i64* in, i64* out, i64 n);
void scan_i32_to_i64(Ctx& c, const i32* in, i64* out, i64 n);
// Stable LSD radix sort of (key, val) pairs on key bits [begin, bits).
void radix_sort_pairs(Ctx& c, u64* keys, i32* vals, i64 n, int bits, int begin = 0);
void radix_sort_pairs(Ctx& c, u64* keys, i64* vals, i64 n, int bits);
void radix_sort_keys(Ctx& c, u64* keys, i64 n, int bits, int begin = 0);
// *dst += *src on the stream (algorithmic-byte counters of timed regions)
void acct_add(Ctx& c, u64* dst, const i64* src);
// sum of int64 values (device result in *out)
void sum_i64(Ctx& c, const i64* in, i64 n, i64* out);
// exact sum of squares of int64 values: out[0] = high word, out[1] = low word
void sum_sq_u128(Ctx& c, const i64* in, i64 n, i64* out);

}  // namespace pggc
