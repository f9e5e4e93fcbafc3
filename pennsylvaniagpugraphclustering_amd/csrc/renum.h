// Internal vertex order of a level for the local mover: vertices renumbered by
// descending degree (in steps of an eighth of a power of two, ties by id), so
// that the records the sweeps gather at random neighbour ids (cluster, gain,
// destination, weight) of the high-degree vertices, which most edges point at,
// sit together in few cache lines, and the vertices without neighbours come
// last.  Results are those of the original order, bit for bit:
//  - every row keeps its entries in the original order, so each per-vertex
//    reduction (the afterburner's FP32 sum) adds the same terms in the same
//    order;
//  - labels stay in the original id space (vertex i' starts in cluster
//    ids[i'] when the clustering starts at singletons);
//  - the afterburner's priority hash is taken of the original id;
//  - new cluster ids go to the NEW_PART movers in the original move order
//    (order class, then original id);
//  - the degree classes, and so every kernel's work split, are unchanged.
// A vertex without neighbours alone in its cluster never moves and no other
// vertex can join it, so a local move of such vertices only runs on the first
// ncore vertices of the copy (renum_core).  On R-MAT scale 24 they are 47% of
// the top level and 84% of the first coarse level, where they also lie between
// the others and spread every gather over six times the cache lines.
#pragma once
#include "graph.h"
#include "localmove.h"

namespace pggc {

struct Renum {
    const void* key = nullptr;  // row offsets of the graph it was built for
    i64 n = 0;
    i64 ncore = 0;  // vertices with neighbours: the first ones
    bool copied = false;  // rows copied (renum_build kept it)
    Buf<i64> rp, vw;
    Buf<i32> col, w32, ids, part;
    Buf<i64> w64;
    DGraph g;       // the renumbered graph
    LevelPlan plan;
    Orders ord;     // orderings of the caller's graph (for the refinement), built on first use
    bool ord_built = false;
    bool built_for(const DGraph& top) const { return key == (const void*)top.rp && n == top.n; }
};

// Builds r for g (no-op when r already holds it).  Without force the copy is
// made only where it pays (RN_MIN_NNZ, RN_HOT in renum.hip); returns whether it
// was made.
bool renum_build(Ctx& c, const DGraph& g, Renum& r, bool force);

// out[i'] = in[ids[i']]: a per-vertex array of the caller's order in the
// renumbered order
void renum_gather(Ctx& c, const Renum& r, const i32* in, i32* out);

// local_move on the renumbered graph: part (caller's order) is read and
// written in place; cons is indexed by label, so it is shared unchanged.
void local_move_renum(Ctx& c, MoveScratch& s, Renum& r, i32* part, RefineData& best, bool is_initial,
                      bool constrained, i32* cons, bool SA, MoveStats* st);

}  // namespace pggc
