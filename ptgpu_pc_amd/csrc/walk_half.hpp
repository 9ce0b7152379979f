// walk_half.hpp -- the walk of one query (closest or any hit) over binary16 four-wide nodes, as the
// per-lane-state megakernel and the batch queries run it: a step that advances every lane of a wave
// by one node, and a sparse phase in which the lanes of a wave share the few queries it still holds.
//
// Trees walked here come from this library's builders or from a caller's BVH whose links were checked
// (every node has one parent, every index is in range), so a walk ends by itself and no reference is
// checked again.
#pragma once

#include "half_bounds.hpp"
#include "render_device.hpp"

namespace ptgpu {

// The short traversal-stack class of the binary16 walk: 36 entries per lane, so a workgroup's stack
// takes 36 KB of LDS and four workgroups fit on a CU (three with the 48-entry class).  A walk that
// would push past it ends with sp = kOverflowSp and is walked again (half_finish_overflowed).
constexpr int kStackShort = 36;
constexpr int kStackTiny = 8;   // a test class: nearly every walk outgrows it (tuning short_stack 2)
constexpr int kOverflowSp = 1 << 20;
constexpr int kLeafMin = 24;
template <int STACK>
constexpr bool kIsShort = STACK == kStackShort || STACK == kStackTiny;

// Entries of a `stack`-entry stack above the need of a depth-first walk of the tree (three pushes per two
// levels); half_sparse may use them.  Of a tree whose height was not known before the launch (a recording right after
// its build), the height it was built with is read: with none to spare, a recorded rebuild and 97x61 frame of the
// 65,538-shape soup took 0.78 ms where the same calls took 0.57; now 0.47.  The
// short classes hold less than that need, and walks that take one entry at a time stay far below it; those of
// half_sparse reach it where many boxes overlap, and are then walked again.  A margin of 16 entries is
// kept: with more, fewer walks start again, but all take more steps (97x61x1 spp of the 65,538-shape soup: 0.31 ms, with
// a margin of 24 0.44, with 32 0.56; of 65,536 triangles with vertices within 0.2 of their centres 1.5, 1.6 and 1.7).
__device__ __forceinline__ int half_slack(int stack, const DevAccel &A) {
    if (stack == kStackShort || stack == kStackTiny) return stack - 16;
    const int depth = A.height_check ? (int)A.height_check[2] : A.depth;
    return stack - 3 * ((depth + 2) / 2);
}

// A pointer read from device memory (a batch's job table) or moved between lanes is a generic
// pointer to the compiler, and loads through it become flat loads, which count against both memory
// wait counters and make every wait cover all outstanding LDS and scalar accesses too.  Every buffer
// the render kernels read or write lives in device (global) memory, so the per-lane pointers of
// the render loop are held as global-address-space pointers (gmem): loads and stores through them
// are global ones, also after a generic-pointer helper is inlined on from_gmem's result.  to_gmem
// goes through the address bits: a cast would fold with from_gmem's back into the generic pointer.
template <class T>
using gmem = __attribute__((address_space(1))) T;
template <class T>
__device__ __forceinline__ gmem<T> *to_gmem(T *p) {
    return reinterpret_cast<gmem<T> *>(reinterpret_cast<unsigned long long>(p));
}
template <class T>
__device__ __forceinline__ T *from_gmem(gmem<T> *p) { return (T *)p; }

// One lane's query.
struct HalfWalk {
    f3 o, d;
    RaySlab rs;
    float tb;        // closest: best t so far; any hit: the query's limit
    int bid;         // closest: the best shape so far (-1 none); any hit: >= 0 once occluded
    int node;        // the node to visit next (negative: none)
    int leaf;        // a leaf to test beside it, as the reference ~first (not negative: none)
    int sp;          // entries on the lane's stack: node references (>= 0) and leaf references (~first)
    bool any;
};
// The tree a query walks.
struct HalfTree {
    gmem<const TNode4H> *nodes;
    gmem<const Prim> *prims;
    int nprims;
    int skip;        // any-hit queries ignore this shape
};

// a new query along (o, d), with any and tb already set
__device__ __forceinline__ void half_start(HalfWalk &W, int root) {
    W.bid = -1;
    W.rs = ray_slab(W.o, W.d);
    W.node = root;
    W.leaf = 0;
    W.sp = 0;
}

// The next node and, beside it, the next leaf from the stack's top two entries (read together: one LDS round
// trip): the top entry is taken, and the one below it too if one of the two is a node and the other a
// leaf.  True when the stack is empty.
__device__ __forceinline__ bool half_refill(HalfWalk &W, const int *stk) {
    const int n = W.sp;
    const int e1 = stk[(n > 1 ? n - 1 : 0) * 256], e2 = stk[(n > 1 ? n - 2 : 0) * 256];
    const bool both = n > 1 && (e1 ^ e2) < 0;
    const int x = both ? e2 : e1;
    W.node = e1 > x ? e1 : x;
    W.leaf = e1 < x ? e1 : x;
    W.sp = n - (both ? 2 : 1);
    return n == 0;
}
// The same in a step without leaf tests: a lane whose leaf waits takes the top entry only if that is a node.
__device__ __forceinline__ bool half_refill_waiting(HalfWalk &W, const int *stk) {
    const int n = W.sp;
    const int e1 = stk[(n > 1 ? n - 1 : 0) * 256], e2 = stk[(n > 1 ? n - 2 : 0) * 256];
    const bool waits = W.leaf < 0;
    const bool both = !waits && n > 1 && (e1 ^ e2) < 0;
    const int x = both ? e2 : e1;
    const int node = e1 > x ? e1 : x;
    W.node = n > 0 ? node : -1;
    W.leaf = waits ? W.leaf : e1 < x ? e1 : x;
    W.sp = n - (both ? 2 : waits && (e1 < 0 || n == 0) ? 0 : 1);
    return n == 0 && !waits;
}

// The children of a node that the ray enters go on the stack without a branch: child k's place above the old top is
// the number of children it is nearer than, so the nearest hit ends on top, and a miss (key 0 and its slot) ends
// above every hit, past the new top.  Returns the new top; kOverflowSp where the short stack cannot hold them.
template <int STACK>
__device__ __forceinline__ int half_push(const uint4 &q0, const uint4 &q1, const uint4 &q2, const uint4 &q3,
                                         const RaySlab &rs, float tb, int *stk, int sp) {
    const unsigned t0 = slab_hn(q0.x, q0.y, q0.z, rs, tb), t1 = slab_hn(q1.x, q1.y, q1.z, rs, tb);
    const unsigned t2 = slab_hn(q2.x, q2.y, q2.z, rs, tb), t3 = slab_hn(q3.x, q3.y, q3.z, rs, tb);
    const unsigned k0 = t0 & ~3u, k1 = (t1 & ~3u) | 1u, k2 = (t2 & ~3u) | 2u, k3 = t3 | 3u;
    const int c01 = k0 < k1, c02 = k0 < k2, c03 = k0 < k3, c12 = k1 < k2, c13 = k1 < k3, c23 = k2 < k3;
    const int p0 = c01 + c02 + c03, p1 = 1 - c01 + c12 + c13, p2 = 2 - c02 - c12 + c23, p3 = 3 - c03 - c13 - c23;
    const int nh = (t0 != 0u) + (t1 != 0u) + (t2 != 0u) + (t3 != 0u);
    if (kIsShort<STACK> && sp > STACK - 4) return kOverflowSp;   // (the other classes hold every walk of their trees)
    int *const top = stk + sp * 256;
    top[p0 * 256] = (int)q0.w;
    top[p1 * 256] = (int)q1.w;
    top[p2 * 256] = (int)q2.w;
    top[p3 * 256] = (int)q3.w;
    return sp + nh;
}

// One step of one lane: the current node (if any) and the pending leaf run (if any), loaded together: a
// hit leaf is not tested in the step that finds it but in the next one, beside the next node's
// loads, so a step costs one memory round trip, not two.  True when the query is decided.
//
// Every lane issues both loads, the run's primitive first: a lane with no run reads primitive 0 and
// one with no node reads node 0 (both exist in a tree with binary16 nodes), and ignores them.  With no
// branch around the loads the wait for the primitive leaves the node's four loads in flight, so the
// triangle test overlaps the node's latency.
//
// WAIT: leaves wait until kLeafMin lanes have one, or an eighth of the lanes can do nothing else, and a lane whose
// leaf waits goes on with its nodes.  The test takes as long for one lane as for all, and longer where leaves hold
// several primitives (KD trees): 640x480x4 of a 20,492-shape SAH tree 3.04 -> 2.75 ms,
// a million queries of a 20,000-shape one 0.64 -> 0.51 ms.  A leaf of one primitive is not
// worth the wait, which leaves the box tests a stale limit (327,692-shape mesh: 18.2 -> 18.8 ms).
template <int STACK, bool STATS, bool WAIT>
__device__ __forceinline__ bool half_step(HalfWalk &W, const HalfTree &T, int *stk, unsigned *st_nodes,
                                          unsigned *st_prims) {
    constexpr bool kShort = kIsShort<STACK>;
    bool test = true;
    if (WAIT) {
        const unsigned long long leaves = __ballot(W.leaf < 0), nodes = __ballot(W.node >= 0);
        test = __popcll(leaves) >= kLeafMin || 8 * __popcll(leaves & ~nodes) >= __popcll(leaves | nodes);
    }
    const int first = ~W.leaf;
    const Prim *pp = from_gmem(T.prims) + (first > 0 ? first : 0);
    float4 a0, a1, a2;
    if (test) {
        a0 = pp->p0;
        a1 = pp->p1;
        a2 = pp->p2;
    }
    // compiler-only barrier (no operands, no instruction): the primitive's loads stay
    // here, ahead of the node's, instead of sinking into the branch that tests them
    asm volatile("" ::: "memory");
    const TNode4H *np = from_gmem(T.nodes) + (W.node > 0 ? W.node : 0);
    const uint4 q0 = np->c[0], q1 = np->c[1], q2 = np->c[2], q3 = np->c[3];
    bool done = false;
    // the pending run (one primitive per LBVH leaf), before the boxes so tb is tight
    if (test && W.leaf < 0) {
        // true: the run ends here (an occluder found, or its last primitive)
        auto test_prim = [&](const float4 &b0, const float4 &b1, const float4 &b2) -> bool {
            int id;
            bool last;
            const float t = prim_isect_vals(b0, b1, b2, W.o, W.d, &id, &last);
            if (STATS) (*st_prims)++;
            if (W.any) {
                if (t != 0.f && t < W.tb && id != T.skip) { W.bid = 1; done = true; return true; }
            } else if (t != 0.f && (t < W.tb || (t == W.tb && id > W.bid))) {
                W.tb = t;
                W.bid = id;
            }
            return last;
        };
        // the first primitive outside the loop: the loop's own loads issue in another
        // order, and a shared loop head would make this test wait for the node too
        if (!test_prim(a0, a1, a2)) {
            for (int q = first + 1;; q++) {
                const Prim *tq = from_gmem(T.prims) + q;
                const float4 b0 = tq->p0, b1 = tq->p1, b2 = tq->p2;
                if (test_prim(b0, b1, b2)) break;
            }
        }
    }
    if (!done && W.node >= 0) {
        if (STATS)
            *st_nodes += (q0.x != kEmptyHalf) + (q1.x != kEmptyHalf) + (q2.x != kEmptyHalf) + (q3.x != kEmptyHalf);
        W.sp = half_push<STACK>(q0, q1, q2, q3, W.rs, W.tb, stk, W.sp);
        done = kShort && W.sp == kOverflowSp;
    }
    if (!done) done = test ? half_refill(W, stk) : half_refill_waiting(W, stk);
    return done;
}

// Walks that outgrew the short stack start again at the root, one entry at a time and from the best hit found so far.
// Where even that does not fit, the lane tests every primitive.  The closest hit is the least (t, then the higher id)
// whatever the order of the tests, and an occluder ends an any-hit query, so the result is the walk's.  Only
// half_sparse's walks outgrow the stack in practice, a few in a hundred thousand where many boxes overlap: 97x61x1 spp of
// 65,536 triangles with vertices within 0.2 of their centres, every primitive at once / the walk again: 28.3 / 1.5 ms.
// Called between traversal phases.
template <int STACK, bool STATS>
__device__ __forceinline__ void half_finish_overflowed(HalfWalk &W, const HalfTree &T, int root, int *stk, unsigned *st_prims) {
    if (!kIsShort<STACK> || W.sp != kOverflowSp) return;
    // true: the run ends here (an occluder found, or its last primitive)
    auto test_prim = [&](int q) -> bool {
        const Prim *tq = from_gmem(T.prims) + q;
        int id;
        bool last;
        const float t = prim_isect_vals(tq->p0, tq->p1, tq->p2, W.o, W.d, &id, &last);
        if (STATS) (*st_prims)++;
        if (W.any) {
            if (t != 0.f && t < W.tb && id != T.skip) { W.bid = 1; return true; }
        } else if (t != 0.f && (t < W.tb || (t == W.tb && id > W.bid))) {
            W.tb = t;
            W.bid = id;
        }
        return last;
    };
    int sp = 1;
    stk[0] = root;
    while (sp > 0 && sp != kOverflowSp && !(W.any && W.bid >= 0)) {
        const int ref = stk[--sp * 256];
        if (ref < 0) {
            for (int q = ~ref; !test_prim(q); q++) {}
        } else {
            const TNode4H *np = from_gmem(T.nodes) + ref;
            sp = half_push<STACK>(np->c[0], np->c[1], np->c[2], np->c[3], W.rs, W.tb, stk, sp);
        }
    }
    if (sp == kOverflowSp)
        for (int q = 0; q < T.nprims && !(W.any && W.bid >= 0); q++) test_prim(q);
    W.sp = 0;
}

// The sparse phase: a wave whose traversing lanes (`trav`) are 16 or fewer lends its idle lanes to the
// queries in flight.  The wave splits into equal groups of 4, 8, 16, 32 or 64 lanes, as many as there
// are queries; the k-th traversing lane's query is walked by group k.  A group is one or more quads,
// and each step pops up to one stack entry per quad: a quad with a node tests its four child boxes, one
// per lane, and a quad with a leaf run tests up to four of its primitives.  The children that are hit
// go back on the stack (the owner lane's LDS column), the top entry's nearest child on top.
//
// What bounds a sparse wave is the number of dependent steps of its queries, one memory round trip and
// some 150 instructions each: a lone query in a wave takes a third of the steps that one node per
// step takes.  Popping several entries visits some nodes a depth-first walk would have culled; the
// closest hit and the occlusion do not depend on the order.
//
// Stack: popping m entries may push 4m.  `slack` is what the stack class leaves above a depth-first
// walk's need: with sp + 3m within it, a walk that goes on one entry at a time still fits (m = 1 is
// the depth-first walk itself).  The short classes have no such bound, and a walk that does not fit ends
// as overflowed.
//
// Called by the whole wave.  `ready`: lanes already waiting for shading; the phase ends when they and
// the finished queries reach `regroup`, or all queries are finished.  Returns true on a lane whose own
// query is decided.
template <int STACK, bool STATS, bool MULTI>
__device__ __forceinline__ bool half_sparse(HalfWalk &W, const HalfTree &T, int slack, bool mine,
                                            unsigned long long trav, unsigned ready, unsigned regroup, int *s_stack,
                                            unsigned *st_nodes, unsigned *st_prims) {
    constexpr bool kShort = kIsShort<STACK>;
    const int lane = (int)__lane_id();
    const int nq = __popcll(trav);
    const int lg = nq <= 1 ? 6 : nq <= 2 ? 5 : nq <= 4 ? 4 : nq <= 8 ? 3 : 2;
    const int gsize = 1 << lg;
    const int gi = lane >> lg, qj = (lane & (gsize - 1)) >> 2, qc = lane & 3;
    int *const my_stk = s_stack + threadIdx.x;
    const int rank_me = __popcll(trav & lanemask_lt());
    // the query's pending node and leaf join its stack
    if (mine) {
        if (kShort && W.sp > STACK - 2) {
            W.sp = kOverflowSp;
        } else {
            if (W.node >= 0) my_stk[(W.sp++) * 256] = W.node;
            if (W.leaf < 0) my_stk[(W.sp++) * 256] = W.leaf;
        }
    }
    // group leaders learn their owner lanes (lane 1 is never a leader: it takes the rest), then the
    // group reads the owner's query
    const int at_leader = __builtin_amdgcn_ds_permute(4 * (mine ? rank_me << lg : 1), lane);
    const int owner = __shfl(at_leader, lane & ~(gsize - 1));
    const bool inq = gi < nq;
    f3 o, d;
    o.x = __shfl(W.o.x, owner); o.y = __shfl(W.o.y, owner); o.z = __shfl(W.o.z, owner);
    d.x = __shfl(W.d.x, owner); d.y = __shfl(W.d.y, owner); d.z = __shfl(W.d.z, owner);
    const RaySlab rs = ray_slab(o, d);
    float tb = __shfl(W.tb, owner);
    int bid = __shfl(W.bid, owner), sp = __shfl(W.sp, owner);
    const bool any = __shfl((int)W.any, owner) != 0;
    HalfTree Q = T;
    if (MULTI) {   // a batch's lanes walk different trees
        auto shp = [&](const void *ptr) -> const void * {
            const unsigned long long v = reinterpret_cast<unsigned long long>(ptr);
            const unsigned lo = (unsigned)__shfl((int)(unsigned)v, owner);
            const unsigned hi = (unsigned)__shfl((int)(unsigned)(v >> 32), owner);
            return reinterpret_cast<const void *>(((unsigned long long)hi << 32) | lo);
        };
        Q.nodes = to_gmem(static_cast<const TNode4H *>(shp(from_gmem(T.nodes))));
        Q.prims = to_gmem(static_cast<const Prim *>(shp(from_gmem(T.prims))));
        Q.nprims = __shfl(T.nprims, owner);
        Q.skip = __shfl(T.skip, owner);
        slack = __shfl(slack, owner);
    }
    int *const stk = s_stack + (threadIdx.x & ~63u) + owner;
    bool end = !inq || (kShort && sp == kOverflowSp);
    const unsigned long long gm = gsize == 64 ? ~0ull : ((1ull << gsize) - 1ull) << (gi << lg);
    for (;;) {
        const unsigned fin = (unsigned)__popcll(__ballot(inq && end && (lane & (gsize - 1)) == 0));
        if (ready + fin >= regroup || fin >= (unsigned)nq) break;
        // how many entries this step pops
        int m = gsize >> 2;
        if (m > sp) m = sp;
        if (STATS) m = 1;   // the counts are those of a one-entry walk, whatever the stack class
        else if (m > 1) {
            const int fit = (slack - sp) / 3;
            if (m > fit) m = fit > 1 ? fit : 1;
        }
        const bool valid = !end && qj < m;
        const int at = sp - 1 - qj;
        const int ref = valid ? stk[at * 256] : 0;
        const bool leaf = valid && ref < 0, inner = valid && ref >= 0;
        int pi = ~ref + qc;
        if (pi > Q.nprims - 1) pi = Q.nprims - 1;
        const Prim *pp = from_gmem(Q.prims) + (leaf ? pi : 0);
        const float4 a0 = pp->p0, a1 = pp->p1, a2 = pp->p2;
        asm volatile("" ::: "memory");   // compiler-only: keeps the order, as in half_step
        const uint4 w = from_gmem(Q.nodes)[inner ? ref : 0].c[qc];
        float bt = tb;
        int bb = bid;
        bool cand = false;
        int cref = 0;
        unsigned key = 0;   // the order of a quad's children: entry distance, then slot; below 4: none
        if (__ballot(leaf)) {
            const unsigned long long lastm = __ballot(leaf && (__float_as_int(a1.w) & kLastInLeaf));
            const unsigned lq = (unsigned)(lastm >> (lane & ~3)) & 15u;      // this quad's last flags
            if (leaf && !(lq & ((1u << qc) - 1u))) {
                int id;
                bool last;
                const float t = prim_isect_vals(a0, a1, a2, o, d, &id, &last);
                if (STATS) (*st_prims)++;
                if (any) {
                    cand = t != 0.f && t < tb && id != Q.skip;
                } else if (t != 0.f && (t < tb || (t == tb && id > bid))) {
                    cand = true;
                    bt = t;
                    bb = id;
                }
            }
            if (leaf && qc == 0 && !lq) {   // the run goes on: its next four primitives
                key = 4;
                cref = ~(~ref + 4);
            }
            const unsigned long long cm = __ballot(cand);
            if (cm) {
                if (any) {
                    if (cm & gm) {
                        bid = 1;
                        end = true;
                    }
                }
                // closest: the least (t, then the higher id) of the group
                for (int x = 1; x < gsize; x <<= 1) {
                    const float ot = __shfl_xor(bt, x);
                    const int oi = __shfl_xor(bb, x);
                    if (ot < bt || (ot == bt && oi > bb)) { bt = ot; bb = oi; }
                }
                if (!any) {
                    tb = bt;
                    bid = bb;
                }
            }
        }
        if (inner) {
            cref = (int)w.w;
            key = slab_hn(w.x, w.y, w.z, rs, tb);
            if (STATS) *st_nodes += w.x != kEmptyHalf;
        }
        const bool hit = key != 0u;
        key = (key & ~3u) | (unsigned)qc;
        const unsigned long long hm = __ballot(hit) & gm;
        const unsigned long long rest = hm >> (lane & ~3);   // from this quad's bits up
        const unsigned k1 = (unsigned)qrot<1>((int)key), k2 = (unsigned)qrot<2>((int)key),
                       k3 = (unsigned)qrot<3>((int)key);
        const int place = (k1 > key) + (k2 > key) + (k3 > key);   // farther children of the same entry
        const int below = __popcll(rest >> 4);                    // children of the entries below this quad's
        const int nsp = sp - m + __popcll(hm);
        if (!end) {
            if (kShort && nsp > STACK) {
                sp = kOverflowSp;
                end = true;
            } else {
                if (hit) stk[(sp - m + below + place) * 256] = cref;
                sp = nsp;
                end = nsp == 0;
            }
        }
    }
    // hand each query back to its owner, which reads its group's leader
    const int src = rank_me << lg;
    const int b_sp = __shfl(sp, src), b_bid = __shfl(bid, src);
    const float b_tb = __shfl(tb, src);
    const bool b_end = __shfl((int)end, src) != 0;
    bool done = false;
    if (mine) {
        W.sp = b_sp;
        W.bid = b_bid;
        W.tb = b_tb;
        done = b_end;
        W.rs = ray_slab(W.o, W.d);   // again, so that the phase does not hold it beside its group's
        if (!done) done = half_refill(W, my_stk);
    }
    return done;
}

}  // namespace ptgpu
