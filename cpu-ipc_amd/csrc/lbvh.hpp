// This Source Code Form is subject to the terms of the Mozilla Public License, v. 2.0.
// If a copy of the MPL was not distributed with this file, You can obtain one at
// https://mozilla.org/MPL/2.0/.  Parts of this file restate expressions of CPU-IPC
// (MPL-2.0) in the reference's operation order; each such part cites the source it follows.
// Traversal of the device LBVH (packed Node records and four-wide records, see common.hpp).
#pragma once
#include "common.hpp"

namespace cipc {

// Workgroups are dispatched to the 8 XCDs of the device round-robin.  xcd_block maps the
// physical index so that XCD k runs the k-th contiguous slice of the logical range: queries
// taken in Morton order then walk nearby subtrees out of the same L2.
constexpr int kXcds = 8;
__device__ inline int xcd_block(int b, int nb) {
    const int q = nb / kXcds, r = nb % kXcds, k = b % kXcds;
    return k * q + (k < r ? k : r) + b / kXcds;
}

struct TreeView {
    int n;
    const Node* nodes;
    const Node4* wide;
    const int* leafpos = nullptr;   // leaf position of each primitive (the walks with After)
};

// The query box of a wide walk: widened by the gap and rounded outward to float, so that a
// child is tested with six float comparisons instead of six conversions and double
// subtractions (which took a fifth of the walk's time).  It never rejects what the exact test accepts: that
// one accepts lo - hi <= gap as rounded in double, within 2^-53 (|lo| + |hi| + gap) of the
// sum compared here, which the 1e-12 margin covers.
struct WalkBox {
    float lo[3], hi[3];
};
__device__ inline float walk_hi(double h, double gap) { return __double2float_ru(h + gap + 1e-12 * (fabs(h) + gap)); }
__device__ inline float walk_lo(double l, double gap) { return __double2float_rd(l - gap - 1e-12 * (fabs(l) + gap)); }
__device__ inline WalkBox walk_box(const Box& q, double gap) {
    return WalkBox{{walk_lo(q.lo.x, gap), walk_lo(q.lo.y, gap), walk_lo(q.lo.z, gap)},
                   {walk_hi(q.hi.x, gap), walk_hi(q.hi.y, gap), walk_hi(q.hi.z, gap)}};
}
__device__ inline bool overlaps_f(const WalkBox& q, const float* lo, const float* hi) {
    return !((lo[0] > q.hi[0]) | (lo[1] > q.hi[1]) | (lo[2] > q.hi[2]) | (hi[0] < q.lo[0]) | (hi[1] < q.lo[1]) | (hi[2] < q.lo[2]));
}

// Walk of the tree by a group of lanes: a query has 4 << bits lanes (bits 0..4: 1 to 16 records
// a step, 16 to 1 queries a wavefront) and one stack in LDS.  A step takes as many records off
// the stack as the group holds, one lane tests one child, and the children that overlap go back
// on the stack.  A walk is a chain of dependent record loads, so what counts is how many steps
// it takes; a lane walking a subtree of its own took one record a step, eight 16-byte loads of
// it in each lane, and as many steps as the longest of 64 such walks.  Measured alone, each at
// its best lanes per query: the active set's edge walk 81 -> 25 us on four 20^3 cubes, 104 -> 40
// on four 32^3, 392 -> 59 on a folded 128^2 cloth, 135 -> 79 on a batch of 40 scenes.
//
// Every lane of the wavefront takes part (inactive queries with active false); q, after and
// active are the same in a group.  While more(), step(hit) calls hit(yes, primitive) by all 64
// lanes together, each with its own leaf or yes = false, for a superset of the leaves that
// overlap q with `gap` (float boxes); with After only for leaves after position `after`, so that
// in a symmetric pair search, where every primitive queries the same tree, each unordered pair
// is met once.  A query whose stack or step bound runs out, and any query of a one-leaf tree,
// is walked again over the exact boxes by its first lane (depth first along the skip pointers,
// CPULinearBVH::query semantics, LBVH.cpp:252-282, without the final sort), after the others:
// exact() is true for its group from then on, and what it met before is met again.
constexpr int kWalkInts = 1024;   // stack entries of a wavefront, kWalkDepth << bits of each query
constexpr int kWalkDepth = 64;
// order of the wavefront's own LDS accesses (they execute in issue order)
__device__ inline void walk_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// a query's lanes in the wavefront; fewer entries than there is room for only where the evaluation
// entry point asks for them, to make walks run out
struct WalkGroup {
    int bits, g, l, cap;   // group, lane in the group, stack entries of a query
    __device__ explicit WalkGroup(int b, int depth = kWalkDepth)
        : bits(b), g((threadIdx.x & 63) >> (b + 2)), l(threadIdx.x & ((4 << b) - 1)), cap(depth << b) {}
    // the group's part of a ballot, and how many of its bits come before this lane
    __device__ unsigned long long part(unsigned long long m) const {
        const int lanes = 4 << bits;
        m >>= g * lanes;
        return lanes == 64 ? m : m & ((1ull << lanes) - 1);
    }
    __device__ int before(unsigned long long part) const { return __popcll(part & ((1ull << l) - 1)); }
};
// a group's query among n, in the order perm: -1 past the last
__device__ inline int walk_query(const WalkGroup& G, int wave, int n, const int* __restrict__ perm) {
    const int t = (wave << (4 - G.bits)) + G.g;
    return t < n ? perm[t] : -1;
}
template <bool After>
class GroupWalk {
    const TreeView& t;
    const WalkGroup& G;
    const Box& q;
    const double gap;
    const int after;
    int* stk;
    WalkBox w;
    int sp, left, bin;   // stack entries; steps left; next node of the exact walk (-1: none)
    bool over;

public:
    __device__ GroupWalk(const TreeView& t_, const WalkGroup& G_, bool active, const Box& q_, double gap_, int after_, int* lds)
        : t(t_), G(G_), q(q_), gap(gap_), after(after_), stk(lds + G_.g * (kWalkDepth << G_.bits)), w(walk_box(q_, gap_)), sp(0), left(t_.n),
          bin(-1), over(false) {
        if (active && t.n > 1) {
            if (G.l == 0) stk[0] = 0;
            sp = 1;
        } else if (active && t.n == 1) {
            restart();
        }
        walk_order();
    }
    __device__ bool more() const { return __any(sp > 0 || bin >= 0); }
    __device__ bool exact() const { return over; }
    template <typename F>
    __device__ void step(F&& hit) {
        bool yes = false;
        int prim = 0;
        if (__any(sp > 0)) {
            const int slot = G.l >> 2, k = G.l & 3;
            const int n = min(sp, 1 << G.bits);
            const bool on = slot < n;
            const int node = on ? stk[sp - 1 - slot] : 0;
            sp -= n;
            walk_order();
            WideChild c;
            c.child = kNoChild;
            if (on) {
                const float4* r = reinterpret_cast<const float4*>(&t.wide[node].c[k]);
                const float4 a = r[0], b = r[1];
                c.lo[0] = a.x; c.lo[1] = a.y; c.lo[2] = a.z; c.child = __float_as_int(a.w);
                c.hi[0] = b.x; c.hi[1] = b.y; c.hi[2] = b.z; c.last = __float_as_int(b.w);
            }
            const bool ov = on && c.child != kNoChild && overlaps_f(w, c.lo, c.hi) && (!After || c.last > after);
            const bool in = ov && c.child >= 0;
            const unsigned long long m = G.part(__ballot(in));
            const int add = __popcll(m);
            if (sp + add > G.cap || (--left <= 0 && sp + add > 0)) {
                restart();
            } else {
                if (in) stk[sp + G.before(m)] = c.child;
                sp += add;
            }
            yes = ov && c.child < 0;
            prim = -c.child - 1;
            walk_order();
        } else if (bin >= 0) {
            const int nodes = 2 * t.n - 1;
            const Node r = t.nodes[bin];
            const bool ov = overlaps(q, Box{r.lo, r.hi}, gap), leaf = bin >= t.n - 1;
            yes = ov && leaf && (!After || bin - (t.n - 1) > after);
            prim = r.left;
            bin = ov && !leaf ? r.left : r.skip;
            if (bin >= nodes || --left <= 0) bin = -1;
        }
        hit(yes, prim);
    }

private:
    __device__ void restart() {
        over = true;
        sp = 0;
        bin = G.l == 0 ? 0 : -1;
        left = 4 * t.n;   // every step moves forward in depth-first order
    }
};

// Pairs queued in LDS for a wavefront's lanes to take 64 at a time: n entries, the same in every
// lane, at most 63 before a push.
constexpr int kPairQueue = 128;
struct PairQueue {
    int2* q;
    int n;
    __device__ void push(bool yes, int2 p) {
        const unsigned long long m = __ballot(yes);
        if (yes) q[n + __popcll(m & ((1ull << (threadIdx.x & 63)) - 1))] = p;
        n += __popcll(m);
    }
    // up to 64 pairs off the queue, one a lane; false in a lane without one
    __device__ bool pop(int2& p) {
        walk_order();
        const int m = min(n, 64), lane = threadIdx.x & 63;
        n -= m;
        p = lane < m ? q[n + lane] : make_int2(0, 0);
        walk_order();
        return lane < m;
    }
};

// Walk, filter and test of pairs: the leaves that query `id` (-1: none) may overlap are queued
// as (id, primitive); keep(pair) filters 64 at a time, whichever query found them, and
// test(on, pair) takes what is left, 64 at a time, all lanes together.  A pair can be passed
// twice (an exact walk).
template <bool After, typename K, typename T>
__device__ inline void pair_walk(const TreeView& t, const WalkGroup& G, int id, const Box& q, int after, int* lds, int2* met_q,
                                 int2* kept_q, K&& keep, T&& test) {
    GroupWalk<After> W(t, G, id >= 0, q, 0.0, after, lds);
    PairQueue met{met_q, 0}, kept{kept_q, 0};
    for (;;) {
        bool more;
        while ((more = W.more()) && met.n < 64) W.step([&](bool yes, int prim) { met.push(yes, make_int2(id, prim)); });
        int2 p;
        if (met.n > 0) {
            const bool on = met.pop(p);
            kept.push(on && keep(p), p);
        }
        const bool last = !more && met.n == 0;
        if (kept.n >= 64 || (last && kept.n > 0)) {
            const bool on = kept.pop(p);
            test(on, p);
        }
        if (last && kept.n == 0) break;
    }
}

}  // namespace cipc
