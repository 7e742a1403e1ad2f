// This Source Code Form is subject to the terms of the Mozilla Public License, v. 2.0.
// If a copy of the MPL was not distributed with this file, You can obtain one at
// https://mozilla.org/MPL/2.0/.  Parts of this file restate expressions of CPU-IPC
// (MPL-2.0) in the reference's operation order; each such part cites the source it follows.
// Broad phase and active set on the device.  Compiled with -ffp-contract=off.
//
// Reference: CPULinearBVH::build / query and CPUBroadPhaseBVH::build / buildSwept
// (CPU IPC/LBVH.cpp:163-339), SpatialHash::calculateActivateSet
// (CollisionBroadPhase.cpp:765-1059), Ground::calculateActivateSet (:1076-1092).
//
// Tree topology: scene box reduction -> 30-bit Morton codes of box centres normalised to
// the scene box -> stable radix sort of (code, primitive) -> unique keys code << 32 |
// primitive -> Karras splits, one thread per internal node -> skip pointers for stackless
// depth-first traversal.  Refit (every build): leaf boxes in leaf order -> internal boxes
// as unions of power-of-two leaf ranges (no inter-work-group synchronisation).  Query
// results do not depend on the topology, so it is rebuilt only every kMaxRefits fits.
//
// Active set: each surface vertex (point-triangle) and surface edge (edge-edge) query walks the
// tree with a group of lanes (GroupWalk) that buffers its first candidates; a second pass
// packs them (walking again only where they did not fit); one thread per candidate places it by
// its primitive id, as the reference's query sorts them, and classifies it.
// Compaction reproduces the reference's serial order: partial-CCD pairs, then Self_ActiveSet =
// point-triangle entries, edge-edge entries, and the point-point/point-edge entries
// deduplicated in std::map key order with multiplicity; Self_EE_ActiveSet for mollified
// entries; Environment_ActiveSet in ascending surface order.
#include "context.hpp"
#include "contact.hpp"
#include "lbvh.hpp"

#include <hipcub/hipcub.hpp>
#include <type_traits>

namespace cipc {

// ---------------------------------------------------------------------------------
// LBVH build
// ---------------------------------------------------------------------------------
__device__ inline unsigned expand_bits(unsigned v) {       // LBVH.cpp:17-24
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}
__device__ inline unsigned morton3(double x, double y, double z) {  // LBVH.cpp:26-37
    const double res = 1024.0;
    auto q = [&](double v) { v = fmax(0.0, fmin(v * res, res - 1.0)); return (unsigned)v; };
    return (expand_bits(q(x)) << 2) | (expand_bits(q(y)) << 1) | expand_bits(q(z));
}

constexpr int kRedBlock = 256;
constexpr int kRedParts = 256;
__global__ __launch_bounds__(kRedBlock) void box_reduce_partial(int n, const Box* __restrict__ b, Box* __restrict__ part) {
    __shared__ Box sh[kRedBlock];
    Box acc{{1.7976931348623157e308, 1.7976931348623157e308, 1.7976931348623157e308},
            {-1.7976931348623157e308, -1.7976931348623157e308, -1.7976931348623157e308}};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        acc = Box{vmin(acc.lo, b[i].lo), vmax(acc.hi, b[i].hi)};
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            sh[threadIdx.x] = Box{vmin(sh[threadIdx.x].lo, sh[threadIdx.x + s].lo), vmax(sh[threadIdx.x].hi, sh[threadIdx.x + s].hi)};
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}
__global__ void morton_keys(int n, const Box* __restrict__ b, const Box* __restrict__ part, int nparts,
                            unsigned* __restrict__ codes, int* __restrict__ ids) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Box sc = part[0];
    for (int k = 1; k < nparts; ++k) sc = Box{vmin(sc.lo, part[k].lo), vmax(sc.hi, part[k].hi)};
    const d3 ext = sc.hi - sc.lo;  // nparts == 1: the partials were reduced beforehand
    const d3 c = 0.5 * (b[i].lo + b[i].hi);
    const d3 off = c - sc.lo;
    const double x = ext.x > 0.0 ? off.x / ext.x : 0.0;
    const double y = ext.y > 0.0 ? off.y / ext.y : 0.0;
    const double z = ext.z > 0.0 ? off.z / ext.z : 0.0;
    codes[i] = morton3(x, y, z);
    ids[i] = i;
}
// Unique keys (code << 32 | primitive).  The radix sort of (code, primitive) pairs is stable
// and the primitives enter in ascending order, so these keys come out sorted exactly as a
// sort of the 64-bit keys would order them.
__global__ void join_keys(int n, const unsigned* __restrict__ codes, const int* __restrict__ ids, unsigned long long* __restrict__ keys) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = ((unsigned long long)codes[i] << 32) | (unsigned)ids[i];
}
__device__ inline int prefix(const unsigned long long* k, int n, int a, int b) {
    if (b < 0 || b >= n) return -1;
    return __clzll(k[a] ^ k[b]);
}
// Karras 2012 topology (LBVH.cpp:62-119,213-228): internal node i covers the key range
// [first, last] and splits it at the highest differing bit.
__global__ void karras_kernel(int n, const unsigned long long* __restrict__ k, Node* __restrict__ nodes, int* __restrict__ range_first, int* __restrict__ range_last, int* __restrict__ split_right) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    int first, last;
    if (i == 0) { first = 0; last = n - 1; }
    else {
        const int lp = prefix(k, n, i, i - 1), rp = prefix(k, n, i, i + 1);
        const int dir = rp > lp ? 1 : -1;
        const int minp = lp < rp ? lp : rp;
        int lmax = 2;
        while (prefix(k, n, i, i + dir * lmax) > minp) lmax <<= 1;
        int len = 0;
        for (int st = lmax >> 1; st > 0; st >>= 1)
            if (prefix(k, n, i, i + dir * (len + st)) > minp) len += st;
        const int other = i + dir * len;
        first = i < other ? i : other;
        last = i < other ? other : i;
    }
    int split;
    const unsigned long long fc = k[first], lc = k[last];
    if (fc == lc) split = (first + last) >> 1;
    else {
        const int common = __clzll(fc ^ lc);
        int s = first, step = last - first;
        do {
            step = (step + 1) >> 1;
            const int cand = s + step;
            if (cand < last && __clzll(fc ^ k[cand]) > common) s = cand;
        } while (step > 1);
        split = s;
    }
    const int l = (split == first) ? split + n - 1 : split;
    const int r = (split + 1 == last) ? split + 1 + n - 1 : split + 1;
    nodes[i].left = l;
    nodes[i].right = r;
    range_first[i] = first;
    range_last[i] = last;
    split_right[split] = r;
}
__global__ void leaf_ids(int n, const int* __restrict__ order, Node* __restrict__ nodes, int* __restrict__ leafpos) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    nodes[n - 1 + s].left = order[s];
    leafpos[order[s]] = s;
}
__global__ void skip_kernel(int n, const int* __restrict__ range_last, const int* __restrict__ split_right, Node* __restrict__ nodes) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * n - 1) return;
    const int last = (i < n - 1) ? range_last[i] : i - (n - 1);
    nodes[i].skip = (last >= n - 1) ? -1 : split_right[last];
}
// Internal boxes.  Node i of the Karras tree covers the sorted leaves [first, last], so its
// box is the union of that range.  Power-of-two reduction levels over the sorted leaf boxes
// (level l node j = leaves [j 2^l, (j+1) 2^l)) are built 8 levels per launch in LDS; each
// internal box is then the union of at most 2 log2(n) level nodes.  No inter-work-group
// communication is needed.
constexpr int kSegBlock = 256;
constexpr int kSegLevels = 8;   // log2(kSegBlock)
__device__ inline Box empty_box() {
    return Box{{1.7976931348623157e308, 1.7976931348623157e308, 1.7976931348623157e308},
               {-1.7976931348623157e308, -1.7976931348623157e308, -1.7976931348623157e308}};
}
// Primitive boxes: static (CPUBroadPhaseBVH::build, LBVH.cpp:284-305) or swept along -p
// with the step whose bits are at *abits (buildSwept, LBVH.cpp:307-339).  The step is read
// on the device, so building the swept trees needs no host round trip.
__device__ inline double step_of(const unsigned long long* abits) { return __longlong_as_double((long long)*abits); }
// Where a tree's primitive boxes come from: a face or an edge of the surface, static (the
// box of the positions) or swept (the box of x and x - a p, a the scene's step in abits).
struct PrimSrc {
    int kind = 0;   // 0: the prim array holds them; 1: faces; 2: surface edges
    const int4* faces = nullptr;
    const int2* se = nullptr;
    const double* x = nullptr;
    const double* p = nullptr;
    const unsigned long long* abits = nullptr;
    const int* vs = nullptr;
};
__device__ inline Box prim_box(const PrimSrc& s, int i) {
    if (s.kind == 1) {
        const int4 v = s.faces[i];
        if (s.abits == nullptr) return box_tri(ld3(s.x, v.x), ld3(s.x, v.y), ld3(s.x, v.z));
        const double a = step_of(s.vs ? s.abits + kSlots * s.vs[v.x] : s.abits);
        Box b = swept_pt(ld3(s.x, v.x), ld3(s.p, v.x), a);
        b = box_union(b, swept_pt(ld3(s.x, v.y), ld3(s.p, v.y), a));
        b = box_union(b, swept_pt(ld3(s.x, v.z), ld3(s.p, v.z), a));
        return b;
    }
    const int2 v = s.se[i];
    if (s.abits == nullptr) return box_edge(ld3(s.x, v.x), ld3(s.x, v.y));
    const double a = step_of(s.vs ? s.abits + kSlots * s.vs[v.x] : s.abits);
    return box_union(swept_pt(ld3(s.x, v.x), ld3(s.p, v.x), a), swept_pt(ld3(s.x, v.y), ld3(s.p, v.y), a));
}

__global__ void prim_boxes(int n, PrimSrc src, Box* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = prim_box(src, i);
}

// Box of the sorted leaves [a, b]: the union of at most 2 log2(n) level nodes (exact: the
// union is a min / max).
__device__ inline Box range_box(int a, int b, const SegLevels& L, const Box* __restrict__ seg) {
    int l = 0;
    Box acc = empty_box();
    while (a <= b && l < 40) {
        if (a & 1) { const Box x = seg[L.offset[l] + a]; acc = Box{vmin(acc.lo, x.lo), vmax(acc.hi, x.hi)}; ++a; }
        if (a <= b && !(b & 1)) { const Box x = seg[L.offset[l] + b]; acc = Box{vmin(acc.lo, x.lo), vmax(acc.hi, x.hi)}; --b; }
        a >>= 1; b >>= 1; ++l;
    }
    return acc;
}
// A box into its slot of a four-wide record: slot code (record << 2 | k), or -1 for none.
__device__ inline void put_wide_box(Node4* __restrict__ wide, int code, const Box& x) {
    if (code < 0) return;
    WideChild& c = wide[code >> 2].c[code & 3];
    c.lo[0] = __double2float_rd(x.lo.x); c.lo[1] = __double2float_rd(x.lo.y); c.lo[2] = __double2float_rd(x.lo.z);
    c.hi[0] = __double2float_ru(x.hi.x); c.hi[1] = __double2float_ru(x.hi.y); c.hi[2] = __double2float_ru(x.hi.z);
}
// A tree's refit, for one tree or two at once (a work-group range each):
//   leaves: the leaf boxes in leaf order (node records and level 0) and reduction levels
//     1..kSegLevels, each work-group over its kSegBlock leaves; with a primitive source the
//     primitive boxes are computed here too (and stored, for the exact leaf tests).
//   upper: the next kSegLevels levels from the last built, one launch per kSegLevels
//     levels (one for up to 2^16 leaves).
//   internal: each internal node's box, the union of the level boxes that cover its leaf
//     range (range_box).
// No work-group waits for another inside a launch: on this GPU that would take a device-wide
// fence, which writes back and invalidates an XCD's L2.
// Each box also goes, rounded outward to float, into the four-wide record slots that hold
// its node (wslot, set with the topology), so the records need no launch of their own.
struct RefitTree {
    int n = 0, levels = 0, leaf_blocks = 0, int_blocks = 0;
    const int* order = nullptr;
    Box* prim = nullptr;
    PrimSrc src;
    Node* nodes = nullptr;
    Node4* wide = nullptr;
    const int* first = nullptr;
    const int* last = nullptr;
    Box* seg = nullptr;
    const int2* wslot = nullptr;
    SegLevels L;
};
struct RefitSet {
    RefitTree t[2];
    int ntrees = 1;
};
__global__ __launch_bounds__(kSegBlock) void refit_leaves(RefitSet rs) {
    const int which = (rs.ntrees > 1 && (int)blockIdx.x >= rs.t[0].leaf_blocks) ? 1 : 0;
    const RefitTree& t = rs.t[which];
    const int blk = (int)blockIdx.x - (which ? rs.t[0].leaf_blocks : 0);
    __shared__ Box sh[kSegBlock];
    const int n = t.n;
    const int g = blk * kSegBlock + threadIdx.x;
    Box b = empty_box();
    if (g < n) {
        const int q = t.order[g];
        if (t.src.kind != 0) {
            b = prim_box(t.src, q);
            t.prim[q] = b;
        } else {
            b = t.prim[q];
        }
        Node& r = t.nodes[n - 1 + g];
        r.lo = b.lo;
        r.hi = b.hi;
        t.seg[g] = b;
        const int2 ws = t.wslot[n - 1 + g];
        put_wide_box(t.wide, ws.x, b);
        put_wide_box(t.wide, ws.y, b);
    }
    sh[threadIdx.x] = b;
    __syncthreads();
    for (int l = 1; l <= kSegLevels; ++l) {
        const int half = 1 << (l - 1);
        if ((threadIdx.x & ((1 << l) - 1)) == 0) {
            const Box a = sh[threadIdx.x], c = sh[threadIdx.x + half];
            sh[threadIdx.x] = Box{vmin(a.lo, c.lo), vmax(a.hi, c.hi)};
        }
        __syncthreads();
        if (l < 40 && t.L.count[l] > 0 && (threadIdx.x & ((1 << l) - 1)) == 0) {
            const int j = g >> l;
            if (j < t.L.count[l]) t.seg[t.L.offset[l] + j] = sh[threadIdx.x];
        }
    }
}
// Levels l0+1 .. l0+kSegLevels from level l0, for every tree of the set that has them: the
// trees' work-groups one after the other (blocks_for(count[l0], kSegBlock) each).
__device__ inline int upper_blocks(const RefitTree& t, int l0) {
    return t.levels > l0 ? (t.L.count[l0] + kSegBlock - 1) / kSegBlock : 0;
}
__global__ __launch_bounds__(kSegBlock) void refit_upper(RefitSet rs, int l0) {
    const int b0 = upper_blocks(rs.t[0], l0);
    const int which = (rs.ntrees > 1 && (int)blockIdx.x >= b0) ? 1 : 0;
    const RefitTree& t = rs.t[which];
    const int blk = (int)blockIdx.x - (which ? b0 : 0);
    __shared__ Box sh[kSegBlock];
    const int nsrc = t.L.count[l0];
    const Box* src = t.seg + t.L.offset[l0];
    const int g = blk * kSegBlock + threadIdx.x;
    sh[threadIdx.x] = g < nsrc ? src[g] : empty_box();
    __syncthreads();
    for (int l = 1; l <= kSegLevels; ++l) {
        const int half = 1 << (l - 1);
        if ((threadIdx.x & ((1 << l) - 1)) == 0) {
            const Box a = sh[threadIdx.x], c = sh[threadIdx.x + half];
            sh[threadIdx.x] = Box{vmin(a.lo, c.lo), vmax(a.hi, c.hi)};
        }
        __syncthreads();
        const int lv = l0 + l;
        if (lv < 40 && t.L.count[lv] > 0 && (threadIdx.x & ((1 << l) - 1)) == 0) {
            const int j = g >> l;
            if (j < t.L.count[lv]) t.seg[t.L.offset[lv] + j] = sh[threadIdx.x];
        }
    }
}
__global__ void refit_internal(RefitSet rs) {
    const int which = (rs.ntrees > 1 && (int)blockIdx.x >= rs.t[0].int_blocks) ? 1 : 0;
    const RefitTree& t = rs.t[which];
    const int blk = (int)blockIdx.x - (which ? rs.t[0].int_blocks : 0);
    const int i = blk * blockDim.x + threadIdx.x;
    if (i >= t.n - 1) return;
    const Box own = range_box(t.first[i], t.last[i], t.L, t.seg);
    t.nodes[i].lo = own.lo;
    t.nodes[i].hi = own.hi;
    put_wide_box(t.wide, t.wslot[i].y, own);
}

// The parts of the four-wide records that depend on the topology only, once per topology:
// what each slot holds and, for every node, the slots its box goes to (wslot.x: the record
// of its parent, for a leaf child; wslot.y: the record of its grandparent).  A record holds
// its node's grandchildren, or the children themselves where those are leaves; unused slots
// hold an empty box.
__global__ void fill_int2(int2* __restrict__ p, int n, int2 v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void wide_static(int n, const Node* __restrict__ nodes, const int* __restrict__ range_last, Node4* __restrict__ wide,
                            int2* __restrict__ wslot) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    int ch[4], via[4], m = 0;
    const int c2[2] = {nodes[i].left, nodes[i].right};
    for (int k = 0; k < 2; ++k) {
        const int c = c2[k];
        if (c < n - 1) {
            ch[m] = nodes[c].left; via[m++] = 1;
            ch[m] = nodes[c].right; via[m++] = 1;
        } else {
            ch[m] = c; via[m++] = 0;
        }
    }
    Node4 r;
    for (int k = 0; k < 4; ++k) {
        WideChild& x = r.c[k];
        x.lo[0] = x.lo[1] = x.lo[2] = __int_as_float(0x7f800000);
        x.hi[0] = x.hi[1] = x.hi[2] = __int_as_float(0xff800000);
        if (k < m) {
            const int c = ch[k];
            x.child = c >= n - 1 ? -(nodes[c].left + 1) : c;
            x.last = c >= n - 1 ? c - (n - 1) : range_last[c];
            if (via[k]) wslot[c].y = i << 2 | k;
            else wslot[c].x = i << 2 | k;
        } else {
            x.child = kNoChild;
            x.last = -1;
        }
    }
    wide[i] = r;
}

// Topology from the current primitive boxes.
void build_topology(Context& c, LBVH& t, int n, hipStream_t st, DBuf<unsigned char>& tmp) {
    ++c.topo_gen;
    t.n = n;
    t.age = 0;
    const int nodes = 2 * n - 1;
    t.nodes.resize(nodes); t.wide.resize(std::max(n - 1, 1));
    t.range_first.resize(std::max(n - 1, 1)); t.range_last.resize(std::max(n - 1, 1)); t.split_right.resize(std::max(n - 1, 1));
    t.codes.resize(n); t.codes_sorted.resize(n); t.order.resize(2 * (size_t)n); t.keys_sorted.resize(n);
    // level l of the box reduction holds ceil(n / 2^l) boxes; level 0 is the leaves
    SegLevels L{};
    long long total = 0;
    int levels = 0;
    for (int l = 0; l < 40; ++l) {
        const long long cnt = ((long long)n + (1ll << l) - 1) >> l;
        L.count[l] = (int)cnt;
        L.offset[l] = total;
        total += cnt;
        levels = l;
        if (cnt == 1) break;
    }
    for (int l = levels + 1; l < 40; ++l) { L.count[l] = 0; L.offset[l] = total; }
    t.L = L;
    t.levels = levels;
    t.seg.resize((size_t)total);
    const int parts = std::min<int>(kRedParts, (int)blocks_for(n, kRedBlock));
    t.scene_partial.resize(parts);
    hipLaunchKernelGGL(box_reduce_partial, dim3(parts), dim3(kRedBlock), 0, st, n, t.prim.p, t.scene_partial.p);
    CIPC_CHECK_LAUNCH();
    if (parts > 1) {
        hipLaunchKernelGGL(box_reduce_partial, dim3(1), dim3(kRedBlock), 0, st, parts, t.scene_partial.p, t.scene_partial.p);
        CIPC_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(morton_keys, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, t.prim.p, t.scene_partial.p, 1, t.codes.p,
                       t.order.p + n);
    CIPC_CHECK_LAUNCH();
    sort_u32_pairs(t.codes.p, t.codes_sorted.p, t.order.p + n, t.order.p, n, 30, st, tmp);
    hipLaunchKernelGGL(join_keys, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, t.codes_sorted.p, t.order.p, t.keys_sorted.p);
    CIPC_CHECK_LAUNCH();
    if (n > 1) {
        hipLaunchKernelGGL(karras_kernel, dim3(blocks_for(n - 1, 256)), dim3(256), 0, st, n, t.keys_sorted.p, t.nodes.p,
                           t.range_first.p, t.range_last.p, t.split_right.p);
        CIPC_CHECK_LAUNCH();
    }
    t.leafpos.resize(n);
    hipLaunchKernelGGL(leaf_ids, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, t.order.p, t.nodes.p, t.leafpos.p);
    hipLaunchKernelGGL(skip_kernel, dim3(blocks_for(nodes, 256)), dim3(256), 0, st, n, t.range_last.p, t.split_right.p, t.nodes.p);
    t.wslot.resize(nodes);
    hipLaunchKernelGGL(fill_int2, dim3(blocks_for(nodes, 256)), dim3(256), 0, st, t.wslot.p, nodes, make_int2(-1, -1));
    if (n > 1)
        hipLaunchKernelGGL(wide_static, dim3(blocks_for(n - 1, 256)), dim3(256), 0, st, n, t.nodes.p, t.range_last.p, t.wide.p,
                           t.wslot.p);
    CIPC_CHECK_LAUNCH();
}

// Boxes of the current primitive boxes on the existing topologies: one tree, or two in the
// same two launches.
static RefitTree refit_view(LBVH& t, const PrimSrc& src) {
    RefitTree r;
    r.n = t.n; r.levels = t.levels;
    r.leaf_blocks = (int)blocks_for(t.n, kSegBlock);
    r.int_blocks = t.n > 1 ? (int)blocks_for(t.n - 1, 256) : 0;
    r.order = t.order.p; r.prim = t.prim.p; r.src = src; r.nodes = t.nodes.p; r.wide = t.wide.p;
    r.first = t.range_first.p; r.last = t.range_last.p; r.seg = t.seg.p; r.wslot = t.wslot.p; r.L = t.L;
    return r;
}
static void refit_set(const RefitSet& rs, hipStream_t st) {
    int lb = 0, ib = 0, levels = 0;
    for (int k = 0; k < rs.ntrees; ++k) {
        lb += rs.t[k].leaf_blocks;
        ib += rs.t[k].int_blocks;
        levels = std::max(levels, rs.t[k].levels);
    }
    if (lb > 0) hipLaunchKernelGGL(refit_leaves, dim3(lb), dim3(kSegBlock), 0, st, rs);
    for (int l0 = kSegLevels; l0 < levels; l0 += kSegLevels) {
        int ub = 0;
        for (int k = 0; k < rs.ntrees; ++k) ub += rs.t[k].levels > l0 ? (int)blocks_for(rs.t[k].L.count[l0], kSegBlock) : 0;
        if (ub > 0) hipLaunchKernelGGL(refit_upper, dim3(ub), dim3(kSegBlock), 0, st, rs, l0);
    }
    if (ib > 0) hipLaunchKernelGGL(refit_internal, dim3(ib), dim3(256), 0, st, rs);
    CIPC_CHECK_LAUNCH();
}
void refit(Context& c, LBVH& t, const PrimSrc& src, hipStream_t st) {
    (void)c;
    RefitSet rs;
    rs.t[0] = refit_view(t, src);
    rs.ntrees = 1;
    refit_set(rs, st);
    ++t.age;
}
static void refit_two(LBVH& a, const PrimSrc& sa, LBVH& b, const PrimSrc& sb, hipStream_t st) {
    RefitSet rs;
    rs.t[0] = refit_view(a, sa);
    rs.t[1] = refit_view(b, sb);
    rs.ntrees = 2;
    refit_set(rs, st);
    ++a.age;
    ++b.age;
}

// The tree over n > 0 primitives has a topology that the next build refits.
static bool refit_only(const LBVH& t, int n) { return n > 0 && t.n == n && t.age < kMaxRefits; }
// A tree over n primitives whose boxes come from src: a new topology (from boxes computed
// first) when none fits, else a refit that computes the boxes itself.
static void build_tree_from(Context& c, LBVH& t, int n, const PrimSrc& src, hipStream_t st, DBuf<unsigned char>& tmp) {
    if (n <= 0) { t.n = n; return; }
    t.prim.resize(n);
    if (t.n != n || t.age >= kMaxRefits) {
        hipLaunchKernelGGL(prim_boxes, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, src, t.prim.p);
        CIPC_CHECK_LAUNCH();
        build_topology(c, t, n, st, tmp);
        refit(c, t, PrimSrc{}, st);
    } else {
        refit(c, t, src, st);
    }
}
void build_tree(Context& c, LBVH& t, int n) {
    if (n <= 0) { t.n = n; return; }
    if (t.n != n || t.age >= kMaxRefits) build_topology(c, t, n, c.stream, c.tmp);
    refit(c, t, PrimSrc{}, c.stream);
}

// The static face and edge trees, on the context's stream.
void build_static_trees(Context& c) {
    Scene& s = c.sc;
    c.face_tree.prim.resize(std::max(s.F, 1));
    c.edge_tree.prim.resize(std::max(s.Es, 1));
    PrimSrc fs, es;
    fs.kind = 1; fs.faces = s.faces.p; fs.x = s.x.p;
    es.kind = 2; es.se = s.se.p; es.x = s.x.p;
    build_tree_from(c, c.face_tree, s.F, fs, c.stream, c.tmp);
    build_tree_from(c, c.edge_tree, s.Es, es, c.stream, c.tmp);
}
void build_swept_trees(Context& c, const unsigned long long* abits, hipStream_t st) {
    Scene& s = c.sc;
    c.sface_tree.prim.resize(std::max(s.F, 1));
    c.sedge_tree.prim.resize(std::max(s.Es, 1));
    PrimSrc fs, es;
    fs.kind = 1; fs.faces = s.faces.p; fs.x = s.x.p; fs.p = s.dir.p; fs.abits = abits; fs.vs = scene_of_vertex(s);
    es.kind = 2; es.se = s.se.p; es.x = s.x.p; es.p = s.dir.p; es.abits = abits; es.vs = scene_of_vertex(s);
    if (refit_only(c.sface_tree, s.F) && refit_only(c.sedge_tree, s.Es)) {
        refit_two(c.sface_tree, fs, c.sedge_tree, es, st);   // both trees in the same two launches
        return;
    }
    build_tree_from(c, c.sface_tree, s.F, fs, st, c.tmp_sb);
    build_tree_from(c, c.sedge_tree, s.Es, es, st, c.tmp_sb);
}

// ---------------------------------------------------------------------------------
// Active set (CollisionBroadPhase.cpp:765-1059)
// ---------------------------------------------------------------------------------
// candidate categories; kDrop: a box hit that the reference's candidate filters discard
enum : int { kNone = 0, kSelfPT = 1, kMap = 2, kSelfEE = 3, kMolPE = 4, kMolEE = 5, kDrop = 6 };

// Candidate collection.
//   A (traverse): each query walks its tree with 4 << bits lanes; the first kQueryCap leaves
//     whose box overlaps the query box with gap sqrt(Hhat) (for edges only later edges, as
//     queryEdgeForEdgesWithBBoxCheck keeps) are stored and all are counted.  The walk loads
//     nothing but tree nodes.
//   B (compact, the same lanes per query): the query's hits into the packed layout, by a second
//     walk for a query with more than kQueryCap.
//   C (classify, one thread per hit): the hit's rank among its query's hits (primitive order),
//     the reference's incidence and collider filters (CollisionBroadPhase.cpp:769-776,862-870),
//     then the distance-type classification.
// The leaf boxes are the primitives' own boxes (prim_box), so the leaf test
// is the box test of the reference's candidate filter.  Queries are taken in the Morton
// order of their rest positions (perm) so that the queries of a wavefront walk nearby subtrees.
// The lanes per query are chosen per context (the autotuner); the hits and their order do not
// depend on it.
constexpr int kQueryCap = 64;

// Point-triangle hits: filters, then classification (CollisionBroadPhase.cpp:765-857).
__device__ inline void pt_classify(int u, const int* __restrict__ dc, int F, const int* __restrict__ own, const int* __restrict__ off,
                                   const int* __restrict__ sv, const double* __restrict__ x, const int* __restrict__ bt,
                                   const int4* __restrict__ faces, const int* __restrict__ candU, int* __restrict__ cand, double hhat,
                                   double sq, const int* __restrict__ vs, int4* __restrict__ rec, int* __restrict__ cat) {
    if (dc[kDcFlags] || u >= dc[kDcPT]) return;
    // sorted position: the hit's rank among its query's hits (all distinct)
    const int q = own[u], o = off[q], e = off[q + 1];
    const int f = candU[u];
    int k = o;
    for (int j = o; j < e; ++j) k += candU[j] < f;
    cand[k] = f;
    if ((unsigned)f >= (unsigned)F || k >= e) {   // cannot happen for a consistent walk; never index with it
        rec[k < e ? k : o] = make_int4(0, 0, 0, 0);
        cat[k < e ? k : o] = kDrop;
        return;
    }
    const int vI = sv[q];
    const int4 fv = faces[f];
    if ((is_collider(bt[vI]) && is_collider(bt[fv.x]) && is_collider(bt[fv.y]) && is_collider(bt[fv.z])) || vI == fv.x ||
        vI == fv.y || vI == fv.z || (vs && vs[vI] != vs[fv.x])) {   // (scenes of a batch never touch)
        rec[k] = make_int4(0, 0, 0, 0);
        cat[k] = kDrop;
        return;
    }
    const d3 P = ld3(x, vI);
    {
        const d3 A = ld3(x, fv.x), B = ld3(x, fv.y), C = ld3(x, fv.z);
        if (!overlaps(box_pt(P), box_tri(A, B, C), sq)) {   // the walk's float boxes admit a superset
            rec[k] = make_int4(0, 0, 0, 0);
            cat[k] = kDrop;
            return;
        }
        const int dt = dtype_pt(P, A, B, C);
        int4 r = make_int4(0, 0, 0, 0);
        int ct = kNone;
        double d;
        switch (dt) {
        case 0: d = d_PP(P, A); if (d < hhat) { r = make_int4(-vI - 1, fv.x, -1, -1); ct = kMap; } break;
        case 1: d = d_PP(P, B); if (d < hhat) { r = make_int4(-vI - 1, fv.y, -1, -1); ct = kMap; } break;
        case 2: d = d_PP(P, C); if (d < hhat) { r = make_int4(-vI - 1, fv.z, -1, -1); ct = kMap; } break;
        case 3: d = d_PE(P, A, B); if (d < hhat) { r = make_int4(-vI - 1, fv.x, fv.y, -1); ct = kMap; } break;
        case 4: d = d_PE(P, B, C); if (d < hhat) { r = make_int4(-vI - 1, fv.y, fv.z, -1); ct = kMap; } break;
        case 5: d = d_PE(P, C, A); if (d < hhat) { r = make_int4(-vI - 1, fv.z, fv.x, -1); ct = kMap; } break;
        case 6: d = d_PT(P, A, B, C); if (d < hhat) { r = make_int4(-vI - 1, fv.x, fv.y, fv.z); ct = kSelfPT; } break;
        default: break;
        }
        rec[k] = r;
        cat[k] = ct;
    }
}

// Edge-edge hits: filters, then classification (CollisionBroadPhase.cpp:858-1052).
__device__ inline void ee_classify(int u, const int* __restrict__ dc, int Es, const int* __restrict__ own, const int* __restrict__ off,
                                   const int2* __restrict__ se, const double* __restrict__ x, const double* __restrict__ vrest,
                                   const int* __restrict__ bt, const int* __restrict__ candU, int* __restrict__ cand, double hhat,
                                   double sq, const int* __restrict__ vs, int4* __restrict__ rec, int2* __restrict__ aux,
                                   int* __restrict__ cat) {
    if (dc[kDcFlags] || u >= dc[kDcEE]) return;
    const int eI = own[u], o = off[eI] - off[0], e = off[eI + 1] - off[0];
    const int eJ = candU[u];
    int k = o;
    for (int j = o; j < e; ++j) k += candU[j] < eJ;
    cand[k] = eJ;
    if ((unsigned)eJ >= (unsigned)Es || k >= e) {   // cannot happen for a consistent walk; never index with it
        rec[k < e ? k : o] = make_int4(0, 0, 0, 0);
        aux[k < e ? k : o] = make_int2(-1, -1);
        cat[k < e ? k : o] = kDrop;
        return;
    }
    const int2 A = se[eI], B = se[eJ];
    if ((is_collider(bt[A.x]) && is_collider(bt[A.y]) && is_collider(bt[B.x]) && is_collider(bt[B.y])) || A.x == B.x ||
        A.x == B.y || A.y == B.x || A.y == B.y || (vs && vs[A.x] != vs[B.x])) {
        rec[k] = make_int4(0, 0, 0, 0);
        aux[k] = make_int2(-1, -1);
        cat[k] = kDrop;
        return;
    }
    const d3 a0 = ld3(x, A.x), a1 = ld3(x, A.y);
    {
        const d3 b0 = ld3(x, B.x), b1v = ld3(x, B.y);
        if (!overlaps(box_edge(a0, a1), box_edge(b0, b1v), sq)) {   // the walk's float boxes admit a superset
            rec[k] = make_int4(0, 0, 0, 0);
            aux[k] = make_int2(-1, -1);
            cat[k] = kDrop;
            return;
        }
        const int dt = dtype_ee(a0, a1, b0, b1v);
        const double cr = ee_cross_sqn(a0, a1, b0, b1v);
        const double ex = eps_x_of(ld3(vrest, A.x), ld3(vrest, A.y), ld3(vrest, B.x), ld3(vrest, B.y));
        const int add_e = (cr < ex) ? -eJ - 2 : -1;
        int4 r = make_int4(0, 0, 0, 0);
        bool hit = false;
        double d;
        switch (dt) {
        case 0: d = d_PP(a0, b0); if (d < hhat) { r = make_int4(-A.x - 1, B.x, -1, add_e); hit = true; } break;
        case 1: d = d_PP(a0, b1v); if (d < hhat) { r = make_int4(-A.x - 1, B.y, -1, add_e); hit = true; } break;
        case 2: d = d_PE(a0, b0, b1v); if (d < hhat) { r = make_int4(-A.x - 1, B.x, B.y, add_e); hit = true; } break;
        case 3: d = d_PP(a1, b0); if (d < hhat) { r = make_int4(-A.y - 1, B.x, -1, add_e); hit = true; } break;
        case 4: d = d_PP(a1, b1v); if (d < hhat) { r = make_int4(-A.y - 1, B.y, -1, add_e); hit = true; } break;
        case 5: d = d_PE(a1, b0, b1v); if (d < hhat) { r = make_int4(-A.y - 1, B.x, B.y, add_e); hit = true; } break;
        case 6: d = d_PE(b0, a0, a1); if (d < hhat) { r = make_int4(-B.x - 1, A.x, A.y, add_e); hit = true; } break;
        case 7: d = d_PE(b1v, a0, a1); if (d < hhat) { r = make_int4(-B.y - 1, A.x, A.y, add_e); hit = true; } break;
        case 8:
            d = d_EE(a0, a1, b0, b1v);
            if (d < hhat) {
                r = (add_e <= -2) ? make_int4(A.x, A.y, B.x, -B.y - Es - 2) : make_int4(A.x, A.y, B.x, B.y);
                hit = true;
            }
            break;
        default: break;
        }
        int ct = kNone;
        int2 ax = make_int2(-1, -1);
        if (hit) {
            // serial compaction rules, CollisionBroadPhase.cpp:1028-1052
            if (r.w >= 0) ct = kSelfEE;
            else if (r.w == -1) ct = kMap;
            else if (r.w >= -Es - 1) { ax = make_int2(eI, -r.w - 2); r.w = -1; ct = kMolPE; }
            else { r.w = -r.w - Es - 2; ct = kMolEE; }
        }
        rec[k] = r;
        aux[k] = ax;
        cat[k] = ct;
    }
}

// Per-category output positions of the hits (four 0/1 categories each, int4 x, y, z, w): the
// counts of every kCatBlock hits, which the scatter's work-groups then add up themselves, each to
// its own block, and ballots within a block.  Only the hits there are, not the capacity, are
// read, and no position is stored: a device-wide scan over the capacities wrote 16 bytes a
// slot (with the scatter 333 us on a batch of 40 scenes and 55 on a folded 128^2 cloth, now 110 and 19).
// What the work-groups read grows with the square of the blocks, so where the capacities hold
// more than kOwnCounts blocks one work-group adds the counts up once (category_starts).  The
// line lies where a launch costs what the sums do: folded cloths with 920 blocks of hits take 15.6 us
// adding up themselves and 10.8 + 5.0 with the launch, 2,450 blocks 26.5 and 19.5 + 7.0, 12,900 blocks
// 326 and 117 + 23.
constexpr int kCatBlock = 1024, kCatThreads = 256, kOwnCounts = 2048, kStartThreads = 1024;
// Category masks of the point-triangle hits and of the edge-edge hits.
__device__ constexpr unsigned kCatPT[4] = {1u << kSelfPT, 1u << kMap, (1u << kNone) | (1u << kSelfPT) | (1u << kMap), 0u};
__device__ constexpr unsigned kCatEE[4] = {1u << kSelfEE, 1u << kMap, (1u << kMolPE) | (1u << kMolEE),
                                           (1u << kNone) | (1u << kSelfEE) | (1u << kMap) | (1u << kMolPE) | (1u << kMolEE)};
template <bool Pt>
__device__ inline int cat_count(int c, unsigned bit, unsigned long long& m) {
    m = __ballot((Pt ? kCatPT[c] : kCatEE[c]) & bit);
    return __popcll(m);
}
// The counts of a wavefront's hits [i0, i0 + kCatBlock / 4).
template <bool Pt>
__device__ inline int4 wave_counts(const int* __restrict__ cat, int i0, int n) {
    int4 t = make_int4(0, 0, 0, 0);
    unsigned long long m;
#pragma unroll
    for (int r = 0; r < kCatBlock / kCatThreads; ++r) {
        const int i = i0 + 64 * r + (threadIdx.x & 63);
        const unsigned bit = i < n ? 1u << cat[i] : 0u;
        t.x += cat_count<Pt>(0, bit, m);
        t.y += cat_count<Pt>(1, bit, m);
        t.z += cat_count<Pt>(2, bit, m);
        t.w += cat_count<Pt>(3, bit, m);
    }
    return t;
}
__device__ inline int4 add4(int4 p, int4 q) { return make_int4(p.x + q.x, p.y + q.y, p.z + q.z, p.w + q.w); }
__device__ inline int4 wave_add4(int4 v) {
    for (int d = 32; d > 0; d >>= 1)
        v = add4(v, make_int4(__shfl_xor(v.x, d), __shfl_xor(v.y, d), __shfl_xor(v.z, d), __shfl_xor(v.w, d)));
    return v;
}
// Work-groups [0, bPT) the point hits' blocks, the rest the edge hits' (sums from bPT on).
__global__ __launch_bounds__(kCatThreads) void category_counts(const int* __restrict__ dc, int bPT, const int* __restrict__ catPT,
                                                               const int* __restrict__ catEE, int4* __restrict__ sums) {
    __shared__ int4 sh[kCatThreads / 64];
    if (dc[kDcFlags]) return;
    const bool pt = (int)blockIdx.x < bPT;
    const int b = pt ? blockIdx.x : blockIdx.x - bPT, n = dc[pt ? kDcPT : kDcEE], w = threadIdx.x >> 6;
    if (b * kCatBlock >= n) return;
    const int i0 = b * kCatBlock + w * (kCatBlock / 4);
    const int4 t = pt ? wave_counts<true>(catPT, i0, n) : wave_counts<false>(catEE, i0, n);
    if ((threadIdx.x & 63) == 0) sh[w] = t;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = add4(add4(sh[0], sh[1]), add4(sh[2], sh[3]));
}
// Every block's counts become the counts of the blocks of its kind before it; the totals of both
// kinds follow at sums[bPT + bEE].  One work-group.
__global__ __launch_bounds__(kStartThreads) void category_starts(const int* __restrict__ dc, int bPT, int bEE, int4* __restrict__ sums) {
    __shared__ int4 part[kStartThreads / 64], total;
    if (dc[kDcFlags]) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int kind = 0; kind < 2; ++kind) {
        int4* s = sums + (kind ? bPT : 0);
        const int n = (dc[kind ? kDcEE : kDcPT] + kCatBlock - 1) / kCatBlock;
        int4 base = make_int4(0, 0, 0, 0);
        for (int b0 = 0; b0 < n; b0 += kStartThreads) {
            const int b = b0 + threadIdx.x;
            const int4 v = b < n ? s[b] : make_int4(0, 0, 0, 0);
            int4 x = v;   // inclusive over the wavefront
            for (int d = 1; d < 64; d <<= 1) {
                const int4 y = make_int4(__shfl_up(x.x, d), __shfl_up(x.y, d), __shfl_up(x.z, d), __shfl_up(x.w, d));
                if (lane >= d) x = add4(x, y);
            }
            if (lane == 63) part[w] = x;
            __syncthreads();
            if (threadIdx.x == 0) {
                int4 t = make_int4(0, 0, 0, 0);
                for (int k = 0; k < kStartThreads / 64; ++k) {
                    const int4 p = part[k];
                    part[k] = t;
                    t = add4(t, p);
                }
                total = t;
            }
            __syncthreads();
            const int4 at = add4(base, part[w]);
            if (b < n) s[b] = make_int4(at.x + x.x - v.x, at.y + x.y - v.y, at.z + x.z - v.z, at.w + x.w - v.w);
            base = add4(base, total);
            __syncthreads();   // part and total are the next round's
        }
        if (threadIdx.x == 0) sums[bPT + bEE + kind] = base;
    }
}
// PP/PE map key: (c0 + V, c1, c2 + 1) packed with `bits` per field preserves the signed
// lexicographic order of std::map<EncodedContact, int> (all keys have c3 = -1).
__device__ inline unsigned long long map_key(int4 r, int V, int bits) {
    return ((unsigned long long)(r.x + V) << (2 * bits)) | ((unsigned long long)r.y << bits) | (unsigned long long)(r.z + 1);
}
// Point-triangle hit i at positions p -> Self_ActiveSet head (a), map keys (b), partial-CCD pairs (c).
__device__ inline void scatter_pt(int i, int ct, int4 p, const int4* __restrict__ rec, const int* __restrict__ own,
                                  const int* __restrict__ cand, int V, int bits, int4* __restrict__ self_set,
                                  unsigned long long* __restrict__ mkeys, int2* __restrict__ ccd) {
    if (ct == kDrop) return;
    ccd[p.z] = make_int2(-own[i] - 1, cand[i]);
    if (ct == kSelfPT) self_set[p.x] = rec[i];
    else if (ct == kMap) mkeys[p.y] = map_key(rec[i], V, bits);
}
// Edge-edge hit i -> Self_ActiveSet (a), map keys (b), Self_EE_ActiveSet + eIe (c), CCD pairs (d).
// base: the point hits' totals (Self_ActiveSet, map keys, CCD pairs), where the edge hits'
// entries start.
__device__ inline void scatter_ee(int i, int ct, int4 p, int4 base, const int4* __restrict__ rec, const int2* __restrict__ aux,
                                  const int* __restrict__ own, const int* __restrict__ cand, int V, int bits,
                                  int4* __restrict__ self_set, unsigned long long* __restrict__ mkeys, int4* __restrict__ ee_set,
                                  int2* __restrict__ ee_ie, int2* __restrict__ ccd) {
    if (ct == kDrop) return;
    ccd[base.z + p.w] = make_int2(own[i], cand[i]);
    if (ct == kSelfEE) self_set[base.x + p.x] = rec[i];
    else if (ct == kMap) mkeys[base.y + p.y] = map_key(rec[i], V, bits);
    else if (ct == kMolPE || ct == kMolEE) { ee_set[p.z] = rec[i]; ee_ie[p.z] = aux[i]; }
}
// Counts: the per-category totals of both kinds, the ground count the ground scan's total.  The map keys fill [0, nm) of a
// buffer of capM; past nm they are the all-ones key, which sorts last.
__device__ inline void category_totals(int Vs, const int4& a, const int4& b, const int* __restrict__ pg, int capM, int* __restrict__ dc) {
    const int nm = a.y + b.y;
    dc[kDcMapKeys] = nm;
    if (nm > capM) { dc[kDcFlags] |= 4; return; }
    // the output counts are published only for a set that fits: over capacity they stay zero,
    // so that later stages read no entry of an unfinished set
    dc[kDcA] = a.x; dc[kDcA2] = a.y; dc[kDcAK] = a.z;
    dc[kDcB] = b.x; dc[kDcB2] = b.y; dc[kDcMol] = b.z; dc[kDcBK] = b.w;
    dc[kDcCCD] = a.z + b.w;
    dc[kDcEnv] = pg[Vs] - pg[0];
}
__device__ inline void map_tail(int i, int capM, int nm, unsigned long long* __restrict__ mkeys) {
    if (i >= capM) return;
    if (i >= nm) mkeys[i] = ~0ull;
}
// After the run-length encoding of the sorted keys: the runs without the all-ones run (there
// is one exactly when nm < capM) are the merged map entries, decoded after the A and B parts
// of Self_ActiveSet; the first thread publishes the set's size.
__global__ void map_decode(int capM, const int* __restrict__ nruns, int* __restrict__ dc, const unsigned long long* __restrict__ keys,
                           const int* __restrict__ counts, int V, int bits, int4* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (dc[kDcFlags]) return;
    const int base = dc[kDcA] + dc[kDcB];
    const int nM = *nruns - (dc[kDcMapKeys] < capM ? 1 : 0);
    if (i == 0) dc[kDcSelf] = base + nM;
    if (i >= nM) return;
    const unsigned long long k = keys[i], m = (1ull << bits) - 1;
    out[base + i] = make_int4((int)((k >> (2 * bits)) & m) - V, (int)((k >> bits) & m), (int)(k & m) - 1, -counts[i]);
}
// pos: the joint scan's ground starts, offset by its first entry
__device__ inline void ground_scatter(int s, int Vs, const int* __restrict__ sv, const int* __restrict__ flag, const int* __restrict__ pos,
                                      int* __restrict__ out) {
    if (s >= Vs || !flag[s]) return;
    out[pos[s] - pos[0]] = sv[s];
}
// In one launch (the four parts write disjoint entries): work-groups [0, bPT) place the point
// hits, the next bEE the edge hits, the next bG the ground entries, the rest write the map keys'
// all-ones tail.  Every work-group with work adds up the blocks' counts (or, with own_counts 0,
// reads what category_starts made of them); the first publishes the totals (category_totals).  Nothing is placed when a capacity was exceeded: the host builds the
// set again.
struct ScatterArgs {
    int* dc;
    int V, bits, Vs, capM, bPT, bEE, bG, own_counts;
    const int *catPT, *ownPT, *candPT, *catEE, *ownEE, *candEE, *sv, *fg, *pg;
    const int4 *sums, *recPT, *recEE;
    const int2* auxEE;
    int4 *self_set, *ee_set;
    int2 *ee_ie, *ccd;
    unsigned long long* mkeys;
    int* env;
};
// A block's hits with their positions: put(hit, category, position).
template <bool Pt, typename P>
__device__ inline void place_hits(const int* __restrict__ cat, int b, int n, int4 at, int4* sh, P&& put) {
    const int w = threadIdx.x >> 6, i0 = b * kCatBlock + w * (kCatBlock / 4);
    const int4 t = wave_counts<Pt>(cat, i0, n);
    if ((threadIdx.x & 63) == 0) sh[w] = t;
    __syncthreads();
    for (int k = 0; k < w; ++k) at = add4(at, sh[k]);
    const unsigned long long before = (1ull << (threadIdx.x & 63)) - 1;
#pragma unroll
    for (int r = 0; r < kCatBlock / kCatThreads; ++r) {
        const int i = i0 + 64 * r + (threadIdx.x & 63);
        const int ct = i < n ? cat[i] : kDrop;
        const unsigned bit = i < n ? 1u << ct : 0u;
        unsigned long long m0, m1, m2, m3;
        const int4 c = make_int4(cat_count<Pt>(0, bit, m0), cat_count<Pt>(1, bit, m1), cat_count<Pt>(2, bit, m2), cat_count<Pt>(3, bit, m3));
        put(i, ct, make_int4(at.x + __popcll(m0 & before), at.y + __popcll(m1 & before), at.z + __popcll(m2 & before), at.w + __popcll(m3 & before)));
        at = add4(at, c);
    }
}
__global__ __launch_bounds__(kCatThreads) void scatter_all(ScatterArgs a) {
    __shared__ int4 sh[3][kCatThreads / 64], hits[kCatThreads / 64];
    int* dc = a.dc;
    if (dc[kDcFlags] & 3) return;   // the candidates exceeded their capacity (an earlier launch)
    const int nPT = dc[kDcPT], nEE = dc[kDcEE];
    const int b = blockIdx.x;
    const bool first = b == 0, pt = b < a.bPT, ee = !pt && b < a.bPT + a.bEE;
    if (!first && ((pt && b * kCatBlock >= nPT) || (ee && (b - a.bPT) * kCatBlock >= nEE))) return;
    // the totals of both kinds (ta, tb), and the counts before this block (of its kind)
    int4 ta = make_int4(0, 0, 0, 0), tb = ta, at = ta;
    if (!a.own_counts) {
        ta = a.sums[a.bPT + a.bEE];
        tb = a.sums[a.bPT + a.bEE + 1];
        if ((pt && b * kCatBlock < nPT) || ee) at = a.sums[b];
    } else {
        const int4 zero = ta;
        const int kPT = (nPT + kCatBlock - 1) / kCatBlock, kEE = (nEE + kCatBlock - 1) / kCatBlock;
        for (int k = threadIdx.x; k < kPT + kEE; k += kCatThreads) {
            const bool p = k < kPT;
            const int block = p ? k : a.bPT + k - kPT;
            const int4 v = a.sums[block];
            if (p) ta = add4(ta, v);
            else tb = add4(tb, v);
            if (p == pt && block < b) at = add4(at, v);
        }
        if (!pt && !ee) at = zero;
        ta = wave_add4(ta); tb = wave_add4(tb); at = wave_add4(at);
        if ((threadIdx.x & 63) == 0) {
            const int w = threadIdx.x >> 6;
            sh[0][w] = ta; sh[1][w] = tb; sh[2][w] = at;
        }
        __syncthreads();
        ta = add4(add4(sh[0][0], sh[0][1]), add4(sh[0][2], sh[0][3]));
        tb = add4(add4(sh[1][0], sh[1][1]), add4(sh[1][2], sh[1][3]));
        at = add4(add4(sh[2][0], sh[2][1]), add4(sh[2][2], sh[2][3]));
    }
    if (first && threadIdx.x == 0) category_totals(a.Vs, ta, tb, a.pg, a.capM, dc);
    const int nm = ta.y + tb.y;
    if (nm > a.capM) return;
    if (pt) {
        place_hits<true>(a.catPT, b, nPT, at, hits, [&](int i, int ct, int4 p) {
            scatter_pt(i, ct, p, a.recPT, a.ownPT, a.candPT, a.V, a.bits, a.self_set, a.mkeys, a.ccd);
        });
        return;
    }
    if (ee) {
        place_hits<false>(a.catEE, b - a.bPT, nEE, at, hits, [&](int i, int ct, int4 p) {
            scatter_ee(i, ct, p, ta, a.recEE, a.auxEE, a.ownEE, a.candEE, a.V, a.bits, a.self_set, a.mkeys, a.ee_set, a.ee_ie, a.ccd);
        });
        return;
    }
    const int g = b - a.bPT - a.bEE;
    if (g < a.bG) ground_scatter(g * kCatThreads + threadIdx.x, a.Vs, a.sv, a.fg, a.pg, a.env);
    else map_tail((g - a.bG) * kCatThreads + threadIdx.x, a.capM, nm, a.mkeys);
}

// The walks' hit buffers.
void size_active_walks(Context& c) {
    ActiveSetScratch& b = c.as;
    b.bufPT.resize((size_t)std::max(c.sc.Vs, 1) * kQueryCap);
    b.bufEE.resize((size_t)std::max(c.sc.Es, 1) * kQueryCap);
}

// Both walks of the active set in one launch, and both compactions in another: work-groups
// [0, nbp) take point queries with 4 << pb lanes each, the rest edge queries with 4 << eb (a
// work-group is one wavefront, so a wavefront's lanes share a query kind).  The traversal
// maps work-groups to XCDs over the joint grid.
struct BothWalks {
    int Vs, Es, nbp, pb, eb;
    const int *pperm, *sv, *eperm;
    const int2* se;
    const double* x;
    TreeView ft, et;
    double sq, gd, hhat;
    d3 gn;
    int *cntPT, *cntEE, *fg, *bufPT, *bufEE;
    const int *oPT, *oEE;
    int* dc;
    int capPT, capEE;
    int *candUPT, *candUEE, *ownPT, *ownEE;
};
// The hits of one query per group: point query s against the faces, or edge query eI against the
// edges after it in number.  put(i, primitive) stores hit i; returns the number of hits, the
// same in a group.  Deterministic, so a second walk meets the same hits in the same order.
template <typename P>
__device__ inline int query_hits(const TreeView& t, const WalkGroup& G, bool active, const Box& q, double gap, int edge, int* lds, P&& put) {
    GroupWalk<false> W(t, G, active, q, gap, 0, lds);
    int n = 0;
    bool again = false;
    while (W.more()) {
        if (W.exact() && !again) {
            again = true;
            n = 0;
        }
        W.step([&](bool yes, int prim) {
            const bool keep = yes && prim > edge;
            const unsigned long long m = G.part(__ballot(keep));
            if (keep) put(n + G.before(m), prim);
            n += __popcll(m);
        });
    }
    return n;
}
template <typename P>
__device__ inline int point_hits(const BothWalks& a, const WalkGroup& G, int s, int* lds, P&& put) {
    const Box q = s >= 0 ? box_pt(ld3(a.x, a.sv[s])) : Box{};
    return query_hits(a.ft, G, s >= 0, q, a.sq, -1, lds, put);
}
template <typename P>
__device__ inline int edge_hits(const BothWalks& a, const WalkGroup& G, int eI, int* lds, P&& put) {
    Box q{};
    if (eI >= 0) {
        const int2 e = a.se[eI];
        q = box_edge(ld3(a.x, e.x), ld3(a.x, e.y));
    }
    return query_hits(a.et, G, eI >= 0, q, a.sq, eI, lds, put);
}
// The point walk also sets each surface vertex's ground flag (distance^2 to the ground below
// Hhat, Ground::calculateActivateSet, CollisionBroadPhase.cpp:1076-1092), for the same scan.
__global__ __launch_bounds__(64) void traverse_both(BothWalks a) {
    __shared__ int lds[kWalkInts];
    const int mb = xcd_block(blockIdx.x, gridDim.x);
    if (mb < a.nbp) {
        const WalkGroup G(a.pb);
        const int s = walk_query(G, mb, a.Vs, a.pperm);
        const int n = point_hits(a, G, s, lds, [&](int i, int f) {
            if (i < kQueryCap) a.bufPT[(size_t)s * kQueryCap + i] = f;
        });
        if (s >= 0 && G.l == 0) {
            a.cntPT[s] = n;
            const double dist = dot(a.gn, ld3(a.x, a.sv[s])) - a.gd;
            a.fg[s] = (dist * dist < a.hhat) ? 1 : 0;
        }
    } else {
        const WalkGroup G(a.eb);
        const int e = walk_query(G, mb - a.nbp, a.Es, a.eperm);
        const int n = edge_hits(a, G, e, lds, [&](int i, int f) {
            if (i < kQueryCap) a.bufEE[(size_t)e * kQueryCap + i] = f;
        });
        if (e >= 0 && G.l == 0) a.cntEE[e] = n;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) { a.cntPT[a.Vs] = 0; a.fg[a.Vs] = 0; a.cntEE[a.Es] = 0; }   // the scans' tails
    if (a.dc && blockIdx.x == 0 && threadIdx.x < kDcWords) a.dc[threadIdx.x] = 0;   // the iteration's device counts start at zero
}
// The compaction also publishes the candidate totals (the per-query scans' last entries)
// against their capacities; every thread reads them from the scan, so none waits for that write.
// A query's lanes copy its hits side by side (one thread per query part copied them one by
// one: 514 -> 72 us on the folded 128^2 cloth, 20 on a batch of 40 scenes).
__global__ __launch_bounds__(64) void compact_both(BothWalks a) {
    __shared__ int lds[kWalkInts];
    const int b = blockIdx.x;
    const int nPT = a.oPT[a.Vs], nEE = a.oEE[a.Es] - a.oEE[0];
    const int flags = (nPT > a.capPT ? 1 : 0) | (nEE > a.capEE ? 2 : 0);
    if (b == 0 && threadIdx.x == 0) {
        a.dc[kDcPT] = nPT;
        a.dc[kDcEE] = nEE;
        a.dc[kDcFlags] = flags;
    }
    if (flags) return;   // over capacity: the host builds the set again
    const bool pt = b < a.nbp;
    const WalkGroup G(pt ? a.pb : a.eb);
    const int q = pt ? walk_query(G, b, a.Vs, a.pperm) : walk_query(G, b - a.nbp, a.Es, a.eperm);
    const int* off = pt ? a.oPT : a.oEE;
    int* cand = pt ? a.candUPT : a.candUEE;
    int* own = pt ? a.ownPT : a.ownEE;
    int o = 0, c = 0;
    if (q >= 0) {
        o = off[q] - (pt ? 0 : off[0]);   // the joint scan's edge starts begin at the point total
        c = off[q + 1] - off[q];
    }
    const bool again = c > kQueryCap;
    if (__any(again)) {
        auto put = [&](int i, int f) { if (i < c) cand[o + i] = f; };
        if (pt) point_hits(a, G, again ? q : -1, lds, put);
        else edge_hits(a, G, again ? q : -1, lds, put);
    }
    const int* buf = (pt ? a.bufPT : a.bufEE) + (size_t)(q >= 0 ? q : 0) * kQueryCap;
    for (int k = G.l; k < c; k += 4 << G.bits) {
        if (!again) cand[o + k] = buf[k];
        own[o + k] = q;
    }
}
// Both hit kinds' filters and classification in one launch: work-groups [0, nbp) the point
// hits, the rest the edge hits.
struct BothClassify {
    int nbp, F, Es;
    const int *dc, *ownPT, *oPT, *sv, *bt, *candUPT, *ownEE, *oEE, *candUEE, *vs;
    const int4* faces;
    const int2* se;
    const double *x, *vrest;
    double hhat, sq;
    int *candPT, *catPT, *candEE, *catEE;
    int4 *recPT, *recEE;
    int2* auxEE;
};
__global__ void classify_both(BothClassify a) {
    const int b = blockIdx.x;
    if (b < a.nbp)
        pt_classify(b * blockDim.x + threadIdx.x, a.dc, a.F, a.ownPT, a.oPT, a.sv, a.x, a.bt, a.faces, a.candUPT, a.candPT, a.hhat, a.sq,
                    a.vs, a.recPT, a.catPT);
    else
        ee_classify((b - a.nbp) * blockDim.x + threadIdx.x, a.dc, a.Es, a.ownEE, a.oEE, a.se, a.x, a.vrest, a.bt, a.candUEE, a.candEE,
                    a.hhat, a.sq, a.vs, a.recEE, a.auxEE, a.catEE);
}
// The walks (compact = false) or the compactions, of the point queries (pt), the edge queries
// (ee) or both, with 4 << pb and 4 << eb lanes per query, on st.  Only the joint launches reset
// and publish the device counts.
void launch_active_walks(Context& c, bool pt, bool ee, bool compact, int pb, int eb, hipStream_t st) {
    Scene& s = c.sc;
    ActiveSetScratch& b = c.as;
    BothWalks a;
    a.Vs = s.Vs; a.Es = s.Es; a.pb = pb; a.eb = eb;
    a.nbp = pt ? (int)blocks_for((size_t)s.Vs << pb, 16) : 0;
    const int nbe = ee ? (int)blocks_for((size_t)s.Es << eb, 16) : 0;
    a.pperm = s.sv_perm.p; a.sv = s.sv.p; a.eperm = s.se_perm.p; a.se = s.se.p; a.x = s.x.p;
    a.ft = TreeView{c.face_tree.n, c.face_tree.nodes.p, c.face_tree.wide.p};
    a.et = TreeView{c.edge_tree.n, c.edge_tree.nodes.p, c.edge_tree.wide.p};
    a.sq = sqrt(s.hhat); a.gd = s.gd; a.hhat = s.hhat; a.gn = s.gn;
    // the joint count / start arrays: points (Vs + 1), edges (Es + 1), ground flags (Vs + 1)
    a.cntPT = b.cnt_all.p; a.cntEE = a.cntPT + (s.Vs + 1); a.fg = a.cntEE + (s.Es + 1);
    a.bufPT = b.bufPT.p; a.bufEE = b.bufEE.p;
    a.oPT = b.off_all.p; a.oEE = a.oPT + (s.Vs + 1); a.dc = pt && ee ? c.dcnt.p : nullptr; a.capPT = b.capPT; a.capEE = b.capEE;
    a.candUPT = b.candUPT.p; a.candUEE = b.candUEE.p; a.ownPT = b.ownPT.p; a.ownEE = b.ownEE.p;
    const dim3 grid(std::max(a.nbp + nbe, 1));   // (a launch without queries still writes the tails and counts)
    if (compact) hipLaunchKernelGGL(compact_both, grid, dim3(64), 0, st, a);
    else hipLaunchKernelGGL(traverse_both, grid, dim3(64), 0, st, a);
    CIPC_CHECK_LAUNCH();
}

// Buffers of the hits and of the outputs are sized by the capacities, so no stage needs a
// count on the host: every kernel reads its count from dcnt, and does nothing once a
// capacity is exceeded (the host then grows it and builds the set again).  Bounds: a
// category of hits is at most the hits of its type, so the outputs are bounded by the hit
// capacities (Self_ActiveSet head nA + nB, map tail nM <= nm <= capM, Self_EE_ActiveSet
// nE <= nEE, CCD pairs nPTk + nEEk <= nPT + nEE, ground nG <= Vs).
void compute_active_set(Context& c, bool publish) {
    Scene& s = c.sc;
    // Everything on the main stream: both static trees refitted by the same launches, both
    // walks in one launch, both compactions in one, both classifications in one.
    const int Vs = s.Vs, Es = s.Es;
    {
        PrimSrc fs, es;
        fs.kind = 1; fs.faces = s.faces.p; fs.x = s.x.p;
        es.kind = 2; es.se = s.se.p; es.x = s.x.p;
        c.face_tree.prim.resize(std::max(s.F, 1));
        c.edge_tree.prim.resize(std::max(Es, 1));
        if (refit_only(c.face_tree, s.F) && refit_only(c.edge_tree, Es)) refit_two(c.face_tree, fs, c.edge_tree, es, c.stream);
        else build_static_trees(c);
    }
    ActiveSetScratch& b = c.as;
    const double sq = sqrt(s.hhat);
    if (b.capPT == 0) b.capPT = std::max(1024, 4 * Vs);
    if (b.capEE == 0) b.capEE = std::max(1024, 4 * Es);
    if (b.capM == 0) b.capM = 1024;
    const int capPT = b.capPT, capEE = b.capEE, capM = b.capM;
    c.dcnt.resize(kDcWords);
    int* dc = c.dcnt.p;
    // hit counts per point and per edge query and the ground flags, in one array for one scan
    const int nall = (Vs + 1) + (Es + 1) + (Vs + 1);
    b.cnt_all.resize(nall); b.off_all.resize(nall);
    int* cPT = b.cnt_all.p;
    int* cEE = cPT + (Vs + 1);
    int* cG = cEE + (Es + 1);
    const int* oPT = b.off_all.p;
    const int* oEE = oPT + (Vs + 1);
    const int* oG = oEE + (Es + 1);
    size_active_walks(c);
    // A: the walks (the point walk also sets the ground flags; the launch zeroes the scan
    // segments' tails and the device counts)
    launch_active_walks(c, true, true, false, c.tune.as_pt_bits, c.tune.as_ee_bits, c.stream);
    // one scan: the edge and ground segments' starts come out offset by their first entry
    exclusive_scan_int(c, b.cnt_all.p, b.off_all.p, nall);
    // B + C: pack, sort, filter and classify the hits
    b.candUPT.resize(capPT + 1); b.candUEE.resize(capEE + 1);
    b.candPT.resize(capPT + 1); b.recPT.resize(capPT + 1); b.catPT.resize(capPT + 1); b.ownPT.resize(capPT + 1);
    b.candEE.resize(capEE + 1); b.recEE.resize(capEE + 1); b.catEE.resize(capEE + 1); b.auxEE.resize(capEE + 1); b.ownEE.resize(capEE + 1);
    BothClassify cl;
    cl.F = s.F; cl.Es = Es;
    cl.dc = dc; cl.ownPT = b.ownPT.p; cl.oPT = oPT; cl.sv = s.sv.p; cl.bt = s.bt.p; cl.candUPT = b.candUPT.p;
    cl.ownEE = b.ownEE.p; cl.oEE = oEE; cl.candUEE = b.candUEE.p; cl.vs = scene_of_vertex(s); cl.faces = s.faces.p; cl.se = s.se.p;
    cl.x = s.x.p; cl.vrest = s.vrest.p; cl.hhat = s.hhat; cl.sq = sq;
    cl.candPT = b.candPT.p; cl.catPT = b.catPT.p; cl.candEE = b.candEE.p; cl.catEE = b.catEE.p;
    cl.recPT = b.recPT.p; cl.recEE = b.recEE.p; cl.auxEE = b.auxEE.p;
    // the point hits' work-groups, then the edge hits' (none of a kind without queries)
    cl.nbp = Vs > 0 ? (int)blocks_for(capPT, 128) : 0;
    const int nbe = Es > 0 ? (int)blocks_for(capEE, 128) : 0;
    launch_active_walks(c, true, true, true, c.tune.as_pt_bits, c.tune.as_ee_bits, c.stream);
    if (cl.nbp + nbe > 0) hipLaunchKernelGGL(classify_both, dim3(cl.nbp + nbe), dim3(128), 0, c.stream, cl);
    CIPC_CHECK_LAUNCH();
    // category counts of every block of hits
    const int blocksPT = (int)blocks_for(capPT, kCatBlock), blocksEE = (int)blocks_for(capEE, kCatBlock);
    b.cat_sums.resize((size_t)blocksPT + blocksEE + 2);   // then the totals
    hipLaunchKernelGGL(category_counts, dim3(blocksPT + blocksEE), dim3(kCatThreads), 0, c.stream, dc, blocksPT, b.catPT.p, b.catEE.p,
                       b.cat_sums.p);
    const bool own_counts = blocksPT + blocksEE <= kOwnCounts;
    if (!own_counts)
        hipLaunchKernelGGL(category_starts, dim3(1), dim3(kStartThreads), 0, c.stream, dc, blocksPT, blocksEE, b.cat_sums.p);
    CIPC_CHECK_LAUNCH();
    // PP/PE map keys need the vertex count to fit three fields in 64 bits
    int bits = 1;
    while ((1ll << bits) < (long long)s.V + 2) ++bits;
    if (3 * bits > 64) throw Error(CIPC_ERR_OVERFLOW, "vertex count too large for the point-point/point-edge key packing");
    // outputs, sized by their bounds (the map tail of Self_ActiveSet has at most capM entries)
    c.self_set.resize((size_t)capPT + capEE + capM + 1); c.ee_set.resize((size_t)capEE + 1); c.ee_ie.resize((size_t)capEE + 1);
    c.ccd_set.resize((size_t)capPT + capEE + 1); c.env_set.resize((size_t)Vs + 1);
    b.mkeys.resize(capM); b.mkeys_sorted.resize(capM); b.ukeys.resize(capM); b.ucounts.resize(capM); b.nruns.resize(1);
    {
        ScatterArgs a;
        a.dc = dc; a.V = s.V; a.bits = bits; a.Vs = Vs; a.capM = capM;
        a.bPT = blocksPT; a.bEE = blocksEE; a.bG = (int)blocks_for(Vs, kCatThreads); a.own_counts = own_counts; a.sums = b.cat_sums.p;
        a.catPT = b.catPT.p; a.ownPT = b.ownPT.p; a.candPT = b.candPT.p; a.recPT = b.recPT.p;
        a.catEE = b.catEE.p; a.ownEE = b.ownEE.p; a.candEE = b.candEE.p; a.recEE = b.recEE.p; a.auxEE = b.auxEE.p;
        a.sv = s.sv.p; a.fg = cG; a.pg = oG; a.self_set = c.self_set.p; a.ee_set = c.ee_set.p; a.ee_ie = c.ee_ie.p;
        a.ccd = c.ccd_set.p; a.mkeys = b.mkeys.p; a.env = c.env_set.p;
        const int blocks = a.bPT + a.bEE + a.bG + (int)blocks_for(capM, kCatThreads);
        hipLaunchKernelGGL(scatter_all, dim3(blocks), dim3(kCatThreads), 0, c.stream, a);
        CIPC_CHECK_LAUNCH();
    }
    // PP/PE map: sort packed keys, run-length encode (std::map order with multiplicity); the
    // all-ones keys past nm form the last run
    sort_u64(c, b.mkeys.p, b.mkeys_sorted.p, capM, 3 * bits);
    size_t bytes = 0;
    CIPC_HIP(hipcub::DeviceRunLengthEncode::Encode(nullptr, bytes, b.mkeys_sorted.p, b.ukeys.p, b.ucounts.p, b.nruns.p, capM, c.stream));
    c.tmp.reserve(bytes);
    CIPC_HIP(hipcub::DeviceRunLengthEncode::Encode(c.tmp.p, bytes, b.mkeys_sorted.p, b.ukeys.p, b.ucounts.p, b.nruns.p, capM, c.stream));
    hipLaunchKernelGGL(map_decode, dim3(blocks_for(capM, 256)), dim3(256), 0, c.stream, capM, b.nruns.p, dc, b.ukeys.p, b.ucounts.p,
                       s.V, bits, c.self_set.p);
    CIPC_CHECK_LAUNCH();
    // the counts are read with the host's next synchronisation (settle_active_set)
    c.pin_dc.reserve(kDcWords);
    if (publish) CIPC_HIP(hipMemcpyAsync(c.pin_dc.p, dc, kDcWords * sizeof(int), hipMemcpyDeviceToHost, c.stream));
    c.dc_pending = true;
}

namespace {
int grown(int cap, int need) {
    if (need > INT32_MAX / 2) throw Error(CIPC_ERR_OVERFLOW, "active-set count beyond the 32-bit index range");
    return need > cap ? need + need / 4 + 256 : cap;
}
}  // namespace

bool grow_capacities(Context& c) {
    if (!c.dc_pending) return false;
    ActiveSetScratch& b = c.as;
    const int* h = c.pin_dc.p;
    const int flags = h[kDcFlags];
    // the hit counts are final whenever they were counted; the map and contact counts only
    // once the hits fitted
    if (flags & 1) b.capPT = grown(b.capPT, h[kDcPT]);
    if (flags & 2) b.capEE = grown(b.capEE, h[kDcEE]);
    if (flags & 4) b.capM = grown(b.capM, h[kDcMapKeys]);
    if (flags == 0 && h[kDcContactOver]) c.capS = grown(c.capS, h[kDcSelf] + h[kDcMol]);
    return flags != 0 || h[kDcContactOver] != 0;
}

bool settle_active_set(Context& c) {
    if (!c.dc_pending) return false;
    bool rebuilt = false;
    for (int round = 0;; ++round) {
        CIPC_HIP(hipStreamSynchronize(c.stream));
        if (!grow_capacities(c)) break;
        if (round >= 3) throw Error(CIPC_ERR_RUNTIME, "active-set capacities kept overflowing");
        compute_active_set(c);
        rebuilt = true;
    }
    const int* h = c.pin_dc.p;
    c.n_self = h[kDcSelf]; c.n_ee = h[kDcMol]; c.n_ccd = h[kDcCCD]; c.n_env = h[kDcEnv];
    c.dc_pending = false;
    return rebuilt;
}

void active_set_now(Context& c) {
    compute_active_set(c);
    settle_active_set(c);
}

// ---------------------------------------------------------------------------------
// isIntersected (IPCSolver.cpp:476-542): ground gaps of the current
// Environment_ActiveSet, then every surface edge against every face whose static box it
// touches, with IglUtils::segTriIntersect (ContactMechanics.h:47-71).
// ---------------------------------------------------------------------------------
// Eigen 3.4 FullPivLU solve of the 3x3 system of segTriIntersect: complete pivoting on
// the first largest |a_ij| in column-major order, rank threshold 3 eps |max pivot|.
__device__ inline bool seg_tri(d3 e0, d3 e1, d3 t0, d3 t1, d3 t2) {
    const d3 c0 = t1 - t0, c1 = t2 - t0, c2 = e0 - e1;
    const d3 n = cross(c0, c1);
    if (dot(n, e0 - t0) * dot(n, e1 - t0) > 0.0) return false;
    double A[3][3] = {{c0.x, c1.x, c2.x}, {c0.y, c1.y, c2.y}, {c0.z, c1.z, c2.z}};
    const double det = A[0][0] * (A[1][1] * A[2][2] - A[1][2] * A[2][1]) - A[0][1] * (A[1][0] * A[2][2] - A[1][2] * A[2][0])
                     + A[0][2] * (A[1][0] * A[2][1] - A[1][1] * A[2][0]);
    if (det == 0.0) return false;
    int rt[3] = {0, 1, 2}, ct[3] = {0, 1, 2}, nz = 3;
    double maxpiv = 0.0;
    for (int k = 0; k < 3; ++k) {
        int br = k, bc = k;
        double best = fabs(A[k][k]);
        for (int cc = k; cc < 3; ++cc)
            for (int r = k; r < 3; ++r)
                if (fabs(A[r][cc]) > best) { best = fabs(A[r][cc]); br = r; bc = cc; }
        if (best == 0.0) { nz = k; for (int i = k; i < 3; ++i) { rt[i] = i; ct[i] = i; } break; }
        if (best > maxpiv) maxpiv = best;
        rt[k] = br; ct[k] = bc;
        if (br != k) for (int cc = 0; cc < 3; ++cc) { const double t = A[k][cc]; A[k][cc] = A[br][cc]; A[br][cc] = t; }
        if (bc != k) for (int r = 0; r < 3; ++r) { const double t = A[r][k]; A[r][k] = A[r][bc]; A[r][bc] = t; }
        for (int r = k + 1; r < 3; ++r) A[r][k] /= A[k][k];
        for (int cc = k + 1; cc < 3; ++cc)
            for (int r = k + 1; r < 3; ++r) A[r][cc] -= A[r][k] * A[k][cc];
    }
    int rank = 0;
    const double thr = maxpiv * (2.220446049250313e-16 * 3.0);
    for (int i = 0; i < nz; ++i) rank += fabs(A[i][i]) > thr;
    const d3 rhs = e0 - t0;
    double cv[3] = {rhs.x, rhs.y, rhs.z}, xs[3] = {0, 0, 0};
    if (rank > 0) {
        for (int k = 0; k < 3; ++k) { const double t = cv[k]; cv[k] = cv[rt[k]]; cv[rt[k]] = t; }
        for (int i = 0; i < 3; ++i) if (cv[i] != 0.0) for (int r = i + 1; r < 3; ++r) cv[r] -= cv[i] * A[r][i];
        for (int i = rank - 1; i >= 0; --i) {
            if (cv[i] == 0.0) continue;
            cv[i] /= A[i][i];
            for (int r = 0; r < i; ++r) cv[r] -= cv[i] * A[r][i];
        }
        int q[3] = {0, 1, 2};
        for (int k = 0; k < 3; ++k) { const int t = q[k]; q[k] = q[ct[k]]; q[ct[k]] = t; }
        for (int i = 0; i < 3; ++i) xs[q[i]] = (i < rank) ? cv[i] : 0.0;
    }
    return xs[0] >= 0.0 && xs[1] >= 0.0 && xs[0] + xs[1] <= 1.0 && xs[2] >= 0.0 && xs[2] <= 1.0;
}
// hit[0] (one scene) or hit[scene] (batch) is set for a face that an edge crosses.  The edges
// walk the face tree (GroupWalk), a group of lanes each; the pairs whose boxes may overlap are
// queued in LDS and tested 64 at a time, so that the test's lanes are full whatever query found
// them.  One lane per face, walking the binary tree of the edges and testing on the way, took 162 us
// on four 20^3 cubes; this takes 27, and the edge tree needs no refit.
__global__ __launch_bounds__(64) void intersect_kernel(int Es, int bits, const int* __restrict__ perm, const int4* __restrict__ faces,
                                                       const int2* __restrict__ se, const double* __restrict__ x,
                                                       const int* __restrict__ bt, TreeView ft, const Box* __restrict__ fbox,
                                                       const int* __restrict__ vs, int* __restrict__ hit) {
    __shared__ int lds[kWalkInts];
    __shared__ int2 met[kPairQueue], kept[kPairQueue];
    const WalkGroup G(bits);
    const int e = walk_query(G, xcd_block(blockIdx.x, gridDim.x), Es, perm);
    Box q{};
    if (e >= 0) q = box_edge(ld3(x, se[e].x), ld3(x, se[e].y));
    pair_walk<false>(ft, G, e, q, 0, lds, met, kept, [&](int2 pr) {
        const int2 E = se[pr.x];
        const int4 fv = faces[pr.y];
        if (E.x == fv.x || E.x == fv.y || E.x == fv.z || E.y == fv.x || E.y == fv.y || E.y == fv.z) return false;
        if (vs && vs[E.x] != vs[fv.x]) return false;
        if (is_collider(bt[E.x]) && is_collider(bt[E.y]) && is_collider(bt[fv.x]) && is_collider(bt[fv.y]) && is_collider(bt[fv.z]))
            return false;
        return overlaps(box_edge(ld3(x, E.x), ld3(x, E.y)), fbox[pr.y], 0.0);   // the walk's boxes are float
    }, [&](bool on, int2 pr) {
        if (!on) return;
        const int2 E = se[pr.x];
        const int4 fv = faces[pr.y];
        if (seg_tri(ld3(x, E.x), ld3(x, E.y), ld3(x, fv.x), ld3(x, fv.y), ld3(x, fv.z))) atomicOr(hit + (vs ? vs[fv.x] : 0), 1);
    });
}
__global__ void ground_touch_kernel(int n, const int* __restrict__ env, const double* __restrict__ x, d3 gn, double gd,
                                    const int* __restrict__ vs, int* __restrict__ hit) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int v = env[i];
    const double dist = dot(gn, ld3(x, v)) - gd;
    if (dist * dist <= 0.0) atomicOr(hit + (vs ? vs[v] : 0), 1);
}
__global__ void zero_int(int* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

void scene_intersections(Context& c, int* out) {
    Scene& s = c.sc;
    const int S = s.S;
    c.counters.resize(2 * (size_t)S);
    hipLaunchKernelGGL(zero_int, dim3(blocks_for(2 * S, 64)), dim3(64), 0, c.stream, c.counters.p, 2 * S);
    if (c.n_env > 0)
        hipLaunchKernelGGL(ground_touch_kernel, dim3(blocks_for(c.n_env, 256)), dim3(256), 0, c.stream, (int)c.n_env, c.env_set.p,
                           s.x.p, s.gn, s.gd, scene_of_vertex(s), c.counters.p);
    // only the face tree is walked: the edge tree keeps its boxes until its next build
    PrimSrc fs;
    fs.kind = 1; fs.faces = s.faces.p; fs.x = s.x.p;
    c.face_tree.prim.resize(std::max(s.F, 1));
    build_tree_from(c, c.face_tree, s.F, fs, c.stream, c.tmp);
    if (s.F > 0 && s.Es > 0) {
        const int bits = walk_bits(s.Es, kCcdEdges);
        hipLaunchKernelGGL(intersect_kernel, dim3(blocks_for((size_t)s.Es << bits, 16)), dim3(64), 0, c.stream, s.Es, bits, s.se_perm.p,
                           s.faces.p, s.se.p, s.x.p, s.bt.p, TreeView{c.face_tree.n, c.face_tree.nodes.p, c.face_tree.wide.p},
                           c.face_tree.prim.p, scene_of_vertex(s), c.counters.p + S);
    }
    CIPC_CHECK_LAUNCH();
    std::vector<int> h(2 * (size_t)S);
    read_back(c, h.data(), (const int*)c.counters.p, h.size());
    for (int k = 0; k < S; ++k) out[k] = (h[k] != 0 || h[S + k] != 0) ? 1 : 0;
}

// ---------------------------------------------------------------------------------
// Evaluation entry point (tests): the walks over boxes of the caller's
// ---------------------------------------------------------------------------------
// queries: all leaves a query may overlap, in any order (query_hits); null: each box's own query
// for the leaves after its own, the overlapping pairs once or more (pair_walk)
__global__ __launch_bounds__(64) void walk_eval_kernel(TreeView t, const Box* __restrict__ box, int nq, const Box* __restrict__ queries,
                                                       double gap, int bits, int depth, int max_hits, int* __restrict__ counts,
                                                       int* __restrict__ hits) {
    __shared__ int lds[kWalkInts];
    __shared__ int2 met[kPairQueue], kept[kPairQueue];
    const WalkGroup G(bits, depth);
    const int i = (blockIdx.x << (4 - bits)) + G.g, q = i < nq ? i : -1;
    if (queries) {
        const int n = query_hits(t, G, q >= 0, q >= 0 ? queries[q] : Box{}, gap, -1, lds, [&](int k, int prim) {
            if (k < max_hits) hits[(size_t)q * max_hits + k] = prim;
        });
        if (q >= 0 && G.l == 0) counts[q] = n;
        return;
    }
    pair_walk<true>(t, G, q, q >= 0 ? box[q] : Box{}, q >= 0 ? t.leafpos[q] : 0, lds, met, kept,
                    [&](int2 pr) { return overlaps(box[pr.x], box[pr.y], 0.0); },
                    [&](bool on, int2 pr) {
                        if (!on) return;
                        const int k = atomicAdd(counts + pr.x, 1);
                        if (k < max_hits) hits[(size_t)pr.x * max_hits + k] = pr.y;
                    });
}
void eval_walk(int n, const double* boxes, int nq, const double* queries, double gap, int bits, int depth, int max_hits, int* counts,
               int* hits) {
    Context c;
    LBVH t;
    DBuf<Box> q;
    DBuf<int> dc, dh;
    t.prim.resize(n); dc.resize(nq); dh.resize((size_t)nq * max_hits);
    CIPC_HIP(hipMemcpy(t.prim.p, boxes, sizeof(Box) * n, hipMemcpyHostToDevice));
    if (queries) {
        q.resize(nq);
        CIPC_HIP(hipMemcpy(q.p, queries, sizeof(Box) * nq, hipMemcpyHostToDevice));
    }
    hipLaunchKernelGGL(zero_int, dim3(blocks_for(nq, 256)), dim3(256), 0, c.stream, dc.p, nq);
    build_tree(c, t, n);
    hipLaunchKernelGGL(walk_eval_kernel, dim3(blocks_for((size_t)nq << bits, 16)), dim3(64), 0, c.stream,
                       TreeView{t.n, t.nodes.p, t.wide.p, t.leafpos.p}, t.prim.p, nq, q.p, gap, bits, depth, max_hits, dc.p, dh.p);
    CIPC_CHECK_LAUNCH();
    CIPC_HIP(hipMemcpy(counts, dc.p, sizeof(int) * nq, hipMemcpyDeviceToHost));
    CIPC_HIP(hipMemcpy(hits, dh.p, sizeof(int) * nq * (size_t)max_hits, hipMemcpyDeviceToHost));
}

bool any_intersection(Context& c) {
    std::vector<int> r(c.sc.S);
    scene_intersections(c, r.data());
    for (int v : r)
        if (v) return true;
    return false;
}

}  // namespace cipc
