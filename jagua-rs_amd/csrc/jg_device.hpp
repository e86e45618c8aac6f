// Device-side views of the flattened engine and the query item, and the traversal
// primitives shared by every query kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "jg_geom.hpp"

namespace jg {

constexpr uint32_t ENTIRE_BIT = 0x80000000u;
constexpr uint32_t SLOT_MASK = 0x7fffffffu;
constexpr uint32_t COUNT_MASK = 0x3fffffffu;
constexpr uint32_t HIT = 0xffffffffu;

struct DevNode {                      // mirrors FlatNode (32 B)
    float4 bbox;
    int32_t first_child;
    uint32_t haz_begin, haz_info, n_active_edges;
};

struct DevEntry {                     // mirrors FlatEntry (32 B)
    float4 ff;
    uint32_t slot_flags, edge_begin, edge_count, n_edges_total;
};

// Reads of the engine image and the item records.  Their pointers come out of descriptor
// tables, so the compiler sees generic addresses and would issue flat loads, which count
// against the LDS wait counter as well: every LDS read of the traversal would then wait for
// the node and edge loads in flight.  These read through global-address-space pointers
// (global_load) instead.
#if defined(__HIP_DEVICE_COMPILE__)
typedef int jg_i4 __attribute__((ext_vector_type(4)));
typedef int jg_i2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) const jg_i4 jg_gi4;
typedef __attribute__((address_space(1))) const jg_i2 jg_gi2;
typedef __attribute__((address_space(1))) const int jg_gi1;
__device__ __forceinline__ float4 ldg4(const float4* p) {
    const jg_i4 v = *(jg_gi4*)p;
    return make_float4(__int_as_float(v.x), __int_as_float(v.y), __int_as_float(v.z), __int_as_float(v.w));
}
__device__ __forceinline__ float2 ldg2(const float2* p) {
    const jg_i2 v = *(jg_gi2*)p;
    return make_float2(__int_as_float(v.x), __int_as_float(v.y));
}
__device__ __forceinline__ uint2 ldg2u(const uint2* p) {
    const jg_i2 v = *(jg_gi2*)p;
    return make_uint2((uint32_t)v.x, (uint32_t)v.y);
}
__device__ __forceinline__ uint32_t ldg1(const uint32_t* p) { return (uint32_t)*(jg_gi1*)p; }
__device__ __forceinline__ DevNode ldg_node(const DevNode* p) {
    const jg_i4 a = ((jg_gi4*)p)[0], b = ((jg_gi4*)p)[1];
    DevNode n;
    n.bbox = make_float4(__int_as_float(a.x), __int_as_float(a.y), __int_as_float(a.z), __int_as_float(a.w));
    n.first_child = b.x;
    n.haz_begin = (uint32_t)b.y;
    n.haz_info = (uint32_t)b.z;
    n.n_active_edges = (uint32_t)b.w;
    return n;
}
__device__ __forceinline__ DevEntry ldg_ent(const DevEntry* p) {
    const jg_i4 a = ((jg_gi4*)p)[0], b = ((jg_gi4*)p)[1];
    DevEntry e;
    e.ff = make_float4(__int_as_float(a.x), __int_as_float(a.y), __int_as_float(a.z), __int_as_float(a.w));
    e.slot_flags = (uint32_t)b.x;
    e.edge_begin = (uint32_t)b.y;
    e.edge_count = (uint32_t)b.z;
    e.n_edges_total = (uint32_t)b.w;
    return e;
}
#else
__device__ inline float4 ldg4(const float4* p) { return *p; }
__device__ inline float2 ldg2(const float2* p) { return *p; }
__device__ inline uint2 ldg2u(const uint2* p) { return *p; }
__device__ inline uint32_t ldg1(const uint32_t* p) { return *p; }
__device__ inline DevNode ldg_node(const DevNode* p) { return *p; }
__device__ inline DevEntry ldg_ent(const DevEntry* p) { return *p; }
#endif
// The slot | Entire word of an entry (its fifth word).
__device__ __forceinline__ uint32_t ldg_slot_flags(const DevEntry* p) { return ldg1((const uint32_t*)p + 4); }

struct CdeView {
    const DevNode* nodes;
    const uint32_t* node_up;          // parent << 2 | sibling index
    const DevEntry* ent;
    const float4* edges;
    const float4* haz_bbox;
    const float4* haz_poi;            // cx, cy, r, interior
    const uint2* haz_vr;
    const float2* haz_verts;
    const uint32_t* cells;            // the deepest node on the path to each cell of a
                                      // 2^cell_level grid over the root box (row iy, column ix)
    uint32_t n_slots, exterior_slot, cd_threshold, n_nodes;
    uint32_t cell_level;
    CellGrid grid;                    // the deepest table level's grid (circle_cells)
    uint32_t box_bound;               // every hazard but exterior_slot's is collected only where its box is met
    float4 ext_inner;                 // a box inside the container (the exterior hazard's shape):
                                      // its bbox when that shape is an axis-aligned rectangle,
                                      // else empty (x_min > x_max)
};

// A cell table entry: cdepth << 28 | depth << 24 | node, for the deepest node on the path to the
// cell and the depth of the first node on that path where QTNode::collect_collisions tests
// entries (15: none on the path).
constexpr uint32_t CELL_NODE = 0xffffffu;
__device__ __forceinline__ uint32_t cell_depth(uint32_t e) { return (e >> 24) & 15u; }
__device__ __forceinline__ uint32_t cell_cdepth(uint32_t e) { return e >> 28; }

struct ItemView {
    const float2* v;                  // local vertices (CCW)
    const float4* ff;                 // ff poles (cx, cy, r, 0) then piers (x1 y1 x2 y2)
    float4 poi;
    uint32_t n_v, n_poles, n_piers, pad;
};

struct FilterView {
    const uint32_t* mask;             // JG_FILTER_KEYS: bit per slot
    uint32_t kind, seed, threshold, n_words;
};

__device__ __forceinline__ bool irrelevant(const FilterView& f, uint64_t q, uint32_t slot) {
    if (f.kind == 0) return false;
    if (f.kind == 1) return (slot >> 5) < f.n_words && ((f.mask[slot >> 5] >> (slot & 31u)) & 1u);
    return filter_hash(f.seed, q, slot) < f.threshold;
}

__device__ __forceinline__ Mat load_mat(const float* m6, uint64_t i) {
    const float* p = m6 + 6 * i;
    return Mat{p[0], p[1], p[2], p[3], p[4], p[5]};
}

// QTHazardVec::strongest (qt_hazard_vec.rs:60-63): index of the first relevant entry of
// node `nd`, or -1.  Without a filter it is the first entry, whose presence the node record
// carries, so no entry is read.
__device__ __forceinline__ int strongest(const CdeView& c, const DevNode& nd, const FilterView& f, uint64_t q,
                                         bool& entire) {
    const uint32_t cnt = nd.haz_info & COUNT_MASK;
    if (f.kind == 0) {
        entire = (nd.haz_info & ENTIRE_BIT) != 0u;
        return cnt ? (int)nd.haz_begin : -1;
    }
    for (uint32_t i = 0; i < cnt; i++) {
        const uint32_t sf = c.ent[nd.haz_begin + i].slot_flags;
        if (!irrelevant(f, q, sf & SLOT_MASK)) {
            entire = (sf & ENTIRE_BIT) != 0u;
            return (int)(nd.haz_begin + i);
        }
    }
    return -1;
}

// Depth-first descent in the reference's quadrant order without a memory stack: the
// pending-sibling masks of the current path live 4 bits per level in one 64-bit register;
// moving to a sibling or the parent uses the node_up links of the device image.
// visit(node, &first_child) returns HIT to stop, or the mask of children to descend into.
template <class Visit>
__device__ __forceinline__ bool descend(const CdeView& c, int start, Visit visit) {
    int n = start;
    uint32_t d = 0;
    uint64_t pend = 0;
    for (;;) {
        int fc = -1;
        const uint32_t m = visit(n, fc);
        if (m == HIT) return true;
        if (m != 0u) {
            const uint32_t k = (uint32_t)__builtin_ctz(m);
            pend |= (uint64_t)(m & ~(1u << k)) << (4u * d);
            d++;
            n = fc + (int)k;
            continue;
        }
        for (;;) {
            if (d == 0) return false;
            const uint32_t sh = 4u * (d - 1u);
            const uint32_t nib = (uint32_t)(pend >> sh) & 0xfu;
            const uint32_t up = c.node_up[n];
            if (nib != 0u) {
                const uint32_t k = (uint32_t)__builtin_ctz(nib);
                pend &= ~((uint64_t)1 << (sh + k));
                n = n - (int)(up & 3u) + (int)k;
                break;
            }
            n = (int)(up >> 2);
            d--;
        }
    }
}

// CDEngine::get_virtual_root (cd_engine.rs:314-327); children's boxes are the quadrants of
// the node's box (rect.rs:141-151), exactly as the tree built them.  depth: the node's depth.
__device__ __forceinline__ int virtual_root(const CdeView& c, float4 bb, uint32_t& depth) {
    int n = 0;
    depth = 0;
    for (;;) {
        const DevNode nd = ldg_node(c.nodes + n);
        if (nd.first_child < 0) return n;
        const int k = quadrant_surrounding(nd.bbox, bb);
        if (k < 0) return n;
        n = nd.first_child + k;
        depth++;
    }
}
__device__ __forceinline__ int virtual_root(const CdeView& c, float4 bb) {
    uint32_t depth;
    return virtual_root(c, bb, depth);
}

__device__ __forceinline__ uint32_t cell_entry(const CdeView& c, uint32_t l, uint32_t ix, uint32_t iy) {
    return ldg1(c.cells + ((1u << (2u * l)) - 1u) / 3u + ((iy << l) | ix));
}

// virtual_root through the cell tables: at every level above the cell that strictly holds bb, that
// cell's quadrant is the one that surrounds bb, so the search passes the deepest node on the path
// to it; it ends there if that node lies above the cell's level, and goes on through node records
// otherwise.
__device__ __forceinline__ int virtual_root_cells(const CdeView& c, float4 root, float4 bb, uint32_t& depth) {
    const HoldingCell h = holding_cell(c.grid, c.cell_level, root, bb);
    const uint32_t e = cell_entry(c, h.l, h.ix, h.iy);
    int n = (int)(e & CELL_NODE);
    depth = cell_depth(e);
    if (depth < h.l) return n;
    for (;;) {
        const DevNode nd = ldg_node(c.nodes + n);
        if (nd.first_child < 0) return n;
        const int k = quadrant_surrounding(nd.bbox, bb);
        if (k < 0) return n;
        n = nd.first_child + k;
        depth++;
    }
}

// The nodes from which the descent of an edge g (x1 y1 x2 y2), starting at a node n0 of depth d0 that
// holds it, may start instead: the deepest nodes on the paths to its cells (edge_cells), one or
// two of them (n1 = n0 then), when the cells lie below n0.  The edge lies inside the root box.
__device__ __forceinline__ void edge_starts(const CdeView& c, float4 root, uint32_t d0, float4 g, uint32_t& n0, uint32_t& n1) {
    const EdgeCells e = edge_cells_inside(c.grid, c.cell_level, root, g);
    if (e.l > d0) {
        n0 = cell_entry(c, e.l, e.x0, e.y0) & CELL_NODE;
        n1 = e.x0 != e.x1 || e.y0 != e.y1 ? cell_entry(c, e.l, e.x1, e.y1) & CELL_NODE : n0;
    } else {
        n1 = n0;
    }
}

// The node of the deepest table level's cell that holds the circle's centre, or the nearest cell.
__device__ __forceinline__ uint32_t centre_cell(const CdeView& c, float4 root, float cx, float cy) {
    if (!(c.grid.sx > 0.0f)) return 0u;
    const float top = (float)((1u << c.cell_level) - 1u);
    const uint32_t ix = grid_index(cx - root.x, c.grid.sx, top), iy = grid_index(cy - root.y, c.grid.sy, top);
    return ldg1(c.cells + ((1u << (2u * c.cell_level)) - 1u) / 3u + ((iy << c.cell_level) | ix)) & CELL_NODE;
}

// QTNode::collides for a circle (qt_node.rs:99-147; Circle quadrant test qt_traits.rs:10-13)
__device__ __forceinline__ bool collides_circle(const CdeView& c, int start, float cx, float cy, float r,
                                                const FilterView& f, uint64_t q) {
    return descend(c, start, [&](int n, int& fc) -> uint32_t {
        const DevNode nd = c.nodes[n];
        bool entire = false;
        const int s = strongest(c, nd, f, q, entire);
        if (s < 0) return 0u;
        if (entire) return HIT;
        if (nd.first_child >= 0) {
            fc = nd.first_child;
            return circle_quadrants(cx, cy, r, nd.bbox);
        }
        const int he = (int)(nd.haz_begin + (nd.haz_info & COUNT_MASK));
        for (int i = s; i < he; i++) {
            const DevEntry e = c.ent[i];
            if (irrelevant(f, q, e.slot_flags & SLOT_MASK)) continue;
            if (!circle_box(cx, cy, r, e.ff)) continue;
            for (uint32_t j = 0; j < e.edge_count; j++)
                if (circle_edge(cx, cy, r, c.edges[e.edge_begin + j])) return HIT;
        }
        return 0u;
    });
}

// QTNode::collides for an edge (qt_node.rs:99-147; Edge quadrant test qt_traits.rs:19-106)
__device__ __forceinline__ bool collides_edge(const CdeView& c, int start, float4 ed, const FilterView& f, uint64_t q) {
    return descend(c, start, [&](int n, int& fc) -> uint32_t {
        const DevNode nd = c.nodes[n];
        bool entire = false;
        const int s = strongest(c, nd, f, q, entire);
        if (s < 0) return 0u;
        if (entire) return HIT;
        if (nd.first_child >= 0) {
            fc = nd.first_child;
            return edge_quadrants_node(ed, nd.bbox);
        }
        const int he = (int)(nd.haz_begin + (nd.haz_info & COUNT_MASK));
        for (int i = s; i < he; i++) {
            const DevEntry e = c.ent[i];
            if (irrelevant(f, q, e.slot_flags & SLOT_MASK)) continue;
            if (!box_edge(e.ff, ed)) continue;
            for (uint32_t j = 0; j < e.edge_count; j++)
                if (edge_edge(ed, c.edges[e.edge_begin + j])) return HIT;
        }
        return 0u;
    });
}

// ---------------------------------------------------------------------------------------
// Wave-cooperative traversal.  QTNode::collides (qt_node.rs:99-147) answers whether any
// relevant hazard of the subtree collides with the entity; its recursion order only decides
// which hazard is found first.  A wave therefore turns all descents of its entities (up to
// ENT circles or edges, each belonging to one query slot) into two LDS queues: node visits
// (entity, node) and edge tests (entity, hazard edge).  Each step takes 64 items of one kind:
//   node step: the visit's strongest relevant hazard (qt_hazard_vec.rs:60-63) is Entire -> hit;
//              an internal node pushes the colliding quadrants (qt_traits.rs); a leaf pushes one
//              edge test per edge of every relevant Partial hazard whose ff_bbox the entity
//              collides with (qt_partial_hazard.rs:67-72);
//   edge step: one Circle-Edge or Edge-Edge test per lane (circle.rs:109-113, edge.rs:162-228).
// Edge steps run whenever 64 tests are pending, so both kinds of step keep every lane busy.
// A query's verdict is the OR of its entities' hits, exactly the reference's verdict.
//
// Kernels using it run one wavefront per workgroup: lanes exchange queue entries and hit flags
// through LDS only across wave_sync(), a workgroup barrier, which the compiler must reach with
// all lanes together; queue depths are wave-uniform values read from lane 63 of scans.

// Entity kinds of a traversal: KIND_EDGE and KIND_CIRCLE are fixed at compile time;
// KIND_MIXED reads the per-entity kind (surrogates with both poles and piers).
enum : int { KIND_EDGE = 0, KIND_CIRCLE = 1, KIND_MIXED = 2 };

constexpr int WL_EDGE_BITS = 10;          // edge tests one leaf visit pushes: fewer than 2^WL_EDGE_BITS
static_assert(64u * ((1u << WL_EDGE_BITS) - 1u) < 65536u, "a wave's edge pushes must fit 16 bits");
constexpr uint32_t WL_RESERVE = 3u * (JG_MAX_QT_DEPTH + 1u);   // node slots a depth-first walk may need
constexpr uint32_t WL_NODE_MASK = 0xffffffu;
constexpr uint32_t WL_MAX_NODES = 1u << 24;
constexpr uint32_t WL_CIRCLE = 0x80u;     // WorkList::ent_slot flag: the entity is a circle
// An edge-test entry names up to 8 consecutive hazard edges: the first edge's index in its low
// 29 bits, the count less one in the top 3.
constexpr uint32_t WL_EDGE_INDEX = 0x1fffffffu;
constexpr uint32_t WL_MAX_EDGES = WL_EDGE_INDEX + 1u;

// A wave's work list in LDS: NCAP_ node visits, ECAP_ edge tests, ENT_ entities.
template <uint32_t NCAP_, uint32_t ECAP_, uint32_t ENT_>
struct WorkList {
    static constexpr uint32_t NCAP = NCAP_, ECAP = ECAP_, ENT = ENT_;
    uint32_t nodes[NCAP];                 // entity << 24 | node
    uint32_t edges[ECAP];                 // hazard edges (WL_EDGE_INDEX)
    float4 geom[ENT];                     // circle (cx, cy, r, -) or edge (x1 y1 x2 y2)
    uint32_t hit[64];                     // per query slot
    uint32_t qidx[64];                    // per query slot: query index (hashed filters)
    uint8_t edge_ent[ECAP];               // entity of the edge test
    uint8_t ent_slot[ENT];                // query slot (0..63) | WL_CIRCLE
};

template <bool FILT>
__device__ __forceinline__ bool irrel(const FilterView& f, uint64_t q, uint32_t slot) {
    return FILT && irrelevant(f, q, slot);
}

template <bool FILT>
__device__ __forceinline__ int strongest_t(const CdeView& c, const DevNode& nd, const FilterView& f, uint64_t q,
                                           bool& entire) {
    if (!FILT) {
        entire = (nd.haz_info & ENTIRE_BIT) != 0u;
        return (nd.haz_info & COUNT_MASK) ? (int)nd.haz_begin : -1;
    }
    return strongest(c, nd, f, q, entire);
}

// QTHazPartial::collides_with's ff_bbox pre-test (qt_partial_hazard.rs:67-72)
__device__ __forceinline__ bool ff_pass(const DevEntry& e, bool circle, float4 g) {
    return circle ? circle_box(g.x, g.y, g.z, e.ff) : box_edge(e.ff, g);
}

__device__ __forceinline__ bool edge_hit(bool circle, float4 g, float4 he) {
    return circle ? circle_edge(g.x, g.y, g.z, he) : edge_edge(g, he);
}

// The workgroup is a single wavefront: a convergent barrier ordering its lanes' LDS accesses.
__device__ __forceinline__ void wave_sync() { __syncthreads(); }

// Number of set bits of m below this lane.
__device__ __forceinline__ uint32_t lanes_below(uint64_t m, uint32_t lane) {
    return (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull));
}

// Inclusive prefix sum of x over the 64 lanes of a wave with every lane active: DPP row shifts
// within rows of 16 lanes, then the row broadcasts of lanes 15 and 31 (GFX9 DPP).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x, uint32_t lane) {
    const uint32_t rl = lane & 15u;
    uint32_t v = x;
    uint32_t t = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x111, 0xf, 0xf, false);   // row_shr:1
    if (rl >= 1u) v += t;
    t = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x112, 0xf, 0xf, false);            // row_shr:2
    if (rl >= 2u) v += t;
    t = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x114, 0xf, 0xf, false);            // row_shr:4
    if (rl >= 4u) v += t;
    t = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x118, 0xf, 0xf, false);            // row_shr:8
    if (rl >= 8u) v += t;
    t = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x142, 0xf, 0xf, false);            // row_bcast:15
    if ((lane & 31u) >= 16u) v += t;
    t = (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x143, 0xf, 0xf, false);            // row_bcast:31
    if (lane >= 32u) v += t;
    return v;
}

// The node visits and edge tests of a wave's entities.  W.hit[slot] is set for every query slot one
// of whose entities collides.  Callers queue visits with push_root or make an entity's first from
// registers (visit_start); run() works the queues off.
// An edge-test item holds up to EG consecutive edges of one hazard entry: a leaf visit pushes one
// item per EG edges, so the lanes of a node step loop over a few pushes each instead of one per
// edge (a leaf of the benchmark layout holds about 7 edges a circle may meet), and an edge step
// tests up to EG edges per item.
//
// A round's chain of dependent reads is what a small launch waits for, and the steps' instructions on
// half-empty waves what a large one does; a first visit from registers saves a step of both, and an
// internal start node is left to run(), whose code is there once (in copies per set-up: 591 us per
// benchmark step against 564).
template <bool FILT, int KIND, int EG, class Lds>
struct WaveTraversal {
    static_assert(EG >= 1 && EG <= 8, "one to eight edges per edge-test item");
    static constexpr uint32_t NCAP = Lds::NCAP, ECAP = Lds::ECAP, ENT = Lds::ENT;
    static constexpr uint32_t EDGE_LIMIT = 1u << WL_EDGE_BITS;   // edge tests one visit may push: fewer
    static constexpr uint32_t ROOT_ROOM = NCAP - WL_RESERVE - 3u;   // node visits that callers may queue

    const CdeView& c;
    const FilterView& f;
    Lds& W;
    const uint32_t lane;
    uint32_t nn = 0, ne = 0;                      // queued node visits and edge tests

    __device__ __forceinline__ WaveTraversal(const CdeView& c_, const FilterView& f_, Lds& W_, uint32_t lane_)
        : c(c_), f(f_), W(W_), lane(lane_) {}

    // Queues one visit (entity << 24 | node) per lane with `want` set; callers keep nn within
    // ROOT_ROOM.
    __device__ __forceinline__ void push_root(bool want, uint32_t item) {
        const uint64_t b = __ballot(want);
        if (want) W.nodes[nn + lanes_below(b, lane)] = item;
        nn += (uint32_t)__builtin_popcountll(b);
    }

    // The entities' first visits, one per lane with `act` set, from registers: the start node's record
    // nd, the entity's query slot, kind and geometry (also in W.geom).  Most start nodes are leaves, and
    // most of those empty; a leaf's edge tests are queued, and what is more than that (an internal
    // node, more edges than the queue takes) queues the visit itself for run().
    __device__ __forceinline__ void visit_start(bool act, uint32_t item, const DevNode& nd, uint32_t slot, bool circle, float4 g) {
        uint32_t n_edges = 0, p_beg = 0, p_cnt = 0, n_pass = 0;
        bool later = false;
        int he = 0, s = -1;
        uint64_t q = 0;
        act = act && (nd.haz_info & COUNT_MASK) != 0u;
        if (act && !(KIND == KIND_EDGE || !circle || (item & WL_NODE_MASK) == 0u)) act = circle_box(g.x, g.y, g.z, nd.bbox);
        if (act) {
            if (FILT) q = W.qidx[slot];
            bool entire = false;
            s = strongest_t<FILT>(c, nd, f, q, entire);
            if (s >= 0 && entire) {
                W.hit[slot] = 1u;
            } else if (s >= 0 && nd.first_child >= 0) {
                later = true;
            } else if (s >= 0) {
                he = (int)(nd.haz_begin + (nd.haz_info & COUNT_MASK));
                for (int i = s; i < he; i++) {
                    const DevEntry e = ldg_ent(c.ent + i);
                    if (!irrel<FILT>(f, q, e.slot_flags & SLOT_MASK) && ff_pass(e, circle, g)) {
                        if (n_pass == 0u) {
                            p_beg = e.edge_begin;
                            p_cnt = e.edge_count;
                        }
                        n_pass++;
                        n_edges += (e.edge_count + (uint32_t)EG - 1u) / (uint32_t)EG;
                    }
                }
            }
        }
        // a leaf of several passing entries is left to run() as well
        later = later || n_edges >= EDGE_LIMIT || n_pass > 1u;
        if (later) n_edges = 0;
        const uint32_t incl = wave_incl_scan(n_edges, lane);
        const uint32_t e_tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        const bool fits = ne + e_tot <= ECAP;
        if (n_edges && fits) {
            uint32_t at = ne + incl - n_edges;
            for (uint32_t j = 0; j < p_cnt; j += EG, at++) {
                const uint32_t k = p_cnt - j < (uint32_t)EG ? p_cnt - j : (uint32_t)EG;
                W.edges[at] = (p_beg + j) | ((k - 1u) << 29);
                W.edge_ent[at] = (uint8_t)(item >> 24);
            }
        }
        if (fits) ne += e_tot;
        push_root(later || (n_edges != 0u && !fits), item);
    }

    __device__ __forceinline__ void run() {
        while (nn + ne != 0u) {
            wave_sync();                              // pushes and hit flags of the last step are visible
            if (ne >= 64u || nn == 0u) {
                // edge step: an item's edges are read before any is evaluated
                const uint32_t take = ne < 64u ? ne : 64u;
                const uint32_t at = lane < take ? ne - 1u - lane : 0u;
                const uint32_t eo = W.edge_ent[at];
                const uint32_t v = lane < take ? W.edges[at] : 0u;
                const uint32_t e0 = v & WL_EDGE_INDEX, cnt = (v >> 29) + 1u;
                float4 hedge[EG];
#pragma unroll
                for (int k = 0; k < EG; k++) hedge[k] = ldg4(c.edges + e0 + ((uint32_t)k < cnt ? (uint32_t)k : 0u));
                if (lane < take) {
                    const uint32_t es = W.ent_slot[eo];
                    const uint32_t slot = es & 63u;
                    if (!W.hit[slot]) {
                        const bool circle = KIND == KIND_CIRCLE || (KIND == KIND_MIXED && (es & WL_CIRCLE) != 0u);
                        const float4 gm = W.geom[eo];
                        bool h = false;
#pragma unroll
                        for (int k = 0; k < EG; k++) h = h || ((uint32_t)k < cnt && edge_hit(circle, gm, hedge[k]));
                        if (h) W.hit[slot] = 1u;
                    }
                }
                ne -= take;
                continue;
            }
            // node step.  An item pushes at most 4 children, 3 more slots than it frees, so taking t
            // items grows the queue by at most 3t: steps take no more than keeps WL_RESERVE slots
            // free.  Within the reserve, single-item steps walk depth-first, which grows the queue by
            // at most 3 per level below where the walk began; the reserve covers the deepest tree.
            // The queue therefore never overflows and every step makes progress.
            uint32_t take = 1u;
            if (nn + 3u + WL_RESERVE <= NCAP) {
                const uint32_t room = (NCAP - WL_RESERVE - nn) / 3u;
                take = nn < 64u ? nn : 64u;
                take = take < room ? take : room;
            }
            const uint32_t base = nn - take;
            const uint32_t item = lane < take ? W.nodes[nn - 1u - lane] : 0u;
            const uint32_t o = item >> 24;
            const DevNode nd = ldg_node(c.nodes + (item & WL_NODE_MASK));
            uint32_t m = 0, n_edges = 0, slot = 0;
            uint32_t p_beg = 0, p_cnt = 0, n_pass = 0;    // a leaf's first passing entry's edges; passing entries
            int fc = 0, s = -1, he = 0;
            bool circle = KIND == KIND_CIRCLE;
            float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            uint64_t q = 0;
            if (lane < take) {
                const uint32_t es = W.ent_slot[o];
                slot = es & 63u;
                if (!W.hit[slot]) {
                    g = W.geom[o];
                    if (KIND == KIND_MIXED) circle = (es & WL_CIRCLE) != 0u;
                    if (FILT) q = W.qidx[slot];
                    bool entire = false;
                    // a circle's start node is visited only if the circle meets its box (circle_cells);
                    // a pushed quadrant's box has passed the same test
                    if (KIND == KIND_EDGE || !circle || (item & WL_NODE_MASK) == 0u || circle_box(g.x, g.y, g.z, nd.bbox))
                        s = strongest_t<FILT>(c, nd, f, q, entire);
                    if (s >= 0 && entire) {
                        W.hit[slot] = 1u;
                        s = -1;
                    } else if (s >= 0 && nd.first_child >= 0) {
                        fc = nd.first_child;
                        m = circle ? circle_quadrants(g.x, g.y, g.z, nd.bbox) : edge_quadrants_node(g, nd.bbox);
                        s = -1;
                    } else if (s >= 0) {
                        // leaf: count the edge tests of its relevant Partial hazards
                        he = (int)(nd.haz_begin + (nd.haz_info & COUNT_MASK));
                        for (int i = s; i < he; i++) {
                            const DevEntry e = ldg_ent(c.ent + i);
                            if (!irrel<FILT>(f, q, e.slot_flags & SLOT_MASK) && ff_pass(e, circle, g)) {
                                if (n_pass == 0u) {
                                    p_beg = e.edge_begin;
                                    p_cnt = e.edge_count;
                                }
                                n_pass++;
                                n_edges += (e.edge_count + (uint32_t)EG - 1u) / (uint32_t)EG;
                            }
                        }
                    }
                }
            }
            // more edge tests than one push carries: this lane tests the leaf's edges itself
            bool inl = n_edges >= EDGE_LIMIT;
            if (inl) n_edges = 0;
            // one scan for both pushes: child counts in the low 16 bits, edge counts in the high
            // 16; neither sum over the wave carries out of its half
            const uint32_t packed = (uint32_t)__builtin_popcount(m) | (n_edges << 16);
            const uint32_t incl = wave_incl_scan(packed, lane);
            const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            const uint32_t excl = incl - packed;
            const uint32_t n_tot = tot & 0xffffu, e_tot = tot >> 16;
            wave_sync();                              // every lane has read its item before pushes overwrite
            {
                uint32_t at = base + (excl & 0xffffu);     // base + n_tot <= NCAP by the choice of take
                for (uint32_t b = m; b; b &= b - 1u)
                    W.nodes[at++] = (item & ~WL_NODE_MASK) | (uint32_t)(fc + __builtin_ctz(b));
                nn = base + n_tot;
            }
            const bool fits = ne + e_tot <= ECAP;
            inl = inl || (!fits && n_edges != 0u);        // or the edge queue is full
            if (n_edges && !inl) {
                uint32_t at = ne + (excl >> 16);
                // one passing entry (the common leaf): its edges from the count above
                const bool one = n_pass == 1u;
                for (int i = one ? he - 1 : s; i < he; i++) {
                    uint32_t beg = p_beg, cnt = p_cnt;
                    if (!one) {
                        const DevEntry e = ldg_ent(c.ent + i);
                        beg = e.edge_begin;
                        cnt = !irrel<FILT>(f, q, e.slot_flags & SLOT_MASK) && ff_pass(e, circle, g) ? e.edge_count : 0u;
                    }
                    for (uint32_t j = 0; j < cnt; j += EG, at++) {
                        const uint32_t k = cnt - j < (uint32_t)EG ? cnt - j : (uint32_t)EG;
                        W.edges[at] = (beg + j) | ((k - 1u) << 29);
                        W.edge_ent[at] = (uint8_t)o;
                    }
                }
            }
            if (inl) {
                bool h = false;
                for (int i = s; i < he && !h; i++) {
                    const DevEntry e = ldg_ent(c.ent + i);
                    if (irrel<FILT>(f, q, e.slot_flags & SLOT_MASK) || !ff_pass(e, circle, g)) continue;
                    for (uint32_t j = 0; j < e.edge_count && !h; j++) h = edge_hit(circle, g, ldg4(c.edges + e.edge_begin + j));
                }
                if (h) W.hit[slot] = 1u;
            }
            if (fits) ne += e_tot;
        }
        wave_sync();
    }
};

// Hazard-polygon point-in-polygon (simple_polygon.rs:255-292) over the hazard's full shape.
__device__ __forceinline__ bool pip_hazard(const CdeView& c, uint32_t slot, float px, float py) {
    const float4 bb = c.haz_bbox[slot];
    if (!box_has_point(bb, px, py)) return false;
    const float ray_x = bb.z + (bb.z - bb.x);
    const uint2 vr = c.haz_vr[slot];
    const float2* v = c.haz_verts + vr.x;
    int cnt = 0;
    float2 a = v[0];
    for (uint32_t i = 0; i < vr.y; i++) {
        const float2 b = v[i + 1 == vr.y ? 0 : i + 1];
        cnt += pip_edge(px, py, ray_x, a.x, a.y, b.x, b.y);
        a = b;
    }
    return (cnt & 1) == 1;
}

// Query-polygon point-in-polygon on the transformed query (vertices transformed on the fly).
__device__ __forceinline__ bool pip_query(const ItemView& it, const Mat& m, float4 qbb, float px, float py) {
    if (!box_has_point(qbb, px, py)) return false;
    const float ray_x = qbb.z + (qbb.z - qbb.x);
    int cnt = 0;
    float2 a = xform(m, it.v[0].x, it.v[0].y);
    const float2 first = a;
    for (uint32_t i = 0; i < it.n_v; i++) {
        const float2 b = i + 1 == it.n_v ? first : xform(m, it.v[i + 1].x, it.v[i + 1].y);
        cnt += pip_edge(px, py, ray_x, a.x, a.y, b.x, b.y);
        a = b;
    }
    return (cnt & 1) == 1;
}

// CDEngine::detect_containment_collision (cd_engine.rs:231-255)
__device__ __forceinline__ bool containment(const CdeView& c, uint32_t slot, const ItemView& it, const Mat& m,
                                            float4 qbb, float2 qpoi) {
    const int rel = box_almost_relation(c.haz_bbox[slot], qbb);
    bool contained = false;
    if (rel == REL_SURROUNDING) {
        contained = pip_hazard(c, slot, qpoi.x, qpoi.y);
    } else if (rel == REL_ENCLOSED) {
        const float4 hp = c.haz_poi[slot];
        contained = pip_query(it, m, qbb, hp.x, hp.y);
    }
    const bool interior = c.haz_poi[slot].w != 0.0f;
    return interior ? contained : !contained;
}

// Sum of v over the 64 lanes (all active).
__device__ __forceinline__ int wave_sum_i32(int v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// pip_hazard / pip_query with the wave's 64 lanes splitting the polygon's edges (lane l takes
// edges l, l + 64, ...).  Each edge's crossing count is the sequential loop's, and their sum is
// an integer, so the parity is the same.  All 64 lanes call them with the same arguments.
__device__ __forceinline__ bool pip_hazard_wave(const CdeView& c, uint32_t slot, float px, float py, uint32_t lane) {
    const float4 hb = ldg4(c.haz_bbox + slot);
    if (!box_has_point(hb, px, py)) return false;
    const float ray_x = hb.z + (hb.z - hb.x);
    const uint2 vr = ldg2u(c.haz_vr + slot);
    const float2* v = c.haz_verts + vr.x;
    int cnt = 0;
    for (uint32_t i = lane; i < vr.y; i += 64u) {
        const float2 a = ldg2(v + i), b = ldg2(v + (i + 1 == vr.y ? 0 : i + 1));
        cnt += pip_edge(px, py, ray_x, a.x, a.y, b.x, b.y);
    }
    return (wave_sum_i32(cnt) & 1) == 1;
}
__device__ __forceinline__ bool pip_query_wave(const ItemView& it, const Mat& m, float4 qbb, float px, float py,
                                               uint32_t lane) {
    if (!box_has_point(qbb, px, py)) return false;
    const float ray_x = qbb.z + (qbb.z - qbb.x);
    int cnt = 0;
    for (uint32_t i = lane; i < it.n_v; i += 64u) {
        const uint32_t k = i + 1 == it.n_v ? 0 : i + 1;
        const float2 vi = ldg2(it.v + i), vk = ldg2(it.v + k);
        const float2 a = xform(m, vi.x, vi.y), b = xform(m, vk.x, vk.y);
        cnt += pip_edge(px, py, ray_x, a.x, a.y, b.x, b.y);
    }
    return (wave_sum_i32(cnt) & 1) == 1;
}

// Transformed bounding box of the query (simple_polygon.rs:122-133 after transform_from).
__device__ __forceinline__ float4 query_bbox(const ItemView& it, const Mat& m) {
    float4 b = make_float4(3.40282347e+38f, 3.40282347e+38f, -3.40282347e+38f, -3.40282347e+38f);
    for (uint32_t i = 0; i < it.n_v; i++) {
        const float2 p = xform(m, it.v[i].x, it.v[i].y);
        b.x = mn(b.x, p.x);
        b.y = mn(b.y, p.y);
        b.z = mx(b.z, p.x);
        b.w = mx(b.w, p.y);
    }
    return b;
}

}  // namespace jg
