// Pole searches of many polygons at once on the GPU: SPolygon::new's pole of inaccessibility
// (simple_polygon.rs:41-71 via fail_fast/pole.rs:52-80) and generate_surrogate_poles
// (fail_fast/pole.rs:12-47), bit for bit with the sequential host search.
//
// The reference search pops cells from a FIFO; every split pushes four children to the back,
// so cells are visited level by level, in order.  Within a level the running best radius
// after cell i is max(best before the level, d_0..d_i), a prefix maximum, and cell i splits
// iff radius_i + d_i exceeds it.  One workgroup per polygon therefore evaluates a level's
// cells in parallel, takes a workgroup-wide prefix max and a prefix sum of the split flags, and
// writes the children of the split cells in order into the next level's frontier.
//
// What bounds it: a polygon's searches follow one another, each a chain of 11 levels, and a
// cell's distance to the border takes every edge.  A polygon of 256 vertices runs up to 100
// searches of about 5000 cells, but over 23000 distinct cells only: the searches differ in their
// poles alone, and a cell's distance to the border does not depend on them.  So the cells are
// kept as a tree over the polygon's searches (PoleNode): a cell met before costs the poles added
// since, a new one its edges, split over the lanes that the level's new cells leave free.
// A call with 192 polygons of 8-256 vertices took 108 ms with every cell evaluated anew by one thread and
// takes 5.8 ms, 3.8 of it here; one with a polygon of 1024 vertices 1800 and 27 ms.
//
// The arithmetic per edge and pole is pole_cell's (jg_geom.hpp).  Minima may be taken in any
// order, the square root of the least squared distance is the least distance (sqrtf is
// monotone), and crossing counts are integers, so every comparison gives the host's verdict.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <memory>
#include <string>
#include <thread>
#include <vector>

#include "../../include/jagua_amd.h"
#include "jg_internal.hpp"

using namespace jg;

namespace {

constexpr uint32_t FRONTIER_CAP = 8192;       // cells per level held per workgroup
constexpr uint32_t MAX_POLES = 1000;          // generate_surrogate_poles' assertion (pole.rs:40-43)

// Nodes of a polygon's cell tree: one search visits at most the root and 10 levels of
// FRONTIER_CAP cells, so an emptied tree holds any search.
constexpr uint32_t NODE_CAP = 98304;
static_assert(NODE_CAP >= 4u + (uint32_t)POLE_LEVELS * FRONTIER_CAP, "an empty tree must hold one search");

struct PoleJob {
    uint32_t v_begin, n;
    float area;
    uint32_t out;             // index of the polygon in the batch
    float4 bbox;
};

enum : uint32_t { PJ_OK = 0, PJ_FAIL = 1, PJ_HOST = 2, PJ_FULL = 3 };

// A cell over the searches of a polygon: the least distance of its centre to the border and to
// the poles seen so far, and first child block (0: none) | poles seen << 15 | flags.
struct PoleNode {
    float d;
    uint32_t link;
};
constexpr uint32_t PN_CHILD = 0x7fffu, PN_SEEN_SHIFT = 15, PN_SEEN = 0x3ffu;
constexpr uint32_t PN_INSIDE = 1u << 25, PN_POLE = 1u << 26;   // centre inside the border; inside a pole
constexpr uint32_t PN_NEW = PN_SEEN << PN_SEEN_SHIFT;          // not evaluated yet
static_assert(NODE_CAP / 4u <= PN_CHILD + 1u && MAX_POLES < PN_SEEN, "a node's link packs both");

// Per workgroup in device memory: the frontier cells past the LDS part, and the cell tree.
struct PoleSpill {
    float4 box[2][FRONTIER_CAP];
    uint32_t id[2][FRONTIER_CAP];
    float d[FRONTIER_CAP];
    PoleNode nodes[NODE_CAP];
};

struct PoleArgs {
    const PoleJob* jobs;
    const float2* verts;
    float4* poles;            // [n_jobs][pole_cap]: the POI, then the surrogate's further poles
    uint32_t* n_poles;
    uint32_t* status;
    PoleSpill* spill;         // [grid]
    uint32_t* counter;        // jobs taken, trees emptied
    uint32_t n_jobs, pole_cap, surrogate;
    uint32_t blocks;          // node blocks per tree, at most NODE_CAP / 4
    uint32_t lim_n[3];
    float lim_cov[3];
};

// A workgroup of NT threads keeps the first FL cells of a frontier, VL vertices and PL poles in LDS.
template <uint32_t NT, uint32_t FL, uint32_t VL>
struct PoleLds {
    static constexpr uint32_t W = NT / 64u, PL = 128, ML = 1024;
    float4 box[2][FL];
    uint32_t id[2][FL];
    float d[FL];
    float2 v[VL];
    float4 P[PL];
    uint64_t split[FRONTIER_CAP / 64u];
    uint16_t miss[ML];        // the level's new cells
    float wmax[W];
    uint32_t wsplit[W];
    float2 best;
    uint32_t n_miss, n_blocks, job;
};

template <int CTRL>
__device__ __forceinline__ float dpp_min(float x) {
    return fminf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false)));
}
// Minimum over aligned groups of T lanes (T a power of two <= 64), every lane active.
__device__ __forceinline__ float group_min(float x, uint32_t T) {
    if (T >= 2u) x = dpp_min<0xb1>(x);     // quad_perm [1, 0, 3, 2]
    if (T >= 4u) x = dpp_min<0x4e>(x);     // quad_perm [2, 3, 0, 1]
    if (T >= 8u) x = dpp_min<0x141>(x);    // row_half_mirror
    if (T >= 16u) x = dpp_min<0x140>(x);   // row_mirror
    if (T >= 32u) x = fminf(x, __shfl_xor(x, 16, 64));
    if (T >= 64u) x = fminf(x, __shfl_xor(x, 32, 64));
    return x;
}

__device__ __forceinline__ float wave_incl_max(float x, uint32_t lane) {
    for (int o = 1; o < 64; o <<= 1) {
        const float y = __shfl_up(x, o, 64);
        if ((int)lane >= o) x = fmaxf(x, y);
    }
    return x;
}

// One polygon's searches, by the whole workgroup.
template <uint32_t NT, uint32_t FL, uint32_t VL>
struct PoleSearch {
    using Lds = PoleLds<NT, FL, VL>;
    static constexpr uint32_t W = Lds::W;
    Lds& L;
    PoleSpill& S;
    const PoleJob job;
    const float2* gv;          // its vertices
    const float4* gP;          // its poles
    const uint32_t blocks;     // of its tree
    const uint32_t tid, lane, wv;

    __device__ float4 box(uint32_t b, uint32_t i) const { return i < FL ? L.box[b][i] : S.box[b][i]; }
    __device__ uint32_t id(uint32_t b, uint32_t i) const { return i < FL ? L.id[b][i] : S.id[b][i]; }
    __device__ float dist(uint32_t i) const { return i < FL ? L.d[i] : S.d[i]; }
    __device__ void put_cell(uint32_t b, uint32_t i, float4 x, uint32_t n) {
        if (i < FL) {
            L.box[b][i] = x;
            L.id[b][i] = n;
        } else {
            S.box[b][i] = x;
            S.id[b][i] = n;
        }
    }
    // the cell's value: its node's distance, negative unless the centre is inside the border
    // and outside every pole
    __device__ void put_value(uint32_t i, float d, uint32_t link) {
        const float x = (link & (PN_INSIDE | PN_POLE)) == PN_INSIDE ? d : -d;
        if (i < FL) L.d[i] = x;
        else S.d[i] = x;
    }
    __device__ float2 vert(uint32_t k) const { return job.n <= VL ? L.v[k] : gv[k]; }
    __device__ float4 pole(uint32_t k) const { return k < Lds::PL ? L.P[k] : gP[k]; }

    // one pole's share of a cell's value (circle.rs:95-107, 154-163)
    __device__ void see_pole(float4 c, float cx, float cy, float& d, bool& in) const {
        const float ex = cx - c.x, ey = cy - c.y;
        const float sq = ex * ex + ey * ey;
        in = in || sq <= c.z * c.z;
        const float dc = sqrtf(sq);
        d = mn(d, dc <= c.z ? c.z - dc : dc - c.z);
    }

    __device__ void start() {
        if (tid == 0) {
            L.n_blocks = 1;
            L.n_miss = 0;
        }
        S.nodes[tid & 3u] = PoleNode{0.0f, PN_NEW};       // block 0: the root
    }

    // compute_pole (pole.rs:52-80) against poles 0..np-1; PJ_OK with the best circle, PJ_FAIL when no
    // cell had a positive distance, PJ_HOST on frontier overflow, PJ_FULL when the tree is full
    // (to be emptied and the search repeated).
    __device__ uint32_t search(uint32_t np, float4& best) {
        float best_r = 0.0f;
        bool have = false;
        uint32_t cur = 0, nF = 1;
        if (tid == 0) put_cell(0, 0, box_inflate_to_square(job.bbox), 0u);
        __syncthreads();
        for (int level = POLE_LEVELS; level >= 0 && nF > 0; level--) {
            // cells met before: the poles added since.  New cells go to the miss list (or, past its
            // end, are evaluated by this thread).
            for (uint32_t i = tid; i < nF; i += NT) {
                const uint32_t ni = id(cur, i);
                const PoleNode nd = S.nodes[ni];
                const float4 b = box(cur, i);
                uint32_t seen = (nd.link >> PN_SEEN_SHIFT) & PN_SEEN;
                if (seen == PN_SEEN) {
                    const uint32_t at = atomicAdd(&L.n_miss, 1u);
                    if (at < Lds::ML) {
                        L.miss[at] = (uint16_t)i;
                        continue;
                    }
                    eval(i, ni, b, np);
                    continue;
                }
                float d = nd.d;
                bool in = (nd.link & PN_POLE) != 0u;
                const float cx = (b.x + b.z) / 2.0f, cy = (b.y + b.w) / 2.0f;
                for (; seen < np; seen++) see_pole(pole(seen), cx, cy, d, in);
                const uint32_t link = (nd.link & (PN_CHILD | PN_INSIDE)) | (np << PN_SEEN_SHIFT) | (in ? PN_POLE : 0u);
                S.nodes[ni] = PoleNode{d, link};
                put_value(i, d, link);
            }
            __syncthreads();
            {
                // T lanes per new cell, its edges and poles split over them
                const uint32_t M = L.n_miss < Lds::ML ? L.n_miss : Lds::ML;
                uint32_t T = 64;
                while (T > 1u && M * T > NT) T >>= 1;
                const uint32_t per = NT / T, g = tid / T, sub = tid & (T - 1u);
                for (uint32_t c0 = 0; c0 < M; c0 += per) {
                    if (c0 + (tid & ~63u) / T >= M) break;            // no cell for this wave
                    const uint32_t m = c0 + g;
                    const bool valid = m < M;
                    const uint32_t i = valid ? L.miss[m] : 0u;
                    eval_group(i, id(cur, i), box(cur, i), np, valid, sub, T);
                }
            }
            __syncthreads();
            // prefix max: each wave takes a contiguous segment of the level
            const uint32_t seg = ((nF + NT - 1u) / NT) * 64u;
            const uint32_t s0 = wv * seg, s1 = s0 + seg < nF ? s0 + seg : nF;
            float m = -INFINITY;
            for (uint32_t i = s0 + lane; i < s1; i += 64u) m = fmaxf(m, dist(i));
            m = wave_incl_max(m, lane);
            if (lane == 63u) L.wmax[wv] = m;
            if (tid == 0) L.n_miss = 0;
            __syncthreads();
            float pre = best_r, top = L.wmax[0];
            uint32_t first = 0;                           // the first wave holding the level's max
            for (uint32_t k = 0; k < W; k++) {
                const float x = L.wmax[k];
                if (k < wv) pre = fmaxf(pre, x);
                if (x > top) {
                    top = x;
                    first = k;
                }
            }
            uint32_t n_split = 0;
            bool found = !(top > best_r) || wv != first;
            for (uint32_t c = s0; c < s1; c += 64u) {
                const uint32_t i = c + lane;
                const bool valid = i < s1;
                const float d = valid ? dist(i) : -INFINITY;
                float4 b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (valid) b = box(cur, i);
                const float incl = wave_incl_max(d, lane);
                const float bx = b.z - b.x, by = b.w - b.y;
                const float radius = sqrtf(bx * bx + by * by) / 2.0f;
                const uint64_t sp = __ballot(valid && level > 0 && (radius + d > fmaxf(pre, incl)));
                if (lane == 0) L.split[i >> 6] = sp;
                n_split += (uint32_t)__builtin_popcountll(sp);
                if (!found) {                             // the first cell reaching the level's max
                    const uint64_t eq = __ballot(valid && d == top);
                    if (eq != 0ull) {
                        found = true;
                        if (lane == (uint32_t)__builtin_ctzll(eq))
                            L.best = make_float2((b.x + b.z) / 2.0f, (b.y + b.w) / 2.0f);
                    }
                }
                pre = fmaxf(pre, __shfl(incl, 63, 64));
            }
            if (lane == 0) L.wsplit[wv] = n_split;
            __syncthreads();
            if (top > best_r) {
                best = make_float4(L.best.x, L.best.y, top, 0.0f);
                best_r = top;
                have = true;
            }
            uint32_t at = 0, tot = 0;
            for (uint32_t k = 0; k < W; k++) {
                if (k < wv) at += L.wsplit[k];
                tot += L.wsplit[k];
            }
            if (tot * 4u > FRONTIER_CAP) return PJ_HOST;
            // the children of the split cells in order; a cell split for the first time takes a
            // block of new nodes (their numbers decide nothing)
            for (uint32_t c = s0; c < s1; c += 64u) {
                const uint64_t sp = L.split[c >> 6];
                if ((sp >> lane) & 1ull) {
                    const uint32_t i = c + lane;
                    const uint32_t ni = id(cur, i);
                    uint32_t link = S.nodes[ni].link;
                    uint32_t blk = link & PN_CHILD;
                    if (blk == 0u) {
                        blk = atomicAdd(&L.n_blocks, 1u);
                        if (blk < blocks) {
                            S.nodes[ni].link = link | blk;
                            for (uint32_t k = 0; k < 4u; k++) S.nodes[4u * blk + k] = PoleNode{0.0f, PN_NEW};
                        }
                    }
                    if (blk < blocks) {
                        const float4 b = box(cur, i);
                        const uint32_t o = 4u * (at + lanes_below(sp, lane));
                        for (uint32_t k = 0; k < 4u; k++) put_cell(cur ^ 1u, o + k, box_quadrant(b, (int)k), 4u * blk + k);
                    }
                }
                at += (uint32_t)__builtin_popcountll(sp);
            }
            __syncthreads();
            if (L.n_blocks > blocks) return PJ_FULL;
            cur ^= 1u;
            nF = tot * 4u;
        }
        return have ? PJ_OK : PJ_FAIL;
    }

    // POINode::new (pole.rs:93-127), as pole_cell: this lane's share (edges and poles sub, sub + T, ...)
    __device__ void share(float cx, float cy, uint32_t np, uint32_t sub, uint32_t T, float& sq, float& dp, uint32_t& cross,
                          bool& in) const {
        sq = INFINITY;
        dp = 3.40282347e+38f;
        cross = 0;
        in = false;
        const uint32_t n = job.n;
        const bool inside_box = box_has_point(job.bbox, cx, cy);
        const float ray_x = job.bbox.z + (job.bbox.z - job.bbox.x);
        // an edge whose y interval is further than this from the ray counts nothing: approx_eq
        // reaches 4 ulps or 2^-23 (pip_edge), and edge_edge needs overlapping boxes
        const float reach = fabsf(cy) * 1e-6f + 2.5e-7f;
        for (uint32_t k = sub; k < n; k += T) {
            const float2 a = vert(k), b = vert(k + 1u == n ? 0u : k + 1u);
            sq = mn(sq, edge_point_sq_dist(make_float4(a.x, a.y, b.x, b.y), cx, cy));
            const bool off = cy < mn(a.y, b.y) - reach || cy > mx(a.y, b.y) + reach;
            if (inside_box && !off) cross += (uint32_t)pip_edge(cx, cy, ray_x, a.x, a.y, b.x, b.y);
        }
        for (uint32_t k = sub; k < np; k += T) see_pole(pole(k), cx, cy, dp, in);
    }
    __device__ void put_node(uint32_t i, uint32_t ni, uint32_t np, float sq, float dp, bool inside, bool in) {
        const float d = mn(mn(3.40282347e+38f, sqrtf(sq)), dp);
        const uint32_t link = (np << PN_SEEN_SHIFT) | (inside ? PN_INSIDE : 0u) | (in ? PN_POLE : 0u);
        S.nodes[ni] = PoleNode{d, link};
        put_value(i, d, link);
    }
    __device__ void eval(uint32_t i, uint32_t ni, float4 b, uint32_t np) {
        float sq, dp;
        uint32_t cross;
        bool in;
        share((b.x + b.z) / 2.0f, (b.y + b.w) / 2.0f, np, 0u, 1u, sq, dp, cross, in);
        put_node(i, ni, np, sq, dp, (cross & 1u) != 0u, in);
    }
    __device__ void eval_group(uint32_t i, uint32_t ni, float4 b, uint32_t np, bool valid, uint32_t sub, uint32_t T) {
        float sq, dp;
        uint32_t cross;
        bool in;
        share((b.x + b.z) / 2.0f, (b.y + b.w) / 2.0f, np, sub, T, sq, dp, cross, in);
        sq = group_min(sq, T);
        dp = group_min(dp, T);
        const uint64_t gm = T == 64u ? ~0ull : ((1ull << T) - 1ull);
        const uint32_t g0 = lane & ~(T - 1u);
        const bool inside = (__builtin_popcountll((__ballot(cross & 1u) >> g0) & gm) & 1) != 0;
        const bool any = ((__ballot(in) >> g0) & gm) != 0ull;
        if (valid && sub == 0u) put_node(i, ni, np, sq, dp, inside, any);
    }
};

template <uint32_t NT, uint32_t FL, uint32_t VL>
__global__ __launch_bounds__(NT) void k_poles(PoleArgs a) {
    __shared__ PoleLds<NT, FL, VL> L;
    const uint32_t tid = threadIdx.x;
    const float PI_F = 3.14159265358979323846f;
    for (;;) {
        if (tid == 0) L.job = atomicAdd(a.counter, 1u);
        __syncthreads();
        const uint32_t j = L.job;
        if (j >= a.n_jobs) return;
        const PoleJob job = a.jobs[j];
        float4* P = a.poles + (size_t)job.out * a.pole_cap;
        PoleSearch<NT, FL, VL> ps{L, a.spill[blockIdx.x], job, a.verts + job.v_begin, P, a.blocks, tid, tid & 63u, tid >> 6};
        if (job.n <= VL)
            for (uint32_t k = tid; k < job.n; k += NT) L.v[k] = ps.gv[k];
        ps.start();
        float covered = 0.0f;
        uint32_t np = 0, st;
        bool emptied = false;
        for (;;) {
            float4 best = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            __syncthreads();                              // the pole (or the new tree) of the last round
            st = ps.search(np, best);
            if (st == PJ_FULL && !emptied) {              // an empty tree holds any search
                __syncthreads();
                ps.start();
                if (tid == 0) atomicAdd(&a.counter[1], 1u);
                emptied = true;
                continue;
            }
            emptied = false;
            if (st == PJ_FULL) st = PJ_HOST;              // (but for the smaller trees of the tests)
            if (st != PJ_OK) break;
            if (tid == 0) {
                P[np] = best;
                if (np < PoleLds<NT, FL, VL>::PL) L.P[np] = best;
            }
            np++;
            covered = np == 1u ? best.z * best.z * PI_F : covered + best.z * best.z * PI_F;
            if (!a.surrogate) break;
            if (np > 1u) {
                // generate_surrogate_poles: the POI, then poles until a count/coverage limit holds
                const float coverage = covered / job.area;
                bool any = false;
                uint32_t limit = 0;
                for (int i = 0; i < 3; i++)
                    if (coverage > a.lim_cov[i] && (!any || a.lim_n[i] < limit)) {
                        limit = a.lim_n[i];
                        any = true;
                    }
                if (any && np >= limit) break;
                if (np >= MAX_POLES) { st = PJ_FAIL; break; }
            }
            if (np >= a.pole_cap) { st = PJ_HOST; break; }
        }
        if (tid == 0) {
            a.status[job.out] = st;
            a.n_poles[job.out] = np;
        }
        __syncthreads();
    }
}

template <class F>
void parallel_for(size_t n, F fn) {
    const size_t nt = std::max<size_t>(1, std::min<size_t>({(size_t)std::thread::hardware_concurrency(), 16, n}));
    std::vector<std::thread> th;
    for (size_t t = 0; t < nt; t++)
        th.emplace_back([&, t] {
            for (size_t i = t; i < n; i += nt) fn(i);
        });
    for (auto& x : th) x.join();
}

}  // namespace

// blocks: node blocks per cell tree; n_emptied (may be null): how many trees were full and emptied.
static jg_status new_batch(const float* xy, const uint32_t* offsets, uint32_t n_polys, const jg_surrogate_config* cfg,
                           jg_spolygon** out, uint32_t* n_host_completed, uint32_t blocks, uint32_t* n_emptied) {
    if (!out || (n_polys && (!xy || !offsets))) return fail(JG_ERR_INVALID_ARG, "null argument");
    if (n_host_completed) *n_host_completed = 0;
    if (n_polys == 0) return JG_OK;
    for (uint32_t i = 0; i < n_polys; i++)
        if (offsets[i + 1] < offsets[i]) return fail(JG_ERR_INVALID_ARG, "offsets must be non-decreasing");
    // SPolygon::new up to the pole search, on host threads
    std::vector<Polygon> polys(n_polys);
    std::vector<std::string> errs(n_polys);
    std::vector<char> ok(n_polys, 0);
    parallel_for(n_polys, [&](size_t i) {
        ok[i] = polygon_prepare(xy + 2 * (size_t)offsets[i], offsets[i + 1] - offsets[i], polys[i], errs[i]) ? 1 : 0;
    });
    for (uint32_t i = 0; i < n_polys; i++)
        if (!ok[i]) return fail(JG_ERR_POLYGON, "polygon " + std::to_string(i) + ": " + errs[i]);
    jg_status st = device_ready();
    if (st != JG_OK) return st;

    uint32_t pole_cap = 1;
    if (cfg) {
        pole_cap = 2;
        for (int i = 0; i < 3; i++) pole_cap = std::max(pole_cap, cfg->n_pole_limits_n[i]);
        pole_cap = std::min(pole_cap, MAX_POLES);
    }
    std::vector<PoleJob> jobs(n_polys);
    std::vector<float2> verts;
    verts.reserve(offsets[n_polys] - offsets[0]);
    for (uint32_t i = 0; i < n_polys; i++) {
        jobs[i] = PoleJob{(uint32_t)verts.size(), polys[i].n(), polys[i].area, i, polys[i].bbox};
        verts.insert(verts.end(), polys[i].v.begin(), polys[i].v.end());
    }
    // largest first: a polygon's searches are one chain, so a large one taken last would be the tail
    std::stable_sort(jobs.begin(), jobs.end(), [](const PoleJob& a, const PoleJob& b) { return a.n > b.n; });
    int dev = 0, cus = 256;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    // 1024 threads per polygon while every polygon has half a compute unit to itself, as its chain
    // of levels is what takes the time; 512 where polygons queue, as the lanes that a short level
    // leaves idle are then missed.  ms per call at 1024 / 512 threads: one polygon of 1024 vertices 26.9 /
    // 37.7, 192 of 8-256 vertices 5.3 / 6.0, 513 of them 5.9 / 6.5, 1500 11.2 / 9.8, 2000 concave ones
    // of 64-1024 vertices 37.2 / 35.7.  (256 threads, measured earlier: 61 for the first, 12.5 for the 1500.)
    const bool wide = n_polys <= 2u * (uint32_t)cus;
    const uint32_t want = std::max<uint32_t>(1u, std::min<uint32_t>(n_polys, (wide ? 2u : 3u) * (uint32_t)cus));

    const size_t b_jobs = sizeof(PoleJob) * n_polys;
    const size_t o_verts = (b_jobs + 255) & ~(size_t)255;
    const size_t o_poles = (o_verts + sizeof(float2) * verts.size() + 255) & ~(size_t)255;
    const size_t o_np = (o_poles + sizeof(float4) * (size_t)pole_cap * n_polys + 255) & ~(size_t)255;
    const size_t o_st = (o_np + 4 * (size_t)n_polys + 255) & ~(size_t)255;
    const size_t o_ctr = (o_st + 4 * (size_t)n_polys + 255) & ~(size_t)255;
    const size_t o_fr = o_ctr + 256;
    // 1.15 MB per workgroup for the length of the call, 0.88 GB at most; fewer workgroups where the
    // device has less to give
    DevBlob blob;
    const uint32_t grid = fit_workgroups(want, o_fr, sizeof(PoleSpill), [&](uint64_t bytes) {
        st = blob.reserve_exact((size_t)bytes);
        if (st != JG_OK) (void)hipGetLastError();     // or the launch below would report it
        return st == JG_OK;
    });
    if (grid == 0) return st;
    uint8_t* base = (uint8_t*)blob.ptr;
    st = hip_check(hipMemcpy(base, jobs.data(), b_jobs, hipMemcpyHostToDevice), "hipMemcpy pole jobs");
    if (st == JG_OK)
        st = hip_check(hipMemcpy(base + o_verts, verts.data(), sizeof(float2) * verts.size(), hipMemcpyHostToDevice),
                       "hipMemcpy pole vertices");
    if (st == JG_OK) st = hip_check(hipMemset(base + o_ctr, 0, 256), "hipMemset pole counter");
    if (st != JG_OK) return st;
    PoleArgs a{};
    a.jobs = (const PoleJob*)base;
    a.verts = (const float2*)(base + o_verts);
    a.poles = (float4*)(base + o_poles);
    a.n_poles = (uint32_t*)(base + o_np);
    a.status = (uint32_t*)(base + o_st);
    a.spill = (PoleSpill*)(base + o_fr);
    a.counter = (uint32_t*)(base + o_ctr);
    a.blocks = blocks;
    a.n_jobs = n_polys;
    a.pole_cap = pole_cap;
    a.surrogate = cfg ? 1u : 0u;
    for (int i = 0; i < 3; i++) {
        a.lim_n[i] = cfg ? cfg->n_pole_limits_n[i] : 0u;
        a.lim_cov[i] = cfg ? cfg->n_pole_limits_cov[i] : 0.0f;
    }
    if (wide) hipLaunchKernelGGL((k_poles<1024, 1024, 2048>), dim3(grid), dim3(1024), 0, nullptr, a);
    else hipLaunchKernelGGL((k_poles<512, 512, 2048>), dim3(grid), dim3(512), 0, nullptr, a);
    st = hip_check(hipGetLastError(), "pole search launch");
    if (st == JG_OK) st = hip_check(hipDeviceSynchronize(), "pole search");
    std::vector<float4> poles((size_t)pole_cap * n_polys);
    std::vector<uint32_t> np(n_polys), status(n_polys);
    if (st == JG_OK)
        st = hip_check(hipMemcpy(poles.data(), base + o_poles, sizeof(float4) * poles.size(), hipMemcpyDeviceToHost),
                       "hipMemcpy poles");
    if (st == JG_OK) st = hip_check(hipMemcpy(np.data(), base + o_np, 4 * (size_t)n_polys, hipMemcpyDeviceToHost), "hipMemcpy");
    if (st == JG_OK)
        st = hip_check(hipMemcpy(status.data(), base + o_st, 4 * (size_t)n_polys, hipMemcpyDeviceToHost), "hipMemcpy");
    if (st == JG_OK && n_emptied) st = hip_check(hipMemcpy(n_emptied, base + o_ctr + 4, 4, hipMemcpyDeviceToHost), "hipMemcpy");
    if (st != JG_OK) return st;

    // finish: the POI, the surrogate from its poles; polygons whose search outgrew the device
    // buffers are searched by the host routine instead
    uint32_t n_host = 0;
    for (uint32_t i = 0; i < n_polys; i++) {
        if (status[i] == PJ_FAIL) return fail(JG_ERR_POLYGON, "polygon " + std::to_string(i) + ": no pole found");
        if (status[i] == PJ_HOST) n_host++;
    }
    // piers of the polygons whose poles came from the device, on the device as well
    std::vector<std::vector<float4>> piers;
    std::vector<uint8_t> pier_host;
    std::vector<uint32_t> pier_of(n_polys, 0xffffffffu);
    if (cfg && cfg->n_ff_piers > 0) {
        std::vector<const Polygon*> pp;
        std::vector<std::vector<float4>> rel;
        for (uint32_t i = 0; i < n_polys; i++) {
            if (status[i] != PJ_OK) continue;
            const float4* P = poles.data() + (size_t)i * pole_cap;
            const uint32_t n_ff = std::min(cfg->n_ff_poles, np[i]);
            polys[i].poi = P[0];
            pier_of[i] = (uint32_t)pp.size();
            pp.push_back(&polys[i]);
            rel.emplace_back(P, P + n_ff);
        }
        st = piers_batch(pp, rel, cfg->n_ff_piers, piers, pier_host);
        if (st != JG_OK) return st;
        for (uint8_t h : pier_host) n_host += h;
    }
    parallel_for(n_polys, [&](size_t i) {
        Polygon& p = polys[i];
        std::string& err = errs[i];
        ok[i] = 1;
        if (status[i] == PJ_HOST) {
            Polygon q;
            const uint32_t n = offsets[i + 1] - offsets[i];
            if (!polygon_new(xy + 2 * (size_t)offsets[i], n, q, err) ||
                (cfg && !polygon_generate_surrogate(q, *cfg, err)))
                ok[i] = 0;
            p = std::move(q);
            return;
        }
        const float4* P = poles.data() + (size_t)i * pole_cap;
        p.poi = P[0];
        const std::vector<float4>* dev_piers =
            pier_of[i] != 0xffffffffu && !pier_host[pier_of[i]] ? &piers[pier_of[i]] : nullptr;
        if (cfg && !surrogate_finish(p, *cfg, std::vector<float4>(P, P + np[i]), err, dev_piers)) ok[i] = 0;
    });
    for (uint32_t i = 0; i < n_polys; i++)
        if (!ok[i]) return fail(JG_ERR_SURROGATE, "polygon " + std::to_string(i) + ": " + errs[i]);
    for (uint32_t i = 0; i < n_polys; i++) {
        auto h = std::make_unique<jg_spolygon>();
        h->poly = std::move(polys[i]);
        out[i] = h.release();
    }
    if (n_host_completed) *n_host_completed = n_host;
    return JG_OK;
}

extern "C" jg_status jg_spolygon_new_batch(const float* xy, const uint32_t* offsets, uint32_t n_polys,
                                           const jg_surrogate_config* cfg, jg_spolygon** out,
                                           uint32_t* n_host_completed) {
    return new_batch(xy, offsets, n_polys, cfg, out, n_host_completed, NODE_CAP / 4u, nullptr);
}

// For the tests, which no polygon takes to a full tree: jg_spolygon_new_batch with trees of `blocks`
// node blocks.  A search that a smaller tree cannot hold is left to the host routine.
extern "C" jg_status jg_check_spolygon_new_batch(const float* xy, const uint32_t* offsets, uint32_t n_polys,
                                                 const jg_surrogate_config* cfg, jg_spolygon** out,
                                                 uint32_t* n_host_completed, uint32_t blocks, uint32_t* n_emptied) {
    if (blocks < 1u || blocks > NODE_CAP / 4u || !n_emptied) return fail(JG_ERR_INVALID_ARG, "tree size out of range");
    return new_batch(xy, offsets, n_polys, cfg, out, n_host_completed, blocks, n_emptied);
}
