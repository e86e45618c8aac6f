// Records of a batched plan's device table and the work-claiming helpers shared by the batched
// detection (jg_batched.hip) and the batched hazard collection (jg_collect.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/jagua_amd.h"
#include "jg_device.hpp"

namespace jg {

struct SetDesc {
    CdeView cde;
    ItemView item;
    FilterView filter;
    uint64_t first;
    uint32_t flags;
    uint32_t lanes;        // lanes per query in the polygon stage (power of two, 1..64)
    const uint32_t* seed;  // collection: slots every query's collector starts with (ascending)
    uint32_t n_seed;
    uint32_t pad;
};

struct Unit {              // 16 B
    uint32_t set;
    uint32_t q0;           // first query, relative to the set
    uint32_t count;        // <= 64
    uint32_t pad;
};

struct Group {             // 16 B: surviving queries q0 + i for the set bits i of mask
    uint32_t set;
    uint32_t q0;
    uint64_t mask;
};

// Work is shared out over 16 streams, each with its own counters on their own 128-byte lines:
// thousands of waves taking work with atomics on a single address queue behind each other
// (measured: 1.81 ms against 1.30 ms per configuration-2 step for the survivor groups alone).
// Items x + 16 j of a list, work units or survivor groups, are stream x's; a wave claims from its own
// stream (workgroup index mod 16) alone, and a launch of at least as many workgroups as items takes
// them without a claim.  Looking at the other streams once the own one is dry costs more than the
// balance it brings, as thousands of waves then end with atomics or loads on the same few lines:
// us per step without / with a try of each stream / with a look at all counters first, 488 / 543 /
// 647 on the benchmark's 2000-item sheet, 275 / 337 / 401 on concave items.  For that reason no
// wave counts itself out either (a batch of 6400 queries took 111 us with both, 70 without).  8 / 16 /
// 32 streams: 471 / 465 / 472.
//   C_USTREAM0 + 32 x counts the units claimed from stream x, C_STREAM0 + 32 x the groups.
//   The survivor groups of the units of unit stream y are appended to their own region of the group
//   array (base gbase[y]); C_GCOUNT0 + 32 (16 p + y) counts them in the launches of parity p.
//   The regions one after another are the list of groups.
//   C_EPOCH counts the surrogate stages, C_EPOCH + 1 the polygon stages of the table.  Each stage
//   takes the parity from the other's count, which stands still meanwhile; the polygon stage
//   clears the other parity's counts, for the next launch.
// C_OVERFLOW counts the queries the batched collection hands to the per-query collector;
// C_DONE counts the waves of a launch that have finished (the last one clears counters).
// Every launch sequence leaves the table's counters ready for the next, and a new table, all zero,
// is.
constexpr uint32_t N_STREAMS = 16, STREAM_STRIDE = 32;
constexpr uint32_t C_STREAM0 = 0;
constexpr uint32_t C_USTREAM0 = C_STREAM0 + STREAM_STRIDE * N_STREAMS;
constexpr uint32_t C_GCOUNT0 = C_USTREAM0 + STREAM_STRIDE * N_STREAMS;
constexpr uint32_t C_OVERFLOW = C_GCOUNT0 + 2u * STREAM_STRIDE * N_STREAMS;
constexpr uint32_t C_DONE = C_OVERFLOW + STREAM_STRIDE;
constexpr uint32_t C_EPOCH = C_DONE + STREAM_STRIDE;
constexpr uint32_t N_COUNTER_WORDS = C_EPOCH + STREAM_STRIDE;

// The calling wave's exit from a launch of gridDim.x one-wave workgroups: true in the last
// wave to leave, once every other wave has left (C_DONE is then back at zero).
__device__ __forceinline__ bool last_wave_out(uint32_t* counters, uint32_t lane) {
    uint32_t last = 0;
    if (lane == 0) {
        last = atomicAdd(&counters[C_DONE], 1u) == gridDim.x - 1u ? 1u : 0u;
        if (last) counters[C_DONE] = 0u;
    }
    return __builtin_amdgcn_readfirstlane(last) != 0u;
}

constexpr uint32_t WAVE = 64;

// The device table of a batched launch, in one buffer: set descriptors, work units, the claim
// counters, the survivor-group region bases of the streams and the survivor groups.
struct TableLayout {
    size_t o_units = 0, o_ctr = 0, o_gbase = 0, o_grp = 0, total = 0;
    uint32_t n_units = 0, grid_s = 0, grid_p = 0;
    uint32_t stages = 2;
    bool filtered = false;            // some set has a filter (kernels with the filter test)
    int kind = KIND_CIRCLE;           // entity kinds of the surrogate stage over all sets
    uint32_t max_slot_words = 0;      // largest engine's slot bitmask, 32-bit words
    uint64_t n_queries = 0;           // over all sets
};

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// Lane 0's f32 value, bit for bit, in a scalar register (readfirstlane moves 32-bit integers).
__device__ __forceinline__ float uniform_f32(float x) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

template <typename T>
__device__ __forceinline__ T wave_bcast(T v) {
    // lane 0's value in a scalar register: what is derived from it (work-unit records, the set
    // descriptor and the engine's pointers) stays wave-uniform and is read with scalar loads
    return (T)__builtin_amdgcn_readfirstlane((int)v);
}

// A wave's items of a list of n, counters from word base on: the next item's index, n when there is
// none for this wave.  Every item is taken: its stream's workgroups claim until the stream is dry,
// and a launch of fewer workgroups than streams goes through all streams.
struct Claims {
    uint32_t x, tried;
    bool fresh;                                   // nothing has been taken yet
    __device__ __forceinline__ Claims() : x(blockIdx.x & (N_STREAMS - 1u)), tried(0u), fresh(true) {}
    __device__ __forceinline__ uint32_t next(uint32_t* counters, uint32_t base, uint32_t n, uint32_t lane) {
        if (n <= gridDim.x) {                     // a workgroup per item
            const bool mine = fresh && blockIdx.x < n;
            fresh = false;
            return mine ? blockIdx.x : n;
        }
        for (;;) {
            uint32_t t = 0;
            if (lane == 0) t = atomicAdd(&counters[base + STREAM_STRIDE * x], 1u);
            const uint64_t i = (uint64_t)x + (uint64_t)N_STREAMS * (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
            if (i < n) return (uint32_t)i;
            if (gridDim.x >= N_STREAMS || ++tried == N_STREAMS) return n;
            x = (x + 1u) & (N_STREAMS - 1u);
        }
    }
};

// Sum of v over the G lanes of this lane's aligned group (G a power of two <= 64).
__device__ __forceinline__ int group_sum_i32(int v, uint32_t G) {
    for (uint32_t o = G >> 1; o > 0; o >>= 1) v += __shfl_xor(v, (int)o, 64);
    return v;
}

// pip_hazard / pip_query with the G lanes of a group splitting the polygon's edges (lane sub
// takes edges sub, sub + G, ...).  Each edge's crossing count is the sequential loop's, and
// their sum is an integer, so the parity is the same.  The group's lanes call them together
// with the same arguments.
__device__ __forceinline__ bool pip_hazard_group(const CdeView& c, uint32_t slot, float px, float py, uint32_t sub,
                                                 uint32_t G) {
    const float4 hb = ldg4(c.haz_bbox + slot);
    if (!box_has_point(hb, px, py)) return false;
    const float ray_x = hb.z + (hb.z - hb.x);
    const uint2 vr = ldg2u(c.haz_vr + slot);
    const float2* v = c.haz_verts + vr.x;
    int cnt = 0;
    for (uint32_t i = sub; i < vr.y; i += G) {
        const float2 a = ldg2(v + i), b = ldg2(v + (i + 1 == vr.y ? 0 : i + 1));
        cnt += pip_edge(px, py, ray_x, a.x, a.y, b.x, b.y);
    }
    return (group_sum_i32(cnt, G) & 1) == 1;
}
__device__ __forceinline__ bool pip_query_group(const ItemView& it, const Mat& m, float4 qbb, float px, float py,
                                                uint32_t sub, uint32_t G) {
    if (!box_has_point(qbb, px, py)) return false;
    const float ray_x = qbb.z + (qbb.z - qbb.x);
    int cnt = 0;
    for (uint32_t i = sub; i < it.n_v; i += G) {
        const uint32_t k = i + 1 == it.n_v ? 0 : i + 1;
        const float2 vi = ldg2(it.v + i), vk = ldg2(it.v + k);
        const float2 a = xform(m, vi.x, vi.y), b = xform(m, vk.x, vk.y);
        cnt += pip_edge(px, py, ray_x, a.x, a.y, b.x, b.y);
    }
    return (group_sum_i32(cnt, G) & 1) == 1;
}

// The batched detection's two stages over one set, described by value (jg_batched.hip): no table,
// no allocation, one launch.  The traversal packs node numbers into 24 bits and hazard edges into
// 29; detect_direct_fits says whether an engine and a batch are within them.
bool detect_direct_fits(const jg_cde* c, uint64_t n);
jg_status detect_direct_launch(const CdeView& cde, const ItemView& item, const FilterView& filter, uint32_t flags,
                               const float* d_m6, uint64_t n, uint8_t* d_status, hipStream_t stream);

// The batched hazard collection over a plan's table (jg_collect.hip): verdict-free, one set
// per query.  ovf is a device list of n_queries (set, query) entries for the queries whose
// sets outgrow the batched kernel's collector.
jg_status collect_launch(const TableLayout& L, uint8_t* base, const float* d_m6, uint32_t cap, uint32_t* d_count,
                         uint64_t* d_hash, uint32_t* d_keys, uint64_t* ovf, uint32_t n_cus, hipStream_t stream);

// The batched collection over one set, described by value: no table, no allocation.  A query whose
// set may outgrow the batched kernel's collector is left with a count of COUNT_OVERFLOW.
constexpr uint32_t COUNT_OVERFLOW = 0xffffffffu;
jg_status collect_direct_launch(const CdeView& cde, const ItemView& item, const float* d_m6, uint64_t n, uint32_t cap,
                                uint32_t* d_count, uint64_t* d_hash, uint32_t* d_keys, uint32_t n_cus, hipStream_t stream);

// The per-query collector for the queries the batched collection handed over (jg_api.hip).
void collect_overflow_launch(const SetDesc* sets, uint32_t* counters, const uint64_t* ovf, const float* m6,
                             uint32_t words, uint32_t cap, uint32_t* count, uint64_t* hash, uint32_t* keys,
                             uint32_t grid, hipStream_t stream);

}  // namespace jg
