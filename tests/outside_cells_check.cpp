// CPU check of the start cells of what lies partly or wholly outside the root box (holding_cell and
// edge_cells in jg_geom.hpp): random boxes and edges around a root box, and a few ulps beside
// its bounds.  A box's holding cell is level 0 wherever no quadrant of the root surrounds it;
// elsewhere the search through the surrounding quadrants passes it.  An edge's descent from its
// cells, or from the root at level 0, reaches exactly the leaves of a random quadtree that its
// descent from the root reaches; so does that of an edge with a NaN among its coordinates.
// Usage: outside_cells_check <seed> <cases>; prints
// "ok <boxes outside> <boxes inside> <edges that leave the box> <with cells> <with a NaN>".
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <set>

#include "../jagua-rs_amd/csrc/jg_geom.hpp"

using namespace jg;

static uint64_t g_state;
static uint64_t u64() {                      // splitmix64
    uint64_t z = (g_state += 0x9e3779b97f4a7c15ull);
    return mix64(z);
}
static double urand() { return (double)(u64() >> 11) * (1.0 / 9007199254740992.0); }

static float ulps(float v, int n) {
    for (; n > 0; n--) v = std::nextafterf(v, INFINITY);
    for (; n < 0; n++) v = std::nextafterf(v, -INFINITY);
    return v;
}

// a coordinate around [lo, hi]: inside, outside, far outside, or within a few ulps of a bound
static float around(float lo, float hi) {
    const float w = hi - lo;
    switch (u64() % 6) {
        case 0: return lo + w * (float)urand();
        case 1: return lo + w * (float)(3.0 * urand() - 1.0);
        case 2: return lo + w * (float)((urand() - 0.5) * 1e4);
        case 3: return ulps(u64() & 1u ? lo : hi, (int)(u64() % 9) - 4);
        case 4: return u64() & 1u ? lo - w * (float)(0.2 * urand()) : hi + w * (float)(0.2 * urand());
        default: return lo + w * (float)(u64() % 33) / 32.0f;
    }
}

struct Tree {                                // a node splits by a hash of its place
    float4 root;
    uint32_t depth, table;
    uint64_t salt;
    bool split(uint32_t l, uint32_t x, uint32_t y) const {
        return l < depth && (mix64(salt + (((uint64_t)l << 40) | ((uint64_t)y << 20) | x)) & 15u) != 0u;
    }
};
static void child(int k, uint32_t& x, uint32_t& y) {
    x = 2 * x + (k == 0 || k == 3);
    y = 2 * y + (k == 0 || k == 1);
}
typedef std::set<uint64_t> Leaves;

static void descend(const Tree& t, uint32_t l, uint32_t x, uint32_t y, float4 box, float4 e, Leaves& out) {
    if (!t.split(l, x, y)) {
        out.insert(((uint64_t)l << 40) | ((uint64_t)y << 20) | x);
        return;
    }
    const uint32_t m = edge_quadrants_node(e, box);
    for (int k = 0; k < 4; k++)
        if ((m >> k) & 1u) {
            uint32_t a = x, b = y;
            child(k, a, b);
            descend(t, l + 1, a, b, box_quadrant(box, k), e, out);
        }
}

// the descent from the deepest node on the path to cell (x, y) of level l
static void from_cell(const Tree& t, uint32_t l, uint32_t x, uint32_t y, float4 e, Leaves& out) {
    uint32_t d = 0, a = 0, b = 0;
    float4 box = t.root;
    for (; d < l && t.split(d, a, b); d++) {
        const uint32_t s = l - d - 1;
        const bool right = (x >> s) & 1u, up = (y >> s) & 1u;
        const int k = up ? (right ? 0 : 1) : (right ? 3 : 2);
        child(k, a, b);
        box = box_quadrant(box, k);
    }
    descend(t, d, a, b, box, e, out);
}

int main(int argc, char** argv) {
    g_state = argc > 1 ? strtoull(argv[1], nullptr, 10) : 1;
    const uint64_t cases = argc > 2 ? strtoull(argv[2], nullptr, 10) : 20000;
    uint64_t outside = 0, inside = 0, leave = 0, cells = 0, nans = 0;
    for (uint64_t i = 0; i < cases; i++) {
        const float w = (float)std::exp(std::log(1e-2) + urand() * std::log(1e7)), h = i % 3 ? w : w * (float)(0.2 + urand());
        const float ox = (float)((urand() - 0.5) * (i % 4 ? 2.0 : 200.0)) * w, oy = (float)((urand() - 0.5) * 2.0) * h;
        const float4 root = make_float4(ox, oy, ox + w, oy + h);
        const uint32_t level = (uint32_t)(u64() % 10);
        const CellGrid g = cell_grid(root, level);
        for (int q = 0; q < 40; q++) {
            const float x = around(root.x, root.z), y = around(root.y, root.w);
            const float s = q % 4 == 0 ? 0.0f : (float)(w * std::exp(std::log(1e-6) + urand() * std::log(1e7)));
            const float x1 = q % 4 == 1 ? around(root.x, root.z) : x + s,
                        y1 = q % 4 == 1 ? around(root.y, root.w) : y + s * (float)urand();
            const float4 b = make_float4(mn(x, x1), mn(y, y1), mx(x, x1), mx(y, y1));
            const HoldingCell hc = holding_cell(g, level, root, b);
            if (hc.l > level || hc.ix >> hc.l || hc.iy >> hc.l) {
                std::printf("cell out of range\n");
                return 1;
            }
            (quadrant_surrounding(root, b) < 0 ? outside : inside)++;
            uint32_t cx = 0, cy = 0;
            float4 box = root;
            for (uint32_t l = 0; l < hc.l; l++) {
                const int k = quadrant_surrounding(box, b);
                if (k < 0) {
                    std::printf("no quadrant surrounds the box at level %u of %u: box %.9g %.9g %.9g %.9g, root %.9g %.9g %.9g %.9g\n",
                                l, hc.l, b.x, b.y, b.z, b.w, root.x, root.y, root.z, root.w);
                    return 1;
                }
                child(k, cx, cy);
                box = box_quadrant(box, k);
            }
            if (cx != hc.ix || cy != hc.iy) {
                std::printf("the surrounding path differs\n");
                return 1;
            }
        }
        const Tree t{root, (uint32_t)(u64() % 8), level, u64()};
        const CellGrid tg = cell_grid(root, t.depth < level ? t.depth : level);
        const uint32_t table = t.depth < level ? t.depth : level;
        for (int q = 0; q < 40; q++) {
            const float len = (float)(w * std::exp(std::log(1e-5) + urand() * std::log(1e5)));
            const double a = q % 8 == 1 ? 0.0 : q % 8 == 3 ? M_PI / 2 : 2.0 * M_PI * urand();
            float4 e = make_float4(around(root.x, root.z), around(root.y, root.w), 0.0f, 0.0f);
            e.z = q % 5 == 0 ? around(root.x, root.z) : e.x + (float)(len * std::cos(a));
            e.w = q % 5 == 0 ? around(root.y, root.w) : e.y + (float)(len * std::sin(a));
            if (q % 2) e = make_float4(e.z, e.w, e.x, e.y);
            const bool in = box_has_point(root, e.x, e.y) && box_has_point(root, e.z, e.w);
            const bool nan = q % 4 == 2;
            if (nan) {                                       // one coordinate, or one of each endpoint
                float* p = &e.x;
                p[u64() % 4] = NAN;
                if (u64() & 1u) p[u64() % 4] = NAN;
            }
            const EdgeCells c = edge_cells(tg, table, root, e);
            if (c.l > table || c.x1 >> c.l || c.y1 >> c.l || ((nan || !in) && c.l != 0u)) {
                std::printf("edge cells out of range, or of an edge that has none\n");
                return 1;
            }
            Leaves ref, got;
            descend(t, 0, 0, 0, root, e, ref);
            from_cell(t, c.l, c.x0, c.y0, e, got);
            if (c.x0 != c.x1 || c.y0 != c.y1) from_cell(t, c.l, c.x1, c.y1, e, got);
            if (ref != got) {
                std::printf("edge leaves differ: case %llu, %zu and %zu, edge %.9g %.9g %.9g %.9g, root %.9g %.9g %.9g %.9g\n",
                            (unsigned long long)i, ref.size(), got.size(), e.x, e.y, e.z, e.w, root.x, root.y, root.z, root.w);
                return 1;
            }
            if (nan) nans++;
            else if (!in) leave++;
            if (c.l) cells++;
        }
    }
    std::printf("ok %llu %llu %llu %llu %llu\n", (unsigned long long)outside, (unsigned long long)inside,
                (unsigned long long)leave, (unsigned long long)cells, (unsigned long long)nans);
    return 0;
}
