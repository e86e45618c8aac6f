// CPU check of the start nodes of circles and edges (circle_cells and edge_cells in jg_geom.hpp): over
// random quadtrees the leaves that a circle's (an edge's) descent from the root reaches, through
// circle_quadrants (edge_quadrants_node) at every internal node, are exactly those reached from
// the nodes of its cells, a circle's each taken only if circle_box holds for it.  Circles lie
// anywhere in and around the box, with radii over seven decades, and with their bounds on cell
// bounds and a few ulps beside them; edges likewise inside it.
// Usage: start_cells_check <seed> <cases>; prints "ok <leaves> <on bounds> <edges with two cells>".
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "../jagua-rs_amd/csrc/jg_geom.hpp"

using namespace jg;

static uint64_t g_state;
static uint64_t u64() {                      // splitmix64
    uint64_t z = (g_state += 0x9e3779b97f4a7c15ull);
    return mix64(z);
}
static double urand() { return (double)(u64() >> 11) * (1.0 / 9007199254740992.0); }

struct Tree {                                // a node splits by a hash of its place
    float4 root;
    uint32_t depth, table, keep;
    uint64_t salt;
    bool split(uint32_t l, uint32_t x, uint32_t y) const {
        return l < depth && (mix64(salt + (((uint64_t)l << 40) | ((uint64_t)y << 20) | x)) & 255u) < keep;
    }
    static void child(int k, uint32_t& x, uint32_t& y) {
        x = 2 * x + (k == 0 || k == 3);
        y = 2 * y + (k == 0 || k == 1);
    }
};
typedef std::set<uint64_t> Leaves;

static void descend(const Tree& t, uint32_t l, uint32_t x, uint32_t y, float4 box, float cx, float cy, float r, Leaves& out) {
    if (!t.split(l, x, y)) {
        out.insert(((uint64_t)l << 40) | ((uint64_t)y << 20) | x);
        return;
    }
    const uint32_t m = circle_quadrants(cx, cy, r, box);
    for (int k = 0; k < 4; k++)
        if ((m >> k) & 1u) {
            uint32_t a = x, b = y;
            Tree::child(k, a, b);
            descend(t, l + 1, a, b, box_quadrant(box, k), cx, cy, r, out);
        }
}

static void descend(const Tree& t, uint32_t l, uint32_t x, uint32_t y, float4 box, float4 e, Leaves& out) {
    if (!t.split(l, x, y)) {
        out.insert(((uint64_t)l << 40) | ((uint64_t)y << 20) | x);
        return;
    }
    const uint32_t m = edge_quadrants_node(e, box);
    for (int k = 0; k < 4; k++)
        if ((m >> k) & 1u) {
            uint32_t a = x, b = y;
            Tree::child(k, a, b);
            descend(t, l + 1, a, b, box_quadrant(box, k), e, out);
        }
}

// the deepest node on the path to cell (x, y) of level l
static float4 deepest(const Tree& t, uint32_t l, uint32_t x, uint32_t y, uint32_t& d, uint32_t& a, uint32_t& b) {
    a = b = d = 0;
    float4 box = t.root;
    while (d < l && t.split(d, a, b)) {
        const uint32_t s = l - d - 1;
        const bool right = (x >> s) & 1u, up = (y >> s) & 1u;
        const int k = up ? (right ? 0 : 1) : (right ? 3 : 2);
        Tree::child(k, a, b);
        box = box_quadrant(box, k);
        d++;
    }
    return box;
}

static void from_cell(const Tree& t, uint32_t l, uint32_t x, uint32_t y, float4 e, Leaves& out) {
    uint32_t d, a, b;
    const float4 box = deepest(t, l, x, y, d, a, b);
    descend(t, d, a, b, box, e, out);
}

static void from_cell(const Tree& t, uint32_t l, uint32_t x, uint32_t y, float cx, float cy, float r, Leaves& out) {
    uint32_t d, a, b;
    const float4 box = deepest(t, l, x, y, d, a, b);
    if (d == 0 || circle_box(cx, cy, r, box)) descend(t, d, a, b, box, cx, cy, r, out);
}

static float ulps(float v, int n) {
    for (; n > 0; n--) v = std::nextafterf(v, INFINITY);
    for (; n < 0; n++) v = std::nextafterf(v, -INFINITY);
    return v;
}

int main(int argc, char** argv) {
    g_state = argc > 1 ? strtoull(argv[1], nullptr, 10) : 1;
    const uint64_t cases = argc > 2 ? strtoull(argv[2], nullptr, 10) : 20000;
    uint64_t leaves = 0, on = 0, two = 0;
    for (uint64_t i = 0; i < cases; i++) {
        Tree t;
        const float w = (float)std::exp(std::log(1e-2) + urand() * std::log(1e7)), h = i % 3 ? w : w * (float)(0.2 + urand());
        const float ox = (float)((urand() - 0.5) * (i % 4 == 0 ? 2000.0 : i % 4 == 1 ? 0.0 : 2.0)) * w, oy = (float)((urand() - 0.5) * 2.0) * h;
        t.root = make_float4(ox, oy, ox + w, oy + h);
        t.depth = (uint32_t)(u64() % 11);
        t.table = t.depth < 9 ? t.depth : 9;
        t.keep = i % 5 ? 200u + (uint32_t)(u64() % 57) : 256u;
        t.salt = u64();
        const CellGrid g = cell_grid(t.root, t.table);
        for (int q = 0; q < 20; q++) {
            float r = (float)(w * std::exp(std::log(1e-6) + urand() * std::log(1e7)));
            // keep the leaf sets small: a wide circle only over a shallow tree
            if (t.depth > 4u) r = fminf(r, 3.0f * w / (float)(1u << t.depth) * (float)(0.2 + urand()));
            float cx = ox + w * (float)(1.4 * urand() - 0.2), cy = oy + h * (float)(1.4 * urand() - 0.2);
            if (q % 2) {
                // a bound of the circle on (or a few ulps beside) a bound of a cell, followed as the tree does
                float4 b = t.root;
                for (uint32_t l = 0; l < 1 + u64() % 9; l++) b = box_quadrant(b, (int)(u64() % 4));
                const int side = (int)(u64() % 4);
                if (side == 0) cx = ulps(b.x - r, (int)(u64() % 7) - 3);
                if (side == 1) cx = ulps(b.z + r, (int)(u64() % 7) - 3);
                if (side == 2) cy = ulps(b.y - r, (int)(u64() % 7) - 3);
                if (side == 3) cy = ulps(b.w + r, (int)(u64() % 7) - 3);
                on++;
            }
            if (q == 18) cx = NAN;
            if (q == 19 && i % 2) r = 0.0f;
            Leaves ref, got;
            descend(t, 0, 0, 0, t.root, cx, cy, r, ref);
            const CircleCells c = circle_cells(g, t.table, t.root, cx, cy, r);
            if (c.l > t.table || c.x1 - c.x0 > 1u || c.y1 - c.y0 > 1u || c.x1 >> c.l || c.y1 >> c.l) {
                std::printf("cells out of range\n");
                return 1;
            }
            for (uint32_t y = c.y0; y <= c.y1; y++)
                for (uint32_t x = c.x0; x <= c.x1; x++) from_cell(t, c.l, x, y, cx, cy, r, got);
            if (ref != got) {
                std::printf("leaves differ: case %llu, %zu and %zu, circle %.9g %.9g %.9g, box %.9g %.9g %.9g %.9g\n",
                            (unsigned long long)i, ref.size(), got.size(), cx, cy, r, t.root.x, t.root.y, t.root.z, t.root.w);
                return 1;
            }
            leaves += ref.size();
        }
        for (int q = 0; q < 40; q++) {
            // an edge inside the box, its length over five decades; every other one with a coordinate on
            // (or a few ulps beside) a bound of a cell, some along an axis
            const float len = (float)(w * std::exp(std::log(1e-6) + urand() * std::log(1e6)) * (t.depth > 6 ? 0.1 : 1.0));
            float4 e = make_float4(ox + w * (float)urand(), oy + h * (float)urand(), 0.0f, 0.0f);
            if (q % 2) {
                float4 b = t.root;
                for (uint32_t l = 0; l < 1 + u64() % 9; l++) b = box_quadrant(b, (int)(u64() % 4));
                if (u64() & 1u) e.x = ulps(u64() & 1u ? b.x : b.z, (int)(u64() % 9) - 4);
                else e.y = ulps(u64() & 1u ? b.y : b.w, (int)(u64() % 9) - 4);
            }
            const double a = q % 8 == 1 ? 0.0 : q % 8 == 3 ? M_PI / 2 : 2.0 * M_PI * urand();
            e.z = e.x + (float)(len * std::cos(a));
            e.w = e.y + (float)(len * std::sin(a));
            if (q % 8 == 1) e.w = e.y;
            if (q % 8 == 3) e.z = e.x;
            const float4 r = t.root;
            e.x = fminf(fmaxf(e.x, r.x), r.z); e.z = fminf(fmaxf(e.z, r.x), r.z);
            e.y = fminf(fmaxf(e.y, r.y), r.w); e.w = fminf(fmaxf(e.w, r.y), r.w);
            if (u64() & 1u) e = make_float4(e.z, e.w, e.x, e.y);
            Leaves ref, got;
            descend(t, 0, 0, 0, t.root, e, ref);
            const float4 eb = make_float4(mn(e.x, e.z), mn(e.y, e.w), mx(e.x, e.z), mx(e.y, e.w));
            const EdgeCells c = edge_cells(g, t.table, t.root, eb);
            const HoldingCell hc = holding_cell(g, t.table, t.root, eb);
            if (c.l > t.table || c.x1 >> c.l || c.y1 >> c.l || hc.l > c.l) {
                std::printf("edge cells out of range\n");
                return 1;
            }
            from_cell(t, c.l, c.x0, c.y0, e, got);
            if (c.x0 != c.x1 || c.y0 != c.y1) {
                from_cell(t, c.l, c.x1, c.y1, e, got);
                two++;
            }
            if (ref != got) {
                std::printf("edge leaves differ: case %llu, %zu and %zu, edge %.9g %.9g %.9g %.9g, box %.9g %.9g %.9g %.9g\n",
                            (unsigned long long)i, ref.size(), got.size(), e.x, e.y, e.z, e.w, r.x, r.y, r.z, r.w);
                return 1;
            }
            // the virtual root's path: the quadrant that surrounds the box, as the search takes it
            // an edge of NaNs has no cell of its own, and a box that is empty along an axis no holding cell
            const float4 en = make_float4(q & 1 ? NAN : eb.x, q & 2 || !(q & 1) ? NAN : eb.y, q & 1 ? NAN : eb.z, q & 2 || !(q & 1) ? NAN : eb.w);
            const float4 bn = make_float4(en.x == en.x ? en.x : FLT_MAX, en.y == en.y ? en.y : FLT_MAX,
                                          en.z == en.z ? en.z : -FLT_MAX, en.w == en.w ? en.w : -FLT_MAX);
            if (edge_cells(g, t.table, t.root, en).l != 0u || holding_cell(g, t.table, t.root, bn).l != 0u) {
                std::printf("a NaN edge or an empty box has a cell\n");
                return 1;
            }
            uint32_t d, x, y;
            deepest(t, hc.l, hc.ix, hc.iy, d, x, y);
            uint32_t rx = 0, ry = 0;
            float4 box = t.root;
            for (uint32_t l = 0; l < d; l++) {
                const int k = quadrant_surrounding(box, eb);
                if (k < 0) {
                    std::printf("no quadrant surrounds the box at level %u of %u\n", l, d);
                    return 1;
                }
                Tree::child(k, rx, ry);
                box = box_quadrant(box, k);
            }
            if (rx != x || ry != y) {
                std::printf("the surrounding path differs\n");
                return 1;
            }
        }
    }
    std::printf("ok %llu %llu %llu\n", (unsigned long long)leaves, (unsigned long long)on, (unsigned long long)two);
    return 0;
}
