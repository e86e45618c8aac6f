// CPU check of the start cells of what lies partly or wholly outside the root box (holding_cell in
// jg_geom.hpp): random boxes around a root box, and a few ulps beside its bounds.  The holding
// cell is level 0 wherever no quadrant of the root surrounds the box; elsewhere the search
// through the surrounding quadrants passes it.
// Usage: outside_cells_check <seed> <cases>; prints "ok <boxes outside> <boxes inside>".
#include <cmath>
#include <cstdio>
#include <cstdlib>

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

int main(int argc, char** argv) {
    g_state = argc > 1 ? strtoull(argv[1], nullptr, 10) : 1;
    const uint64_t cases = argc > 2 ? strtoull(argv[2], nullptr, 10) : 20000;
    uint64_t outside = 0, inside = 0;
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
                cx = 2u * cx + (k == 0 || k == 3);
                cy = 2u * cy + (k == 0 || k == 1);
                box = box_quadrant(box, k);
            }
            if (cx != hc.ix || cy != hc.iy) {
                std::printf("the surrounding path differs\n");
                return 1;
            }
        }
    }
    std::printf("ok %llu %llu\n", (unsigned long long)outside, (unsigned long long)inside);
    return 0;
}
