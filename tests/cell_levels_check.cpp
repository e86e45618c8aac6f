// CPU check of how many levels the cell tables have (image_cells): all that the tree's depth gives in a full
// layout, CELL_LEVELS_MIN in a sparse one, whose updates would rewrite large tables for
// nothing; and that patches of tables of every number of levels leave each entry as a fresh
// walk of the tree gives it.
// Usage: cell_levels_check; prints "ok <levels of each engine> ...".
#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

#include "../jagua-rs_amd/csrc/jg_host.hpp"

using namespace jg;

static uint64_t g_state = 5;
static double urand() {
    g_state += 0x9e3779b97f4a7c15ull;
    return (double)(mix64(g_state) >> 11) * (1.0 / 9007199254740992.0);
}
static Polygon ngon(float cx, float cy, float r, int nv) {
    std::vector<float> xy;
    for (int i = 0; i < nv; i++) {
        xy.push_back(cx + r * (float)std::cos(2.0 * M_PI * (i + 0.1) / nv));
        xy.push_back(cy + r * (float)std::sin(2.0 * M_PI * (i + 0.1) / nv));
    }
    Polygon p;
    std::string err;
    if (!polygon_new(xy.data(), (uint32_t)nv, p, err)) std::exit(2);
    return p;
}

struct Engine {
    SlotMap map;
    QuadTree qt;
    PoolImage im;
    std::vector<jg_hazkey> keys;
    Engine(uint32_t depth, int across) {
        qt.init((uint8_t)depth, make_float4(0.0f, 0.0f, 1000.0f, 1000.0f), 16);
        put(500.0f, 500.0f, 480.0f, 4, JG_ENTITY_EXTERIOR);
        for (int i = 0; i < across * across; i++) {
            const float g = 640.0f / (float)across;
            put(180.0f + g * ((float)(i % across) + 0.5f), 180.0f + g * ((float)(i / across) + 0.5f), 0.42f * g, 7, JG_ENTITY_PLACED_ITEM);
        }
    }
    void put(float x, float y, float r, int nv, uint32_t kind) {
        HazardRec rec;
        rec.entity = jg_hazard_entity{};
        rec.entity.kind = kind;
        rec.shape = ngon(x, y, r, nv);
        keys.push_back(map.insert(std::move(rec)));
        qt.register_hazard(0, root_entry(map.slots[keys.back().idx].rec.shape, keys.back()), map);
    }
    void drop(size_t i) {
        const jg_hazkey k = keys[i];
        map.remove(k);
        qt.deregister_hazard(0, k.idx, k.version);
        keys.erase(keys.begin() + (long)i);
    }
    // every entry of every level against a walk of the tree
    bool cells_right() const {
        for (uint32_t l = 0; l <= im.cell_level; l++)
            for (uint32_t y = 0; y < 1u << l; y++)
                for (uint32_t x = 0; x < 1u << l; x++) {
                    int32_t n = 0;
                    uint32_t d = 0, cd = collects_at(qt, 0) ? 0 : CELL_NO_CDEPTH;
                    while (d < l && qt.pool[(size_t)n].child >= 0) {
                        const bool right = (x >> (l - d - 1)) & 1u, up = (y >> (l - d - 1)) & 1u;
                        n = qt.pool[(size_t)n].child + (up ? (right ? 0 : 1) : (right ? 3 : 2));
                        d++;
                        if (cd == CELL_NO_CDEPTH && collects_at(qt, n)) cd = d;
                    }
                    const size_t at = (((size_t)1 << (2 * l)) - 1) / 3 + (((size_t)y << l) | x);
                    if (im.cells[at] != ((cd << 28) | (d << 24) | (uint32_t)n)) return false;
                }
        return true;
    }
};

int main() {
    std::string line = "ok";
    for (int e = 0; e < 6; e++) {
        static const struct { uint32_t depth; int across; uint32_t level; } cases[] = {
            {5, 0, 5}, {8, 1, 7}, {10, 2, 7}, {10, 4, 8}, {10, 40, 9}, {8, 24, 8}};
        Engine g(cases[e].depth, cases[e].across);
        image_build(g.im, g.qt, g.map);
        line += " " + std::to_string(g.im.cell_level);
        if (g.im.cell_level != cases[e].level || !g.cells_right()) {
            std::printf("engine %d: %u levels, not %u, or wrong cells\n", e, g.im.cell_level, cases[e].level);
            return 1;
        }
        std::vector<uint8_t> staging;
        std::vector<ImageSeg> segs;
        uint64_t cells_bytes = 0;
        for (int step = 0; step < 24; step++) {
            const uint32_t level = g.im.cell_level;
            if (step % 2 == 0) g.put((float)(100.0 + 800.0 * urand()), (float)(100.0 + 800.0 * urand()), (float)(5.0 + 60.0 * urand()), 9, JG_ENTITY_PLACED_ITEM);
            else g.drop(1 + (size_t)(urand() * (double)(g.keys.size() - 1)));
            if (!image_patch(g.im, g.qt, g.map, staging, segs)) image_build(g.im, g.qt, g.map);
            else if (g.im.cell_level != level) return 1;
            for (const ImageSeg& s : segs) cells_bytes += s.dst >= g.im.o_ce ? s.bytes : 0;
            if (!g.cells_right()) {
                std::printf("engine %d step %d: wrong cells\n", e, step);
                return 1;
            }
        }
        line += "/" + std::to_string(cells_bytes / 24);
    }
    std::printf("%s\n", line.c_str());
    return 0;
}
