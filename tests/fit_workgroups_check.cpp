// CPU check of fit_workgroups (jg_host.hpp): with memory for every workgroup it asks once; with less it halves
// until the memory suffices, down to one workgroup; without memory for one it gives none, and
// what was granted is what was asked for last.
#include <cstdio>

#include "../jagua-rs_amd/csrc/jg_host.hpp"

int main() {
    const uint64_t fixed = 1000, per = 1u << 20;
    for (uint32_t want = 1; want <= 1024; want++)
        for (uint64_t have = 0; have <= fixed + per * 1030; have += have < 4 * per ? per / 8 : 7 * per + 13) {
            uint32_t calls = 0;
            uint64_t last = 0;
            const uint32_t g = jg::fit_workgroups(want, fixed, per, [&](uint64_t bytes) {
                calls++;
                last = bytes;
                return bytes <= have;
            });
            bool ok = g <= want && calls <= 11u;
            if (g) ok = ok && last == fixed + per * g && last <= have && (g == want ? calls == 1 : fixed + per * (2ull * g + 1) > have);
            else ok = ok && fixed + per > have;
            if (!ok) {
                std::printf("want %u, have %llu: %u after %u\n", want, (unsigned long long)have, g, calls);
                return 1;
            }
        }
    std::printf("ok\n");
    return 0;
}
