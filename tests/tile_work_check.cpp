// Host check of the work of the stem scans (csrc/cd_tile.h, and with the
// argument "diag" csrc/cd_scan.h): reads sequences of nucleotide codes from
// stdin (one per line, digits 0-3), scans the tiles (the anti-diagonals) of
// each as a workgroup of 256 lanes does (stem_tiles in cd_kernels.hip) and
// prints "l p q calls tiles": the longest stem, the function calls of the scan
// (compiled with -finstrument-functions) and its number of tiles.
#include <cstdio>
#include <iostream>
#include <string>
#include <vector>

#include "cd_tile.h"

static long calls = 0;
extern "C" {
__attribute__((no_instrument_function)) void __cyg_profile_func_enter(void *, void *) { ++calls; }
__attribute__((no_instrument_function)) void __cyg_profile_func_exit(void *, void *) {}
}

int main(int argc, char **argv) {
    constexpr int NT = 256;
    const bool diag = argc > 1 && std::string(argv[1]) == "diag";
    std::string seq;
    while (std::getline(std::cin, seq)) {
        const int n = (int)seq.size(), nw = cd::scan_words(n);
        std::vector<uint2> s(nw, make_uint2(0, 0)), r(nw, make_uint2(0, 0));
        for (int i = 0; i < n; ++i) {
            const int a = seq[i] - '0', b = (seq[n - 1 - i] - '0') ^ 3;
            s[i >> 5].x |= (uint32_t)(a & 1) << (i & 31);
            s[i >> 5].y |= (uint32_t)(a >> 1) << (i & 31);
            r[i >> 5].x |= (uint32_t)(b & 1) << (i & 31);
            r[i >> 5].y |= (uint32_t)(b >> 1) << (i & 31);
        }
        const uint2 *sp = s.data(), *rp = r.data();
        const int TT = 2 * cd::tile_prefix(n, cd::tile_blocks(n));
        std::vector<cd::TileCursor> cur(NT);
        std::vector<int> K(NT, diag ? 1 : cd::TILE_MIN_RUN);
        auto share = [&](int w) {  // the lanes of wave w share the largest K
            int top = 0;
            for (int t = w; t < w + 64; ++t) top = K[t] > top ? K[t] : top;
            for (int t = w; t < w + 64; ++t) K[t] = top;
        };
        uint64_t best = 0;
        calls = 0;
        for (int j = 0; diag ? 5 + j * NT <= 2 * n - 3 : j < (TT + NT - 1) / NT; ++j)
            for (int w = 0; w < NT; w += 64) {
                for (int t = w; t < w + 64; ++t) {
                    if (diag) {
                        if (5 + t + j * NT <= 2 * n - 3) cd::scan_diagonal(sp, rp, n, 5 + t + j * NT, 4, K[t], best);
                        continue;
                    }
                    const int t0 = (int)((int64_t)t * TT / NT), t1 = (int)((int64_t)(t + 1) * TT / NT);
                    if (t0 + j < t1) {
                        if (j == 0) cd::tile_seek(sp, rp, n, t0, cur[t]);
                        cd::tile_step(sp, rp, n, cur[t], K[t], best);
                    }
                }
                share(w);
            }
        const long work = calls;
        const int l = (int)(best >> 40);
        std::printf("%d %d %d %ld %d\n", l, l ? 0xFFFFF - (int)((best >> 20) & 0xFFFFF) : 0,
                    l ? 0xFFFFF - (int)(best & 0xFFFFF) : 0, work, TT);
    }
    return 0;
}
