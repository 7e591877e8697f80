// Host check of the engine's word search (csrc/cd_seek.h): reads CDS from
// stdin, one per line -- "sequence K" (digits 0-3) for a whole search at K, or
// "sequence l p q mask" for the search of the changed part of a CDS whose
// parent's longest stem (l, p, q) still pairs, mask a 0/1 per codon -- and runs
// the search as a workgroup does (seek_run in cd_kernels.hip): the index, the
// chunks looked up, the chains walked, the matches measured.  Prints "l p q" of
// the best stem found, and on stderr how many positions were looked up.  Planes,
// index and mask are allocated at exactly their documented size so that the
// address sanitizer catches any access outside them.
#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <sstream>
#include <string>
#include <vector>

#include "cd_seek.h"

int main(int argc, char **argv) {
    const int HEADS = argc > 1 ? std::stoi(argv[1]) : 1024;
    std::string line;
    long looked = 0, total = 0;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string seq, maskstr;
        int K = 0, pp = 0, pq = 0;
        in >> seq >> K >> pp >> pq >> maskstr;
        const bool changed = !maskstr.empty();
        const int n = (int)seq.size(), L = n / 3, nw = cd::scan_words(n);
        std::vector<uint2> sp(nw, make_uint2(0, 0)), rp(nw, make_uint2(0, 0));
        for (int i = 0; i < n; ++i) {
            const int a = seq[i] - '0', b = (seq[n - 1 - i] - '0') ^ 3;
            sp[i >> 5].x |= (uint32_t)(a & 1) << (i & 31);
            sp[i >> 5].y |= (uint32_t)(a >> 1) << (i & 31);
            rp[i >> 5].x |= (uint32_t)(b & 1) << (i & 31);
            rp[i >> 5].y |= (uint32_t)(b >> 1) << (i & 31);
        }
        std::vector<uint32_t> chg(cd::sk_mask_words(L), 0);
        for (int k = 0; k < (int)maskstr.size(); ++k)
            if (maskstr[k] == '1') chg[k >> 5] |= 1u << (k & 31);
        uint64_t best = changed ? cd::scan_key(K, pp, pq) : 0;
        if (cd::sk_takes(n, K)) {
            const int Q = cd::sk_word(n, K), st = cd::sk_stride(n, K), NI = cd::sk_count(n, K);
            if (NI > cd::sk_count_max(n)) {
                std::printf("index larger than its LDS share n=%d K=%d\n", n, K);
                return 1;
            }
            const uint32_t mask = (1u << Q) - 1u;
            std::vector<uint32_t> bits(cd::SK_BITWORDS, 0), head(HEADS, cd::SK_NIL);
            std::vector<uint16_t> next(NI);
            for (int k = 0; k < NI; ++k) cd::sk_insert(rp.data(), st, mask, k, bits.data(), head.data(), HEADS,
                                                          next.data());
            const int xe = cd::sk_positions(n, K, changed), nch = (xe + 7) >> 3;
            total += nch;
            for (int ch = 0; ch < nch; ++ch) {
                if (changed && !cd::sk_chunk_changed(chg.data(), L, K, ch)) continue;
                ++looked;
                for (uint32_t hit = cd::sk_chunk_lookup(sp.data(), bits.data(), mask, ch, xe); hit; hit &= hit - 1u) {
                    const int a = 8 * ch + __builtin_ctz(hit);
                    const uint32_t w = cd::sk_number_at(sp.data(), a, mask);
                    for (uint32_t e = head[cd::sk_chain(w, HEADS)]; e != cd::SK_NIL; e = next[e]) {
                        int ma = a, mb = st * (int)e;
                        if (cd::sk_number_at(rp.data(), mb, mask) != w || !cd::sk_half(n, Q, changed, ma, mb)) continue;
                        cd::qg_measure(sp.data(), rp.data(), n, ma, mb, K, best);
                    }
                }
            }
        }
        const int l = (int)(best >> 40);
        std::printf("%d %d %d\n", l, l ? 0xFFFFF - (int)((best >> 20) & 0xFFFFF) : 0, l ? 0xFFFFF - (int)(best & 0xFFFFF) : 0);
    }
    std::fprintf(stderr, "chunks %ld of %ld\n", looked, total);
    return 0;
}
