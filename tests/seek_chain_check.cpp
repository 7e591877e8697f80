// Host check of a CDS's whole stem search as a workgroup of four waves runs it
// (seek_cds in cd_kernels.hip over csrc/cd_seek.h): the first length, the
// searches at it and after it, their budgets, and the tiles and anti-diagonals
// where the searches end without a stem.  Reads CDS from stdin, one per line:
// "sequence" (digits 0-3; initialisation), or "sequence l p q mask" (a child:
// its parent's longest stem, and 0/1 per codon that changed).  An argument
// replaces every wave's budget.  Prints "l p q searches tiled".  A line "after n K
// all found seed parent" prints the length of the next search.
#include <algorithm>
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>
#include <vector>

#include "cd_seek.h"
#include "cd_tile.h"

static constexpr int NW = 4, NT = 64 * NW, HEADS = 2048;
static int g_budget = -1;

struct Cds {
    std::vector<uint2> s, r;
    std::vector<uint32_t> chg;
    int n, L;
    int base(int p) const { return (int)(((s[p >> 5].x >> (p & 31)) & 1u) | (((s[p >> 5].y >> (p & 31)) & 1u) << 1)); }
};

// stem_seed
static int seed_of(const Cds &c, int l, int p, int q, bool &intact) {
    uint64_t m = 0;
    for (int k = 0; k < 64; ++k) {
        const int i = p + l - 1 - k, j = q + k;
        if (l > 0 && i >= 0 && j < c.n && (c.base(i) ^ c.base(j)) == 3) m |= 1ull << k;
    }
    intact = l > 0 && l <= 64 && (~m & (~0ull >> (64 - l))) == 0;
    int run = 0;
    for (; m; m &= m >> 1) ++run;
    return run;
}

// seek_run by wave w: false when it stops early
static bool wave_search(const Cds &c, int w, int K, bool changed, const std::vector<uint32_t> &bits,
                        const std::vector<uint32_t> &head, const std::vector<uint16_t> &next, uint64_t &best) {
    const int n = c.n, Q = cd::sk_word(n, K), st = cd::sk_stride(n, K);
    const uint32_t mask = (1u << Q) - 1u;
    const int xe = cd::sk_positions(n, K, changed), nch = (xe + 7) >> 3;
    int steps = g_budget >= 0 ? g_budget : cd::sk_budget(n);
    std::vector<int> cand, list;
    std::vector<std::pair<int, int>> match;
    auto measure = [&](size_t from) {
        for (size_t i = from; i < match.size(); ++i)
            cd::qg_measure(c.s.data(), c.r.data(), n, match[i].first, match[i].second, K, best);
        match.resize(from);
    };
    int c0 = w * 64;
    for (bool last = false; !last;) {
        std::vector<int> chunks;
        if (changed) {
            while (list.size() < 64 && c0 < nch) {
                for (int x = c0; x < c0 + 64 && x < nch; ++x)
                    if (cd::sk_chunk_changed(c.chg.data(), c.L, K, x)) list.push_back(x);
                c0 += NT;
            }
            const size_t take = std::min<size_t>(list.size(), 64);
            chunks.assign(list.end() - (long)take, list.end());
            list.resize(list.size() - take);
            last = list.empty() && c0 >= nch;
        } else {
            for (int x = c0; x < c0 + 64 && x < nch; ++x) chunks.push_back(x);
            c0 += NT;
            last = c0 >= nch;
        }
        for (int ch : chunks)
            for (uint32_t h = cd::sk_chunk_lookup(c.s.data(), bits.data(), mask, ch, xe); h; h &= h - 1u)
                cand.push_back(8 * ch + __builtin_ctz(h));
        while (cand.size() >= 64 || (last && !cand.empty())) {
            const size_t take = std::min<size_t>(cand.size(), 64);
            std::vector<int> a(cand.end() - (long)take, cand.end());
            cand.resize(cand.size() - take);
            std::vector<uint32_t> word(take), e(take);
            for (size_t i = 0; i < take; ++i) {
                word[i] = cd::sk_number_at(c.s.data(), a[i], mask);
                e[i] = head[cd::sk_chain(word[i], HEADS)];
            }
            for (;;) {
                bool any = false;
                for (uint32_t x : e) any |= x != cd::SK_NIL;
                if (!any) break;
                if (--steps < 0) return false;
                for (size_t i = 0; i < take; ++i) {
                    if (e[i] == cd::SK_NIL) continue;
                    int ma = a[i], mb = st * (int)e[i];
                    const uint32_t v = cd::sk_number_at(c.r.data(), mb, mask);
                    e[i] = next[e[i]];
                    if (v == word[i] && cd::sk_half(n, Q, changed, ma, mb)) match.push_back({ma, mb});
                }
                if (match.size() >= 64) {
                    measure(match.size() - 64);
                    if (cd::sk_stops(K, best)) return false;
                }
            }
        }
    }
    measure(0);
    return true;
}

// stem_tiles
static uint64_t tiles(const Cds &c, int seed) {
    const int n = c.n, TT = 2 * cd::tile_prefix(n, cd::tile_blocks(n));
    uint64_t best = 0;
    for (int t = 0; t < NT; ++t) {
        int K = std::max(seed, cd::TILE_MIN_RUN);
        const int t0 = (int)((int64_t)t * TT / NT), t1 = (int)((int64_t)(t + 1) * TT / NT);
        cd::TileCursor cur;
        for (int j = t0; j < t1; ++j) {
            if (j == t0) cd::tile_seek(c.s.data(), c.r.data(), n, t0, cur);
            cd::tile_step(c.s.data(), c.r.data(), n, cur, K, best);
        }
    }
    if (seed < cd::TILE_MIN_RUN && (int)(best >> 40) < cd::TILE_MIN_RUN) {
        best = 0;
        int K = 1;
        for (int S = 5; S <= 2 * n - 3; ++S) cd::scan_diagonal(c.s.data(), c.r.data(), n, S, 4, K, best);
    }
    return best;
}

int main(int argc, char **argv) {
    if (argc > 1) g_budget = std::stoi(argv[1]);
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string seq, maskstr;
        int pl = 0, pp = 0, pq = 0;
        in >> seq;
        if (seq == "after") {
            int a[6];
            for (int &x : a) in >> x;
            std::printf("%d\n", cd::sk_after_k(a[0], a[1], a[2] != 0, a[3], a[4], a[5] != 0));
            continue;
        }
        in >> pl >> pp >> pq >> maskstr;
        Cds c;
        const int n = c.n = (int)seq.size();
        c.L = n / 3;
        c.s.assign(cd::scan_words(n), make_uint2(0, 0));
        c.r = c.s;
        c.chg.assign(cd::sk_mask_words(c.L), 0);
        for (int i = 0; i < n; ++i) {
            const int a = seq[i] - '0', b = (seq[n - 1 - i] - '0') ^ 3;
            c.s[i >> 5].x |= (uint32_t)(a & 1) << (i & 31);
            c.s[i >> 5].y |= (uint32_t)(a >> 1) << (i & 31);
            c.r[i >> 5].x |= (uint32_t)(b & 1) << (i & 31);
            c.r[i >> 5].y |= (uint32_t)(b >> 1) << (i & 31);
        }
        for (int k = 0; k < (int)maskstr.size(); ++k)
            if (maskstr[k] == '1') c.chg[k >> 5] |= 1u << (k & 31);
        // seek_cds
        const bool parent = !maskstr.empty();
        bool intact = false;
        int seed = parent ? seed_of(c, pl, pp, pq, intact) : 0;
        intact = intact && cd::sk_takes(n, pl);
        int K = intact ? pl : parent ? cd::sk_first_k(n, seed, pl) : cd::sk_blind_k(n);
        uint64_t best = 0;
        int searches = 0;
        bool done = false;
        while (K && cd::sk_takes(n, K)) {
            ++searches;
            const int Q = cd::sk_word(n, K), st = cd::sk_stride(n, K), NI = cd::sk_count(n, K);
            std::vector<uint32_t> bits(cd::SK_BITWORDS, 0), head(HEADS, cd::SK_NIL);
            std::vector<uint16_t> next(NI);
            for (int k = 0; k < NI; ++k)
                cd::sk_insert(c.r.data(), st, (1u << Q) - 1u, k, bits.data(), head.data(), HEADS, next.data());
            best = intact ? cd::scan_key(pl, pp, pq) : 0;
            bool all = true;
            uint64_t top = best;
            for (int w = 0; w < NW; ++w) {
                uint64_t b = best;
                all &= wave_search(c, w, K, intact, bits, head, next, b);
                top = std::max(top, b);
            }
            best = top;
            const int found = (int)(best >> 40);
            if (all && found >= K) {
                done = true;
                break;
            }
            K = cd::sk_after_k(n, K, all, found, seed, parent);
            seed = std::max(seed, found);
        }
        if (!done) best = tiles(c, seed);
        const int l = (int)(best >> 40);
        std::printf("%d %d %d %d %d\n", l, l ? 0xFFFFF - (int)((best >> 20) & 0xFFFFF) : 0,
                    l ? 0xFFFFF - (int)(best & 0xFFFFF) : 0, searches, done ? 0 : 1);
    }
    return 0;
}
