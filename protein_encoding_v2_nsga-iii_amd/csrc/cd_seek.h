// cd_seek.h -- longest hairpin stem of one CDS by exact short-word matches
// when a stem length K >= 5 is known or guessed (calMaximumSL,
// utils.cuh:712-888).
//
// As in cd_tile.h, stems are runs along the diagonals of the s-versus-rc match
// matrix: s[a+t] == rc[b+t] pairs bases (a+t, n-1-b-t), and the pair is valid
// (j - i > 4) while a + b + 2t <= n - 6.  Words of Q = min(7, K-1) bases of rc
// (K-2 for long CDS) are indexed at the positions b = 0, st, 2st, ... with
// st = K - Q + 1 >= 2; a
// valid run of R >= K matches holds st consecutive word starts, so one of them
// is indexed.  Looking a position a of s up finds the runs through its word;
// every match whose word is valid is measured exactly along its diagonal, so
// with K at most the longest stem the maximum of the keys is exact including
// the tie rule (longest, then smallest p, then smallest q).
//
// Whole search: every a is looked up and the valid half of the matrix (i < j)
// is measured.
//
// Search of the changed part: a child's CDS differs from its parent's in a few
// codons.  When the parent's longest stem (length K) still pairs, a run of K
// or more that holds no changed base was a run of the parent, no longer and
// not before the parent's stem in the tie order; so besides that stem only the
// runs through a changed base count.  Such a run has a subrun of K through the
// changed base x, whose words in the arm that holds x start at x-K+1 .. x+K-Q:
// only those positions a are looked up, on both arms (a match in the invalid
// half is the same run read from the other arm, and is measured from there).
//
// The index is a bitmap of the words present (2 KiB, exact: 14 bits a word),
// which about NI / 16384 of the lookups pass, and chains of the indexed
// positions by a hash of the word, which only those walk.  A search stops at a
// budget of chain steps (a periodic sequence can match itself everywhere) or at
// a stem far above K, and is taken up again at the length found (sk_after_k); the
// tiles are scanned where no search comes to an end.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cd_qgram.h"
#include "cd_scan.h"

namespace cd {

constexpr int SK_KMIN = 5;               // smallest K searched
constexpr int SK_BITWORDS = 512;         // bitmap: 2^14 words of at most 7 bases
constexpr uint32_t SK_NIL = 0xFFFFu;     // end of a chain

// Smallest stride of a search on n bases: 2, or 3 for long CDS, whose links
// would otherwise take the LDS of two workgroups in ten (their stems of 8 or
// less are rare).
__host__ __device__ inline int sk_stride_min(int n) { return n > 3072 ? 3 : 2; }
// Bases of a word (Q) and stride of the indexed positions (st) at K.
__host__ __device__ inline int sk_word(int n, int K) {
    const int q = K + 1 - sk_stride_min(n);
    return q < 7 ? q : 7;
}
__host__ __device__ inline int sk_stride(int n, int K) { return K - sk_word(n, K) + 1; }
// Indexed positions b = 0, st, ... with b + Q <= n (n >= Q).
__host__ __device__ inline int sk_count(int n, int K) { return (n - sk_word(n, K)) / sk_stride(n, K) + 1; }
// Most index entries of any search (Q >= 4).
__host__ __device__ inline int sk_count_max(int n) { return n >= 4 ? (n - 4) / sk_stride_min(n) + 1 : 0; }

// Whether the search takes a CDS of n bases at K: words of at least 4 bases, a
// stem of K fits, positions fit 16 bits.
__host__ __device__ inline bool sk_takes(int n, int K) { return sk_word(n, K) >= 4 && (n - 4) / 2 >= K && n <= 0xFFFF; }

// Number (14 bits) of the word whose low and high bits start at bit 0 of lo and
// hi; mask = 2^Q - 1.
__host__ __device__ inline uint32_t sk_number(uint32_t lo, uint32_t hi, uint32_t mask) {
    return ((hi & mask) << 7) | (lo & mask);
}
// The number of plane P's word at position a (a + Q <= n: words a/32 and
// a/32+1 are inside scan_words(n)).
__host__ __device__ inline uint32_t sk_number_at(const uint2 *P, int a, uint32_t mask) {
    const uint2 p0 = P[a >> 5], p1 = P[(a >> 5) + 1];
    return sk_number(scan_funnel(p1.x, p0.x, a & 31), scan_funnel(p1.y, p0.y, a & 31), mask);
}
// Its chain, of `heads` (a power of two from 512 to 4096): the high bits of the
// number folded over the low ones.
__host__ __device__ inline uint32_t sk_chain(uint32_t number, int heads) {
    return (number ^ (number >> 9)) & (uint32_t)(heads - 1);
}

// Insert entry k (rc position st*k): its bit, and the head of its chain.
__host__ __device__ inline void sk_insert(const uint2 *rp, int st, uint32_t mask, int k, uint32_t *bits, uint32_t *head,
                                          int heads, uint16_t *next) {
    const uint32_t w = sk_number_at(rp, st * k, mask);
#if defined(__HIP_DEVICE_COMPILE__)
    atomicOr(bits + (w >> 5), 1u << (w & 31u));
    next[k] = (uint16_t)atomicExch(head + sk_chain(w, heads), (uint32_t)k);
#else
    bits[w >> 5] |= 1u << (w & 31u);
    next[k] = (uint16_t)head[sk_chain(w, heads)];
    head[sk_chain(w, heads)] = (uint32_t)k;
#endif
}

// Positions of s that are looked up: below this (a word that fits, and for
// the whole search one with a valid partner).
__host__ __device__ inline int sk_positions(int n, int K, bool changed) {
    const int Q = sk_word(n, K), fit = n - Q + 1, valid = n - 6 - 2 * (Q - 1) + 1;
    return changed ? fit : (valid < fit ? (valid > 0 ? valid : 0) : fit);
}

// Words of a change mask (bit k: codon k changed) of L codons, one zero word
// past the last.
__host__ __device__ inline int sk_mask_words(int L) { return ((L + 31) >> 5) + 1; }

// Whether a position of chunk ch (8ch .. 8ch+7) is looked up in the search of
// the changed part: some changed codon k has 3k-K+1 <= a <= 3k+2+K-Q.
__host__ __device__ inline bool sk_chunk_changed(const uint32_t *chg, int L, int K, int ch) {
    const int x0 = 8 * ch, lo = x0 - K + sk_word(3 * L, K);
    const int k0 = lo > 0 ? lo / 3 : 0, kl = (x0 + 6 + K) / 3, k1 = kl < L - 1 ? kl : L - 1;
    const int len = k1 - k0 + 1;
    if (len <= 0) return false;
    if (len > 31) return true;
    const int w = k0 >> 5;
    return (scan_funnel(chg[w + 1], chg[w], k0 & 31) & ((1u << len) - 1u)) != 0u;
}

// The positions of chunk ch below xe whose words are indexed (bit j: 8ch + j).
__host__ __device__ inline uint32_t sk_chunk_lookup(const uint2 *sp, const uint32_t *bits, uint32_t mask, int ch, int xe) {
    const int x0 = 8 * ch;
    const uint2 p0 = sp[x0 >> 5], p1 = sp[(x0 >> 5) + 1];
    const uint32_t lo = scan_funnel(p1.x, p0.x, x0 & 31), hi = scan_funnel(p1.y, p0.y, x0 & 31);
    uint32_t hit = 0u;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t w = sk_number(lo >> j, hi >> j, mask);
        hit |= ((bits[w >> 5] >> (w & 31u)) & 1u) << j;
    }
    const int left = xe - x0;
    return left >= 8 ? hit : hit & ((1u << (left > 0 ? left : 0)) - 1u);
}

// A match of the words at a (s) and b (rc): (a, b) where the run is measured
// from, with its first Q pairs valid; false where the word is in neither half.
__host__ __device__ inline bool sk_half(int n, int Q, bool changed, int &a, int &b) {
    if (a + b + 2 * (Q - 1) <= n - 6) return true;
    if (!changed || a + b < n + 4) return false;
    const int t = a;
    a = n - Q - b;  // the same pairs from the other arm
    b = n - Q - t;
    return true;
}

// Chain steps a wave may take before the tiles are faster.
__host__ __device__ inline int sk_budget(int n) { return 160 + (n >> 4); }

// A length of which about 6 to 24 runs are expected in a random sequence of n
// bases (n^2 / 2 places, a run of K or more starts at 3 in 4^(K+1)): the first
// K without a parent.
__host__ __device__ inline int sk_blind_k(int n) {
    int K = 0;
    for (uint64_t e = (uint64_t)n * n / 16; e >= 4; e >>= 2) ++K;
    return K > SK_KMIN ? K : SK_KMIN;
}
// K of the first search of a changed CDS whose parent's longest stem has
// length parent_l and of which a run of `seed` is known to pair; and of the
// search after one at K found no stem of K (a guess).  A broken stem far
// longer than the others says nothing of the next longest, so the guess is at
// most sk_blind_k; guesses go down one by one, because each base less makes
// four times the matches.
__host__ __device__ inline int sk_first_k(int n, int seed, int parent_l) {
    const int kb = sk_blind_k(n), g = parent_l - 1 < kb ? parent_l - 1 : kb;
    const int k = g > seed ? g : seed;
    return k > SK_KMIN ? k : SK_KMIN;
}
__host__ __device__ inline int sk_next_k(int K, int seed) {
    if (K <= SK_KMIN) return 0;  // the tiles follow
    return K - 1 > seed ? K - 1 : seed;
}
// Whether a wave of a search at K stops at its best key so far: a stem of twice
// K, of a repeat, whose runs are many and long to measure.
__host__ __device__ inline bool sk_stops(int K, uint64_t best) { return (int)(best >> 40) >= 2 * K; }
// K of the search after one at K, 0: the tiles.  A search that stopped early
// (all false: out of budget, or sk_stops) is taken up again at the
// length it had found, if that is longer by half at least: the entries and the
// matches fall with K.  Without a parent one lower guess is made: two fruitless
// ones say that the CDS is no random one, and its stems may be as short as one
// pair.  Initialisation of 64 designs of 1500 residues of FK (stems of 2200): 160
// us, 8.6 ms when every search that stopped went to the tiles; of 600 of K (none):
// 86 us, 92 with a guess at every length.
// The chain ends whatever a search returns: K falls, or grows by half and can
// only grow from there, because `seed` is then the length met.
__host__ __device__ inline int sk_after_k(int n, int K, bool all, int found, int seed, bool parent) {
    if (!all) return 2 * found >= 3 * K ? found : 0;
    const int next = parent || K >= sk_blind_k(n) ? sk_next_k(K, seed) : 0;
    return next < K ? next : 0;
}

// LDS of a search on n bases by `waves` waves with `heads` chains: bitmap, chain heads, links, per
// wave the candidates (a half step of 256 over a kept rest of 63), the matches
// to measure (64 over 63) and the chunks to look up (64 over 63).
constexpr int SK_CAND = 320, SK_LIST = 128, SK_MATCH = 128;
__host__ __device__ inline int sk_link_bytes(int n) { return (2 * sk_count_max(n) + 15) & ~15; }
__host__ __device__ inline int sk_lds_bytes(int n, int heads, int waves) {
    return (SK_BITWORDS + heads) * 4 + sk_link_bytes(n) + waves * (SK_MATCH * 4 + (SK_CAND + SK_LIST) * 2);
}

}  // namespace cd
