// cd_kernels.hip -- HIP kernels of the codon-design engine for gfx950.
//
// One generation is these launches over every resident job:
//   k_design<OFFSPRING>  one workgroup per child: parent from the survivor
//                        mask, survivor copy, mutation, objectives 0-4
//                        (mutationKernel, main.cu:121-240)
//   k_stem_each          longest stem of each CDS the mutation changed
//   (k_stem_list)        (calMaximumSL), for small (large) launches
//   k_dominance          objective 5 of the children, bit-packed
//                        eps-domination matrix (sorting.cuh:994-1023), the
//                        pool's ideal and worst points
//   k_front0             the first front, its maxima and ASF minima, many
//                        workgroups per job
//   k_fronts             one workgroup per job: further fronts, extreme
//                        points, hyperplane/MNDF nadir (sorting.cuh:974-1089,
//                        132-972)
//   k_associate          nearest reference line per ranked design and the
//                        niche counts (sorting.cuh:1105-1180)
//   k_front_associate    the three above in one launch, for few and small
//                        pools (fuse_fronts)
//   [k_levels]           the niche levels, when the reference points do not
//                        fit in LDS (else k_place settles them)
//   k_place              level-0 picks, whole buckets, the cut list
//   k_niche              the cut buckets ranked by priority
//                        (sorting.cuh:1182-1279); ends the generation
//   k_place_niche        the two above in one workgroup per job, for pools up
//                        to 2048
// Hand-offs between workgroups happen at kernel boundaries; atomics that
// fold per-job quantities are reduced over the workgroup first (same-address
// atomics serialise at the device's coherence point).
// Work lists map blockIdx.x to (job, item) so the same kernels advance one
// job or a batch of uneven jobs.
#include <cfloat>
#include <mutex>

#include "cd_device.h"
#include "cd_kernels.h"
#include "cd_qgram.h"
#include "cd_scan.h"
#include "cd_seek.h"
#include "cd_tile.h"

namespace cd {

__host__ __device__ constexpr int align16(int x) { return (x + 15) & ~15; }

// k_design's dynamic LDS: log weights by codon code lw6 [64] (int64) and
// synonym words by code [64] (u64), then the design's code rows [m][Ls]
// (stride Ls = row_stride(L)), then the CDS statistics [m].  Rows are 16-byte
// aligned, so the genome moves between HBM and LDS in 16-byte words and four
// codes share a 32-bit word in the sums.  Holding the pool as codes instead of
// synonym indices halves this (no index rows, no per-position synonym ranges)
// and saves the conversion of every codon of every child: 1.4 us a workgroup.
constexpr int DL_SYN = 512, DL_ROWS = 1024;

// The change masks of the CDS (sk_mask_words(L) words each) follow the
// statistics.
size_t design_lds_bytes(int L, int m) {
    return DL_ROWS + (size_t)m * (row_stride(L) + sizeof(CdsStat) + 4 * sk_mask_words(L)) + 16;
}

// Jobs are accepted up to this size: 160 KiB for m synonym and code rows, the
// synonym ranges and the statistics of a design.
__host__ __device__ inline int plane_stage_bytes(int L) { return align16((scan_words(3 * L) + 1) * 8); }
size_t design_bytes_accepted(int L, int m) {
    const int a = row_stride(L), b = plane_stage_bytes(L);
    return (size_t)576 + 2 * a + (size_t)m * ((a > b ? a : b) + a) + align16(m * (int)sizeof(CdsStat)) + 16;
}

// one CDS's bit planes as k_design leaves them: the sequence's, scan_words(3L)
// words of (low bits, high bits) of the nucleotide codes, then the change mask
// (bit k: codon k changed) in whole 8-byte words
__host__ __device__ inline int plane_words(int L) { return scan_words(3 * L) + ((sk_mask_words(L) + 1) >> 1); }
size_t cds_plane_bytes(int L) { return (size_t)plane_words(L) * sizeof(uint2); }

// An entry of k_stem_list's list: CDS and child below; the buffer the child is
// in and its job above.
__device__ __forceinline__ uint64_t stem_entry(uint32_t job, uint32_t child, uint32_t c, uint32_t buf) {
    return (uint64_t)((child << 4) | c) | ((uint64_t)((job << 1) | buf) << 32);
}

// dynamic LDS of the stem kernels: a CDS's planes, its reverse complement's and
// the change mask, then the word search's index (the launchers add the chain
// heads and the waves' queues)
__host__ __device__ inline int stem_index_at(int L) { return align16((scan_words(3 * L) + plane_words(L)) * (int)sizeof(uint2)); }
size_t stem_lds_bytes(int L) { return (size_t)stem_index_at(L) + sk_lds_bytes(3 * L, 0, 0); }
static size_t seek_more_bytes(int heads, int threads) {
    return (size_t)sk_lds_bytes(0, heads, threads / 64) - sk_lds_bytes(0, 0, 0);
}

constexpr int HITQ = 192;  // a wave's queue of hits: a full batch of 64 and one step's 128
// k_design's static LDS for a workgroup of NW waves.
template <int NW>
struct DesignShared {
    float pobj[NOBJ];
    int32_t pidx[2 * NOBJ];
    int32_t ppql[4];
    int32_t dirty[MAX_M];  // CDS the operator changed
    int32_t hd[MAX_M * (MAX_M - 1) / 2];
    uint16_t hitq[NW][HITQ];  // per wave: codons that passed an operator's test, awaiting their work
};

// CdsStat records in global memory, four 16-byte words through the global
// address space (an aggregate copy would go through flat accesses).
struct CdsWords {
    u32x4 w[4];
};
static_assert(sizeof(CdsWords) == sizeof(CdsStat), "a CdsStat record is four 16-byte words");
__device__ __forceinline__ CdsStat gload_stat(const CdsStat *p) {
    const u32x4 *q = (const u32x4 *)p;
    CdsWords v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v.w[i] = gload(q + i);
    return __builtin_bit_cast(CdsStat, v);
}
__device__ __forceinline__ void gstore_stat(CdsStat *p, const CdsStat &s) {
    u32x4 *q = (u32x4 *)p;
    const CdsWords v = __builtin_bit_cast(CdsWords, s);
#pragma unroll
    for (int i = 0; i < 4; ++i) gstore(q + i, v.w[i]);
}

// Facts of codons given by their codes (first base << 4 | second << 2 | third).
// Third base C (1) or G (2).
__device__ __forceinline__ int code_gc3(int a) { return (a ^ (a >> 1)) & 1; }
// Hidden stop codons read across the junction a|b: a[1] a[2] b[0] and
// a[2] b[0] b[1] (countRightSideHSC, utils.cuh:138-161).
__device__ __forceinline__ int code_hidden(uint64_t stop6, int a, int b) {
    return (int)((stop6 >> (((a & 15) << 2) | (b >> 4))) & 1u) + (int)((stop6 >> (((a & 3) << 4) | (b >> 2))) & 1u);
}
// Nucleotide mismatches of the codons whose codes are the bytes of x ^ y:
// a byte's three 2-bit fields differ when either bit of the field is set.
__device__ __forceinline__ int code_mismatch4(uint32_t x) { return __popc((x | (x >> 1)) & 0x15151515u); }
__device__ __forceinline__ int code_mismatch(int a, int b) { return code_mismatch4((uint32_t)(a ^ b)); }
// Base p of a CDS given as a row of codes.
__device__ __forceinline__ int code_base(const uint8_t *row, int p) {
    const unsigned k = (unsigned)p / 3u;
    return (row[k] >> (4 - 2 * (p - 3 * (int)k))) & 3;
}
// ---------------------------------------------------------------------------
// Longest stem of one CDS held as bit planes in LDS (calMaximumSL,
// utils.cuh:712-888; the planes are built by k_design): word searches
// (cd_seek.h) at a known or guessed length, a lower guess after a fruitless
// one and the length met after one that stopped early, and the tiles (cd_tile.h)
// for a CDS whose stems are all shorter than 5 or that the searches give up on.
// A CDS with no run of 4 and no seed of 4 is scanned exactly along its
// anti-diagonals (cd_scan.h).  Each search takes the maximum key (longest, then
// smallest p, then smallest q).
// ---------------------------------------------------------------------------
// The seed: the longest run of pairs (i - k, j + k), k < 64, that
// still pair in the child, with (i, j) = (p + l - 1, q) the parent's
// innermost pair.  Each such run is a stem of the child (its pairs lie on one
// anti-diagonal and enclose at least the parent's loop), so its length bounds
// the longest stem from below.  intact: every pair of the parent's stem still
// pairs.
__device__ __forceinline__ int plane_base(const uint2 *sp, int p) {
    const uint2 w = sp[p >> 5];
    const int b = p & 31;
    return (int)(((w.x >> b) & 1u) | (((w.y >> b) & 1u) << 1));
}
__device__ __forceinline__ int stem_seed(const uint2 *sp, int n, int l, int p, int q, int lane, bool &intact) {
    const int i = p + l - 1, j = q;
    const bool pair = l > 0 && lane <= i && j + lane < n && ((plane_base(sp, i - lane) ^ plane_base(sp, j + lane)) == 3);
    uint64_t m = __ballot(pair);
    intact = l > 0 && l <= 64 && (~m & (~0ull >> (64 - l))) == 0;
    int run = 0;
    while (m) {  // each round removes the last pair of every run
        ++run;
        m &= m >> 1;
    }
    return run;
}

// The tiled scan of a CDS with a stem of `seed` known (0: none) by a
// workgroup, and its exact scan when there is neither a seed of 4 nor a run of
// 4; returns the workgroup's maximum key.  Out of line, for the search's rare
// fallback: inlined, its registers would raise the pressure of the search
// path.  The LDS pointers keep their address space, so the scan's loads stay
// LDS loads.
typedef __attribute__((address_space(3))) uint2 lds_uint2;
typedef __attribute__((address_space(3))) uint64_t lds_uint64;
__device__ __noinline__ uint64_t stem_tiles(int n, const lds_uint2 *planes, int seed, lds_uint64 *lds_redu) {
    const int tid = threadIdx.x, NT = blockDim.x;
    const uint2 *sp = (const uint2 *)planes, *rp = sp + scan_words(n);
    uint64_t *redu = (uint64_t *)lds_redu;
    // Every lane's K is a length some stem of this CDS has, so the wave may
    // share the largest after each step.  Trip counts are the same for every
    // lane, so every lane takes part in the exchanges.
    int K = max(seed, TILE_MIN_RUN);
    uint64_t best = 0;
    {
        const int TT = 2 * tile_prefix(n, tile_blocks(n));
        const int t0 = (int)((int64_t)tid * TT / NT), t1 = (int)((int64_t)(tid + 1) * TT / NT);
        const int trips = (TT + NT - 1) / NT;
        TileCursor cur;
        for (int j = 0; j < trips; ++j) {
            if (t0 + j < t1) {
                if (j == 0) tile_seek(sp, rp, n, t0, cur);
                tile_step(sp, rp, n, cur, K, best);
            }
            K = wave_max_nonneg(K);
        }
    }
    best = block_max_u64(best, redu);
    // With a seed of 4 or more the longest stem is at least 4 long, so the
    // tiles measured it; without one and with no run of 4, the exact scan.
    if (seed < TILE_MIN_RUN && (int)(best >> 40) < TILE_MIN_RUN) {
        best = 0;
        K = 1;
        const int S0 = MIN_HAIRPIN + 1 + tid, Sw = MIN_HAIRPIN + 1 + (tid & ~63), last = 2 * n - 3;
        const int trips = Sw <= last ? (last - Sw) / NT + 1 : 0;
        for (int j = 0; j < trips; ++j) {
            const int S = S0 + j * NT;
            if (S <= last) scan_diagonal(sp, rp, n, S, MIN_HAIRPIN, K, best);
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) K = max(K, __shfl_xor(K, o, 64));
        }
        best = block_max_u64(best, redu);
    }
    return best;
}

// LDS of the word search (cd_seek.h).
struct SeekLds {
    uint32_t *bits, *head;
    uint16_t *next;
    uint32_t *match;         // match, cand, list: the wave's own
    uint16_t *cand, *list;
    const uint32_t *chg;     // the CDS's change mask (offspring)
};
template <int HEADS>
__device__ __forceinline__ SeekLds seek_lds(uint8_t *base, int n, int wid, const uint32_t *chg) {
    SeekLds S;
    S.bits = (uint32_t *)base;
    S.head = S.bits + SK_BITWORDS;
    S.next = (uint16_t *)(S.head + HEADS);
    S.match = (uint32_t *)((uint8_t *)S.next + sk_link_bytes(n) + wid * (SK_MATCH * 4 + (SK_CAND + SK_LIST) * 2));
    S.cand = (uint16_t *)(S.match + SK_MATCH);
    S.list = S.cand + SK_CAND;
    S.chg = chg;
    return S;
}
// Empties the bitmap and the chains (the next barrier makes it visible).
template <int NT, int HEADS>
__device__ __forceinline__ void seek_clear(const SeekLds &S) {
    u32x4 *b = (u32x4 *)S.bits;
    const u32x4 zero = {0u, 0u, 0u, 0u}, nil = {SK_NIL, SK_NIL, SK_NIL, SK_NIL};
#pragma unroll
    for (int i = 0; i < SK_BITWORDS / 4; i += NT)
        if (SK_BITWORDS / 4 % NT == 0 || i + (int)threadIdx.x < SK_BITWORDS / 4) b[i + threadIdx.x] = zero;
#pragma unroll
    for (int i = 0; i < HEADS / 4; i += NT)
        if (HEADS / 4 % NT == 0 || i + (int)threadIdx.x < HEADS / 4) b[SK_BITWORDS / 4 + i + threadIdx.x] = nil;
}

// A CDS's planes and change mask from the job's plane buffer g into LDS
// (planes of the sequence, planes of the reverse complement, mask) by NT
// threads: the first NT words' loads on construction, the rest and all stores
// in place().  Bit b of the reverse complement is position n-1-b complemented:
// a word of it is 32 positions of the sequence turned round.
template <int NT>
struct PlaneLoad {
    const uint64_t *g;
    int n, W, words;
    uint64_t fwd, r0, r1, mask;
    __device__ __forceinline__ int turn_at(int i) const { return max(n - 32 - 32 * i, 0) >> 5; }
    __device__ __forceinline__ uint64_t turned(int i, uint64_t a, uint64_t b) const {
        const int e = n - 32 * i, st = e - 32;  // positions st .. e-1
        uint32_t lo, hi, keep = ~0u;
        if (st >= 0) {
            lo = scan_funnel((uint32_t)b, (uint32_t)a, st & 31);
            hi = scan_funnel((uint32_t)(b >> 32), (uint32_t)(a >> 32), st & 31);
        } else {
            keep = e > 0 ? (1u << e) - 1u : 0u;
            lo = (uint32_t)a << (-st & 31);
            hi = (uint32_t)(a >> 32) << (-st & 31);
        }
        return (uint64_t)(~__builtin_bitreverse32(lo) & keep) | ((uint64_t)(~__builtin_bitreverse32(hi) & keep) << 32);
    }
    __device__ __forceinline__ PlaneLoad(const uint64_t *gp, int L) : g(gp), n(3 * L), W(scan_words(n)), words(plane_words(L)) {
        const int tid = (int)threadIdx.x, i = min(tid, W - 1), t = turn_at(i);
        fwd = gload(g + i);
        r0 = gload(g + t);
        r1 = gload(g + t + 1);
        mask = gload(g + min(W + tid, words - 1));
    }
    __device__ __forceinline__ void place(uint64_t *planes) const {
        const int tid = (int)threadIdx.x;
        if (tid < W) {
            planes[tid] = fwd;
            planes[W + tid] = turned(tid, r0, r1);
        }
        if (W + tid < words) planes[2 * W + tid] = mask;
        for (int i = tid + NT; i < W; i += NT) {
            const int t = turn_at(i);
            const uint64_t f = gload(g + i), a = gload(g + t), b = gload(g + t + 1);
            planes[i] = f;
            planes[W + i] = turned(i, a, b);
        }
        for (int i = W + tid + NT; i < words; i += NT) planes[W + i] = gload(g + i);
    }
};

// Lanes of `bal` below the calling one.
__device__ __forceinline__ int lanes_below(uint64_t bal) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
}

// One search of a workgroup of NT threads at K (cd_seek.h), the index emptied
// before and planes and index ready behind a barrier.  Every wave looks up its
// chunks of 8 positions, 64 chunks a step (of the changed part only the chunks
// near a changed codon, gathered first), queues the positions whose words are
// indexed, walks their chains 64 positions at a time and queues the matches,
// which are measured 64 at a time: the lanes stay busy whatever share of the
// lookups, positions and chain entries passes, and no barrier stands between.
// best: the lane's largest key.  Returns false in a wave that ran out of
// budget or stopped at a far longer stem (sk_stops).
template <int NT, int HEADS>
__device__ __forceinline__ bool seek_run(const SeekLds &S, const uint2 *sp, const uint2 *rp, int n, int L, int K,
                                         bool changed, uint64_t &best) {
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int Q = sk_word(n, K), st = sk_stride(n, K), NI = sk_count(n, K);
    const uint32_t mask = (1u << Q) - 1u;
    for (int k = tid; k < NI; k += NT) sk_insert(rp, st, mask, k, S.bits, S.head, HEADS, S.next);
    lds_barrier();
    const int xe = sk_positions(n, K, changed), nch = (xe + 7) >> 3;
    // (the same in every lane) chain steps left; positions, matches and chunks queued
    int steps = sk_budget(n), cnt = 0, nm = 0, listed = 0;
    int c0 = wid * 64;
    for (bool last = false; !last;) {
        int ch = nch;  // the lane's chunk of this step
        if (changed) {
            while (listed < 64 && c0 < nch) {
                const int c = c0 + lane;
                const bool act = c < nch && sk_chunk_changed(S.chg, L, K, c);
                const uint64_t bal = __ballot(act);
                if (act) S.list[listed + lanes_below(bal)] = (uint16_t)c;
                listed += (int)__popcll(bal);
                c0 += NT;
            }
            wave_lds_sync();
            const int take = min(listed, 64);
            listed -= take;
            if (lane < take) ch = S.list[listed + lane];
            last = listed == 0 && c0 >= nch;
        } else {
            ch = min(c0 + lane, nch);
            c0 += NT;
            last = c0 >= nch;
        }
        uint32_t hit = ch < nch ? sk_chunk_lookup(sp, S.bits, mask, ch, xe) : 0u;
        // queue the lane's positions: all together when they fit (a step has
        // some twenty), else in two halves
        uint32_t rest = 0u;
        int mine = __popc(hit), incl = wave_scan_i32(mine), got = __builtin_amdgcn_readlane(incl, 63);
        const bool halves = cnt + got > SK_CAND;
        if (halves) {
            rest = hit & 0xF0u;
            hit &= 0x0Fu;
            mine = __popc(hit);
            incl = wave_scan_i32(mine);
            got = __builtin_amdgcn_readlane(incl, 63);
        }
        for (bool more = true; more;) {
            int at = cnt + incl - mine;
            while (hit) {
                S.cand[at++] = (uint16_t)(8 * ch + __builtin_ctz(hit));
                hit &= hit - 1u;
            }
            cnt += got;
            wave_lds_sync();
            more = __any(rest != 0u);
            const bool drain = last && !more;
            while (cnt >= 64 || (drain && cnt > 0)) {
                const int take = min(cnt, 64);
                cnt -= take;
                const int a = lane < take ? (int)S.cand[cnt + lane] : 0;
                const uint32_t w = sk_number_at(sp, a, mask);
                uint32_t e = lane < take ? S.head[sk_chain(w, HEADS)] : SK_NIL;
                while (__any(e != SK_NIL)) {
                    if (--steps < 0) return false;
                    int ma = a, mb = 0;
                    bool ok = false;
                    if (e != SK_NIL) {
                        mb = st * (int)e;
                        const uint32_t v = sk_number_at(rp, mb, mask);
                        e = S.next[e];
                        ok = v == w && sk_half(n, Q, changed, ma, mb);
                    }
                    const uint64_t bal = __ballot(ok);
                    if (ok) S.match[nm + lanes_below(bal)] = qg_pack(ma, mb);
                    nm += (int)__popcll(bal);
                    if (nm >= 64) {
                        wave_lds_sync();
                        nm -= 64;
                        const uint32_t v = S.match[nm + lane];
                        qg_measure(sp, rp, n, (int)(v >> 16), (int)(v & 0xFFFFu), K, best);
                        if (__any(sk_stops(K, best))) return false;
                    }
                }
            }
            if (more) {  // the second half
                hit = rest;
                rest = 0u;
                mine = __popc(hit);
                incl = wave_scan_i32(mine);
                got = __builtin_amdgcn_readlane(incl, 63);
            }
        }
    }
    if (nm > 0) {
        wave_lds_sync();
        if (lane < nm) {
            const uint32_t v = S.match[lane];
            qg_measure(sp, rp, n, (int)(v >> 16), (int)(v & 0xFFFFu), K, best);
        }
    }
    return true;
}

// The search(es) of one CDS by a workgroup of NT threads: planes in LDS at sp
// and rp, the index emptied, all behind a barrier.  parent: whether (pl, pp,
// pq) is the longest stem of the CDS's parent, from which it differs in the
// codons of S.chg.  Returns the workgroup's largest key; every thread holds it.
template <int NT, int HEADS>
__device__ __forceinline__ uint64_t seek_cds(const SeekLds &S, const uint2 *sp, const uint2 *rp, int n, int L,
                                             bool parent, int pl, int pp, int pq, uint64_t *redu, int32_t *flag) {
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    bool intact = false;
    int seed = parent ? stem_seed(sp, n, pl, pp, pq, lane, intact) : 0;  // every wave itself
    intact = intact && sk_takes(n, pl);
    int K = intact ? pl : parent ? sk_first_k(n, seed, pl) : sk_blind_k(n);
    bool fresh = true;
    while (K && sk_takes(n, K)) {
        if (!fresh) {
            lds_barrier();  // the search before has read the index
            seek_clear<NT, HEADS>(S);
            lds_barrier();
        }
        fresh = false;
        uint64_t best = intact && lane == 0 ? scan_key(pl, pp, pq) : 0ull;
        const bool ok = seek_run<NT, HEADS>(S, sp, rp, n, L, K, intact, best);
        best = wave_max_u64(best);
        if (lane == 0) {
            redu[wid] = best;
            flag[wid] = ok;
        }
        lds_barrier();
        bool all = true;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) {
            best = redu[w] > best ? redu[w] : best;
            all &= flag[w] != 0;
        }
        const int found = (int)(best >> 40);  // (a stem of the CDS, also where the budget ran out)
        if (all && found >= K) return best;
        K = sk_after_k(n, K, all, found, seed, parent);
        seed = max(seed, found);
        lds_barrier();  // redu and flag are read
    }
    lds_barrier();
    return stem_tiles(n, (const lds_uint2 *)sp, seed, (lds_uint64 *)redu);
}

// ---------------------------------------------------------------------------
// Evaluation of a design's code rows in LDS (calMinimumCAI/CBP/HSC/HD,
// calMaximumGC3, utils.cuh:271-626), in three kinds of task, one wave a task
// and no barrier between them:
//   sums of one CDS        CAI and CPB sums, hidden stops, GC3 codons, then the
//                          CDS's values; four codons to a 32-bit word
//   planes of one CDS      its bit planes for the stem search
//   Hamming distance of one pair of CDS
// With the whole workgroup on one CDS at a time (a barrier and a cross-wave
// sum after each) the reductions cost about as much as the sums.  With the
// code rows, the tasks and the operators' synonym words the offspring launch
// went from 608 to 395 us on the 64-job mix (42 240 children), 161 to 98 us for
// 4096 children of 12 008 codons, 32 to 23 us for 1024 of 2004; the remaining
// bound is VALU issue, about a quarter of it the operators' Philox draws.
// ---------------------------------------------------------------------------
// Per-CDS values of the sums: CAI, CPB, the HSC quotient and the GC3 fraction.
__device__ __forceinline__ void cds_values(CdsStat &s, int L) {
    s.ov[0] = (float)det_exp(((double)s.cai * 0x1p-40) / (double)L);
    s.ov[1] = (float)(((double)s.cpb * 0x1p-40) / (double)(L - 2));
    s.ov[2] = (float)s.hsc / (float)(L - 1);
    s.ov[3] = (float)s.gc3 / (float)L;
}

// Bytes of v (each below 64) that are stop codes: UAA, UAG, UGA are 48, 50
// and 56 (the job's table keeps the standard code), the bytes whose bits 5
// and 4 are set, 2 and 0 clear, and 3 and 1 not both set.
__device__ __forceinline__ int stops4(uint32_t v) {
    const uint32_t t = v ^ 0x30303030u;
    const uint32_t z = (t & 0x35353535u) | (t & (t >> 2) & 0x02020202u);  // 0 in a stop's byte
    return 4 - __popc((z + 0x7F7F7F7Fu) & 0x80808080u);
}

// Sums of the CDS in row w (nwd words): a word's four codons and their four
// junctions a step.  Padding codons are code 0: they add the log weight and
// the pair score of code 0, taken off at the end, and no GC3; their junctions
// are masked off, and a stop scores no pairs.
__device__ __forceinline__ void task_sums(const DevJob &J, const int64_t *lw6, const uint32_t *w, int L, int nwd,
                                          CdsStat *rec, bool have_parent) {
    const int lane = threadIdx.x & 63, n4 = (L + 3) >> 2;
    const int64_t *const pair6 = J.cpfx6;
    int64_t cai = 0, cpb = 0;
    uint32_t hg = 0;  // hidden stops in the high half, GC3 codons in the low half (both below 2^16)
#pragma unroll 1
    for (int q = lane; q < n4; q += 64) {
        const uint32_t a = w[q], nx = q + 1 < nwd ? w[q + 1] : 0u;
        const uint32_t b = __builtin_amdgcn_alignbit(nx, a, 8);  // the codons one further on
        const uint32_t e = ((a & 0x003F003Fu) << 9) | ((b & 0x003F003Fu) << 3);  // byte offsets of pairs 0 and 2
        const uint32_t o = (((a >> 8) & 0x003F003Fu) << 9) | (((b >> 8) & 0x003F003Fu) << 3);  // of 1 and 3
        const char *const pb = (const char *)pair6;
        const int64_t p0 = gload((const int64_t *)(pb + (e & 0xFFFFu))), p1 = gload((const int64_t *)(pb + (o & 0xFFFFu)));
        const int64_t p2 = gload((const int64_t *)(pb + (e >> 16))), p3 = gload((const int64_t *)(pb + (o >> 16)));
        cai += (lw6[a & 63u] + lw6[(a >> 8) & 63u]) + (lw6[(a >> 16) & 63u] + lw6[a >> 24]);
        const uint32_t gc = (a ^ (a >> 1)) & 0x01010101u;  // third base C (1) or G (2)
        // junctions a|b: a[1] a[2] b[0] and a[2] b[0] b[1]
        // (countRightSideHSC, utils.cuh:138-161); the last codon has none
        const int left = L - 1 - 4 * q;
        const uint32_t keep = left >= 4 ? ~0u : (1u << (8 * max(left, 0))) - 1u;
        const uint32_t j1 = ((a & 0x0F0F0F0Fu) << 2) | ((b >> 4) & 0x03030303u);
        const uint32_t j2 = ((a & 0x03030303u) << 4) | ((b >> 2) & 0x0F0F0F0Fu);
        hg += ((uint32_t)(stops4(j1 & keep) + stops4(j2 & keep)) << 16) + (uint32_t)__popc(gc);
        cpb += (p0 + p1) + (p2 + p3);
    }
    cai = wave_sum_i64(cai);
    cpb = wave_sum_i64(cpb);
    hg = (uint32_t)wave_sum_i32((int)hg);
    const int pads = 4 * n4 - L;
    CdsStat s = *rec;
    if (!have_parent) s.l = s.p = s.q = 0;
    s.cai = cai - pads * lw6[0];
    s.cpb = cpb - pads * gload(pair6);
    s.hsc = (int)(hg >> 16);
    s.gc3 = (int)(hg & 0xFFFFu);
    s.pad = 1;
    s.key = 0;
    cds_values(s, L);
    if (lane == 0) *rec = s;
}

// Twelve bits of four codons (three to a byte, bytes in order) packed in a row.
__device__ __forceinline__ uint32_t pack12(uint32_t x) {
    const uint32_t t = x | (x >> 5);
    return (t & 0x3Fu) | ((t >> 10) & 0xFC0u);
}

// Bit planes of the CDS in row w into the job's plane buffer, then its change
// mask: bit p is position p, positions past n are zero; a word is (low bits,
// high bits) of 32 positions.  A lane builds a word from the eleven or twelve
// codons it meets, which start at any byte; the reverse complement's planes
// are made from these where they are used (PlaneLoad).  A lane per 32 codons
// and both planes took a fifth of k_design's vector instructions: 64-job mix
// 410 -> 379 us, 4096 children of 12 008 codons 106 -> 91, 128 of 202 13.5 ->
// 11.9, and 2 to 6 us more in the stem kernels of the first two.
__device__ __forceinline__ void task_planes(const uint32_t *w, int L, int nwd, const uint32_t *chg, uint2 *sp) {
    const int n = 3 * L, W = scan_words(n), lane = threadIdx.x & 63;
    for (int i = lane; i < W; i += 64) {
        const uint32_t k0 = 32u * (uint32_t)i / 3u, r = 32u * (uint32_t)i - 3u * k0;
        const int q = (int)(k0 >> 2);
        uint32_t d[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) d[t] = w[min(q + t, nwd - 1)];
#pragma unroll
        for (int t = 0; t < 4; ++t) d[t] = q + t < nwd ? d[t] : 0u;  // (the row's padding codes are 0)
        uint32_t l[3], h[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const uint32_t c = __builtin_amdgcn_alignbyte(d[t + 1], d[t], k0 & 3u);
            // per byte the three bases' low (high) bits in position order
            l[t] = pack12(((c >> 4) & 0x01010101u) | ((c >> 1) & 0x02020202u) | ((c << 2) & 0x04040404u));
            h[t] = pack12(((c >> 5) & 0x01010101u) | ((c >> 2) & 0x02020202u) | ((c << 1) & 0x04040404u));
        }
        const uint32_t lo = __builtin_amdgcn_alignbit(l[2] >> 8, l[0] | (l[1] << 12) | (l[2] << 24), r);
        const uint32_t hi = __builtin_amdgcn_alignbit(h[2] >> 8, h[0] | (h[1] << 12) | (h[2] << 24), r);
        gstore((uint64_t *)(sp + i), (uint64_t)lo | ((uint64_t)hi << 32));
    }
    uint32_t *const mk = (uint32_t *)(sp + W);
    for (int i = lane; i < sk_mask_words(L); i += 64) gstore(mk + i, chg[i]);
}

// Hamming distance of the CDS in rows a and b (nv 16-byte words; the padding
// codes are 0 in every CDS and add nothing), wave-uniform.
__device__ __forceinline__ int task_pair(const uint32_t *a, const uint32_t *b, int nv) {
    const u32x4 *a4 = (const u32x4 *)a, *b4 = (const u32x4 *)b;
    int acc = 0;
    for (int q = threadIdx.x & 63; q < nv; q += 64) {
        const u32x4 x = a4[q] ^ b4[q];
#pragma unroll
        for (int v = 0; v < 4; ++v) acc += code_mismatch4(x[v]);
    }
    return wave_sum_i32(acc);
}

// The tasks of a design whose CDS in dmask changed (all of them without a
// parent): wave wid of nw takes every nw-th.  The pairs are those of the one
// changed CDS, or every pair when more changed (sh.hd holds the parent's
// distances on entry).
template <class SH>
__device__ __forceinline__ void design_tasks(const DevJob &J, const int64_t *lw6, const uint32_t *rows, uint32_t dmask, bool have_parent,
                             const uint32_t *chg, CdsStat *cst, SH &sh, uint2 *planes, int wid, int nw) {
    const int L = J.L, m = J.m, nwd = J.Ls >> 2, lane = threadIdx.x & 63, PW = plane_words(L);
    const int nd = __popc(dmask), npair = nd == 1 ? m - 1 : (nd ? m * (m - 1) / 2 : 0);
    uint32_t left = dmask;  // the CDS of task t, for t rising
    int t0 = 0;
    int i = 0, j = 0, p0 = -1;  // the last pair enumerated
    for (int t = wid; t < 2 * nd + npair; t += nw) {
        if (t < 2 * nd) {
            const int r = t < nd ? t : t - nd;
            if (r < t0) {
                left = dmask;
                t0 = 0;
            }
            for (; t0 < r; ++t0) left &= left - 1u;
            const int c = __builtin_ctz(left);
            if (t < nd)
                task_sums(J, lw6, rows + c * nwd, L, nwd, cst + c, have_parent);
            else
                task_planes(rows + c * nwd, L, nwd, chg + c * sk_mask_words(L), planes + (size_t)c * PW);
            continue;
        }
        const int p = t - 2 * nd;  // pair p of the list
        int a, b, q;
        if (nd == 1) {
            const int c = __builtin_ctz(dmask), o = p < c ? p : p + 1;
            a = min(c, o);
            b = max(c, o);
            q = a * (2 * m - a - 1) / 2 + b - a - 1;
        } else {
            for (; p0 < p; ++p0)  // pairs (i, j), i < j, in lexicographic order
                if (p0 < 0)
                    j = 1;
                else if (++j == m) {
                    ++i;
                    j = i + 1;
                }
            a = i;
            b = j;
            q = p;
        }
        const int d = task_pair(rows + a * nwd, rows + b * nwd, nwd >> 2);
        if (lane == 0) sh.hd[q] = d;
    }
}

// Largest v of lanes 0-15 (one DPP row), and the last lane below m holding it.
__device__ __forceinline__ int last_max16(float v, int m) {
    float x = v;
    x = fmaxf(x, dpp_f32<0x111, 0xf>(x, -FLT_MAX));
    x = fmaxf(x, dpp_f32<0x112, 0xf>(x, -FLT_MAX));
    x = fmaxf(x, dpp_f32<0x114, 0xf>(x, -FLT_MAX));
    x = fmaxf(x, dpp_f32<0x118, 0xf>(x, -FLT_MAX));
    x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 15));
    const uint64_t at = __ballot(v == x && (int)(threadIdx.x & 63) < m);
    return 63 - (int)__builtin_clzll(at);
}

// Objectives 0-4 of the design and their indices, by one wave, stored to
// oobj and oidx (entry 10, the stem's CDS, is left to the stem search): each
// is the largest of the CDS's (pairs') values, ties to the last CDS (pair) --
// a serial sweep that takes every value at least as large as the one it holds
// (utils.cuh:271-626).  The values are finite, and all zeros of one objective
// have one sign.  The smallest distance is the largest negated quotient:
// distinct distances below 2^24 have distinct quotients.
template <class SH>
__device__ __forceinline__ void design_objectives(const DevJob &J, const CdsStat *cst, const SH &sh, float *oobj, int8_t *oidx) {
    const int m = J.m, n = 3 * J.L, lane = threadIdx.x & 63, npair = m * (m - 1) / 2;
    const float gc3_ref = J.gc3_ref;
    const bool cl = lane < m;
    const CdsStat &sc = cst[cl ? lane : 0];
    const float v0 = sc.ov[0], v1 = sc.ov[1], v2 = sc.ov[2], v3 = sc.ov[3];
    const float k0 = cl ? -v0 : -FLT_MAX, k1 = cl ? -v1 : -FLT_MAX, k2 = cl ? -v2 : -FLT_MAX;
    const float k4 = cl ? fabsf(v3 - gc3_ref) : -FLT_MAX;
    int dist = 0x7FFFFFFF, pair = 0;
    for (int q = lane; q < npair; q += 64) {  // at most two a lane; ties to the later pair
        const int d = sh.hd[q];
        if (d <= dist) {
            dist = d;
            pair = q;
        }
    }
    const int dmin = wave_min_i32(dist);
    const int qh = wave_max_i32(dist == dmin ? pair : -1);
    const int c0 = last_max16(k0, m), c1 = last_max16(k1, m), c2 = last_max16(k2, m), c4 = last_max16(k4, m);
    int i = 0, r = qh;  // pair qh of the lexicographic order
    while (r >= m - 1 - i) {
        r -= m - 1 - i;
        ++i;
    }
    const int j = i + 1 + r;
    const float dev = lane_of(v3, c4) - gc3_ref;
    if (lane < 2 * NOBJ && lane != 10) {
        const int v = lane == 0 ? c0 : lane == 2 ? c1 : lane == 4 ? c2 : lane == 6 ? i : lane == 7 ? j
                      : lane == 8 ? c4 : lane == 9 ? (dev < 0 ? GC_UP : GC_DOWN) : 0;
        gstore(oidx + lane, (int8_t)v);
    }
    if (lane < NOBJ - 1) {
        const float o0 = -lane_of(v0, c0), o1 = -lane_of(v1, c1), o2 = -lane_of(v2, c2);
        const float o3 = -((float)dmin / (float)n), o4 = fabsf(dev);
        gstore(oobj + lane, lane == 0 ? o0 : lane == 1 ? o1 : lane == 2 ? o2 : lane == 3 ? o3 : o4);
    }
}

// ---------------------------------------------------------------------------
// Mutation operators (include/mutation.cuh) on the code rows in LDS.  A
// codon's code names its amino acid, so one table word per code (SynWord)
// holds its synonyms' codes, their number and its own place among them.  Each
// thread owns whole codons; operators that read neighbours only touch codons
// of the other parity or of other CDS, as in the reference.  Draws: the i-th
// slot an operator visits in CDS c takes words 2(i&1) (the mutation test) and
// 2(i&1)+1 (the choice, or the shuffle) of Philox(gen, child, c*L + (i >> 1),
// TAG_MUT), so one call serves two slots and a thread takes the two slots of
// one call.
// ---------------------------------------------------------------------------

struct MutArgs {
    const DevJob *J;
    const uint64_t *syn;  // [64] synonym words by code
    uint8_t *rows;        // [m][Ls] codes
    uint32_t *chg;        // [m][sk_mask_words(L)] changed codons
    int Ls, CW;
    uint32_t gen, child;
};

// A code's synonym word (the 64 after J.lw6's log weights): codes of synonyms 0-4 in six-bit fields of
// the low half, of synonym 5 in bits 0-5 of the high half, their number in
// bits 8-10 and the code's own index in bits 12-14 of it.
struct SynWord {
    uint32_t lo, hi;
    __device__ __forceinline__ explicit SynWord(uint64_t v) : lo((uint32_t)v), hi((uint32_t)(v >> 32)) {}
    __device__ __forceinline__ int num() const { return (int)((hi >> 8) & 7u); }
    __device__ __forceinline__ int own() const { return (int)((hi >> 12) & 7u); }
    __device__ __forceinline__ int code(int j) const { return (int)((j < 5 ? lo >> (6 * j) : hi) & 63u); }
};

// Codon k of CDS c becomes `code`.
__device__ __forceinline__ void set_code(const MutArgs &A, int c, int k, int code) {
    A.rows[c * A.Ls + k] = (uint8_t)code;
    atomicOr(A.chg + c * A.CW + (k >> 5), 1u << (k & 31));
}

// The pick-th (0-based) set bit of a candidate mask.
__device__ __forceinline__ int nth_bit(uint32_t mask, uint32_t pick) {
    for (uint32_t q = 0; q < pick; ++q) mask &= mask - 1u;
    return __builtin_ctz(mask);
}

__device__ __forceinline__ void pair_draws(const MutArgs &A, int c, int q, uint32_t r[4]) {
    philox(A.gen, A.child, (uint32_t)(c * A.J->L + q), TAG_MUT, A.J->seed, r);
}

// The codons of an operator whose work per accepted codon is long, in
// batches: wave w tests the draw pairs q = 64w + lane, 64w + 256 + lane, ...
// (test(q) returns bit h set when codon h of pair q passes the operator's
// Bernoulli test), queues the codons that pass (slot 2q + h) in its segment of
// sh.hitq, and runs work(slot) one codon a lane whenever 64 are queued, then on
// the rest.  Accepted codons change only themselves and the tests and the work
// of other codons read only codons no test of this operator accepts, so the
// order of the work does not matter.  Wave-local: the waves never wait for
// each other.
template <class Test, class Work>
__device__ __forceinline__ void hits_by_wave(int npairs, uint16_t *seg, Test test, Work work) {
    const int lane = threadIdx.x & 63;
    int cnt = 0;  // the same in every lane of the wave
    for (int q0 = (int)(threadIdx.x & ~63u); q0 < npairs; q0 += blockDim.x) {
        const int q = q0 + lane;
        const uint32_t hm = q < npairs ? test(q) : 0u;
        const uint64_t b0 = __ballot(hm & 1u), b1 = __ballot(hm & 2u);
        const int r0 = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b0 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b0, 0u));
        const int r1 = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b1 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b1, 0u));
        const int n0 = (int)__popcll(b0);
        if (hm & 1u) seg[cnt + r0] = (uint16_t)(2 * q);
        if (hm & 2u) seg[cnt + n0 + r1] = (uint16_t)(2 * q + 1);
        cnt += n0 + (int)__popcll(b1);
        while (cnt >= 64) {  // at most 63 + 128 queued: within HITQ
            work((int)seg[cnt - 64 + lane]);
            cnt -= 64;
        }
    }
    if (lane < cnt) work((int)seg[lane]);
}

// mutationRandom, mutation.cuh:16-63: every codon of every CDS; a thread
// takes codons 2q and 2q+1 of CDS c for its (c, q) pairs
__device__ __forceinline__ void mut_random(const MutArgs &A, int32_t *dirty) {
    const DevJob &J = *A.J;
    const int L = J.L, Ls = A.Ls, hL = (L + 1) >> 1, total = J.m * hL;
    int c = (int)((unsigned)threadIdx.x / (unsigned)hL), q = (int)threadIdx.x - c * hL;
    for (int t = threadIdx.x; t < total; t += blockDim.x) {
        uint32_t r[4];
        pair_draws(A, c, q, r);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 2 * q + h;
            if (k >= L || !bern(r[2 * h], J.thr_pm)) continue;
            const SynWord e(A.syn[A.rows[c * Ls + k]]);
            const int ns = e.num(), cur = e.own();
            if (ns == 1) continue;
            int nw = (int)uniform_int(r[2 * h + 1], (uint32_t)(ns - 1));
            if (nw >= cur) ++nw;
            set_code(A, c, k, e.code(nw));
            dirty[c] = 1;
        }
        q += blockDim.x;
        while (q >= hL) {
            q -= hL;
            ++c;
        }
    }
}

// mutationCAI with SELECT_UPPER_RANDOM, mutation.cuh:65-142
__device__ __forceinline__ void mut_cai(const MutArgs &A, int cds, int32_t *dirty) {
    const DevJob &J = *A.J;
    const int L = J.L;
    const uint8_t *const row = A.rows + cds * A.Ls;
    for (int q = threadIdx.x; 2 * q < L; q += blockDim.x) {
        uint32_t r[4];
        pair_draws(A, cds, q, r);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 2 * q + h;
            if (k >= L || !bern(r[2 * h], J.thr_pm)) continue;
            const SynWord e(A.syn[row[k]]);
            const int ns = e.num(), cur = e.own();
            if (cur != ns - 1) {
                set_code(A, cds, k, e.code(cur + 1 + (int)uniform_int(r[2 * h + 1], (uint32_t)(ns - 1 - cur))));
                dirty[cds] = 1;
            }
        }
    }
}

// mutationCBP with SELECT_UPPER_RANDOM, mutation.cuh:144-262: the codons
// k = 2i + parity below L-1; a thread takes i = 2q, 2q+1 (k = 4q + parity,
// 4q + parity + 2)
__device__ __forceinline__ void mut_cbp(const MutArgs &A, int cds, int32_t *dirty, uint16_t *seg) {
    const DevJob &J = *A.J;
    const int L = J.L, parity = (int)(A.gen & 1u);
    const uint64_t thr = J.thr_2pm, stop6 = J.stop6;
    const float *const cps6 = J.cps6;
    const uint8_t *const row = A.rows + cds * A.Ls;
    const int npairs = L - 1 - parity > 0 ? (L - 1 - parity + 3) >> 2 : 0;  // 4q + parity < L - 1
    auto test = [&](int q) -> uint32_t {
        uint32_t r[4];
        pair_draws(A, cds, q, r);
        uint32_t hm = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 4 * q + parity + 2 * h;
            if (k < L - 1 && bern(r[2 * h], thr)) hm |= 1u << h;
        }
        return hm;
    };
    auto work = [&](int slot) {
        const int q = slot >> 1, h = slot & 1, k = 4 * q + parity + 2 * h;
        const SynWord e(A.syn[row[k]]);
        const int left = (k > 0) ? (int)row[k - 1] : 0;
        const int right = row[k + 1];
        const int ns = e.num(), cur = e.own();
        if (ns == 1) return;
        // every synonym's score, the pair-score loads issued together (a
        // missing neighbour adds nothing; stop codes score 0 in the table)
        const bool hl = k > 0, hr = !((stop6 >> right) & 1u);
        const float *rowl = cps6 + left * 64, *colr = cps6 + right;
        float sc[MAX_SYN];
#pragma unroll
        for (int j = 0; j < MAX_SYN; ++j) {
            const int g = j < ns ? e.code(j) : e.code(0);
            const float a = gload(rowl + g), b = gload(colr + g * 64);
            float v = 0.f;
            v += hl ? a : 0.f;
            v += hr ? b : 0.f;
            sc[j] = v;
        }
        float curv = sc[0];
#pragma unroll
        for (int j = 1; j < MAX_SYN; ++j) curv = j == cur ? sc[j] : curv;
        uint32_t cand = 0;  // synonyms scoring above the current codon, in order
#pragma unroll
        for (int j = 0; j < MAX_SYN; ++j)
            if (j < ns && j != cur && sc[j] > curv) cand |= 1u << j;
        if (cand) {
            uint32_t r[4];
            pair_draws(A, cds, q, r);
            set_code(A, cds, k, e.code(nth_bit(cand, uniform_int(h ? r[3] : r[1], (uint32_t)__popc(cand)))));
            dirty[cds] = 1;
        }
    };
    hits_by_wave(npairs, seg, test, work);
}

// mutationHSC with SELECT_UPPER_RANDOM, mutation.cuh:264-388: the codons
// k = 2i + parity below L, two per thread as in mut_cbp
__device__ __forceinline__ void mut_hsc(const MutArgs &A, int cds, int32_t *dirty, uint16_t *seg) {
    const DevJob &J = *A.J;
    const int L = J.L, parity = (int)(A.gen & 1u);
    const uint64_t thr = J.thr_2pm;
    const uint8_t *const row = A.rows + cds * A.Ls;
    const uint64_t stop6 = J.stop6;
    const int npairs = L - parity > 0 ? (L - parity + 3) >> 2 : 0;  // 4q + parity < L
    auto test = [&](int q) -> uint32_t {
        uint32_t r[4];
        pair_draws(A, cds, q, r);
        uint32_t hm = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 4 * q + parity + 2 * h;
            if (k < L && bern(r[2 * h], thr)) hm |= 1u << h;
        }
        return hm;
    };
    auto work = [&](int slot) {
        const int q = slot >> 1, h = slot & 1, k = 4 * q + parity + 2 * h;
        const SynWord e(A.syn[row[k]]);
        const int left = (k > 0) ? (int)row[k - 1] : -1;
        const int right = (k < L - 1) ? (int)row[k + 1] : -1;
        const int ns = e.num(), cur = e.own();
        auto count = [&](int g) -> int {
            int v = 0;
            if (left >= 0) v += code_hidden(stop6, left, g);
            if (right >= 0) v += code_hidden(stop6, g, right);
            return v;
        };
        const int curv = count(row[k]);
        uint32_t cand = 0;
        for (int j = 0; j < ns; ++j)
            if (j != cur && count(e.code(j)) > curv) cand |= 1u << j;
        if (cand) {
            uint32_t r[4];
            pair_draws(A, cds, q, r);
            set_code(A, cds, k, e.code(nth_bit(cand, uniform_int(h ? r[3] : r[1], (uint32_t)__popc(cand)))));
            dirty[cds] = 1;
        }
    };
    hits_by_wave(npairs, seg, test, work);
}

// indexArrayShuffling, utils.cuh:203-218: Fisher-Yates over the n <= 6
// synonyms, entries i = n-1 .. 1 swapped with j_i, the mixed-radix digits
// (radix i+1) of uniform_int(x, n!).  Digits by multiplication: for r < 720,
// (r * (65536/d + 1)) >> 16 is r / d for d = 2..6.  The order is packed in
// 4-bit fields (entry i at bits 4i) so that it stays in registers.
__device__ __forceinline__ uint32_t shuffle(uint32_t x, int n) {
    const uint32_t fact = n == 6 ? 720u : n == 5 ? 120u : n == 4 ? 24u : n == 3 ? 6u : n == 2 ? 2u : 1u;
    uint32_t r = uniform_int(x, fact);
    uint32_t perm = 0x543210u;
#pragma unroll
    for (int i = 5; i > 0; --i) {
        if (i >= n) continue;
        const uint32_t d = (uint32_t)(i + 1), q = (r * (65536u / d + 1u)) >> 16, j = r - q * d;
        r = q;
        const uint32_t vi = (perm >> (4 * i)) & 0xFu, vj = (perm >> (4 * j)) & 0xFu;
        perm &= ~((0xFu << (4 * i)) | (0xFu << (4 * j)));
        perm |= (vj << (4 * i)) | (vi << (4 * j));
    }
    return perm;
}
__device__ __forceinline__ int perm_at(uint32_t perm, int j) { return (int)((perm >> (4 * j)) & 0xFu); }

// mutationHD, mutation.cuh:390-534: codons of cds1, scored against all CDS
__device__ __forceinline__ void mut_hd(const MutArgs &A, int cds1, int cds2, int32_t *dirty, uint16_t *seg) {
    const DevJob &J = *A.J;
    const int L = J.L, m = J.m, Ls = A.Ls;
    const uint64_t thr = J.thr_pm;
    const uint8_t *const row = A.rows + cds1 * Ls;
    auto test = [&](int q) -> uint32_t {
        uint32_t r[4];
        pair_draws(A, cds1, q, r);
        uint32_t hm = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (2 * q + h < L && bern(r[2 * h], thr)) hm |= 1u << h;
        return hm;
    };
    auto work = [&](int k) {
        const SynWord e(A.syn[row[k]]);
        const int ns = e.num(), cur = e.own();
        if (ns == 1) return;
        uint32_t r[4];
        pair_draws(A, cds1, k >> 1, r);
        const uint32_t order = shuffle((k & 1) ? r[3] : r[1], ns);
        const int g2 = A.rows[cds2 * Ls + k];
        // every candidate's codes (the synonyms in shuffled order, slot
        // MAX_SYN the current codon) first, then the smallest distance
        // to the other CDS's codons at k (only cds1's codons change here,
        // each by its own lane) and the distance to cds2's codon
        int gc[MAX_SYN + 1], mn[MAX_SYN + 1], pr[MAX_SYN + 1];
#pragma unroll
        for (int j = 0; j <= MAX_SYN; ++j) {
            gc[j] = e.code(j == MAX_SYN ? cur : perm_at(order, j < ns ? j : ns - 1));
            mn[j] = 127;
            pr[j] = code_mismatch(gc[j], g2);
        }
        for (int o = 0; o < m; ++o) {
            if (o == cds1) continue;
            const int oc = A.rows[o * Ls + k];
#pragma unroll
            for (int j = 0; j <= MAX_SYN; ++j) mn[j] = min(mn[j], code_mismatch(gc[j], oc));
        }
        const int cur_pair = pr[MAX_SYN], cur_mhd = mn[MAX_SYN];
        int best_pair = -1, best_mhd = -1, best = -1;
#pragma unroll
        for (int j = 0; j < MAX_SYN; ++j) {
            const int sh = perm_at(order, j);
            if (j >= ns || sh == cur) continue;
            const int np_ = pr[j], nm = mn[j];
            if (nm > cur_mhd && nm > best_mhd) {
                best_mhd = nm;
                best = sh;
            } else if (best_mhd == -1 && nm == cur_mhd && np_ > cur_pair && np_ > best_pair) {
                best_pair = np_;
                best = sh;
            }
        }
        if (best_mhd != -1 || best_pair != -1) {
            set_code(A, cds1, k, e.code(best));
            dirty[cds1] = 1;
        }
    };
    hits_by_wave((L + 1) >> 1, seg, test, work);
}

// mutationGC3, mutation.cuh:536-653 (probability = the parent's GC3 deviation)
__device__ __forceinline__ void mut_gc3(const MutArgs &A, int cds, int dir, float dev, int32_t *dirty, uint16_t *seg) {
    const DevJob &J = *A.J;
    const int L = J.L;
    const uint64_t thr = bern_threshold(dev);
    const uint8_t *const row = A.rows + cds * A.Ls;
    auto test = [&](int q) -> uint32_t {
        uint32_t r[4];
        pair_draws(A, cds, q, r);
        uint32_t hm = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (2 * q + h < L && bern(r[2 * h], thr)) hm |= 1u << h;
        return hm;
    };
    auto work = [&](int k) {
        const int g = row[k];
        const SynWord e(A.syn[g]);
        const int ns = e.num(), cur = e.own();
        if (ns == 1) return;
        uint32_t r[4];
        pair_draws(A, cds, k >> 1, r);
        const uint32_t order = shuffle((k & 1) ? r[3] : r[1], ns);
        const int curg = code_gc3(g);
        for (int j = 0; j < ns; ++j) {
            const int sh = perm_at(order, j);
            if (sh == cur) continue;
            const int ng = code_gc3(e.code(sh));
            if ((dir == GC_UP && ng > curg) || (dir == GC_DOWN && ng < curg)) {
                set_code(A, cds, k, e.code(sh));
                dirty[cds] = 1;
                break;
            }
        }
    };
    hits_by_wave((L + 1) >> 1, seg, test, work);
}

// mutationSL, mutation.cuh:775-969, by one wave.  The accept test of the
// reference (mutation.cuh:843,896,947) compares the parent's SL objective with
// the integer quotient l_new / ((n-4)/2); it only needs to know whether the
// CDS still has any stem and whether it is one full-length hairpin.  The first
// and last 64 bases nearly always decide both: a complementary pair more than
// the loop apart is a stem, one mismatch rules a full hairpin out.  The rest
// of the CDS is read only when they do not.
template <class SH>
__device__ __forceinline__ void mut_sl(const MutArgs &A, SH &sh, int32_t *dirty) {
    const DevJob &J = *A.J;
    const int L = J.L, n = 3 * L, lane = threadIdx.x & 63;
    const int cds = sh.pidx[10];
    const uint8_t *const row = A.rows + cds * A.Ls;
    const int P0 = sh.ppql[0], Lst = sh.ppql[2];
    const int l_idx = P0 / 3, r_idx = (P0 + Lst - 1) / 3;
    const int mid = (r_idx + l_idx) / 2;
    const int stem_len = r_idx - l_idx + 1, half = stem_len / 2;
    const bool odd = (stem_len % 2) == 1;
    const int l_st0 = odd ? mid - 1 : mid, r_st0 = mid + 1;
    const int den = J.den_sl;
    const float parent_sl = sh.pobj[5];
    const int trials = (odd ? 1 : 0) + 2 * half;
    int cur_l = Lst;
    for (int t = 0; t < trials; ++t) {
        int pos;
        if (odd && t == 0) {
            pos = mid;
        } else {
            const int u = t - (odd ? 1 : 0);
            pos = (u & 1) ? r_st0 + (u >> 1) : l_st0 - (u >> 1);
        }
        uint32_t r[4];
        philox(A.gen, A.child, (uint32_t)t, TAG_SL, J.seed, r);
        const int saved = row[pos];
        const SynWord e(A.syn[saved]);
        const int ns = e.num();
        const bool changed = bern(r[0], J.thr_pm) && ns > 1;
        if (changed) {
            int nw = (int)uniform_int(r[1], (uint32_t)(ns - 1));
            if (nw == e.own()) ++nw;  // mutation.cuh:827 compares with ==
            if (lane == 0) set_code(A, cds, pos, e.code(nw));  // (a codon put back stays marked)
        }
        wave_lds_sync();
        // the first and last 64 bases
        const int lc = min(lane, n - 1);
        const int f = code_base(row, lc), b = code_base(row, n - 1 - lc);
        bool any = false;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const uint64_t F = __ballot(f == a), B = __ballot(b == (a ^ 3));
            if (F && B && n - 1 - (int)__builtin_ctzll(B) - (int)__builtin_ctzll(F) > MIN_HAIRPIN) any = true;
        }
        // the full hairpin's pairs (i, n-1-i), and for odd n (i, n-2-i) or (1+i, n-1-i)
        auto pairs_hold = [&](int i) -> int {
            const int x = code_base(row, i), y = code_base(row, n - 1 - i);
            int ok = (x ^ y) == 3 ? 1 : 0;
            if (n & 1) {
                ok |= ((x ^ code_base(row, n - 2 - i)) == 3) ? 2 : 0;
                ok |= ((code_base(row, 1 + i) ^ y) == 3) ? 4 : 0;
            }
            return ok;
        };
        int full = 0;
        {
            const int ok = lane < den ? pairs_hold(lane) : 7;
#pragma unroll
            for (int q = 0; q < 3; ++q) full |= __ballot(!((ok >> q) & 1)) == 0 ? 1 << q : 0;
        }
        if (!any) {  // every base
            int first[4] = {0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF}, last[4] = {-1, -1, -1, -1};
            for (int i = lane; i < n; i += 64) {
                const int x = code_base(row, i);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (x == q) {
                        first[q] = min(first[q], i);
                        last[q] = i;
                    }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                first[q] = wave_min_i32(first[q]);
                last[q] = wave_max_i32(last[q]);
            }
#pragma unroll
            for (int a = 0; a < 4; ++a)
                if (first[a] != 0x7FFFFFFF && last[a ^ 3] >= 0 && last[a ^ 3] - first[a] > MIN_HAIRPIN) any = true;
        }
        if (full && den > 64) {  // every pair
            int ok = 7;
            for (int i = lane; i < den; i += 64) ok &= pairs_hold(i);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (__ballot(!((ok >> q) & 1))) full &= ~(1 << q);
        }
        bool is_full = false;
        if (den > 0) {
            if ((full & 1) && (n - 1 - 2 * (den - 1)) > MIN_HAIRPIN) is_full = true;
            if ((n & 1) && (full & 6) && (n - 2 - 2 * (den - 1)) > MIN_HAIRPIN) is_full = true;
        }
        if (any) cur_l = is_full ? den : 0;
        const float rhs = (float)(den > 0 ? cur_l / den : 0);
        const bool done = parent_sl > rhs;
        if (changed) {
            if (done)
                dirty[cds] = 1;
            else if (lane == 0)
                A.rows[cds * A.Ls + pos] = (uint8_t)saved;
        }
        wave_lds_sync();
        if (done) break;
    }
}

// The niche arrays the association counts into, cleared from entry i0 on in
// steps.
__device__ __forceinline__ void clear_niche(const DevJob &J, int i0, int step) {
    const int R = J.R;
    if (i0 >= R) return;
    const NicheView g = niche_view(J.niche, R);
    for (int r = i0; r < R; r += step) {
        gstore((uint64_t *)g.cr + r, (uint64_t)0);
        gstore(g.fill + r, 0);
        gstore(g.nearest + r, ~0ull);
    }
}

// The index of the c-th survivor (0-based, ascending pool index) in the
// survivor mask of W words: wave-uniform, every lane of the wave takes part.
__device__ __forceinline__ int survivor_at(const uint64_t *selm, int W, int c, uint64_t first) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    uint64_t x = lane < W ? first : 0ull;  // (word `lane` of the mask, loaded by the caller)
    for (int w0 = 0; w0 < W; w0 += 64) {
        if (w0) {
            const int w = w0 + lane;
            x = w < W ? gload(selm + w) : 0ull;
        }
        const int incl = wave_scan_i32((int)__popcll(x));  // inclusive prefix of the words' counts
        const uint64_t hit = __ballot(base + incl > c);
        if (hit) {
            const int q = (int)__builtin_ctzll(hit);  // wave-uniform: read lane q directly
            uint64_t y = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), q) << 32) |
                         (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, q);
            int k = c - (base + __builtin_amdgcn_readlane(incl, q) - (int)__popcll(y));  // rank within the word
            int pos = 0;
#pragma unroll
            for (int h = 32; h > 0; h >>= 1) {  // the k-th set bit of y
                const uint64_t low = (1ull << h) - 1ull;
                const int n = (int)__popcll(y & low);
                if (k >= n) {
                    k -= n;
                    y >>= h;
                    pos += h;
                } else {
                    y &= low;
                }
            }
            return (w0 + q) * 64 + pos;
        }
        base += __builtin_amdgcn_readlane(incl, 63);
    }
    return 0;  // fewer than c + 1 survivors: not reached
}

// ---------------------------------------------------------------------------
// k_design: one workgroup per design.
//   INIT       random genome (design 0: best-CAI codons), genPopulation,
//              utils.cuh:1047-1104, then evaluation into buffer 0
//   EVAL       evaluation of genome[0][d] (synonym indices) into buffer 0
//   OFFSPRING  survivor copy, mutation, evaluation (mutationKernel)
// A design's genome row is m CDS rows of codon codes, of stride Ls; it moves
// between HBM and LDS in 16-byte words.  item_base of INIT: 1 when the pool
// has not been written yet (rows N .. 2N-1 are then set to every codon's first
// synonym).
// ---------------------------------------------------------------------------
template <int MODE, int NT, int WAVES>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WAVES))) void k_design(const DevJob *__restrict__ jobs, const int2 *__restrict__ items,
                                                uint2 *__restrict__ stem_list, int32_t *stem_ctl, int stem_group,
                                                int stem_cap, int item_base) {
    extern __shared__ __align__(16) uint8_t dyn[];
    __shared__ DesignShared<NT / 64> sh;
    const int2 it = items[blockIdx.x];
    const DevJob &J = jobs[it.x];
    const int L = J.L, m = J.m, Ls = J.Ls, N = J.N;
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G16 = (m * Ls) >> 4;  // 16-byte words of a design row
    const int64_t *lw6 = (const int64_t *)dyn;
    const uint64_t *syn6 = (const uint64_t *)(dyn + DL_SYN);
    uint8_t *rows = dyn + DL_ROWS;
    CdsStat *cst = (CdsStat *)(rows + m * Ls);
    uint32_t *const chg = (uint32_t *)(cst + m);
    const int CW = sk_mask_words(L), npair = m * (m - 1) / 2;

    // The descriptor fields of the staging phase, read before its stores (a
    // store through a pool pointer could alias the descriptor as far as the
    // compiler knows, and would make every later field a reload).
    int8_t *const genome0 = J.genome[0], *const genome1 = J.genome[1];
    float *const obj0 = J.obj[0], *const obj1 = J.obj[1];
    int8_t *const oidx0 = J.oidx[0], *const oidx1 = J.oidx[1];
    int32_t *const pql0 = J.pql[0], *const pql1 = J.pql[1];
    CdsStat *const cst0 = J.cst[0], *const cst1 = J.cst[1];
    int32_t *const hdp0 = J.hdp[0], *const hdp1 = J.hdp[1];
    int32_t *const np = J.np;
    SelAcc *const acc = J.acc;
    // Every load of the set-up is issued before the first LDS store (a store
    // under a branch would wait for its own load first): the two tables (the
    // log weights, then the synonym words: 128 8-byte words together), the
    // generation counter and the first words of the survivor mask.
    const int64_t *p_tab = J.lw6;
    const uint64_t *p_sel = J.selm;
    const SelState *p_st = J.st;
    int W = J.W;
    asm volatile("" : "+s"(p_tab), "+s"(p_sel), "+s"(p_st), "+s"(W));
    int64_t v_tab = gload(p_tab + (tid & 127));
    uint32_t g0 = 0;
    uint64_t sel0 = 0;
    if (MODE == 2) {
        g0 = gload(&p_st->gen);
        sel0 = gload(p_sel + min(lane, W - 1));
    }
    // (taken here, so that no load is moved into the branches below)
    asm volatile("" : "+v"(v_tab), "+v"(sel0));
    if (tid < 128) ((int64_t *)dyn)[tid] = v_tab;
    if (tid < MAX_M) sh.dirty[tid] = (MODE != 2);
    for (int i = tid; i < m * CW; i += NT) chg[i] = 0u;
    uint32_t gen = 0;
    int dst = 0, out_slot = it.y, src = 0, parent = 0;
    if (MODE == 2) {
        gen = __builtin_amdgcn_readfirstlane(g0);
        src = (int)(gen & 1u);
        dst = src ^ 1;
        out_slot = N + it.y;
        parent = survivor_at(p_sel, W, it.y, sel0);
    }
    u32x4 *rows4 = (u32x4 *)rows;
    if (MODE == 0) {
        const int d = it.y;
        const uint8_t *const pos = J.pos, *const ctab = J.code;
        uint8_t *const base = (uint8_t *)genome0 + (size_t)(N + d) * m * Ls;
        for (int c = 0; c < m; ++c)
            for (int k = tid; k < Ls; k += NT) {
                int v = 0, first = 0;
                if (k < L) {
                    const int g = (int)gload(pos + k), ns = (int)gload(pos + Ls + k);
                    int s = ns - 1;
                    if (d != 0) {
                        uint32_t r[4];
                        philox(0u, (uint32_t)d, (uint32_t)(c * L + k), TAG_INIT, J.seed, r);
                        s = (int)uniform_int(r[0], (uint32_t)ns);
                    }
                    v = (int)gload(ctab + g + s);
                    first = (int)gload(ctab + g);
                }
                rows[c * Ls + k] = (uint8_t)v;
                if (item_base && N + d < J.P) gstore(base + c * Ls + k, (uint8_t)first);
            }
    } else if (MODE == 1) {
        // synonym indices to codes, four a word; the padding positions are
        // forced to code 0
        const uint8_t *const pos = J.pos, *const ctab = J.code;
        const uint32_t *sg = (const uint32_t *)genome0;  // rows of L bytes, packed, in the caller's pinned memory; it has a word past them
        const int nwd = Ls >> 2;
        uint32_t *c4 = (uint32_t *)rows;
        for (int c = 0; c < m; ++c)
            for (int q = tid; q < nwd; q += NT) {
                const int left = L - 4 * q;  // positions of the word below L
                const uint32_t keep = left >= 4 ? ~0u : (left <= 0 ? 0u : (1u << (8 * left)) - 1u);
                const size_t at = ((size_t)it.y * m + c) * L + (left > 0 ? 4 * q : 0);
                // (the next word is the next lane's; only the wave's and the
                // row's last lane read it: the rows come over the link)
                const uint32_t s0 = gload(sg + (at >> 2));
                uint32_t s1 = __shfl_down(s0, 1, 64);
                if (lane == 63 || left <= 4) s1 = gload(sg + (at >> 2) + 1);
                const uint32_t sw = __builtin_amdgcn_alignbyte(s1, s0, (uint32_t)at & 3u);
                const uint32_t g = (sw & keep) + gload((const uint32_t *)pos + q);  // bytewise
                uint32_t code = 0;
#pragma unroll
                for (int b = 0; b < 4; ++b) code |= (uint32_t)gload(ctab + ((g >> (8 * b)) & 0x3Fu)) << (8 * b);
                c4[c * nwd + q] = code & keep;
            }
    } else {
        const int c = it.y;
        // the survivor copy (copySolution, utils.cuh:1106-1147): every load
        // is issued before the stores, at clamped indices
        const float *const obj_s = src ? obj1 : obj0;
        float *const obj_d = src ? obj0 : obj1;
        const int8_t *const oidx_s = src ? oidx1 : oidx0;
        int8_t *const oidx_d = src ? oidx0 : oidx1;
        const int32_t *const pql_s = src ? pql1 : pql0;
        int32_t *const pql_d = src ? pql0 : pql1;
        const CdsStat *const cst_s = src ? cst1 : cst0;
        CdsStat *const cst_d = src ? cst0 : cst1;
        const int32_t *const hdp_s = src ? hdp1 : hdp0;
        int32_t *const hdp_d = src ? hdp0 : hdp1;
        const u32x4 *pg = (const u32x4 *)((src ? genome1 : genome0) + (size_t)parent * m * Ls);
        u32x4 *sg = (u32x4 *)((dst ? genome1 : genome0) + (size_t)c * m * Ls);
        // the records' loads first (lanes of wave 0), then the genome row's
        float vo = 0.f;
        int8_t vi = 0;
        int32_t vp = 0;
        CdsStat cs{};
        int32_t vh = 0;
        const int hp = tid - 64;  // lanes 64 .. 64 + npair - 1: the pairs' distances
        if (hp >= 0 && hp < npair) vh = gload(hdp_s + (size_t)parent * npair + hp);
        if (tid < 16) {
            vo = gload(obj_s + (size_t)parent * NOBJ + min(tid, NOBJ - 1));
            vi = gload(oidx_s + (size_t)parent * 2 * NOBJ + min(tid, 2 * NOBJ - 1));
            vp = gload(pql_s + (size_t)parent * 4 + min(tid, 3));
            cs = gload_stat(cst_s + (size_t)parent * m + min(tid, m - 1));
        }
        for (int i0 = tid; i0 < G16; i0 += 4 * NT) {
            u32x4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = gload(pg + min(i0 + u * NT, G16 - 1));
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (i0 + u * NT < G16) {
                    gstore(sg + i0 + u * NT, v[u]);
                    rows4[i0 + u * NT] = v[u];
                }
        }
        if (tid < 16) {
            if (tid < NOBJ) {
                gstore(obj_d + (size_t)c * NOBJ + tid, vo);
                sh.pobj[tid] = vo;
            }
            if (tid < 2 * NOBJ) {
                gstore(oidx_d + (size_t)c * 2 * NOBJ + tid, vi);
                sh.pidx[tid] = vi;
            }
            if (tid < 4) {
                gstore(pql_d + (size_t)c * 4 + tid, vp);
                sh.ppql[tid] = vp;
            }
            if (tid < m) {
                cs.pad = 0;
                gstore_stat(cst_d + (size_t)c * m + tid, cs);
                cst[tid] = cs;
            }
        }
        if (hp >= 0 && hp < npair) {
            gstore(hdp_d + (size_t)c * npair + hp, vh);
            sh.hd[hp] = vh;
        }
        if (tid == NT - 1) {  // the sort of this generation starts from cleared counts
            gstore(np + c, 0);
            gstore(np + N + c, 0);
        }
        if (c == 0 && tid < ACC_WORDS) gstore((uint32_t *)acc + tid, acc_clear_word(tid));
        clear_niche(J, c * NT + tid, N * NT);  // (and the association from cleared niche arrays)
    }
    lds_barrier();  // tables, genome row and records
    if (MODE == 2) {
        const int c = it.y;
        uint32_t r[4];
        philox(gen, (uint32_t)c, 0u, TAG_TYPE, J.seed, r);
        const int type = (int)uniform_int(r[0], (uint32_t)(NOBJ + 1));  // main.cu:172-178
        const MutArgs A{&J, syn6, rows, chg, Ls, CW, gen, (uint32_t)c};
        switch (type) {  // main.cu:181-211
        case 0: mut_random(A, sh.dirty); break;
        case 1: mut_cai(A, sh.pidx[0], sh.dirty); break;
        case 2: mut_cbp(A, sh.pidx[2], sh.dirty, sh.hitq[wid]); break;
        case 3: mut_hsc(A, sh.pidx[4], sh.dirty, sh.hitq[wid]); break;
        case 4: mut_hd(A, sh.pidx[6], sh.pidx[7], sh.dirty, sh.hitq[wid]); break;
        case 5:
            if (sh.pidx[9] == GC_UP || sh.pidx[9] == GC_DOWN)
                mut_gc3(A, sh.pidx[8], sh.pidx[9], sh.pobj[4], sh.dirty, sh.hitq[wid]);
            break;
        default:
            if (wid == 0) mut_sl(A, sh, sh.dirty);
            break;
        }
        lds_barrier();
    }
    const uint32_t dmask = (uint32_t)__ballot(lane < m && sh.dirty[min(lane, MAX_M - 1)] != 0);
    // the design's genome row is final: its stores drain during the evaluation
    if (MODE != 1) {
        u32x4 *og = (u32x4 *)((dst ? genome1 : genome0) + (size_t)out_slot * m * Ls);
        for (int i = tid; i < G16; i += NT) gstore(og + i, rows4[i]);
    }
    design_tasks(J, lw6, (const uint32_t *)rows, dmask, MODE == 2, chg, cst, sh,
                 J.planes + (size_t)out_slot * m * plane_words(L), wid, NT / 64);
    lds_barrier();
    if (wid == 0)
        design_objectives(J, cst, sh, (dst ? obj1 : obj0) + (size_t)out_slot * NOBJ,
                          (dst ? oidx1 : oidx0) + (size_t)out_slot * 2 * NOBJ);
    if (tid >= NT - 128) {  // the records, by the wave(s) before the last lane's work below
        const int t = tid - (NT - 128);
        if (t < m) gstore_stat((dst ? cst1 : cst0) + (size_t)out_slot * m + t, cst[t]);
        if (t < npair) gstore((dst ? hdp1 : hdp0) + (size_t)out_slot * npair + t, sh.hd[t]);
    }
    // the unchanged CDS's longest stem; the changed CDS for k_stem_list
    if (wid == NT / 64 - 1) {
        const int l = lane < m && !((dmask >> lane) & 1u) ? cst[lane].l : 0;
        const int lmax = wave_max_nonneg(l);
        if (lane == 0) gstore(J.stem_max + out_slot, lmax);  // (k_dominance counts the offspring's changed CDS)
        if (MODE == MODE_OFFSPRING && dmask && stem_cap) {  // in the child's sublist
            const int item = item_base + (int)blockIdx.x, k = item / stem_group;
            int e = 0;
            if (lane == 0) e = atomicAdd(stem_ctl + k, (int)__popc(dmask));
            e = __builtin_amdgcn_readfirstlane(e) + (int)__popc(dmask & ((1u << (lane & 31)) - 1u));
            if (lane < m && ((dmask >> lane) & 1u) && e < stem_cap)
                gstore((uint64_t *)(stem_list + (size_t)k * stem_cap + e),
                       stem_entry((uint32_t)it.x, (uint32_t)it.y, (uint32_t)lane, (uint32_t)dst));
        }
    }
}

// `words` 16-byte words from the host's pinned memory to the device: what a call
// sets up, some 60 KB, where the copy engine's hand-over to the first kernel
// takes longer than the transfer.
__global__ __launch_bounds__(256) void k_fetch(u32x4 *__restrict__ dst, const u32x4 *__restrict__ src, uint32_t words) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < words) gstore(dst + i, gload(src + i));
}

// What a caller reads of a job, written straight to the host's pinned memory:
// the first gblocks workgroups convert `bytes` bytes from byte `first` on (both
// multiples of 16, or the last) of the pool's packed synonym indices, 16 a
// thread, to `rows`; the others copy the selection state, survivor mask,
// fronts, objectives, their indices and stem positions, word by word, to
// `rest` (ReadRest).  The buffer comes from the generation counter
// here, so nothing is read back before.  Bound by the link: 200 x 2 CDS of
// 351 codons with their records in one launch and one wait, 60 us a call;
// a copy for each array and one for the counter, 186 us.
__global__ __launch_bounds__(256) void k_read(const DevJob *__restrict__ jobs, uint8_t *__restrict__ rows, uint32_t *__restrict__ rest,
                                              uint64_t first, uint64_t bytes, uint32_t gblocks) {
    __shared__ uint8_t own[64];
    const DevJob &J = jobs[0];
    const int b = (int)(gload(&J.st->gen) & 1u);
    if (blockIdx.x >= gblocks) {
        const uint32_t P = (uint32_t)J.P, t = (blockIdx.x - gblocks) * 256 + threadIdx.x;
        const uint32_t ends[6] = {(uint32_t)(sizeof(SelState) / 4), 2u * (uint32_t)J.W, P, 6 * P, 3 * P, 4 * P};
        const uint32_t *from[6] = {(const uint32_t *)J.st, (const uint32_t *)J.selm, (const uint32_t *)J.front_of,
                                   (const uint32_t *)(b ? J.obj[1] : J.obj[0]), (const uint32_t *)(b ? J.oidx[1] : J.oidx[0]),
                                   (const uint32_t *)(b ? J.pql[1] : J.pql[0])};
        uint32_t at = t;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            if (at < ends[k]) {
                gstore(rest + t, gload(from[k] + at));
                return;
            }
            at -= ends[k];
        }
        return;
    }
    const uint32_t L = (uint32_t)J.L, Ls = (uint32_t)J.Ls;
    const uint8_t *const src = (const uint8_t *)(b ? J.genome[1] : J.genome[0]);
    const uint64_t *syn = (const uint64_t *)(J.lw6 + 64);
    if (threadIdx.x < 64) own[threadIdx.x] = (uint8_t)SynWord(gload(syn + threadIdx.x)).own();
    __syncthreads();
    const uint64_t at = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 16;
    if (at >= bytes) return;
    uint64_t r = (first + at) / L;
    uint32_t k = (uint32_t)(first + at - r * L);
    const uint8_t *p = src + r * Ls + k;
    u32x4 v = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (at + i < bytes) v[i >> 2] |= (uint32_t)own[gload(p) & 63] << (8 * (i & 3));
        ++p;
        if (++k == L) {
            k = 0;
            p += Ls - L;
        }
    }
    gstore((u32x4 *)(rows + at), v);  // (room for whole 16-byte words)
}

// ---------------------------------------------------------------------------
// k_stem (initialisation and evaluation): one workgroup per (work item, CDS),
// blockIdx.x = item * mg + c with mg the largest m of the jobs launched: a
// word search at a guessed length (sk_blind_k).  k_stem_finish decodes the key.
// 128 threads and 1024 chains a CDS where there are many, 256 and 2048 where the
// latency of one counts (STEM_FEW).  8192 CDS of 1503 bases: 24.7 us; by the tiles
// of the match matrix 216.
// ---------------------------------------------------------------------------
template <int NT, int HEADS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8))) void k_stem(const DevJob *__restrict__ jobs, const int2 *__restrict__ items, int mg) {
    extern __shared__ __align__(16) uint8_t dyn[];
    __shared__ uint64_t redu[16];
    __shared__ int32_t flag[NT / 64];
    const int2 it = items[blockIdx.x / (unsigned)mg];
    const int c = (int)(blockIdx.x % (unsigned)mg);
    const DevJob &J = jobs[it.x];
    const int L = J.L, m = J.m, n = 3 * L, wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (c >= m) return;
    const size_t rec = (size_t)it.y * m + c;  // (the designs are in buffer 0)
    CdsStat *cs = J.cst[0] + rec;
    uint64_t *planes = (uint64_t *)dyn;
    const PlaneLoad<NT> load((const uint64_t *)(J.planes + rec * plane_words(L)), L);
    load.place(planes);
    const SeekLds S = seek_lds<HEADS>(dyn + stem_index_at(L), n, wid, nullptr);
    seek_clear<NT, HEADS>(S);
    lds_barrier();
    const uint2 *sp = (const uint2 *)planes;
    const uint64_t key = seek_cds<NT, HEADS>(S, sp, sp + scan_words(n), n, L, false, 0, 0, 0, redu, flag);
    if (threadIdx.x == 0) gstore(&cs->key, key);
}

// ---------------------------------------------------------------------------
// The stem of child `child`'s CDS c (offspring generations): the parent's stem
// (it stands in the child's record) and the change mask decide the search
// (seek_cds).  The key goes into the CDS record and the length into the
// design's longest stem (stem_max) with an atomic maximum.  buf: the buffer
// the child is in, or -1: take it from the generation counter, and leave a
// CDS that did not change alone.
// ---------------------------------------------------------------------------
template <int NT, int HEADS>
__device__ __forceinline__ void stem_child(const DevJob &J, int child, int c, int buf, uint8_t *dyn, uint64_t *redu, int32_t *flag) {
    // The descriptor fields first, held in scalar registers; then the record
    // (of both buffers while the counter is on its way), the planes and the
    // mask, loaded together.  The child sits at slot N + child of the next
    // buffer, (gen + 1) & 1.
    const SelState *p_st = J.st;
    CdsStat *cs0 = J.cst[0], *cs1 = J.cst[1];
    const uint2 *p_pl = J.planes;
    int32_t *p_sm = J.stem_max;
    int L = J.L, m = J.m, N = J.N;
    asm volatile("" : "+s"(p_st), "+s"(cs0), "+s"(cs1), "+s"(p_pl), "+s"(p_sm), "+s"(L), "+s"(m), "+s"(N));
    if (buf < 0 && c >= m) return;
    const int n = 3 * L, slot = N + child, tid = (int)threadIdx.x;
    const size_t rec = (size_t)slot * m + c;
    CdsStat *cs = (buf > 0 ? cs1 : cs0) + rec;
    const int32_t *r0 = (const int32_t *)cs;
    int pl = gload(r0 + 6), pp = gload(r0 + 7), pq = gload(r0 + 8), fresh = 1;  // CdsStat::l, p, q
    uint32_t gen = 0;
    int l1 = 0, p1 = 0, q1 = 0, f1 = 0;
    if (buf < 0) {
        gen = gload(&p_st->gen);
        const int32_t *r1 = (const int32_t *)(cs1 + rec);
        fresh = gload(r0 + 9);  // CdsStat::pad
        l1 = gload(r1 + 6), p1 = gload(r1 + 7), q1 = gload(r1 + 8), f1 = gload(r1 + 9);
    }
    const PlaneLoad<NT> load((const uint64_t *)(p_pl + rec * plane_words(L)), L);
    if (buf < 0 && !(__builtin_amdgcn_readfirstlane(gen) & 1u)) {
        cs = cs1 + rec;
        pl = l1, pp = p1, pq = q1, fresh = f1;
    }
    if (__builtin_amdgcn_readfirstlane(fresh) == 0) return;
    uint64_t *planes = (uint64_t *)dyn;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const SeekLds S = seek_lds<HEADS>(dyn + stem_index_at(L), n, wid, (const uint32_t *)(planes + 2 * scan_words(n)));
    if (buf >= 0) lds_barrier();  // the previous entry's LDS is no longer read
    seek_clear<NT, HEADS>(S);
    load.place(planes);
    lds_barrier();
    const uint2 *sp = (const uint2 *)planes;
    const uint64_t key = seek_cds<NT, HEADS>(S, sp, sp + scan_words(n), n, L, true, pl, pp, pq, redu, flag);
    if (tid == 0) {
        gstore(&cs->key, key);
        if (key) atomicMax(&p_sm[slot], (int)(key >> 40));
    }
}

// k_stem_each: a workgroup per CDS of the children, for small launches: the
// unchanged CDS leave after their record, and k_design does not wait for the
// list's counters at its end.  Against the list: 128 children of 202 codons
// 39.2 -> 38.2 us a generation, 777 of 6190 75.2 -> 74.2, 1024 of 2004
// 67.7 -> 62.0 (k_design 25.8 -> 21.1); 4096 of 12008 (32768 CDS) 240.0 ->
// 241.7; the 64-job mix 835 -> 1208, mostly empty workgroups.
template <int NT, int HEADS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8))) void k_stem_each(
    const DevJob *__restrict__ jobs, const int2 *__restrict__ items, int mg) {
    extern __shared__ __align__(16) uint8_t dyn[];
    __shared__ uint64_t redu[16];
    __shared__ int32_t flag[NT / 64];
    const int2 it = items[blockIdx.x / (unsigned)mg];
    stem_child<NT, HEADS>(jobs[it.x], it.y, (int)(blockIdx.x % (unsigned)mg), -1, dyn, redu, flag);
}

// ---------------------------------------------------------------------------
// k_stem_list (offspring generations): the changed CDS k_design listed
// (stem_entry), in `groups` sublists of cap entries with their counts in ctl;
// the entries are numbered sublist by sublist (a prefix sum of the counts),
// which keeps the children list's order, and gridDim.x workgroups of NT threads
// take them round-robin, one CDS a workgroup at a time (stem_child).
// k_dominance clears ctl for the next generation.
// Bound by the searches resident per CU (LDS) and their chain of lookups: the
// scans of the tiles that this search replaced took 502 us on the 64-job mix
// (now 326), 130 us for 4096 children of 12 008 codons (69), 32 us for 777 of
// 6190 (21).
// ---------------------------------------------------------------------------
template <int NT, int HEADS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8))) void k_stem_list(
    const DevJob *__restrict__ jobs, const uint2 *__restrict__ list, const int32_t *__restrict__ ctl, int groups, int cap) {
    extern __shared__ __align__(16) uint8_t dyn[];
    __shared__ uint64_t redu[16];
    __shared__ int32_t flag[NT / 64];
    const int G = (int)gridDim.x, lane = (int)threadIdx.x & 63;
    // Up to 64 sublists (4096 children at 64 each): every wave scans their
    // counts in registers, and the workgroup's entries are fetched one ahead
    // of the one being searched, so no barrier stands before the first search.
    // More: the prefix sums sit where the planes go -- built before each chunk
    // of 64 entries is fetched, overwritten by the planes after -- and are
    // built again only when the workgroup has entries past its first chunk.
    const bool few = groups <= 64;
    int *pre = (int *)dyn;  // [groups + 1]
    __shared__ int red[16], s_carry;
    __shared__ uint64_t s_ent[64];  // the workgroup's next entries, fetched together
    int incl = 0, count = 0, e = (int)blockIdx.x, j = 0;
    uint64_t nxt = 0;
    auto fetch = [&](int q) -> uint64_t {  // entry q of the list (few; q is the same in every lane)
        const int k = (int)__popcll(__ballot(incl <= q));
        const int first = k ? __builtin_amdgcn_readlane(incl, k - 1) : 0;
        return gload((const uint64_t *)(list + (size_t)k * cap + (q - first)));
    };
    if (few) {
        incl = wave_scan_i32(lane < groups ? min(gload(ctl + lane), cap) : 0);
        count = __builtin_amdgcn_readlane(incl, 63);
        if (e < count) nxt = fetch(e);
    }
    for (bool start = true;; start = false, e += G) {
        uint64_t ent;
        if (few) {
            if (e >= count) break;
            ent = nxt;
            if (e + G < count) nxt = fetch(e + G);
        } else {
            if (!start && e >= count) break;
            if (start || j == 64) {
                __syncthreads();  // the previous entries' planes are no longer read
                if (threadIdx.x == 0) s_carry = 0;
                for (int g0 = 0; g0 < groups; g0 += blockDim.x) {  // exclusive prefix of the counts
                    const int g = g0 + (int)threadIdx.x;
                    const int n = g < groups ? min(gload(ctl + g), cap) : 0;
                    int total;
                    const int ex = block_scan_excl(n, red, &total);
                    if (g < groups) pre[g] = s_carry + ex;
                    __syncthreads();
                    if (threadIdx.x == 0) s_carry += total;
                    __syncthreads();
                }
                if (threadIdx.x == 0) pre[groups] = s_carry;
                __syncthreads();
                count = pre[groups];
                if (e >= count) break;
                const int q = e + (int)threadIdx.x * G;
                if (threadIdx.x < 64 && q < count) {
                    int k = 0;  // the last sublist whose entries start at or before q
                    for (int h = STEM_MAX_GROUPS / 2; h > 0; h >>= 1)
                        if (k + h < groups && pre[k + h] <= q) k += h;
                    s_ent[threadIdx.x] = gload((const uint64_t *)(list + (size_t)k * cap + (q - pre[k])));
                }
                j = 0;
                __syncthreads();
            }
            ent = s_ent[j++];
        }
        {
            // (wave-uniform: the descriptor comes by scalar loads)
            const uint32_t ex = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)ent);
            const uint32_t ey = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(ent >> 32));
            stem_child<NT, HEADS>(jobs[ey >> 1], (int)(ex >> 4), (int)(ex & 15u), (int)(ey & 1u), dyn, redu, flag);
        }
    }
}

// Objective 5 of a design: the longest stem over its CDS, ties to the last
// CDS (calMaximumSL's obj5 = l / ((3L-4)/2), utils.cuh:880).  Stores the
// stems k_stem found and clears the marks k_design left.
__device__ int stem_finish_at(CdsStat *cst, float *obj, int8_t *oidx, int32_t *pql, int m, int den_sl, int slot) {
    // a record's 16-byte words 1 (hsc, gc3, l, p) and 2 (q, pad, key), four
    // records' loads issued together
    u32x4 *cs = (u32x4 *)(cst + (size_t)slot * m);
    int bl = 0, bp = 0, bq = 0, bc = m - 1, changed = 0;
    for (int c0 = 0; c0 < m; c0 += 4) {
        u32x4 w1[4], w2[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = min(c0 + u, m - 1);
            w1[u] = gload(cs + 4 * c + 1);
            w2[u] = gload(cs + 4 * c + 2);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = c0 + u;
            if (c >= m) break;
            int l = (int)w1[u].z, p = (int)w1[u].w, q = (int)w2[u].x;
            if (w2[u].y) {  // pad: the stem k_stem found
                stem_unkey((uint64_t)w2[u].z | ((uint64_t)w2[u].w << 32), l, p, q);
                w1[u].z = (uint32_t)l;
                w1[u].w = (uint32_t)p;
                w2[u].x = (uint32_t)q;
                w2[u].y = 0u;
                gstore(cs + 4 * c + 1, w1[u]);
                gstore(cs + 4 * c + 2, w2[u]);
                ++changed;
            }
            if (l >= bl) {
                bl = l;
                bp = p;
                bq = q;
                bc = c;
            }
        }
    }
    gstore(obj + (size_t)slot * NOBJ + 5, (float)bl / (float)den_sl);
    gstore(oidx + (size_t)slot * 2 * NOBJ + 10, (int8_t)bc);
    int32_t *pq = pql + (size_t)slot * 4;
    gstore(pq, bp);
    gstore(pq + 1, bq);
    gstore(pq + 2, bl);
    gstore(pq + 3, 0);
    return changed;
}

// stem_finish_at for every work item's design (initialisation and evaluation,
// in buffer 0; the offspring generation leaves it to k_dominance).
__global__ __launch_bounds__(256) void k_stem_finish(const DevJob *__restrict__ jobs, const int2 *__restrict__ items,
                                                     int n_items) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_items) return;
    const int2 it = items[i];
    const DevJob &J = jobs[it.x];
    stem_finish_at(J.cst[0], J.obj[0], J.oidx[0], J.pql[0], J.m, J.den_sl, it.y);
}

// ---------------------------------------------------------------------------
// Selection
// ---------------------------------------------------------------------------
// The objectives of the pool, buffer (gen + 1) & 1.  Both buffers' pointers
// are read from the descriptor before the choice and held in scalar
// registers, so that the rows' loads wait for the generation counter only,
// not for a further descriptor load at an offset the counter decides.
__device__ __forceinline__ const float *pool_obj(const DevJob &J, uint32_t gen) {
    const float *o0 = J.obj[0], *o1 = J.obj[1];
    asm volatile("" : "+s"(o0), "+s"(o1));
    return (gen & 1u) ? o0 : o1;
}

// The pool's extrema over rows row0 .. row0 + rows - 1 (updateIdealValue /
// updateWorstValue, sorting.cuh:132-426; fminf / fmaxf from FLT_MAX /
// -FLT_MAX), folded into the job's accumulators with one atomic minimum and
// maximum per objective.  One wave; `vals` holds the rows' objectives.
__device__ void pool_extrema(const DevJob &J, int row0, int rows, const float *vals) {
    const int lane = threadIdx.x & 63, P = J.P;
    float mn[NOBJ], mx[NOBJ];
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        mn[k] = FLT_MAX;
        mx[k] = -FLT_MAX;
    }
    for (int t = lane; t < rows && row0 + t < P; t += 64)
#pragma unroll
        for (int k = 0; k < NOBJ; ++k) {
            const float v = vals[t * NOBJ + k];
            mn[k] = fminf(mn[k], v);
            mx[k] = fmaxf(mx[k], v);
        }
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        mn[k] = wave_min_f32(mn[k]);
        mx[k] = wave_max_f32(mx[k]);
    }
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NOBJ; ++k) {
            atomicMin(&J.acc->lo[k], ord_bits(mn[k]));
            atomicMax(&J.acc->hi[k], ord_bits(mx[k]));
        }
}

// The column designs of a wave (cand: the lane's) against WR rows in LDS:
// amask[q] is the word of the lanes that dominate row q, the returned word's
// bit q says that row q dominates the lane's design.
template <int WR>
__device__ __forceinline__ uint64_t dominance_rows(const float *rw, const float *cand, uint64_t *amask) {
    const int lane = threadIdx.x & 63;
    uint64_t col = 0;
#pragma unroll 1
    for (int q0 = 0; q0 < WR; q0 += 16) {  // 16 rows at a time, last row first
        uint32_t c16 = 0;
        uint64_t am[16];  // (wave-uniform: scalar registers)
#pragma unroll
        for (int u = 15; u >= 0; --u) {
            const float *const row = rw + (q0 + u) * NOBJ;
            float hi = cand[0] - row[0], lo = hi;  // (a NaN difference is never significant)
#pragma unroll
            for (int k = 1; k < NOBJ; ++k) {
                const float d = cand[k] - row[k];
                hi = fmaxf(hi, d);
                lo = fminf(lo, d);
            }
            // the lanes whose design has a difference above the precision
            // and those with one below minus the precision (wave-uniform
            // masks); design i dominates the row when only the second holds
            // (the lanes past the pool hold +inf, so the first), and the row
            // dominates design i when only the first holds
            const uint64_t U = __builtin_amdgcn_ballot_w64(hi > F_PRECISION);
            const uint64_t D = __builtin_amdgcn_ballot_w64(lo < -F_PRECISION);
            am[u] = D & ~U;
            c16 = c16 + c16 + (uint32_t)__builtin_amdgcn_inverse_ballot_w64(U & ~D);
        }
        if (lane == 0)
#pragma unroll
            for (int u = 0; u < 16; ++u) amask[q0 + u] = am[u];
        col |= (uint64_t)c16 << q0;
    }
    __builtin_amdgcn_wave_barrier();
    return col;
}

// Bit t of word w of row j is set when design 64w + t dominates design j;
// the matrix is stored word-major, dom[w * P + j], so that the front peeling
// reads one word of consecutive rows per wave.  np[j] counts the dominators.
//
// dominate() (sorting.cuh:94-130) compares |a - b| against the precision
// and the sign of a - b;
// with d = a - b per objective, a dominates b exactly when no d exceeds the
// precision and some d is below minus the precision, and b dominates a
// exactly when the reverse holds (b - a is the negation of a - b, bit for
// bit).  One difference per objective therefore decides both directions,
// and the pool is split into 64 x 64 tiles of (row block b, column block w)
// with b <= w only: item = (job, 64b, w, 0).  Lane t holds column design
// 64w + t.  A tile writes the words of block w of its rows (the ballot of
// its column designs against each row) and, off the diagonal, the words of
// block b of its column designs (each lane gathers one bit per row).  ROWS/64
// tiles per workgroup of four waves, ROWS/4 rows of a tile per wave; the
// partial column words of a tile's waves are combined in LDS.  The diagonal
// tile of a row block also finishes its children's stem records (offspring
// generation) and folds its rows into the pool's extrema.
template <int ROWS>
__global__ __launch_bounds__(256) void k_dominance(const DevJob *__restrict__ jobs, const int4 *__restrict__ items,
                                                   int n_items, bool finish, int32_t *stem_ctl, int ctl_n) {
    static_assert(ROWS == 64 || ROWS == 128 || ROWS == 256, "one, two or four tiles per workgroup");
    constexpr int TPW = ROWS / 64;  // tiles per workgroup
    constexpr int G = 4 / TPW;      // waves per tile
    constexpr int WR = 64 / G;      // rows of a tile per wave
    __shared__ float rows[TPW][64 * NOBJ];
    __shared__ uint64_t part[TPW][G][64];
    __shared__ uint64_t amask[4][WR];  // per wave: the word of block wc of each of its rows
    if (stem_ctl && blockIdx.x == 0)  // k_stem_list has read the counts
        for (int g = threadIdx.x; g < ctl_n; g += blockDim.x) gstore(stem_ctl + g, 0);
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), tl = wv / G, sub = wv % G;
    const int idx = (int)blockIdx.x * TPW + tl;
    const bool have = idx < n_items;  // (the last workgroup may hold fewer tiles)
    const int4 it = items[min(idx, n_items - 1)];
    const DevJob &J = jobs[it.x];
    const int P = J.P, N = J.N, r0 = it.y, wc = it.z, c0 = 64 * wc;
    const bool diag = r0 == c0;
    // the generation counter's load issued, then the descriptor fields read
    // (held in scalar registers: no load waits for the counter's value)
    const uint32_t g0 = gload(&J.st->gen);
    float *o0 = J.obj[0], *o1 = J.obj[1];
    const int32_t *smax = J.stem_max;
    int den = J.den_sl;
    asm volatile("" : "+s"(o0), "+s"(o1), "+s"(smax), "+s"(den));
    // (and those of the stem records' completion below)
    CdsStat *cs0 = J.cst[0], *cs1 = J.cst[1];
    int8_t *oi0 = J.oidx[0], *oi1 = J.oidx[1];
    int32_t *pq0 = J.pql[0], *pq1 = J.pql[1];
    int m = J.m;
    asm volatile("" : "+s"(cs0), "+s"(cs1), "+s"(oi0), "+s"(oi1), "+s"(pq0), "+s"(pq1), "+s"(m));
    const uint32_t gen = __builtin_amdgcn_readfirstlane(g0);
    const int buf = (int)((gen + 1u) & 1u);
    float *const obj = buf ? o1 : o0;
    // (a sort alone has no stem maxima: its loads read the objectives
    // instead, so that they need no branch and issue with the rows')
    if (!finish) smax = (const int32_t *)obj;
    const float den_sl = (float)den;
    // In the offspring generation a child's objective 5 is its longest stem
    // over (3L-4)/2, the value stem_finish stores.  The column design's row
    // and the tile row of the lane are loaded at clamped indices, all before
    // any value is used (the first wave of a tile stages the tile rows).
    const int i = c0 + lane, ic = min(i, P - 1), rr = r0 + lane, rc = min(rr, P - 1);
    float cand[NOBJ], wrow[NOBJ];
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        cand[k] = gload(obj + (size_t)ic * NOBJ + k);
        wrow[k] = gload(obj + (size_t)rc * NOBJ + k);
    }
    const int32_t csm = gload(smax + ic), rsm = gload(smax + rc);
    // the diagonal tiles complete the stem records of their children and
    // count the CDS the children recomputed (before the rows are used, so
    // that the records' loads issue while the rows' are in flight; the
    // objective 5 it stores is the value the rows take below)
    if (finish && diag && sub == 0) {
        int changed = 0;
        if (rr >= N && rr < P && have)
            changed = stem_finish_at(buf ? cs1 : cs0, obj, buf ? oi1 : oi0, buf ? pq1 : pq0, m, den, rr);
        changed = wave_sum_i32(changed);
        if (lane == 0 && changed) atomicAdd(&J.st->cds_scanned, (unsigned long long)changed);
    }
    if (finish && i >= N) cand[NOBJ - 1] = (float)csm / den_sl;
    if (finish && rr >= N) wrow[NOBJ - 1] = (float)rsm / den_sl;
    const bool cv = i < P;
    if (!cv)
#pragma unroll
        for (int k = 0; k < NOBJ; ++k) cand[k] = __builtin_inff();
    if (sub == 0) {
        // rows past the pool hold +inf: no design is dominated by them
        // (d = -inf or NaN in every objective), and their words are not
        // stored
        float *const o = rows[tl] + lane * NOBJ;
#pragma unroll
        for (int k = 0; k < NOBJ; ++k) o[k] = rr < P ? wrow[k] : __builtin_inff();
    }
    __syncthreads();
    // and fold their rows into the pool's extrema
    if (diag && have && sub == G - 1) pool_extrema(J, r0, 64, rows[tl]);
    const float *const rw = rows[tl] + sub * WR * NOBJ;
    // bit q of col: row r0 + sub*WR + q dominates design i
    uint64_t col = dominance_rows<WR>(rw, cand, amask[wv]);
    const uint64_t mine = amask[wv][min(lane, WR - 1)];  // lane q < WR: the word of row r0 + sub*WR + q
    const int r = r0 + sub * WR + lane;
    if (have && lane < WR && r < P) {
        gstore(J.dom + (size_t)wc * P + r, mine);
        if (mine) atomicAdd(&J.np[r], (int)__popcll(mine));
    }
    if (G > 1) {
        part[tl][sub][lane] = col << (sub * WR);
        lds_barrier();
        if (sub == 0)
#pragma unroll
            for (int g = 1; g < G; ++g) col |= part[tl][g][lane];
    }
    if (!diag && have && sub == 0 && cv) {
        gstore(J.dom + (size_t)(r0 >> 6) * P + i, col);
        if (col) atomicAdd(&J.np[i], (int)__popcll(col));
    }
}

// (v, id) becomes (ov, oid) when that pair is smaller: a smaller value, or
// the same value with a smaller index (a NaN value is never taken).  Written
// without short-circuit evaluation so that it compiles to selects.
__device__ __forceinline__ void argmin_pair(float &v, int &id, float ov, int oid) {
    const bool take = (ov < v) | ((ov == v) & (oid < id));
    v = take ? ov : v;
    id = take ? oid : id;
}

// argmin_pair with the pair a DPP step brings from another lane; lanes
// outside a shifted or masked row contribute (FLT_MAX, 0x7FFFFFFF), the start
// value of every lane's fold.
template <int CTRL, int ROWS>
__device__ __forceinline__ void argmin_dpp(float &v, int &id) {
    const float ov = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(FLT_MAX), __float_as_int(v), CTRL, ROWS, 0xf, false));
    const int oid = __builtin_amdgcn_update_dpp(0x7FFFFFFF, id, CTRL, ROWS, 0xf, false);
    argmin_pair(v, id, ov, oid);
}
// The smallest (value, index) pair of a full wave, wave-uniform: the smallest
// value first, then the smallest index among the lanes that hold it (one
// instruction a step each, against eight for the pair's comparison).  Values
// are never NaN; a value above FLT_MAX counts as FLT_MAX with no index, the
// start value of every lane's fold.
__device__ __forceinline__ void wave_argmin(float &v, int &id) {
    const float m = wave_min_f32(v);
    id = wave_min_i32(v == m ? id : 0x7FFFFFFF);
    v = m;
}

// The ASF values (sorting.cuh:428-449) of one design for all six axes.  The clamped differences t[k] are +0
// or at least 0.001 (or NaN, which no comparison takes), and axis a takes the
// strict running maximum of t[a] and t[k] / F_PRECISION over k != a.  A
// correctly rounded division by a positive constant is nondecreasing, so the
// largest of those quotients is the quotient of the largest t[k], k != a: the
// largest and second-largest differences give every axis with two divisions,
// the same values as dividing each difference.
__device__ __forceinline__ void asf_all(const float *x, const float *ideal, float *out) {
    float t[NOBJ];
    float m1 = -FLT_MAX, m2 = -FLT_MAX;  // largest and second-largest difference
    int k1 = -1;
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        t[k] = x[k] - ideal[k];
        if ((double)t[k] < 0.001) t[k] = 0.f;
        const bool top = t[k] > m1, second = !top && t[k] > m2;
        m2 = top ? m1 : (second ? t[k] : m2);
        m1 = top ? t[k] : m1;
        k1 = top ? k : k1;
    }
    const float q1 = m1 == -FLT_MAX ? -FLT_MAX : m1 / F_PRECISION;
    const float q2 = m2 == -FLT_MAX ? -FLT_MAX : m2 / F_PRECISION;
#pragma unroll
    for (int a = 0; a < NOBJ; ++a) {
        const float q = a == k1 ? q2 : q1;
        out[a] = t[a] > q ? t[a] : q;
    }
}

__device__ __forceinline__ unsigned long long asf_key(float v, int id) {
    return ((unsigned long long)ord_bits(v) << 32) | (uint32_t)id;
}

// Extreme points (findExtremePoints, sorting.cuh:601-683) settled axis by
// axis against the previous ones, by one wave.  The candidate rows are the
// previous extremes (0-5) and the rows of the first front's ASF minima of the
// six axes (6-11); lane t (0-11) holds row t's ASF values c[] (never NaN), pv
// and pid the first front's minimum of lane t - 6's axis (lanes 6-11).  Per
// axis the smallest value among the rows the slots (lanes 0-5) hold and the
// first front's minimum wins, ties to the first front, then to the lowest slot
// -- what the serial fold over (value, index) pairs finds, a slot's index being
// above every design's -- and its row and ASF values go to the axis's slot.
// Returns the row held by slot `lane` (lanes 0-5).
__device__ int settle_extremes(float *c, float pv, int pid) {
    const int lane = threadIdx.x & 63;
    int cur = lane;
#pragma unroll
    for (int axis = 0; axis < NOBJ; ++axis) {
        const bool slot = lane < NOBJ, first = lane == NOBJ + axis;
        const float v = slot ? c[axis] : (first ? pv : FLT_MAX);
        // lanes 0-5 and 6-11 lie in one DPP row: its smallest value in lane 15
        float m = v;
        m = fminf(m, dpp_f32<0x111, 0xf>(m, FLT_MAX));
        m = fminf(m, dpp_f32<0x112, 0xf>(m, FLT_MAX));
        m = fminf(m, dpp_f32<0x114, 0xf>(m, FLT_MAX));
        m = fminf(m, dpp_f32<0x118, 0xf>(m, FLT_MAX));
        m = lane_of(m, 15);
        if (!(m < FLT_MAX)) continue;
        const uint64_t at = __ballot(v == m && (slot || (first && pid != 0x7FFFFFFF)));
        const int win = (at >> (NOBJ + axis)) & 1ull ? NOBJ + axis : (int)__builtin_ctzll(at);
        const int held = __builtin_amdgcn_readlane(cur, win);
        if (lane == axis) cur = held;
#pragma unroll
        for (int k = axis + 1; k < NOBJ; ++k) {
            const float o = lane_of(c[k], win);
            if (lane == axis) c[k] = o;
        }
    }
    return cur;
}

// GaussianElimination (sorting.cuh:451-599, E x = 1) by one wave: lane r
// (0-5) holds row r of AB (a[6] the right-hand side) in registers and reads
// the pivot row with v_readlane; every element takes the same operations in
// the same order as the row-by-row elimination, so the solution is the same
// to the bit.  Returns x[lane] in lanes 0-5.
__device__ float gauss_wave(const float *E) {
    const int lane = threadIdx.x & 63;
    const bool row_lane = lane < NOBJ;
    const int r = row_lane ? lane : 0;
    float a[NOBJ + 1];
#pragma unroll
    for (int c = 0; c < NOBJ; ++c) a[c] = E[r * NOBJ + c];
    a[NOBJ] = 1.0f;
#pragma unroll
    for (int col = 0; col < NOBJ; ++col) {
        if (fabsf(lane_of(a[col], col)) <= 1e-6f) {  // add the first row below with a usable entry
            const uint64_t cand = __ballot(row_lane && lane > col && fabsf(a[col]) > 1e-6f);
            if (cand) {
                const int rr = (int)__builtin_ctzll(cand);
#pragma unroll
                for (int c = col; c <= NOBJ; ++c) {
                    const float add = lane_of(a[c], rr);
                    if (lane == col) a[c] += add;
                }
            }
        }
        float prow[NOBJ + 1];
#pragma unroll
        for (int c = col; c <= NOBJ; ++c) prow[c] = lane_of(a[c], col);
        if (row_lane && lane > col) {
            const float f = a[col] / prow[col];
#pragma unroll
            for (int c = col; c <= NOBJ; ++c) a[c] -= f * prow[c];
        }
    }
#pragma unroll
    for (int row = NOBJ - 1; row >= 0; --row) {
        float s = 0.f;
#pragma unroll
        for (int cc = row + 1; cc < NOBJ; ++cc) s += lane_of(a[cc], row);
        float x = lane_of(a[NOBJ], row);
        if (row != NOBJ - 1) x -= s;
        x /= lane_of(a[row], row);
        if (lane == row) {
            a[NOBJ] = x;
            a[row] = 1.0f;
        }
        if (lane < row) a[row] *= x;
    }
    return a[NOBJ];
}

// The first front (designs nobody dominates: their dominator counts are
// complete after k_dominance), one design a thread (grid: jobs x chunks of
// FRONT0_THREADS designs of the largest pool): front_of 0 or -1, the
// first-front words of the ranked mask, and the workgroup's share of the
// first front's size, its maximum per objective (updateNadirValue_MNDF,
// sorting.cuh:685-884) and its per-axis ASF minima against the ideal point
// k_dominance folded (findExtremePoints, sorting.cuh:601-683; the smallest
// value, ties to the lowest index), reduced over the workgroup and folded
// into the job's accumulators with one atomic per quantity.
__global__ __launch_bounds__(FRONT0_THREADS) void k_front0(const DevJob *__restrict__ jobs) {
    const DevJob &J = jobs[blockIdx.x];
    // the descriptor fields held in scalar registers, then the generation
    // counter, the ideal point and the dominator count loaded together (the
    // rows' loads wait for the counter alone)
    SelState *st = J.st;
    SelAcc *acc = J.acc;
    const int32_t *np = J.np;
    const float *o0 = J.obj[0], *o1 = J.obj[1];
    int P = J.P;
    asm volatile("" : "+s"(st), "+s"(acc), "+s"(np), "+s"(o0), "+s"(o1), "+s"(P));
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    constexpr int NW = FRONT0_THREADS / 64;
    const int d0 = blockIdx.y * FRONT0_THREADS;
    if (d0 >= P) return;
    const uint32_t g0 = gload(&st->gen);
    const int d = d0 + tid, dc = min(d, P - 1);
    const int npv = gload(np + dc);
    const uint32_t lo = gload(acc->lo + min(tid, NOBJ - 1));
    const uint32_t gen = __builtin_amdgcn_readfirstlane(g0);
    const float *const obj = (gen & 1u) ? o0 : o1;  // buffer (gen + 1) & 1
    float x[NOBJ];
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) x[k] = gload(obj + (size_t)dc * NOBJ + k);
    __shared__ float ideal[NOBJ], red_v[NW * 2 * NOBJ];
    __shared__ int red_i[NW * NOBJ], s_cnt;
    if (tid < NOBJ) ideal[tid] = ord_float(lo);
    if (tid == 0) s_cnt = 0;
    __syncthreads();
    const bool f0 = d < P && npv == 0;
    if (d < P) gstore(J.front_of + d, f0 ? 0 : -1);
    const uint64_t b = __ballot(f0);  // a wave's 64 designs are one word of the mask
    if (lane == 0 && d0 + 64 * wid < P) {
        gstore(J.ranked + (d0 >> 6) + wid, b);
        if (b) atomicAdd(&s_cnt, (int)__popcll(b));
    }
    float fm[NOBJ], bv[NOBJ];
    int bi[NOBJ];
    asf_all(x, ideal, bv);
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        fm[k] = f0 ? x[k] : -FLT_MAX;
        // an ASF value is never NaN: it is at least -FLT_MAX
        bi[k] = f0 ? d : 0x7FFFFFFF;
        bv[k] = f0 ? bv[k] : FLT_MAX;
        fm[k] = wave_max_f32(fm[k]);
        wave_argmin(bv[k], bi[k]);
    }
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NOBJ; ++k) {
            red_v[wid * 2 * NOBJ + k] = fm[k];
            red_v[wid * 2 * NOBJ + NOBJ + k] = bv[k];
            red_i[wid * NOBJ + k] = bi[k];
        }
    __syncthreads();
    if (tid < NOBJ) {
        float m = -FLT_MAX, v = FLT_MAX;
        int id = 0x7FFFFFFF;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            m = fmaxf(m, red_v[w * 2 * NOBJ + tid]);
            argmin_pair(v, id, red_v[w * 2 * NOBJ + NOBJ + tid], red_i[w * NOBJ + tid]);
        }
        atomicMax(&acc->f0hi[tid], ord_bits(m));
        if (id != 0x7FFFFFFF) atomicMin(&acc->asf[tid], asf_key(v, id));
    }
    if (tid == 0 && s_cnt) atomicAdd(&acc->f0, s_cnt);
}

// Further fronts while fewer than N designs are ranked (nonDominatedSorting's
// peeling, sorting.cuh:1026-1086), by a whole workgroup.  `ranked` and `lastm`
// hold the first front's words and *s_cnt its size on entry, `newm` zeros and
// *s_new zero; on return `ranked` and *s_cnt cover every front, `lastm` is the
// last one.  Returns its index; last_size its size.  front_of is stored when
// `store` is set (one workgroup a job).
template <class Pool>
__device__ int peel_fronts(const Pool &J, bool store, uint64_t *ranked, uint64_t *newm, uint64_t *lastm, int *s_cnt,
                           int *s_new, int &last_size) {
    const int P = J.P, W = J.W, N = J.N;
    const int tid = threadIdx.x, NT = blockDim.x, lane = tid & 63;
    int f = 0;
    last_size = *s_cnt;
    while (*s_cnt < N) {
        ++f;
        // a design joins front f when all its dominators are ranked
        int c = 0;
        for (int r0 = 0; r0 < P; r0 += NT) {  // a wave's 64 designs are one word of the masks
            const int r = r0 + tid;
            bool joins = false;
            if (r < P && !((ranked[r >> 6] >> (r & 63)) & 1ull)) {
                uint64_t any = 0;
                for (int w = 0; w < W; ++w) any |= gload(J.dom + (size_t)w * P + r) & ~ranked[w];
                joins = !any;
            }
            const uint64_t b = __ballot(joins);
            if (joins && store) gstore(J.front_of + r, f);
            if (lane == 0 && b) newm[r >> 6] = b;
            c += __popcll(b);
        }
        if (lane == 0) atomicAdd(s_new, c);
        __syncthreads();
        if (*s_new == 0) {  // a dominance cycle: every remaining design forms the front
            for (int r = tid; r < P; r += NT)
                if (!((ranked[r >> 6] >> (r & 63)) & 1ull)) {
                    atomicOr((unsigned long long *)&newm[r >> 6], 1ull << (r & 63));
                    if (store) gstore(J.front_of + r, f);
                }
            __syncthreads();
            if (tid == 0) *s_new = P - *s_cnt;
            __syncthreads();
        }
        for (int w = tid; w < W; w += NT) {
            lastm[w] = newm[w];
            ranked[w] |= newm[w];
            newm[w] = 0;
        }
        last_size = *s_new;
        __syncthreads();
        if (tid == 0) {
            *s_cnt += *s_new;
            *s_new = 0;
        }
        __syncthreads();
    }
    return f;
}

// What the extreme points and the nadir are settled from, in LDS.
struct SettleShared {
    float ideal[NOBJ], worst[NOBJ], f0max[NOBJ];  // pool extrema, first front's maxima
    float pv[NOBJ];                               // per axis the first front's smallest ASF value
    int pid[NOBJ];                                // and its design (0x7FFFFFFF: none)
    float crow[2 * NOBJ][NOBJ];                   // candidate rows of the extremes
    float ext[NOBJ * NOBJ], nadir[NOBJ];
};

// The extreme points settled against the previous ones (prev: lane i < 36
// holds value i of them) and the nadir point (updateNadirValue_HYP with the
// MNDF fallback, sorting.cuh:911-972), by one wave; stored to `out` with the
// front counts when out is not null.
__device__ void settle_nadir(SettleShared &S, const float *obj, int P, float prev, SelRes *out, int ranked_n, int f,
                             int last_size, bool n_cut) {
    const int lane = threadIdx.x & 63;
    // the candidate rows: the current extreme points and the rows of the first
    // front's ASF minima; lane t (0-11) takes row t's ASF values for every axis
    if (lane < NOBJ * NOBJ) {
        const int c = lane / NOBJ, k = lane % NOBJ, p = S.pid[c];
        S.crow[c][k] = prev;
        S.crow[NOBJ + c][k] = p < P ? gload(obj + (size_t)p * NOBJ + k) : 0.f;
    }
    wave_lds_sync();
    const int row = min(lane, 2 * NOBJ - 1), ax = row >= NOBJ ? row - NOBJ : 0;
    float a[NOBJ];
    asf_all(S.crow[row], S.ideal, a);
    const int held = settle_extremes(a, S.pv[ax], S.pid[ax]);
    const int mine = __shfl(held, lane < NOBJ * NOBJ ? lane / NOBJ : 0, 64);
    if (lane < NOBJ * NOBJ) S.ext[lane] = S.crow[mine][lane % NOBJ];
    wave_lds_sync();
    const float x = gauss_wave(S.ext);  // x[lane], lanes 0-5
    float xs[NOBJ];
#pragma unroll
    for (int i = 0; i < NOBJ; ++i) xs[i] = lane_of(x, i);
    // residuals of every extreme and the intercepts (a lane each)
    bool exc = false;
    float icpt = 0.f;
    if (lane < NOBJ) {
        float res = 0.f;
#pragma unroll
        for (int i = 0; i < NOBJ; ++i) res += xs[i] * (S.ext[lane * NOBJ + i] - S.ideal[i]);
        if (fabsf(res - 1.f) > F_PRECISION || isnan(res) || isinf(res)) exc = true;
        icpt = 1.f / x;
        if (icpt <= F_PRECISION || isnan(icpt) || isinf(icpt)) exc = true;
    }
    const bool hyp = __ballot(exc) != 0;
    if (lane < NOBJ) {
        const float lo = S.ideal[lane], hi = S.f0max[lane];
        const float nad = hyp ? (((hi - lo) > F_PRECISION) ? hi : S.worst[lane]) : lo + icpt;
        S.nadir[lane] = nad;
        if (out) {
            gstore(&out->ideal[lane], lo);
            gstore(&out->worst[lane], S.worst[lane]);
            gstore(&out->nadir[lane], nad);
        }
    }
    if (out) {
        if (lane < NOBJ * NOBJ) gstore(&out->ext[lane], S.ext[lane]);
        if (lane == 0) {
            gstore(&out->hyp, (int32_t)hyp);
            gstore(&out->ranked, ranked_n);
            gstore(&out->last, f);
            gstore(&out->base, (f == 0) ? 0 : ranked_n - last_size);
            gstore(&out->n_cut, (int32_t)n_cut);
        }
    }
}

// One workgroup per job, after k_front0: the selection up to the niching of
// jobs that k_front_associate does not take.
//  * Further fronts while fewer than N designs are ranked.
//  * The extreme points settled against the previous ones and the nadir point,
//    by one wave.
//  * The survivors of the fronts before the last one.
__global__ __launch_bounds__(1024) void k_fronts(const DevJob *__restrict__ jobs) {
    const DevJob &J = jobs[blockIdx.x];
    const int P = J.P, W = J.W, N = J.N;
    const int tid = threadIdx.x, NT = blockDim.x, lane = tid & 63, wid = tid >> 6;
    // the descriptor fields first, held in scalar registers, then every
    // load of the set-up at once
    SelState *st = J.st;
    const SelAcc *acc = J.acc;
    const uint64_t *rk = J.ranked;
    const float *o0 = J.obj[0], *o1 = J.obj[1];
    asm volatile("" : "+s"(st), "+s"(acc), "+s"(rk), "+s"(o0), "+s"(o1));
    const uint32_t g0 = gload(&st->gen);
    __shared__ uint64_t ranked[MAX_W], newm[MAX_W], lastm[MAX_W];
    __shared__ int s_cnt, s_new;
    __shared__ SettleShared S;
    const int ei = min(lane, NOBJ * NOBJ - 1);
    const float e0 = gload(st->res[0].ext + ei), e1 = gload(st->res[1].ext + ei);
    if (tid < NOBJ) {
        S.ideal[tid] = ord_float(gload(acc->lo + tid));
        S.worst[tid] = ord_float(gload(acc->hi + tid));
        S.f0max[tid] = ord_float(gload(acc->f0hi + tid));
        const unsigned long long k = gload(acc->asf + tid);
        S.pv[tid] = k == ~0ull ? FLT_MAX : ord_float((uint32_t)(k >> 32));
        S.pid[tid] = k == ~0ull ? 0x7FFFFFFF : (int)(uint32_t)k;
    }
    if (tid == 0) {
        s_cnt = gload(&acc->f0);
        s_new = 0;
    }
    const uint32_t gen = __builtin_amdgcn_readfirstlane(g0);
    const float *const obj = (gen & 1u) ? o0 : o1;  // buffer (gen + 1) & 1
    for (int w = tid; w < W; w += NT) {
        const uint64_t f0w = gload(rk + w);
        ranked[w] = f0w;
        lastm[w] = f0w;
        newm[w] = 0;
    }
    __syncthreads();
    int last_size;
    const int f = peel_fronts(J, true, ranked, newm, lastm, &s_cnt, &s_new, last_size);
    const int ranked_n = s_cnt;
    const bool n_cut = ranked_n == N;
    // survivors so far: every ranked design when the fronts fill N exactly,
    // else the fronts before the last one
    for (int w = tid; w < W; w += NT) gstore(J.selm + w, n_cut ? ranked[w] : (ranked[w] & ~lastm[w]));
    if (wid == 0)
        settle_nadir(S, obj, P, (gen & 1u) ? e1 : e0, st->res + ((gen + 1u) & 1u), ranked_n, f, last_size, n_cut);
}

// ---------------------------------------------------------------------------
// A sort alone (cd_nds_noalloc), in two launches on arguments by value: no
// descriptor, work list or cleared counts stand before the first.
//   k_sort_tiles   the domination matrix, a tile (b, w), b <= w, a workgroup of
//                  four waves as in k_dominance; instead of counts, word [w][b]
//                  of S.any says which rows of block b some design of block w
//                  dominates (a plain store)
//   k_sort_fronts  one workgroup: the first front from those words, then the
//                  further ones
// 2048 designs, 1024 ranked: 4.9 + 3.1 us (setup, k_dominance, k_front0, k_fronts
// and the count's copy, five launches: 23).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_sort_tiles(SortArgs S) {
    __shared__ float rows[64 * NOBJ];
    __shared__ uint64_t part[4][64], amask[4][16], s_rows[4];
    const int lane = threadIdx.x & 63, sub = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), P = S.P, W = S.W;
    const int t = (int)blockIdx.x;  // tile t: w(w+1)/2 + b
    int w = (int)((sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
    w += (w + 1) * (w + 2) / 2 <= t;
    w -= w * (w + 1) / 2 > t;
    const int b = t - w * (w + 1) / 2, r0 = 64 * b, i = 64 * w + lane, rr = r0 + lane;
    float cand[NOBJ], row[NOBJ];
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        cand[k] = gload(S.obj + (size_t)min(i, P - 1) * NOBJ + k);
        row[k] = gload(S.obj + (size_t)min(rr, P - 1) * NOBJ + k);
    }
    // designs and rows past the pool hold +inf (k_dominance)
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) cand[k] = i < P ? cand[k] : __builtin_inff();
    if (sub == 0)
#pragma unroll
        for (int k = 0; k < NOBJ; ++k) rows[lane * NOBJ + k] = rr < P ? row[k] : __builtin_inff();
    __syncthreads();
    uint64_t col = dominance_rows<16>(rows + sub * 16 * NOBJ, cand, amask[sub]);
    const uint64_t mine = amask[sub][min(lane, 15)];
    const int r = r0 + sub * 16 + lane;
    if (lane < 16 && r < P) gstore(S.dom + (size_t)w * P + r, mine);
    const uint64_t hit = __ballot(lane < 16 && mine != 0);
    if (lane == 0) s_rows[sub] = hit;
    part[sub][lane] = col << (sub * 16);
    lds_barrier();
    if (sub) return;
    if (lane == 0) gstore(S.any + (size_t)w * W + b, s_rows[0] | (s_rows[1] << 16) | (s_rows[2] << 32) | (s_rows[3] << 48));
    if (b == w) return;
#pragma unroll
    for (int g = 1; g < 4; ++g) col |= part[g][lane];
    if (i < P) gstore(S.dom + (size_t)b * P + i, col);
    const uint64_t cols = __ballot(col != 0);
    if (lane == 0) gstore(S.any + (size_t)b * W + w, cols);
}
__global__ __launch_bounds__(1024) void k_sort_fronts(SortArgs S) {
    __shared__ uint64_t ranked[MAX_W], newm[MAX_W], lastm[MAX_W];
    __shared__ int s_cnt, s_new;
    const int tid = threadIdx.x, NT = blockDim.x, P = S.P, W = S.W;
    for (int w = tid; w < W; w += NT) newm[w] = 0;
    if (tid == 0) s_cnt = s_new = 0;
    __syncthreads();
    for (int i = tid; i < W * W; i += NT) {  // word i % W of the rows that are dominated
        const uint64_t x = gload(S.any + i);
        if (x) atomicOr((unsigned long long *)&newm[i % W], (unsigned long long)x);
    }
    __syncthreads();
    for (int w = tid; w < W; w += NT) {
        const uint64_t x = ~newm[w] & (64 * w + 64 <= P ? ~0ull : (1ull << (P & 63)) - 1ull);
        ranked[w] = x;
        lastm[w] = x;
        newm[w] = 0;
        if (x) atomicAdd(&s_cnt, (int)__popcll(x));
    }
    __syncthreads();
    for (int r = tid; r < P; r += NT) gstore(S.front_of + r, (ranked[r >> 6] >> (r & 63)) & 1ull ? 0 : -1);
    __syncthreads();  // (before the further fronts store theirs)
    int last_size;
    const int f = peel_fronts(S, true, ranked, newm, lastm, &s_cnt, &s_new, last_size);
    if (tid == 0) gstore(S.n_fronts, f + 1);
}

// The squared perpendicular distance of f to a reference line, w its weights
// and den the sum of their squares (utils.cuh:1149-1171 before its root).
__device__ __forceinline__ float perp_dist2(const float *f, const float *w, float den) {
    float num = 0.f;
#pragma unroll
    for (int i = 0; i < NOBJ; ++i) num += w[i] * f[i];
    const float k = num / den;
    float d = 0.f;
#pragma unroll
    for (int i = 0; i < NOBJ; ++i) {
        const float t = k * w[i] - f[i];
        d += t * t;
    }
    return d;
}

// The nearest of the reference lines r = sub, sub + LPD, ... below R: the
// smallest distance (the root of perp_dist2), ties to the lowest index, as a
// sweep that takes every strictly smaller root finds it; best stays FLT_MAX
// when no root is below it.  The root is taken once, of the line kept: a
// smaller square has a smaller or equal root, and the roots of two squares
// can only be equal when the squares are within two parts in 2^23, so a
// square below the kept one by more than one part in 2^20 replaces it at
// once and the rare one between compares the roots themselves.
template <int LPD>
__device__ __forceinline__ void nearest_line(const float *f, const float *refpts, int R, int sub, float &best, int &br) {
    float b2 = __builtin_inff();
    br = 0;
    for (int r = sub; r < R; r += LPD) {
        const f32x4 *q = (const f32x4 *)(refpts + (size_t)r * REF_STRIDE);
        const f32x4 a = gload(q), b = gload(q + 1);
        const float w[NOBJ] = {a.x, a.y, a.z, a.w, b.x, b.y};
        const float d2 = perp_dist2(f, w, b.z);
        bool take = d2 < b2 * 0.99999905f;  // 1 - 2^-20
        if (d2 < b2 && !take) take = sqrtf(d2) < sqrtf(b2);
        b2 = take ? d2 : b2;
        br = take ? r : br;
    }
    best = sqrtf(b2);
    if (!(best < FLT_MAX)) {
        best = FLT_MAX;
        br = 0;
    }
}

__device__ __forceinline__ uint64_t niche_prio(const DevJob &J, uint32_t gen, int d) {
    uint32_t r[4];
    philox(gen, (uint32_t)d, 0u, TAG_NICHE, J.seed, r);
    return ((uint64_t)r[0] << 32) | (uint32_t)d;
}

// A design's row normalised by the ideal and nadir points (a zero range maps to 0).
__device__ __forceinline__ void normalise_row(const float *x, const float *ideal, const float *nadir, float *f) {
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        const float den = nadir[k] - ideal[k];
        f[k] = (den == 0.f) ? 0.f : (x[k] - ideal[k]) / den;
    }
}

// Association of one ranked design d (row x) by its LPD lanes (sub 0 .. LPD -
// 1), every lane of the wave or none of a design's lanes taking part:
// its nearest reference line (sorting.cuh:1105-1180), ties to the lowest
// index (the first minimum of a sweep in index order).  The niche arrays are
// folded in with atomics: designs of the fronts before the last count toward
// their niche, those of the last front toward its bucket, with the bucket's
// nearest design as a 64-bit (distance, design) minimum.  A distance is never
// NaN or above FLT_MAX.
template <int LPD>
__device__ __forceinline__ void associate_design(const DevJob &J, uint32_t gen, int d, int sub, const float *f,
                                                 bool is_last) {
    const int R = J.R;
    float best;
    int br;
    nearest_line<LPD>(f, J.refpts, R, sub, best, br);
    bool writer;
    if (LPD == 64) {
        wave_argmin(best, br);  // (every lane of the wave is here: one design a wave)
        writer = sub == 0;
    } else {
        // the design's eight lanes (two quads of a DPP row): the quads by
        // quad permutations, then the first quad into the second by a row
        // shift, whose last lane ends with the design's minimum (the lanes
        // read only their own design's lanes, which are all here)
        argmin_dpp<0xB1, 0xf>(best, br);   // quad_perm [1,0,3,2]
        argmin_dpp<0x4E, 0xf>(best, br);   // quad_perm [2,3,0,1]
        argmin_dpp<0x114, 0xf>(best, br);  // row_shr:4
        writer = sub == 7;
    }
    if (writer) {
        gstore(J.ref_of + d, br);
        const NicheView g = niche_view(J.niche, R);
        if (!is_last) {
            atomicAdd(&g.cr[br].x, 1);
        } else {
            atomicAdd(&g.cr[br].y, 1);
            atomicMin(g.nearest + br, asf_key(best, d));
            gstore(J.prio + d, (uint32_t)(niche_prio(J, gen, d) >> 32));
        }
    }
}

// Nearest reference line of every ranked design: LPD lanes per design (a
// wave, or eight lanes), D designs a workgroup (item = (job, first design)).
template <int D, int LPD>
__global__ __launch_bounds__(D * LPD) void k_associate(const DevJob *__restrict__ jobs,
                                                       const int2 *__restrict__ items) {
    static_assert(LPD == 64 || LPD == 8, "a wave or eight lanes per design");
    const int2 it = items[blockIdx.x];
    const DevJob &J = jobs[it.x];
    const int sub = (int)threadIdx.x % LPD, P = J.P;
    const SelState *st = J.st;
    // everything the wave reads before its first store, loaded together: the
    // selection's result, the design's front and objectives (at a clamped index)
    const uint32_t gen = __builtin_amdgcn_readfirstlane(gload(&st->gen));
    const SelRes *res = st->res + ((gen + 1u) & 1u);
    const int n_cut = gload(&res->n_cut), last = gload(&res->last);
    float ideal[NOBJ], nadir[NOBJ];
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        ideal[k] = gload(&res->ideal[k]);
        nadir[k] = gload(&res->nadir[k]);
    }
    const int d = it.y + (int)threadIdx.x / LPD, dc = min(d, P - 1);
    // the row in 8-byte words (rows are 24 bytes), each feeding two objectives,
    // so that the loads stay ahead of the per-objective branches
    const f32x2 *o2 = (const f32x2 *)(pool_obj(J, gen) + (size_t)dc * NOBJ);
    const f32x2 x01 = gload(o2), x23 = gload(o2 + 1), x45 = gload(o2 + 2);
    const int fr = gload(J.front_of + dc);
    const float x[NOBJ] = {x01.x, x01.y, x23.x, x23.y, x45.x, x45.y};
    float f[NOBJ];
    normalise_row(x, ideal, nadir, f);
    if (n_cut || d >= P || fr < 0) return;  // no niching, or no ranked design (all the design's lanes)
    associate_design<LPD>(J, gen, d, sub, f, fr == last);
}

// k_front0, k_fronts and k_associate in one launch, for pools of at most
// FUSED_POOL designs: D designs a workgroup as in k_associate, and every
// workgroup of a job settles the job's selection itself -- the first front
// from the dominator counts, its maxima and ASF minima, further fronts, the
// extreme points and the nadir -- instead of reading it from two kernels
// before.  The settling is a few microseconds of dependent steps whichever
// workgroup runs it, so doing it side by side costs no time while the
// workgroups fit the chip, and the two launches and their load rounds go.
// The workgroup of the job's first designs stores the result (SelState::res
// of the other parity than the one read, front_of, the survivors so far).
// Measured for the 100-residue job (pool 256, 4 designs a workgroup): 53.7 ->
// 50.4 us a generation; 1237-residue job (pool 1554, 8): 94.8 -> 93.4; 500-
// residue job (pool 2048, 8): 78.8 -> 78.2.  Of its 11.4 us there, the first
// front takes 2.7, its reductions 2.3, the extremes and the nadir 3.3, the
// association 1.7.
template <int D, int LPD>
__global__ __launch_bounds__(D * LPD) void k_front_associate(const DevJob *__restrict__ jobs,
                                                             const int2 *__restrict__ items) {
    constexpr int NT = D * LPD, NW = NT / 64, MW = FUSED_POOL / 64;
    __shared__ uint64_t ranked[MW], newm[MW], lastm[MW];
    __shared__ int s_cnt, s_new;
    __shared__ SettleShared S;
    __shared__ float red_m[NW][NOBJ], red_v[NW][NOBJ];
    __shared__ int red_i[NW][NOBJ], red_c[NW];
    const int2 it = items[blockIdx.x];
    const DevJob &J = jobs[it.x];
    // the descriptor fields held in scalar registers, then the loads that
    // wait for nothing else
    SelState *st = J.st;
    const SelAcc *acc = J.acc;
    const int32_t *np = J.np;
    const float *o0 = J.obj[0], *o1 = J.obj[1];
    int32_t *front_of = J.front_of;
    int P = J.P, W = J.W, N = J.N;
    asm volatile("" : "+s"(st), "+s"(acc), "+s"(np), "+s"(o0), "+s"(o1), "+s"(front_of), "+s"(P), "+s"(W), "+s"(N));
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, sub = tid % LPD;
    const bool first = it.y == 0;  // the workgroup that stores the job's selection
    const uint32_t g0 = gload(&st->gen);
    float ideal[NOBJ];
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) ideal[k] = ord_float(gload(acc->lo + k));
    const uint32_t hi = gload(acc->hi + min(lane, NOBJ - 1));
    const int ei = min(lane, NOBJ * NOBJ - 1);
    const float e0 = gload(st->res[0].ext + ei), e1 = gload(st->res[1].ext + ei);
    const uint32_t gen = __builtin_amdgcn_readfirstlane(g0);
    const float *const obj = (gen & 1u) ? o0 : o1;  // buffer (gen + 1) & 1
    const f32x2 *const rows = (const f32x2 *)obj;
    const int d = it.y + tid / LPD, dc = min(d, P - 1);
    const f32x2 x01 = gload(rows + 3 * dc), x23 = gload(rows + 3 * dc + 1), x45 = gload(rows + 3 * dc + 2);
    // the first front: its words, size, maxima (updateNadirValue_MNDF,
    // sorting.cuh:685-884) and per-axis ASF minima, ties to the lowest index
    // (findExtremePoints, sorting.cuh:601-683); a wave without one skips
    float fm[NOBJ], bv[NOBJ];
    int bi[NOBJ], cnt = 0;
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        fm[k] = -FLT_MAX;
        bv[k] = FLT_MAX;
        bi[k] = 0x7FFFFFFF;
    }
    for (int c0 = 0; c0 < P; c0 += 2 * NT) {  // two designs a thread and round
        int v[2];
        f32x2 r[2][3];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int qc = min(c0 + u * NT + tid, P - 1);
            v[u] = gload(np + qc);
#pragma unroll
            for (int h = 0; h < 3; ++h) r[u][h] = gload(rows + 3 * qc + h);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int q = c0 + u * NT + tid, w0 = (c0 + u * NT) / 64 + wid;  // a wave's designs are word w0
            const bool f0 = q < P && v[u] == 0;
            const uint64_t b = __ballot(f0);
            if (first && q < P) gstore(front_of + q, f0 ? 0 : -1);
            if (lane == 0 && w0 < W) {
                ranked[w0] = b;
                lastm[w0] = b;
                newm[w0] = 0;
            }
            if (!b) continue;
            cnt += (int)__popcll(b);
            const float x[NOBJ] = {r[u][0].x, r[u][0].y, r[u][1].x, r[u][1].y, r[u][2].x, r[u][2].y};
            float a[NOBJ];
            asf_all(x, ideal, a);
#pragma unroll
            for (int k = 0; k < NOBJ; ++k) {
                fm[k] = fmaxf(fm[k], f0 ? x[k] : -FLT_MAX);
                const bool less = f0 && a[k] < bv[k];  // (designs rise: ties keep the first)
                bv[k] = less ? a[k] : bv[k];
                bi[k] = less ? q : bi[k];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) {
        fm[k] = wave_max_f32(fm[k]);
        wave_argmin(bv[k], bi[k]);
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NOBJ; ++k) {
            red_m[wid][k] = fm[k];
            red_v[wid][k] = bv[k];
            red_i[wid][k] = bi[k];
        }
        red_c[wid] = cnt;
    }
    lds_barrier();
    if (tid < NOBJ) {
        float m = -FLT_MAX, v = FLT_MAX;
        int id = 0x7FFFFFFF;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            m = fmaxf(m, red_m[w][tid]);
            argmin_pair(v, id, red_v[w][tid], red_i[w][tid]);
        }
        S.f0max[tid] = m;
        S.pv[tid] = v;
        S.pid[tid] = id;
        S.worst[tid] = ord_float(hi);
        float lo = ideal[0];
#pragma unroll
        for (int k = 1; k < NOBJ; ++k) lo = tid == k ? ideal[k] : lo;
        S.ideal[tid] = lo;
    }
    if (tid == 64) {  // (another wave than the reductions': NW is at least 4)
        int c = 0;
        for (int w = 0; w < NW; ++w) c += red_c[w];
        s_cnt = c;
        s_new = 0;
    }
    lds_barrier();
    int last_size;
    const int f = peel_fronts(J, first, ranked, newm, lastm, &s_cnt, &s_new, last_size);
    const int ranked_n = s_cnt;
    const bool n_cut = ranked_n == N;
    // survivors so far: every ranked design when the fronts fill N exactly,
    // else the fronts before the last one
    if (first)
        for (int w = tid; w < W; w += NT) gstore(J.selm + w, n_cut ? ranked[w] : (ranked[w] & ~lastm[w]));
    else if (n_cut)
        return;  // no niching
    if (wid == 0)
        settle_nadir(S, obj, P, (gen & 1u) ? e1 : e0, first ? st->res + ((gen + 1u) & 1u) : nullptr, ranked_n, f,
                     last_size, n_cut);
    if (n_cut) return;
    lds_barrier();
    const float x[NOBJ] = {x01.x, x01.y, x23.x, x23.y, x45.x, x45.y};
    float nadir[NOBJ], fn[NOBJ];
#pragma unroll
    for (int k = 0; k < NOBJ; ++k) nadir[k] = S.nadir[k];
    normalise_row(x, ideal, nadir, fn);
    if (d >= P || !((ranked[d >> 6] >> (d & 63)) & 1ull)) return;  // no ranked design (all the design's lanes)
    associate_design<LPD>(J, gen, d, sub, fn, (lastm[d >> 6] >> (d & 63)) & 1ull);
}

// The levels of referenceBasedSorting (sorting.cuh:1182-1279) in closed form,
// by wave 0 of a workgroup (every thread calls it; the niche arrays are in
// LDS or global memory).  Picks made through level i: C(i) = sum_r
// clamp(i + 1 - cnt[r], 0, rem[r]), nondecreasing in i; the final level is
// the smallest i with C(i) >= need (or P), found by bisection, where the
// first eligible reference points in index order take one more.  Per
// reference point: its picks, its level-0 pick (an empty niche takes its
// nearest design, ties to the lowest index), and, for a bucket only part of
// whose rest is taken (a cut bucket), its offset in the cut list, a multiple
// of ALIGN (a power of two).  Returns the cut list's size.
template <int ALIGN>
__device__ __forceinline__ int niche_levels(const DevJob &J, int base, const int2 *cr,
                                            const unsigned long long *nearest, int *kp, int *lvl0, int *coff) {
    const int P = J.P, N = J.N, R = J.R, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __shared__ int s_ncut;
    if (wid == 0) {
        const int need = N - base;
        // up to 256 reference points: four a lane, in registers
        const bool small = R <= 256;
        int2 rc[4];
        unsigned long long nr[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int r = min(lane + 64 * k, R - 1);
            const bool in = small && lane + 64 * k < R;
            rc[k] = cr[r];
            nr[k] = nearest[r];
            rc[k].x = in ? rc[k].x : 0;
            rc[k].y = in ? rc[k].y : 0;
        }
        // the bucket taken whole last bounds the final level: with hi its last
        // level, C(hi) is every design of the last front, at least `need`
        int top = 0;
        if (small) {
#pragma unroll
            for (int k = 0; k < 4; ++k) top = max(top, rc[k].y ? rc[k].x + rc[k].y : 0);
        } else {
            for (int r = lane; r < R; r += 64) {
                const int2 c = cr[r];
                top = max(top, c.y ? c.x + c.y : 0);
            }
        }
        int lo = -1, clo = 0, hi = min(P, max(wave_max_nonneg(top) - 1, 0));  // C(lo) < need; C(hi) >= need or hi = P
        while (hi - lo > 1) {
            const int mid = lo + ((hi - lo) >> 1);
            int acc = 0;
            if (small) {
#pragma unroll
                for (int k = 0; k < 4; ++k) acc += min(max(mid + 1 - rc[k].x, 0), rc[k].y);
            } else {
                for (int r = lane; r < R; r += 64) {
                    const int2 c = cr[r];
                    acc += min(max(mid + 1 - c.x, 0), c.y);
                }
            }
            const int C = wave_sum_i32(acc);
            if (C >= need) {
                hi = mid;
            } else {
                lo = mid;
                clo = C;
            }
        }
        const int istar = hi, need_final = need - clo;
        int carry = 0, cut_carry = 0;
        // 64 reference points r = r0 + lane with their counts and nearest design
        auto settle = [&](int r0, int2 c, unsigned long long near) {
            const int r = r0 + lane;
            const bool e = r < R && c.x <= istar && istar < c.x + c.y;
            const uint64_t eb = __ballot(e);
            const int ex = carry + (int)__popcll(eb & ((1ull << lane) - 1ull));
            const int k = min(max(istar - c.x, 0), c.y) + ((e && ex < need_final) ? 1 : 0);
            // level 0 of an empty niche: its nearest design, ties to the
            // lowest index (the reference's fallback to the lowest index, for a
            // NaN distance or none below FLT_MAX, never applies: every distance
            // is at most FLT_MAX and none is NaN)
            const int l0 = (r < R && k > 0 && c.x == 0) ? (int)(uint32_t)near : -1;
            const int h = l0 >= 0 ? 1 : 0;
            const int cut = (r < R && k - h > 0 && k - h < c.y - h) ? c.y : 0;
            const int room = (cut + ALIGN - 1) & ~(ALIGN - 1);
            const int incl = wave_scan_i32(room);  // inclusive prefix of the cut sizes over the wave
            if (r < R) {
                kp[r] = k;
                lvl0[r] = l0;
                coff[r] = cut ? cut_carry + incl - room : -1;
            }
            carry += (int)__popcll(eb);
            cut_carry += __builtin_amdgcn_readlane(incl, 63);
        };
        if (small) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (64 * k < R) settle(64 * k, rc[k], nr[k]);
        } else {
            for (int r0 = 0; r0 < R; r0 += 64) {
                const int r = min(r0 + lane, R - 1);
                settle(r0, cr[r], nearest[r]);
            }
        }
        if (lane == 0) s_ncut = cut_carry;
    }
    __syncthreads();
    return s_ncut;
}

// niche_levels for jobs whose niche arrays do not fit in LDS (R above
// NICHE_STAGE): one workgroup per job, on the arrays in global memory.
__global__ __launch_bounds__(256) void k_levels(const DevJob *__restrict__ jobs) {
    const DevJob &J = jobs[blockIdx.x];
    const SelRes &res = J.st->res[(J.st->gen + 1u) & 1u];
    if (res.n_cut || J.R <= NICHE_STAGE) return;
    const NicheView g = niche_view(J.niche, J.R);
    const int ncut = niche_levels<1>(J, res.base, g.cr, g.nearest, g.kp, g.lvl0, g.coff);
    if (threadIdx.x == 0) J.acc->ncut = ncut;
}

// Every design of the last front, one a thread (grid: jobs x chunks of NT
// designs of the largest pool).  Each workgroup first settles the levels
// itself (niche_levels on the niche arrays staged in LDS; workgroup 0 also
// keeps them for k_niche) when R fits, else reads what k_levels wrote.  A
// design is selected when it is its niche's level-0 pick or when the rest of
// its bucket is taken whole (one atomic OR per wave and word of the survivor
// mask); the designs of a cut bucket get slots in the cut list, bucket by
// bucket, keyed by (priority, design), for k_niche to rank -- the workgroup
// counts its designs per bucket in LDS and claims each bucket's share with
// one atomic (when R fits).
__global__ __launch_bounds__(1024) void k_place(const DevJob *__restrict__ jobs) {
    const DevJob &J = jobs[blockIdx.x];
    const SelRes *const st = J.st->res + ((J.st->gen + 1u) & 1u);
    const int P = J.P, R = J.R, NT = blockDim.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int d0 = blockIdx.y * NT;
    if (d0 >= P) return;
    // the design's own fields, issued with the state's at a clamped index
    // (ref_of and prio are read only for designs of the last front)
    const int d = d0 + tid, dc = min(d, P - 1);
    const int fo = gload(J.front_of + dc), rf = gload(J.ref_of + dc);
    const uint32_t pr = gload(J.prio + dc);
    if (st->n_cut) return;
    const NicheView g = niche_view(J.niche, R);
    const bool staged = R <= NICHE_STAGE;
    __shared__ int2 s_cr[NICHE_STAGE];
    __shared__ unsigned long long s_near[NICHE_STAGE];
    __shared__ int s_kp[NICHE_STAGE], s_l0[NICHE_STAGE], s_co[NICHE_STAGE], l_cnt[NICHE_STAGE], l_base[NICHE_STAGE];
    const int *kp = g.kp, *lvl0 = g.lvl0, *coff = g.coff;
    if (staged) {
        for (int r = tid; r < R; r += NT) {
            s_cr[r] = g.cr[r];
            s_near[r] = gload(g.nearest + r);
            l_cnt[r] = 0;
        }
        __syncthreads();
        const int ncut = niche_levels<1>(J, st->base, s_cr, s_near, s_kp, s_l0, s_co);
        if (blockIdx.y == 0) {
            for (int r = tid; r < R; r += NT) {
                gstore(g.kp + r, s_kp[r]);
                gstore(g.lvl0 + r, s_l0[r]);
                gstore(g.coff + r, s_co[r]);
            }
            if (tid == 0) J.acc->ncut = ncut;
        }
        kp = s_kp;
        lvl0 = s_l0;
        coff = s_co;
    }
    const bool mine = d < P && fo == st->last;
    int r = 0, co = -1, loc = 0;
    bool sel = false;
    if (mine) {
        r = rf;
        const int l0 = lvl0[r];
        co = coff[r];
        sel = d == l0;
        if (co >= 0)
            loc = staged ? atomicAdd(&l_cnt[r], 1) : 0;
        else if (!sel)  // not cut: the rest of the bucket is taken whole, or nothing of it
            sel = kp[r] - (l0 >= 0 ? 1 : 0) > 0;
    }
    if (staged) {
        __syncthreads();
        for (int q = tid; q < R; q += NT)
            if (l_cnt[q]) l_base[q] = atomicAdd(g.fill + q, l_cnt[q]);
        __syncthreads();
    }
    if (mine && co >= 0) {
        const int slot = co + (staged ? l_base[r] + loc : atomicAdd(g.fill + r, 1));
        gstore(J.cutl + slot, ((uint64_t)pr << 32) | (uint32_t)d);
        gstore(J.cutr + slot, r);
    }
    const uint64_t b = __ballot(sel);  // a wave's 64 designs are one word of the mask
    if (lane == 0 && b) atomicOr((unsigned long long *)J.selm + (d0 >> 6) + wid, b);
}

// The designs of the cut buckets, one a thread in cut-list order (grid: jobs
// x chunks of NT designs of the largest pool): a design other than its
// niche's level-0 pick is selected when fewer than kk of the rest of its
// bucket (the bucket without the level-0 pick) have a smaller (priority,
// design) key.  A workgroup stages the keys of every bucket its slots touch
// in LDS (dynamic, 8 bytes a design of the pool).  Workgroup 0 ends the
// generation (nothing here reads the generation count).
__global__ __launch_bounds__(1024) void k_niche(const DevJob *__restrict__ jobs) {
    extern __shared__ __align__(16) uint8_t dyn[];
    uint64_t *keys = (uint64_t *)dyn;
    const DevJob &J = jobs[blockIdx.x];
    SelState *st = J.st;
    const int R = J.R, NT = blockDim.x, tid = threadIdx.x;
    const int s0 = blockIdx.y * NT;
    if (blockIdx.y == 0 && tid == 0) st->gen = st->gen + 1u;
    const int ncut = J.acc->ncut;  // 0 where the fronts filled N exactly
    if (s0 >= ncut) return;
    const NicheView g = niche_view(J.niche, R);
    __shared__ int s_a, s_b;
    const int s = s0 + tid, sc = min(s, ncut - 1);
    const uint64_t my = gload(J.cutl + sc);
    const int r = gload(J.cutr + sc);
    // the bucket's fields, loaded together
    const int co = gload(g.coff + r), nr = gload((const int32_t *)(g.cr + r) + 1), l0 = gload(g.lvl0 + r),
              kr = gload(g.kp + r);
    if (tid == 0) s_a = co;  // the first slot's bucket starts here
    if (s == min(s0 + NT, ncut) - 1) s_b = co + nr;
    __syncthreads();
    const int a = s_a, nk = s_b - s_a;
    for (int u = tid; u < nk; u += NT) keys[u] = gload(J.cutl + a + u);
    __syncthreads();
    if (s < ncut) {
        const int d = (int)(uint32_t)my;
        if (d != l0) {
            const int kk = kr - (l0 >= 0 ? 1 : 0);
            const int off = co - a;
            int rank = 0;
#pragma unroll 4
            for (int u = 0; u < nr; ++u) rank += (int)(keys[off + u] < my);
            // the level-0 pick of the bucket is not part of the rest
            if (l0 >= 0 && ((((uint64_t)gload(J.prio + l0)) << 32) | (uint32_t)l0) < my) --rank;
            if (rank < kk) atomicOr((unsigned long long *)J.selm + (d >> 6), 1ull << (d & 63));
        }
    }
}

// k_place and k_niche in one workgroup per job, for pools of at most
// PLACE_NICHE_POOL designs whose niche arrays fit in LDS (R <= NICHE_STAGE):
// the levels settled in LDS, the designs of the last front placed (designs
// d = tid, tid + NT, ...), the cut buckets' keys (priority, design) and
// buckets kept in LDS (dynamic, place_niche_lds_bytes) instead of the
// global cut list, and the cut designs ranked within their buckets after one
// barrier instead of a kernel boundary.  The same selection as k_place then
// k_niche: a design is selected when it is its niche's level-0 pick, when
// the rest of its bucket is taken whole, or when fewer than kk of the rest of
// its cut bucket have a smaller key.  Ends the generation, as k_niche does.
// The buckets' priorities are ranked four to an LDS read (the lanes of one
// bucket read the same words), and the picks are folded in LDS and stored
// once: with 64-bit keys read one at a time and an atomic on the survivor
// mask per pick, the ranking of the 500-residue job's 1335 cut designs (44
// buckets of up to 63) took 3.1 us, now 2.1, and a pool of 2048 with buckets
// of hundreds 20.7 us in all.
__global__ __launch_bounds__(1024) void k_place_niche(const DevJob *__restrict__ jobs) {
    extern __shared__ __align__(16) uint8_t dyn[];
    const DevJob &J = jobs[blockIdx.x];
    // the descriptor fields first, held in scalar registers, then the state,
    // the reference points' counts and the first designs' rows at once
    SelState *st = J.st;
    int32_t *niche = J.niche;
    const int32_t *front_of = J.front_of, *ref_of = J.ref_of;
    const uint32_t *prio = J.prio;
    uint64_t *selm = J.selm;
    int P = J.P, R = J.R, W = J.W;
    asm volatile("" : "+s"(st), "+s"(niche), "+s"(front_of), "+s"(ref_of), "+s"(prio), "+s"(selm), "+s"(P), "+s"(R), "+s"(W));
    const int NT = blockDim.x, tid = threadIdx.x;
    // (both halves of the selection's results, the counter choosing one)
    const uint32_t g0 = gload(&st->gen);
    const int nc0 = gload(&st->res[0].n_cut), la0 = gload(&st->res[0].last), ba0 = gload(&st->res[0].base);
    const int nc1 = gload(&st->res[1].n_cut), la1 = gload(&st->res[1].last), ba1 = gload(&st->res[1].base);
    int fo[2], rf[2];
    uint32_t pr[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int dc = min(tid + u * NT, P - 1);
        fo[u] = gload(front_of + dc);
        rf[u] = gload(ref_of + dc);
        pr[u] = gload(prio + dc);
    }
    const uint64_t sm = gload(selm + min(tid, W - 1));
    // and the reference points' counts and nearest designs (first chunk)
    const NicheView g = niche_view(niche, R);
    const int rc0 = min(tid, R - 1);
    const uint64_t cr0 = gload((const uint64_t *)g.cr + rc0);  // int2 (x low, y high)
    const unsigned long long nn0 = gload(g.nearest + rc0);
    const bool h1 = ((g0 + 1u) & 1u) != 0;
    const int n_cut = h1 ? nc1 : nc0, last = h1 ? la1 : la0, base = h1 ? ba1 : ba0;
    // the cut buckets' designs, bucket by bucket, each bucket in whole 16-byte
    // words: priorities (pads hold ~0), and (bucket << 16 | design) (pads ~0)
    uint32_t *const kpri = (uint32_t *)dyn, *const kwho = kpri + place_niche_slots(P, R);
    __shared__ int2 s_cr[NICHE_STAGE];
    __shared__ unsigned long long s_near[NICHE_STAGE];
    __shared__ int s_kp[NICHE_STAGE], s_l0[NICHE_STAGE], s_co[NICHE_STAGE], l_cnt[NICHE_STAGE];
    __shared__ uint32_t s_pl0[NICHE_STAGE];  // priority of each bucket's level-0 pick
    __shared__ uint32_t s_sel[PLACE_NICHE_POOL / 32];  // the last front's picks, folded here and stored once
    if (tid < R) {
        s_cr[tid] = make_int2((int)(uint32_t)cr0, (int)(uint32_t)(cr0 >> 32));
        s_near[tid] = nn0;
        l_cnt[tid] = 0;
    }
    for (int r = tid + NT; r < R; r += NT) {
        s_cr[r] = g.cr[r];
        s_near[r] = gload(g.nearest + r);
        l_cnt[r] = 0;
    }
    if (tid < PLACE_NICHE_POOL / 32) s_sel[tid] = 0u;
    __syncthreads();
    if (tid == 0) gstore(&st->gen, g0 + 1u);  // (every thread has read the count)
    if (n_cut) return;
    const int ncut = niche_levels<4>(J, base, s_cr, s_near, s_kp, s_l0, s_co);  // (with the pads)
    for (int r = tid; r < R; r += NT) {
        const int co = s_co[r], nr = s_cr[r].y;
        if (co >= 0)
            for (int i = nr; i & 3; ++i) kpri[co + i] = kwho[co + i] = ~0u;
    }
    // place the designs of the last front
    for (int d0 = 0; d0 < P; d0 += 2 * NT) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int d = d0 + u * NT + tid;
            if (d0) {  // (the first designs' rows were loaded before the levels)
                const int dc = min(d, P - 1);
                fo[u] = gload(front_of + dc);
                rf[u] = gload(ref_of + dc);
                pr[u] = gload(prio + dc);
            }
            if (d >= P || fo[u] != last) continue;
            const int r = rf[u], l0 = s_l0[r], co = s_co[r], kr = s_kp[r];
            bool sel = d == l0;
            if (sel) s_pl0[r] = pr[u];  // (the level-0 pick is a last-front design of its bucket)
            if (co >= 0) {
                const int slot = co + atomicAdd(&l_cnt[r], 1);
                kpri[slot] = pr[u];
                kwho[slot] = ((uint32_t)r << 16) | (uint32_t)d;
            } else if (!sel) {  // not cut: the rest of the bucket is taken whole, or nothing of it
                sel = kr - (l0 >= 0 ? 1 : 0) > 0;
            }
            if (sel) atomicOr(&s_sel[d >> 5], 1u << (d & 31));
        }
    }
    __syncthreads();  // the cut buckets' keys are complete
    // rank the designs of the cut buckets: the smaller priorities of a bucket
    // counted four to an LDS read (the lanes of one bucket read the same
    // words); equal priorities, one pair in 2^32, go by the design
    for (int sl = tid; sl < ncut; sl += NT) {
        const uint32_t who = kwho[sl], my = kpri[sl];
        if (who == ~0u) continue;
        const int r = (int)(who >> 16), d = (int)(who & 0xFFFFu), l0 = s_l0[r];
        const int kk = s_kp[r] - (l0 >= 0 ? 1 : 0), off = s_co[r], nr = s_cr[r].y;
        const uint32_t pl0 = s_pl0[r];
        const u32x4 *kq = (const u32x4 *)(kpri + off);
        int rank = 0, same = 0;
#pragma unroll 4
        for (int i = 0; i < nr; i += 4) {
            const u32x4 k = kq[i >> 2];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                rank += (int)(k[v] < my);
                same += (int)(k[v] == my);
            }
        }
        if (same > 1)
            for (int i = 0; i < nr; ++i) rank += (int)(kpri[off + i] == my && kwho[off + i] < who);
        if (d == l0) continue;
        // the level-0 pick of the bucket is not part of the rest
        if (l0 >= 0 && (pl0 < my || (pl0 == my && l0 < d))) --rank;
        if (rank < kk) atomicOr(&s_sel[d >> 5], 1u << (d & 31));
    }
    __syncthreads();  // the picks are complete
    // (pools of at most PLACE_NICHE_POOL designs: at most 32 words)
    if (tid < W) gstore(selm + tid, sm | (uint64_t)s_sel[2 * tid] | ((uint64_t)s_sel[2 * tid + 1] << 32));
}

// Initial state after k_design<INIT>: the first N designs survive, extreme points
// from the first designs (main.cu:101, 106-113).
__global__ void k_init_state(const DevJob *__restrict__ jobs) {
    const DevJob &J = jobs[blockIdx.x];
    SelState *st = J.st;
    for (int w = threadIdx.x; w < J.W; w += blockDim.x) {
        const int n = J.N - 64 * w;
        J.selm[w] = n >= 64 ? ~0ull : (n > 0 ? (1ull << n) - 1ull : 0ull);
    }
    for (int i = threadIdx.x; i < J.P; i += blockDim.x) J.front_of[i] = -1;
    // (a job initialised again keeps the points of its last selection until
    // the next one)
    const uint32_t from = st->gen & 1u;
    if (threadIdx.x < NOBJ && from) {
        st->res[0].ideal[threadIdx.x] = st->res[1].ideal[threadIdx.x];
        st->res[0].worst[threadIdx.x] = st->res[1].worst[threadIdx.x];
        st->res[0].nadir[threadIdx.x] = st->res[1].nadir[threadIdx.x];
    }
    __syncthreads();
    if (threadIdx.x < NOBJ * NOBJ) {
        const int e = threadIdx.x / NOBJ, k = threadIdx.x % NOBJ;
        st->res[0].ext[threadIdx.x] = (e < J.N) ? J.obj[0][(size_t)e * NOBJ + k] : 0.f;
    }
    if (threadIdx.x == 0) {
        SelRes &r = st->res[0];
        r.n_cut = r.hyp = r.ranked = r.last = r.base = 0;
        st->gen = 0;
        st->cds_scanned = 0;
    }
}

// Clear the dominator counts and selection accumulators before a standalone
// sort (the generation loop clears them
// inside k_design<OFFSPRING>).
__global__ void k_zero_np(const DevJob *__restrict__ jobs) {
    const DevJob &J = jobs[blockIdx.x];
    for (int i = threadIdx.x; i < J.P; i += blockDim.x) J.np[i] = 0;
    if (threadIdx.x < ACC_WORDS) ((uint32_t *)J.acc)[threadIdx.x] = acc_clear_word(threadIdx.x);
    clear_niche(J, threadIdx.x, blockDim.x);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
hipError_t launch_design(int mode, const DevJob *jobs, const int2 *items, int n, size_t lds, hipStream_t s,
                         uint2 *stem_list, int32_t *stem_ctl, StemList sl, int item_base, int threads) {
    if (n <= 0) return hipSuccess;
    switch (mode) {
    case 0: hipLaunchKernelGGL((k_design<0, 256, 6>), dim3(n), dim3(256), lds, s, jobs, items, nullptr, nullptr, 1, 0, item_base); break;
    case 1: hipLaunchKernelGGL((k_design<1, 256, 6>), dim3(n), dim3(256), lds, s, jobs, items, nullptr, nullptr, 1, 0, 0); break;
    default:
        if (!stem_list || !stem_ctl || sl.cap < 0 || sl.group <= 0 || sl.groups > STEM_MAX_GROUPS || item_base < 0)
            return hipErrorInvalidValue;
        if (threads == 256 && n > DESIGN_MANY)
            hipLaunchKernelGGL((k_design<2, 256, 8>), dim3(n), dim3(256), lds, s, jobs, items, stem_list, stem_ctl,
                               sl.group, sl.cap, item_base);
        else if (threads == 256)
            hipLaunchKernelGGL((k_design<2, 256, 6>), dim3(n), dim3(256), lds, s, jobs, items, stem_list, stem_ctl,
                               sl.group, sl.cap, item_base);
        else if (threads == 512)
            hipLaunchKernelGGL((k_design<2, 512, 6>), dim3(n), dim3(512), lds, s, jobs, items, stem_list, stem_ctl,
                               sl.group, sl.cap, item_base);
        else
            return hipErrorInvalidValue;
        break;
    }
    return hipGetLastError();
}
hipError_t launch_fetch(void *dst, const void *src, size_t bytes, hipStream_t s) {
    const uint32_t words = (uint32_t)((bytes + 15) / 16);
    if (!words) return hipSuccess;
    hipLaunchKernelGGL(k_fetch, dim3((words + 255) / 256), dim3(256), 0, s, (u32x4 *)dst, (const u32x4 *)src, words);
    return hipGetLastError();
}
hipError_t launch_read(const DevJob *job, uint8_t *rows, void *rest, size_t rest_bytes, size_t first, size_t bytes, hipStream_t s) {
    const size_t g = (bytes + 4095) / 4096, n = g + (rest ? (rest_bytes + 1023) / 1024 : 0);
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_read, dim3((unsigned)n), dim3(256), 0, s, job, rows, (uint32_t *)rest, (uint64_t)first, (uint64_t)bytes, (uint32_t)g);
    return hipGetLastError();
}
hipError_t launch_stem(const DevJob *jobs, const int2 *items, int n, int mg, size_t lds, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if ((int64_t)n * mg <= STEM_FEW)
        hipLaunchKernelGGL((k_stem<256, 2048>), dim3(n * mg), dim3(256), lds + seek_more_bytes(2048, 256), s, jobs, items, mg);
    else
        hipLaunchKernelGGL((k_stem<128, 1024>), dim3(n * mg), dim3(128), lds + seek_more_bytes(1024, 128), s, jobs, items, mg);
    return hipGetLastError();
}
hipError_t launch_stem_list(const DevJob *jobs, const int2 *items, int n, int mg, int longest, const uint2 *stem_list,
                            const int32_t *stem_ctl, StemList sl, int waves, size_t lds, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (!stem_list || !stem_ctl || waves < 5 || waves > 8 || sl.groups > STEM_MAX_GROUPS) return hipErrorInvalidValue;
    if (sl.cap == 0) {
        hipLaunchKernelGGL((k_stem_each<256, 2048>), dim3(n * mg), dim3(256), lds + seek_more_bytes(2048, 256), s, jobs, items, mg);
        return hipGetLastError();
    }
    const int capacity = sl.groups * sl.cap;
    // workgroups take the entries round-robin, so every one should be
    // resident from the start: per CU, `waves` waves per SIMD or what the
    // registers and the LDS (dynamic and static) hold, as the runtime counts it
    auto go = [&](auto kern, int heads, int threads) -> hipError_t {
        size_t bytes = lds + seek_more_bytes(heads, threads);
        if (bytes < 4 * ((size_t)sl.groups + 1)) bytes = 4 * ((size_t)sl.groups + 1);  // the prefix sums share the planes' LDS
        int fit = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, (const void *)kern, threads, bytes) != hipSuccess || fit < 1) fit = 1;
        const int most = waves * 256 / threads, per_cu = fit < most ? fit : most;
        const int grid = capacity < STEM_CUS * per_cu ? capacity : STEM_CUS * per_cu;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), bytes, s, jobs, stem_list, stem_ctl, sl.groups, sl.cap);
        return hipGetLastError();
    };
    return stem_path(n, mg, longest) == STEM_PATH_FEW ? go(k_stem_list<256, 2048>, 2048, 256) : go(k_stem_list<128, 1024>, 1024, 128);
}
hipError_t launch_stem_finish(const DevJob *jobs, const int2 *items, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stem_finish, dim3((n + 255) / 256), dim3(256), 0, s, jobs, items, n);
    return hipGetLastError();
}
hipError_t launch_sort(const SortArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_sort_tiles, dim3(a.W * (a.W + 1) / 2), dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int threads = a.P <= 256 ? 256 : a.P <= 512 ? 512 : 1024;
    hipLaunchKernelGGL(k_sort_fronts, dim3(1), dim3(threads), 0, s, a);
    return hipGetLastError();
}
hipError_t launch_dominance(const DevJob *jobs, const int4 *items, int n, bool finish, int32_t *stem_ctl, int ctl_n, int rows,
                            hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const int g = (n + rows / 64 - 1) / (rows / 64);
    switch (rows) {
    case 64: hipLaunchKernelGGL(k_dominance<64>, dim3(g), dim3(256), 0, s, jobs, items, n, finish, stem_ctl, ctl_n); break;
    case 128: hipLaunchKernelGGL(k_dominance<128>, dim3(g), dim3(256), 0, s, jobs, items, n, finish, stem_ctl, ctl_n); break;
    case 256: hipLaunchKernelGGL(k_dominance<256>, dim3(g), dim3(256), 0, s, jobs, items, n, finish, stem_ctl, ctl_n); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
hipError_t launch_fronts(const DevJob *jobs, int njobs, int max_pool, int threads, hipStream_t s) {
    if (threads != 256 && threads != 512 && threads != 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_front0, dim3(njobs, (max_pool + FRONT0_THREADS - 1) / FRONT0_THREADS), dim3(FRONT0_THREADS), 0, s,
                       jobs);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_fronts, dim3(njobs), dim3(threads), 0, s, jobs);
    return hipGetLastError();
}
hipError_t launch_associate(const DevJob *jobs, const int2 *items, int n, int designs, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    switch (designs) {
    case 4: hipLaunchKernelGGL((k_associate<4, 64>), dim3(n), dim3(256), 0, s, jobs, items); break;
    case 8: hipLaunchKernelGGL((k_associate<8, 64>), dim3(n), dim3(512), 0, s, jobs, items); break;
    case 16: hipLaunchKernelGGL((k_associate<16, 64>), dim3(n), dim3(1024), 0, s, jobs, items); break;
    case 32: hipLaunchKernelGGL((k_associate<32, 8>), dim3(n), dim3(256), 0, s, jobs, items); break;
    case 64: hipLaunchKernelGGL((k_associate<64, 8>), dim3(n), dim3(512), 0, s, jobs, items); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
hipError_t launch_front_associate(const DevJob *jobs, const int2 *items, int n, int designs, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    switch (designs) {
    case 4: hipLaunchKernelGGL((k_front_associate<4, 64>), dim3(n), dim3(256), 0, s, jobs, items); break;
    case 8: hipLaunchKernelGGL((k_front_associate<8, 64>), dim3(n), dim3(512), 0, s, jobs, items); break;
    case 16: hipLaunchKernelGGL((k_front_associate<16, 64>), dim3(n), dim3(1024), 0, s, jobs, items); break;
    case 32: hipLaunchKernelGGL((k_front_associate<32, 8>), dim3(n), dim3(256), 0, s, jobs, items); break;
    case 64: hipLaunchKernelGGL((k_front_associate<64, 8>), dim3(n), dim3(512), 0, s, jobs, items); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
bool shapes_valid(const Shapes &h) {
    return h.design_split >= 0 && (h.design_threads == 256 || h.design_threads == 512) && h.stem_waves >= 5 &&
           h.stem_waves <= 8 &&
           (h.dom_rows == 64 || h.dom_rows == 128 || h.dom_rows == 256) &&
           (h.fronts_threads == 256 || h.fronts_threads == 512 || h.fronts_threads == 1024) &&
           (h.assoc_designs == 4 || h.assoc_designs == 8 || h.assoc_designs == 16 || h.assoc_designs == 32 ||
            h.assoc_designs == 64) &&
           (h.niche_threads == 256 || h.niche_threads == 512 || h.niche_threads == 1024);
}
size_t niche_lds_bytes(int P) { return (size_t)8 * P; }

// The dynamic-LDS limit of a kernel is an attribute of the process, shared by
// every job, batch and captured graph that launches it, so it only ever
// rises: a job created after a larger one must not lower the limit under the
// larger one's launches.  `held` is the limit set so far for that group of
// kernels; `apply` sets the attribute on each of them.
template <class F>
static hipError_t raise_lds_limit(size_t &held, size_t bytes, F apply) {
    static std::mutex mu;
    std::lock_guard<std::mutex> lk(mu);
    if (bytes <= held) return hipSuccess;
    const hipError_t e = apply((int)bytes);
    if (e == hipSuccess) held = bytes;
    return e;
}
static size_t g_design_lds = 0, g_stem_lds = 0, g_niche_lds = 0, g_place_niche_lds = 0;

hipError_t set_niche_lds_limit(int max_pool, int max_refs) {
    const size_t bytes = niche_lds_need(max_pool, max_refs);
    if (bytes <= NICHE_LDS_PLAIN) return hipSuccess;
    const bool place = takes_place_niche(max_pool, max_refs);
    const void *const kern = place ? (const void *)k_place_niche : (const void *)k_niche;
    return raise_lds_limit(place ? g_place_niche_lds : g_niche_lds, bytes, [kern](int b) {
        return hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, b);
    });
}
hipError_t launch_niche(const DevJob *jobs, int njobs, int max_pool, int max_refs, int threads, hipStream_t s) {
    if (threads != 256 && threads != 512 && threads != 1024) return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    if (max_refs > NICHE_STAGE) {
        hipLaunchKernelGGL(k_levels, dim3(njobs), dim3(256), 0, s, jobs);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (takes_place_niche(max_pool, max_refs)) {  // one workgroup per job
        hipLaunchKernelGGL(k_place_niche, dim3(njobs), dim3(threads), place_niche_lds_bytes(max_pool, max_refs), s, jobs);
        return hipGetLastError();
    }
    const dim3 grid(njobs, (max_pool + threads - 1) / threads);
    hipLaunchKernelGGL(k_place, grid, dim3(threads), 0, s, jobs);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_niche, grid, dim3(threads), niche_lds_bytes(max_pool), s, jobs);
    return hipGetLastError();
}
hipError_t launch_init_state(const DevJob *jobs, int njobs, hipStream_t s) {
    hipLaunchKernelGGL(k_init_state, dim3(njobs), dim3(256), 0, s, jobs);
    return hipGetLastError();
}
hipError_t launch_zero_np(const DevJob *jobs, int njobs, hipStream_t s) {
    hipLaunchKernelGGL(k_zero_np, dim3(njobs), dim3(256), 0, s, jobs);
    return hipGetLastError();
}

hipError_t set_design_lds_limit(size_t bytes) {
    return raise_lds_limit(g_design_lds, bytes, [](int b) {
        const void *fns[] = {(const void *)k_design<0, 256, 6>, (const void *)k_design<1, 256, 6>,
                             (const void *)k_design<2, 256, 6>,
                             (const void *)k_design<2, 256, 8>, (const void *)k_design<2, 512, 6>};
        for (const void *f : fns) {
            const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, b);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    });
}
hipError_t set_stem_lds_limit(size_t bytes) {
    return raise_lds_limit(g_stem_lds, bytes, [](int b) {
        const void *fns[] = {(const void *)k_stem<128, 1024>,      (const void *)k_stem<256, 2048>,
                             (const void *)k_stem_each<256, 2048>, (const void *)k_stem_list<128, 1024>,
                             (const void *)k_stem_list<256, 2048>};
        for (const void *f : fns) {
            const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, b);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    });
}

}  // namespace cd
