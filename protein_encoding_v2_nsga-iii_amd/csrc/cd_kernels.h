// cd_kernels.h -- host-side launchers of the codon-design kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "cd_layout.h"

namespace cd {

enum DesignMode { MODE_INIT = 0, MODE_EVAL = 1, MODE_OFFSPRING = 2 };

constexpr size_t LDS_BYTES = 160 * 1024;  // per workgroup on gfx950
constexpr int DOM_ROWS = 64;               // tile rows per k_dominance workgroup of the standalone sort and selection
constexpr int ASSOC_DESIGNS = 4;           // designs per k_associate workgroup (a wave each), the smallest shape
// The stem kernels' shapes by the CDS of a launch (designs x the largest m).
// Few: the latency of a search counts, 256 threads and 2048 chains each; many:
// the searches resident per CU do, which the LDS bounds: 128 and 1024.
// Listed offspring, 256 x 2048 against 128 x 1024: 1024 children of 2004
// codons 67.7, 69.3 us a generation, 4096 of 12008 (32768 CDS) 240, 247, the
// 64-job mix (42 240 children) 887, 833.  Chains, 256 threads, 512 / 1024 /
// 2048 / 4096: 251 / 242 / 238 / 245 us on the 4096 children.
constexpr int STEM_FEW = 2048;    // initialisation and evaluation
constexpr int STEM_MANY = 65536;  // offspring
// Listed offspring of CDS of at most this many codons take the second shape
// whatever their number: their indexes are small, so twice as many searches
// reside with it.  5 / 16 jobs of 4 x 1024 CDS, 256 x 2048 against 128 x 1024:
// 101 codons 122.8 / 111.4 and 245.7 / 211.3 us a generation, 600 141.4 / 138.1
// and 298.2 / 281.7, 900 147.3 / 140.7 and 333.9 / 308.4, 1300 163.7 / 171.8 and
// 394.1 / 408.3.
constexpr int STEM_SHORT = 1024;
// Offspring launches up to this size have no list of the changed CDS (the
// figures stand at k_stem_each).
constexpr int STEM_EACH = 16384;
constexpr int STEM_CUS = 256;              // compute units of an MI355X: k_stem_list runs a resident grid

// Launch shapes of one generation's kernels.  Every shape gives the same
// results -- a shape only changes how the work is split over workgroups and
// lanes -- so the autotuner may pick any of them while a job runs.
struct Shapes {
    int design_split;    // k_design LDS bytes up to which children launch apart from the rest (0: one launch)
    int design_threads;  // k_design workgroup of the other children (a lone job: all): 256 or 512 threads
    int stem_waves;      // k_stem_list waves per SIMD, at most: 5, 6, 7 or 8
    int dom_rows;        // k_dominance tile rows per workgroup (dom_rows / 64 tiles of 64 x 64): 64, 128 or 256
    int fronts_threads;  // k_fronts workgroup: 256, 512 or 1024 threads
    int assoc_designs;   // designs per k_associate workgroup: 4, 8 or 16 (a wave each), 32 or 64 (eight lanes each)
    int niche_threads;   // niching workgroup (k_place_niche, or k_place and k_niche above 2048 designs): 256, 512 or 1024 threads
};
// Untuned shapes of a lone job, and of a batch or served tick (the k_design
// and k_associate fields by the work's sizes: untuned_shapes).
constexpr Shapes SHAPES_JOB = {0, 512, 8, 64, 512, 4, 1024};
constexpr Shapes SHAPES_BATCH = {0, 256, 8, 128, 1024, 4, 1024};
bool shapes_valid(const Shapes &s);
// More children than this in a launch of 256-thread workgroups (seven a CU
// are resident at 68 VGPRs) and k_design is throughput-bound: it then takes
// the build for eight waves per SIMD, which spills a few registers (64-job
// mix 426 -> 397 us).  Microseconds of k_design for six / eight waves a SIMD,
// children of 202 codons: 1536 of them 15.8 / 16.9, 2100 20.5 / 20.2, 3072 24.6 /
// 24.3, 4096 29.8 / 28.7, 6000 39.4 / 37.2; of 2004: 1536 21.5 / 22.5, 2100 26.7 /
// 26.5, 4096 39.2 / 38.2; of 12 008: 2100 64.7 / 67.6, 3072 76.2 / 78.7, 4096 90.4 /
// 91.0; batches of 50 to 950 residues, 2048 children 23.1 / 23.7, 2560 30.7 / 34.0,
// 4096 42.2 / 41.4, 8192 74.1 / 69.0.
constexpr int DESIGN_MANY = 2048;

size_t design_lds_bytes(int L, int m);
size_t design_bytes_accepted(int L, int m);  // at most LDS_BYTES for a job to be accepted
size_t stem_lds_bytes(int L);
size_t cds_plane_bytes(int L);  // one CDS in the job's plane buffer: its sequence's bit planes and its change mask
hipError_t set_design_lds_limit(size_t bytes);
hipError_t set_stem_lds_limit(size_t bytes);

// The changed CDS of an offspring generation, in sublists of consecutive
// children (`group` of them, at least 64, at most STEM_MAX_GROUPS sublists),
// each with its own count in stem_ctl, so that the children's appends spread
// over many counters and the sublists in order keep the children list's
// order (longest jobs first); a sublist holds `cap` entries.
constexpr int STEM_MAX_GROUPS = 2048;
struct StemList {
    int group, groups, cap;
};
inline StemList stem_list_geom(int n_items, int mg) {
    StemList g;
    g.group = (n_items + STEM_MAX_GROUPS - 1) / STEM_MAX_GROUPS;
    if (g.group < 64) g.group = 64;
    g.groups = (n_items + g.group - 1) / g.group;
    g.cap = g.group * mg;
    return g;
}
// The stem kernel of a generation of n children of up to mg CDS, the longest of
// `longest` codons.
enum StemPath { STEM_PATH_EACH = 0, STEM_PATH_FEW = 1, STEM_PATH_MANY = 2 };  // k_stem_each, k_stem_list's two shapes
inline StemPath stem_path(int n_items, int mg, int longest) {
    const int64_t cds = (int64_t)n_items * mg;
    return cds <= STEM_EACH ? STEM_PATH_EACH : cds <= STEM_MANY && longest > STEM_SHORT ? STEM_PATH_FEW : STEM_PATH_MANY;
}
// The list of a generation's launches; cap 0: none, k_stem_each takes every CDS.
inline StemList stem_list_plan(int n_items, int mg) {
    StemList g = stem_list_geom(n_items, mg);
    if ((int64_t)n_items * mg <= STEM_EACH) g.cap = 0;
    return g;
}
// k_stem_list's dynamic LDS holds the sublists' prefix sums (at most this
// many bytes) before it holds a CDS's planes and tables
constexpr size_t STEM_PRE_BYTES = 4 * (STEM_MAX_GROUPS + 1);
// (and beside them the search's chain heads and the queues of four waves)
inline size_t stem_list_lds(size_t stem_lds) {
    const size_t b = stem_lds + 4 * (2048 + 1408);
    return b > STEM_PRE_BYTES ? b : STEM_PRE_BYTES;
}
inline size_t stem_list_entries(int n_items, int mg) {
    const StemList g = stem_list_geom(n_items, mg);
    return (size_t)g.groups * g.cap;
}
// items: (job, design or child).  The offspring mode lists every changed CDS
// in the sublists (entry ((item_base + item) << 4) | c; sl =
// stem_list_geom of the whole children list) and counts them in stem_ctl;
// the three are required there.  item_base: the position of items[0] in the
// children list k_stem_list reads.  threads: the offspring mode's workgroup,
// 256 or 512 (initialisation and evaluation take 256).
hipError_t launch_design(int mode, const DevJob *jobs, const int2 *items, int n, size_t lds, hipStream_t s,
                         uint2 *stem_list = nullptr, int32_t *stem_ctl = nullptr, StemList sl = StemList{0, 0, 0},
                         int item_base = 0, int threads = 256);
// (MODE_INIT: item_base 1 when the pool has not been written before)
// bytes (rounded up to 16) from pinned host memory to the device, both 16-byte
// aligned
hipError_t launch_fetch(void *dst, const void *src, size_t bytes, hipStream_t s);
// what a caller reads of a job to pinned host memory: the bytes [first, first +
// bytes) of the pool's packed synonym indices to rows (first a multiple of 16;
// room for whole 16-byte words), and, unless rest is null, the arrays of
// ReadRest one after the other
struct ReadRest {
    size_t selm, front, obj, idx, pql, bytes;  // offsets; the selection state comes first
    ReadRest(int P, int W)
        : selm(sizeof(SelState)), front(selm + 8 * (size_t)W), obj(front + 4 * (size_t)P), idx(obj + 24 * (size_t)P),
          pql(idx + 12 * (size_t)P), bytes(pql + 16 * (size_t)P) {}
};
hipError_t launch_read(const DevJob *job, uint8_t *rows, void *rest, size_t rest_bytes, size_t first, size_t bytes, hipStream_t s);
// initialisation and evaluation: a workgroup per (item, CDS c < mg): stem of
// each CDS of the items' designs
hipError_t launch_stem(const DevJob *jobs, const int2 *items, int n, int mg, size_t lds, hipStream_t s);
// offspring generations: stem of each CDS the offspring k_design listed
// (the n items and sl as given to it), on as many workgroups as are resident at
// once (STEM_CUS x what `waves`, 5 to 8 waves per SIMD, and the LDS allow), at
// most the entries there can be; longest: codons of the longest CDS;
// launch_dominance with the same stem_ctl and sl.groups clears the counts
hipError_t launch_stem_list(const DevJob *jobs, const int2 *items, int n, int mg, int longest, const uint2 *stem_list,
                            const int32_t *stem_ctl, StemList sl, int waves, size_t lds, hipStream_t s);
// one thread per item: objective 5, clears the marks
hipError_t launch_stem_finish(const DevJob *jobs, const int2 *items, int n, hipStream_t s);
// a sort of P objective vectors obj [P][6] (device memory) until at least N are
// ranked: front_of [P], *n_fronts; scratch: dom [W][P], any [W][W], W = (P + 63) / 64
struct SortArgs {
    const float *obj;
    int32_t *front_of, *n_fronts;
    uint64_t *dom, *any;
    int P, N, W;
};
hipError_t launch_sort(const SortArgs &a, hipStream_t s);
// items: (job, 64b, w, 0), the 64 x 64 tiles b <= w, rows / 64 (rows: 64, 128 or 256) per workgroup.  finish: the offspring generation, whose children's stem
// objective (and stem records) k_dominance completes in place of
// launch_stem_finish; stem_ctl (or null): the ctl_n changed-CDS counts of
// that generation's k_design, cleared for the next one
hipError_t launch_dominance(const DevJob *jobs, const int4 *items, int n, bool finish, int32_t *stem_ctl, int ctl_n,
                            int rows, hipStream_t s);
// k_front0 (grid: jobs x chunks of FRONT0_THREADS designs of the largest
// pool, max_pool), then k_fronts (one workgroup of `threads` (256, 512 or
// 1024) per job)
constexpr int FRONT0_THREADS = 256;
hipError_t launch_fronts(const DevJob *jobs, int njobs, int max_pool, int threads, hipStream_t s);
// items: (job, first design), `designs` designs per item: 4, 8 or 16 (a wave each), 32 or 64 (eight lanes each)
hipError_t launch_associate(const DevJob *jobs, const int2 *items, int n, int designs, hipStream_t s);
// launch_fronts and launch_associate in one launch, for pools of at most
// FUSED_POOL designs
constexpr int FUSED_POOL = 2048;
// Taken while all jobs' pools together hold at most FUSED_TOTAL designs, 512
// workgroups of 8: each workgroup repeats the job's settling, which costs
// nothing while the workgroups run side by side and more than the two launches
// it saves once they queue.  Microseconds of the fronts and association, fused
// against apart: pool 1024 19.3 / 20.7, 4096 24.8 / 24.6, 8192 37.0 / 28.1.
constexpr int FUSED_TOTAL = 4096;
inline bool fuse_fronts(int max_pool, int pool) { return max_pool <= FUSED_POOL && pool <= FUSED_TOTAL; }
hipError_t launch_front_associate(const DevJob *jobs, const int2 *items, int n, int designs, hipStream_t s);
// Pools of at most PLACE_NICHE_POOL designs with at most NICHE_STAGE
// reference points: k_place_niche (one workgroup of `threads` per job,
// place_niche_lds_bytes(max_pool, max_refs) of dynamic LDS).  Otherwise k_levels (one
// workgroup per job) when some job has more reference points than
// NICHE_STAGE (max_refs), then k_place and k_niche (grid: jobs x chunks of
// `threads` (256, 512 or 1024) designs of the largest pool, max_pool; k_niche
// takes niche_lds_bytes(max_pool) of dynamic LDS)
constexpr int PLACE_NICHE_POOL = 2048;
// slots of its cut list: every design of the pool, and up to three pads a bucket
__host__ __device__ inline int place_niche_slots(int P, int R) { return P + 3 * (R < P ? R : P); }
inline size_t place_niche_lds_bytes(int P, int R) { return (size_t)8 * ((place_niche_slots(P, R) + 3) & ~3); }
size_t niche_lds_bytes(int P);
// The rule above, and the dynamic LDS of the niching kernel it takes; that
// kernel's limit is raised above NICHE_LDS_PLAIN.  Of that kernel only:
// k_place_niche's static arrays take 37 KiB, so it cannot have the 128 KB that
// k_niche takes for a pool of 16384.
constexpr size_t NICHE_LDS_PLAIN = 24 * 1024;
inline bool takes_place_niche(int max_pool, int max_refs) { return max_pool <= PLACE_NICHE_POOL && max_refs <= NICHE_STAGE; }
inline size_t niche_lds_need(int P, int R) {
    return takes_place_niche(P, R) ? place_niche_lds_bytes(P, R) : niche_lds_bytes(P);
}
hipError_t set_niche_lds_limit(int max_pool, int max_refs);
hipError_t launch_niche(const DevJob *jobs, int njobs, int max_pool, int max_refs, int threads, hipStream_t s);
hipError_t launch_init_state(const DevJob *jobs, int njobs, hipStream_t s);
hipError_t launch_zero_np(const DevJob *jobs, int njobs, hipStream_t s);

}  // namespace cd
