// cd_api.hip -- C ABI of the codon-design engine (include/codon_nsga3.h):
// job lifecycle, table preparation, work lists and the per-generation
// hipGraph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <utility>
#include <mutex>
#include <string>
#include <vector>

#include "cd_host.h"

using cdhost::fail;
using cdhost::Launch;

namespace {

const int8_t SYN_START[21] = {0, 4, 6, 8, 10, 12, 16, 18, 21, 23, 29, 30, 32, 36, 38, 44, 50, 54, 58, 59, 61};
const int8_t SYN_NUM[21] = {4, 2, 2, 2, 2, 4, 2, 3, 2, 6, 1, 2, 4, 2, 6, 6, 4, 4, 1, 2, 3};
const char AMINO[] = "ACDEFGHIKLMNPQRSTVWYZ";
// Standard genetic code, codons enumerated U C A G per position ('Z' = stop).
const char CODE[] = "FFLLSSSSYYZZCCZWLLLLPPPPHHQQRRRRIIIMTTTTNNKKSSRRVVVVAAAADDEEGGGG";

int nt_code(char c) {
    switch (c) {
    case 'A': return 0;
    case 'C': return 1;
    case 'G': return 2;
    case 'U': return 3;
    default: return -1;
    }
}

char translate(const uint8_t *c3) {  // codes A0 C1 G2 U3 -> index in U C A G order
    static const int ucag[4] = {2, 1, 3, 0};
    return CODE[ucag[c3[0]] * 16 + ucag[c3[1]] * 4 + ucag[c3[2]]];
}

// Tables of a job indexed by codon code (first base << 4 | second << 2 |
// third, A=0 C=1 G=2 U=3), the form k_design works in.
struct HostTables {
    uint8_t code[64];        // code of each codon of the table
    int64_t lw6[64];         // 2^40-scaled log weights
    uint64_t syn6[64];       // synonym words (DevJob::lw6)
    int64_t cpfx6[64 * 64];  // 2^40-scaled pair scores, 0 where either codon is a stop
    float cps6[64 * 64];     // pair scores, 0 where either codon is a stop
    uint64_t stop6;          // bit per code: the table's last three codons
};

int build_tables(const cd_tables &t, HostTables &h) {
    if (!t.codons || !t.weights || !t.cps) return fail(CD_E_INVALID, "null table pointer");
    uint8_t nt[192];
    for (int i = 0; i < 192; ++i) {
        const int c = nt_code(t.codons[i]);
        if (c < 0) return fail(CD_E_INVALID, "codon table letters must be A, C, G or U");
        nt[i] = (uint8_t)c;
    }
    for (int a = 0; a < 21; ++a)
        for (int g = SYN_START[a]; g < SYN_START[a] + SYN_NUM[a]; ++g)
            if (translate(&nt[3 * g]) != AMINO[a])
                return fail(CD_E_INVALID, "codon table block does not encode its amino acid");
    uint64_t seen = 0;
    for (int g = 0; g < 64; ++g) {
        h.code[g] = (uint8_t)(nt[3 * g] << 4 | nt[3 * g + 1] << 2 | nt[3 * g + 2]);
        seen |= 1ull << h.code[g];
    }
    if (seen != ~0ull) return fail(CD_E_INVALID, "codon table lists a codon twice");
    for (int a = 0; a < 21; ++a)
        for (int j = 0; j < SYN_NUM[a]; ++j) {
            uint64_t v = ((uint64_t)SYN_NUM[a] << 40) | ((uint64_t)j << 44);
            for (int i = 0; i < SYN_NUM[a]; ++i) v |= (uint64_t)h.code[SYN_START[a] + i] << (i < 5 ? 6 * i : 32);
            h.syn6[h.code[SYN_START[a] + j]] = v;
        }
    h.stop6 = 0;
    for (int g = 61; g < 64; ++g) h.stop6 |= 1ull << h.code[g];
    for (int g = 0; g < 64; ++g) {
        const float w = t.weights[g];
        if (!(w > 0.f) || w > 1.f) return fail(CD_E_INVALID, "CAI weights must lie in (0, 1]");
        h.lw6[h.code[g]] = llrint(std::log((double)w) * 0x1p40);
    }
    std::memset(h.cpfx6, 0, sizeof(h.cpfx6));
    std::memset(h.cps6, 0, sizeof(h.cps6));
    for (int a = 0; a < 61; ++a)
        for (int b = 0; b < 61; ++b) {
            const float v = t.cps[a * 61 + b];
            if (!(std::fabs(v) <= 1000.f)) return fail(CD_E_INVALID, "codon-pair scores must be finite and |v| <= 1000");
            h.cps6[h.code[a] * 64 + h.code[b]] = v;
            h.cpfx6[h.code[a] * 64 + h.code[b]] = llrint((double)v * 0x1p40);
        }
    return CD_OK;
}

// Das-Dennis simplex lattice in the order of combinationRepetition
// (sorting.cuh:1285-1354): multisets of H objectives in lexicographic order,
// coordinate = H-fold float sum of 1/H over the objective's multiplicity.
// Rows of REF_STRIDE floats: the coordinates, then the sum of their squares
// in objective order (perp_dist's divisor, rounded term by term as on the
// device: no contraction), then 0.
std::vector<float> das_dennis(int H) {
    std::vector<float> out;
    std::vector<int> x(H, 0);
    const float step = 1.f / (float)H;
    while (true) {
        float v[6] = {0, 0, 0, 0, 0, 0};
        for (int i = 0; i < H; ++i) v[x[i]] += step;
        out.insert(out.end(), v, v + 6);
        float den = 0.f;
        for (float w : v) den += w * w;
        out.push_back(den);
        out.push_back(0.f);
        int i = H - 1;
        while (i >= 0 && x[i] == 5) --i;
        if (i < 0) break;
        const int nv = x[i] + 1;
        for (int j = i; j < H; ++j) x[j] = nv;
    }
    return out;
}

int64_t n_ref(int H) {
    int64_t r = 1;
    for (int i = 1; i <= 5; ++i) r = r * (H + i) / i;
    return r;
}

// Bernoulli threshold: a 32-bit draw x succeeds when x < floor(p * 2^32).
uint64_t bern_threshold_host(float p) {
    double t = (double)p * 4294967296.0;
    if (!(t > 0.0)) return 0;
    if (t >= 18446744073709551615.0) return ~0ull;
    return (uint64_t)t;
}

size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }

struct Sizes {
    size_t total = 0;
    size_t add(size_t b) {
        size_t o = total;
        total += a256(b);
        return o;
    }
};

}  // namespace

namespace {

// What a descriptor is set up for: a job, one evaluation of P designs, or one
// selection from P objective vectors (a sort is the first part of one).
enum class Use { Job, Evaluate, Select };

// Lay out every device buffer of a job in one allocation.  The regions the
// host fills come first, `head` bytes in all, and go up in one transfer; what
// a single selection gives back (st, selm, front) lies together and comes down
// in one.
struct Layout {
    size_t pos, code, lw6, cpfx6, cps6, ref, genome[2], obj[2], oidx[2], pql[2], cst[2], hdp[2], planes, stem_max, slist,
        sctl,
        front,
        np, dom,
        ref_of, niche, st, acc, ranked, selm, prio, cutl, cutr, self, off, domi, asc;
    size_t head, total;
};

Layout layout(int L, int m, int N, int P, int R, int W, int n_dom, int n_asc, Use use) {
    Sizes s;
    Layout o{};
    o.self = s.add(sizeof(cd::DevJob));
    if (use != Use::Select) {
        o.pos = s.add(2 * (size_t)cd::row_stride(L));
        o.code = s.add(64);
        o.lw6 = s.add(128 * 8);
        o.cpfx6 = s.add(64 * 64 * 8);
        o.cps6 = s.add(64 * 64 * 4);
        o.off = s.add((size_t)(use == Use::Job ? N : P) * sizeof(int2));
    }
    if (use != Use::Evaluate) {
        o.ref = s.add((size_t)R * cd::REF_STRIDE * 4);
        o.domi = s.add((size_t)n_dom * sizeof(int4));
        o.asc = s.add((size_t)n_asc * sizeof(int2));
    }
    if (use == Use::Select) {
        o.obj[0] = o.obj[1] = s.add((size_t)P * 6 * 4);
        o.st = s.add(sizeof(cd::SelState));
        o.head = s.total;
        o.selm = s.add((size_t)W * 8);
        o.front = s.add((size_t)P * 4);
    } else {
        o.head = s.total;
        for (int b = 0; b < (use == Use::Job ? 2 : 1); ++b) {
            if (use == Use::Job) {  // (an evaluation's rows and results are in pinned memory)
                o.obj[b] = s.add((size_t)P * 6 * 4);
                o.oidx[b] = s.add((size_t)P * 12);
                o.pql[b] = s.add((size_t)P * 16);
                o.genome[b] = s.add((size_t)P * m * cd::row_stride(L));
            }
            o.cst[b] = s.add((size_t)P * m * sizeof(cd::CdsStat));
            o.hdp[b] = s.add((size_t)P * (m * (m - 1) / 2) * 4);
        }
        o.planes = s.add((size_t)P * m * cd::cds_plane_bytes(L));
        o.stem_max = s.add((size_t)P * 4);
    }
    if (use == Use::Job) {
        o.slist = s.add(cd::stem_list_entries(N, m) * sizeof(uint2));
        o.sctl = s.add((size_t)cd::STEM_MAX_GROUPS * 4);
        o.st = s.add(sizeof(cd::SelState));
        o.selm = s.add((size_t)W * 8);
        o.front = s.add((size_t)P * 4);
    }
    if (use != Use::Evaluate) {
        o.np = s.add((size_t)P * 4);
        o.dom = s.add((size_t)P * W * 8);
        o.ref_of = s.add((size_t)P * 4);
        o.niche = s.add((size_t)cd::NICHE_INTS * R * 4);
        o.acc = s.add(sizeof(cd::SelAcc));
        o.ranked = s.add((size_t)W * 8);
        o.prio = s.add((size_t)P * 4);
        o.cutl = s.add((size_t)P * 8);
        o.cutr = s.add((size_t)P * 4);
    }
    o.total = s.total;
    return o;
}

// Room for the work lists of a job of pool P in any shape (the smallest
// group gives the most items; the domination tiles are the same in every
// shape).
void work_counts(int P, int W, int *n_dom, int *n_asc) {
    (void)P;
    *n_dom = W * (W + 1) / 2;
    *n_asc = (P + cd::ASSOC_DESIGNS - 1) / cd::ASSOC_DESIGNS;
}

// Domination tiles and association groups of one job (job index j) in the
// given shapes.  The tiles are the 64 x 64 blocks (row block b, column block
// w) with b <= w; k_dominance takes dom_rows / 64 of them per workgroup.
void job_lists(int P, int W, const cd::Shapes &sh, std::vector<int4> &dom, std::vector<int2> &asc, int j = 0) {
    for (int w = 0; w < W; ++w)
        for (int b = 0; b <= w; ++b) dom.push_back(make_int4(j, 64 * b, w, 0));
    for (int t = 0; t < (P + sh.assoc_designs - 1) / sh.assoc_designs; ++t)
        asc.push_back(make_int2(j, t * sh.assoc_designs));
}

int validate(const cd_job_desc *d) {
    if (!d) return fail(CD_E_INVALID, "null descriptor");
    // main.cu:485-489
    if (d->N <= 0) return fail(CD_E_INVALID, "population size N must be positive");
    if (d->m < 2 || d->m > cd::MAX_M) return fail(CD_E_INVALID, "CDS count m must be in [2, 16]");
    if (!(d->Pm >= 0.f && d->Pm <= 1.f)) return fail(CD_E_INVALID, "mutation probability must be in [0, 1]");
    if (d->L < 3 || d->L > 100000) return fail(CD_E_INVALID, "L (codons incl. stop) must be in [3, 100000]");
    if (d->H < 1 || n_ref(d->H) > (1 << 20)) return fail(CD_E_INVALID, "H must be >= 1 with at most 2^20 reference points");
    if (2LL * d->N > 64LL * cd::MAX_W) return fail(CD_E_INVALID, "pool 2N exceeds 16384");
    if (!d->aa) return fail(CD_E_INVALID, "null amino-acid sequence");
    for (int k = 0; k < d->L; ++k) {  // findAminoIndex, utils.cuh:60-86
        if (d->aa[k] < 0 || d->aa[k] > 20) return fail(CD_E_INVALID, "amino-acid index out of range");
        if ((d->aa[k] == 20) != (k == d->L - 1)) return fail(CD_E_INVALID, "the stop (20) must be exactly the last codon");
    }
    if (3LL * d->L >= (1 << 20)) return fail(CD_E_INVALID, "sequence too long for stem positions");
    if (cd::design_bytes_accepted(d->L, d->m) > cd::LDS_BYTES || cd::stem_list_lds(cd::stem_lds_bytes(d->L)) > cd::LDS_BYTES)
        return fail(CD_E_INVALID, "m*L too large for one workgroup's LDS (160 KiB)");
    return CD_OK;
}

// Memory a job frees stays in the device's stream-ordered pool for the next
// job instead of going back to the system at each synchronisation (set once
// per device).
hipError_t keep_pool_memory() {
    static std::mutex mu;
    static bool done[64] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= 64) return e;
    std::lock_guard<std::mutex> lk(mu);
    if (done[dev]) return hipSuccess;
    hipMemPool_t pool;
    e = hipDeviceGetDefaultMemPool(&pool, dev);
    uint64_t keep = ~0ull;
    if (e == hipSuccess) e = hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
    if (e == hipSuccess) done[dev] = true;
    return e;
}

// Streams of jobs that have ended, for the next ones: creating and destroying
// one costs about 50 us.  At most STREAMS_IDLE are kept, synchronised.
constexpr size_t STREAMS_IDLE = 16;
struct Streams {
    std::mutex mu;
    std::vector<std::pair<int, hipStream_t>> idle;  // (device, stream)
    hipError_t take(int *dev, hipStream_t *s) {
        const hipError_t e = hipGetDevice(dev);
        if (e != hipSuccess) return e;
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t i = idle.size(); i-- > 0;)
                if (idle[i].first == *dev) {
                    *s = idle[i].second;
                    idle.erase(idle.begin() + (ptrdiff_t)i);
                    return hipSuccess;
                }
        }
        return hipStreamCreateWithFlags(s, hipStreamNonBlocking);
    }
    void give(int dev, hipStream_t s) {
        {
            std::lock_guard<std::mutex> lk(mu);
            if (idle.size() < STREAMS_IDLE) {
                idle.push_back({dev, s});
                return;
            }
        }
        (void)hipStreamDestroy(s);
    }
};
Streams &streams() {  // (never destroyed: the runtime may be gone by then)
    static Streams *p = new Streams();
    return *p;
}

// `allocate` (a HIP allocation), and once more without the idle buffers of the
// one-shot calls (Shots) when memory has run out.
void drop_idle_shots();
template <class F>
hipError_t allocated(F allocate) {
    hipError_t e = allocate();
    if (e == hipSuccess) return e;
    (void)hipGetLastError();  // (or the next launch would report it)
    drop_idle_shots();
    e = allocate();
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

// The sizes of a descriptor's job (J->N, H, L, m, R, P, W), its layout and its
// tables.
int size_job(cd_job *J, const cd_job_desc *d, Use use, int P, Layout &o, HostTables &t) {
    J->selection_only = use == Use::Select;
    J->L = use == Use::Select ? 0 : d->L;
    J->m = use == Use::Select ? 0 : d->m;
    J->N = d->N;
    J->H = d->H;
    J->R = (int)n_ref(d->H);
    J->P = P;
    J->W = (P + 63) / 64;
    work_counts(J->P, J->W, &J->n_dom, &J->n_asc);
    o = layout(J->L, J->m, J->N, J->P, J->R, J->W, J->n_dom, J->n_asc, use);
    return use == Use::Select ? CD_OK : build_tables(d->tables, t);
}

// The descriptor and work lists of J in an allocation at base, and the image
// of its first o.head bytes (cleared by the caller).
void describe_job(cd_job *J, const cd_job_desc *d, Use use, const Layout &o, const HostTables &t, char *base, char *image) {
    auto put = [&](size_t at, const void *src, size_t bytes) { std::memcpy(image + at, src, bytes); };
    const bool designs = use != Use::Select, select = use != Use::Evaluate;
    cd::DevJob &h = J->h;
    h.L = J->L;
    h.m = J->m;
    h.N = J->N;
    h.P = J->P;
    h.R = J->R;
    h.W = J->W;
    h.den_sl = designs ? (3 * J->L - 4) / 2 : 1;
    h.Ls = designs ? cd::row_stride(J->L) : 0;
    h.seed = d->seed;
    h.thr_pm = bern_threshold_host(d->Pm);
    h.thr_2pm = bern_threshold_host(d->Pm * 2.0f);
    h.gc3_ref = d->tables.gc3_ref;
    for (int b = 0; b < 2; ++b) h.obj[b] = (float *)(base + o.obj[use == Use::Job ? b : 0]);
    if (designs) {
        // per position the first codon of its amino acid and its synonym count
        uint8_t *pos = (uint8_t *)image + o.pos;
        for (int k = 0; k < h.Ls; ++k) {
            const int a = k < J->L ? d->aa[k] : -1;
            pos[k] = a >= 0 ? (uint8_t)SYN_START[a] : 0;
            pos[h.Ls + k] = a >= 0 ? (uint8_t)SYN_NUM[a] : 1;
        }
        put(o.code, t.code, 64);
        put(o.lw6, t.lw6, 64 * 8);
        put(o.lw6 + 64 * 8, t.syn6, 64 * 8);
        put(o.cpfx6, t.cpfx6, 64 * 64 * 8);
        put(o.cps6, t.cps6, 64 * 64 * 4);
        h.pos = (const uint8_t *)(base + o.pos);
        h.code = (const uint8_t *)(base + o.code);
        h.lw6 = (const int64_t *)(base + o.lw6);
        h.cpfx6 = (const int64_t *)(base + o.cpfx6);
        h.cps6 = (const float *)(base + o.cps6);
        h.stop6 = t.stop6;
        for (int b = 0; b < 2; ++b) {
            const int u = use == Use::Job ? b : 0;
            h.genome[b] = (int8_t *)(base + o.genome[u]);
            h.oidx[b] = (int8_t *)(base + o.oidx[u]);
            h.pql[b] = (int32_t *)(base + o.pql[u]);
            h.cst[b] = (cd::CdsStat *)(base + o.cst[u]);
            h.hdp[b] = (int32_t *)(base + o.hdp[u]);
        }
        h.planes = (uint2 *)(base + o.planes);
        h.stem_max = (int32_t *)(base + o.stem_max);
        int2 *off = (int2 *)(image + o.off);
        for (int c = 0, n = use == Use::Job ? J->N : J->P; c < n; ++c) off[c] = make_int2(0, c);
        J->d_off = (int2 *)(base + o.off);
        J->lds = cd::design_lds_bytes(J->L, J->m);
        J->stem_lds = cd::stem_lds_bytes(J->L);
    }
    if (use == Use::Job) {
        J->d_slist = (uint2 *)(base + o.slist);  // the counts in d_sctl start at zero with the cleared allocation
        J->d_sctl = (int32_t *)(base + o.sctl);
        // the tuned shapes of this kind of job, if any
        cd_job *self = J;
        cd::Shapes sh;
        J->shapes = cdhost::untuned_shapes(&self, 1);
        if (cdhost::cached_shapes(cdhost::work_signature(&self, 1), &sh)) J->shapes = sh;
    } else {
        J->shapes.dom_rows = cd::DOM_ROWS;
    }
    if (select) {
        const auto ref = das_dennis(d->H);
        put(o.ref, ref.data(), ref.size() * sizeof(float));
        h.refpts = (const float *)(base + o.ref);
        h.front_of = (int32_t *)(base + o.front);
        h.np = (int32_t *)(base + o.np);
        h.dom = (uint64_t *)(base + o.dom);
        h.ref_of = (int32_t *)(base + o.ref_of);
        h.niche = (int32_t *)(base + o.niche);
        h.st = (cd::SelState *)(base + o.st);
        h.acc = (cd::SelAcc *)(base + o.acc);
        h.ranked = (uint64_t *)(base + o.ranked);
        h.selm = (uint64_t *)(base + o.selm);
        h.prio = (uint32_t *)(base + o.prio);
        h.cutl = (uint64_t *)(base + o.cutl);
        h.cutr = (int32_t *)(base + o.cutr);
        std::vector<int4> dom;
        std::vector<int2> asc;
        job_lists(J->P, J->W, J->shapes, dom, asc);
        put(o.domi, dom.data(), dom.size() * sizeof(int4));
        put(o.asc, asc.data(), asc.size() * sizeof(int2));
        J->n_dom = (int)dom.size();
        J->n_asc = (int)asc.size();
        J->d_dom = (int4 *)(base + o.domi);
        J->d_asc = (int2 *)(base + o.asc);
    }
    put(o.self, &h, sizeof(h));
    J->d_self = (cd::DevJob *)(base + o.self);
}

// Raise the kernels' dynamic LDS limits to what J's launches take.
hipError_t job_lds_limits(const cd_job *J, bool select) {
    hipError_t e = hipSuccess;
    if (J->lds > 48 * 1024) e = cd::set_design_lds_limit(J->lds);
    if (e == hipSuccess && cd::stem_list_lds(J->stem_lds) > 48 * 1024)
        e = cd::set_stem_lds_limit(cd::stem_list_lds(J->stem_lds));
    if (e == hipSuccess && select) e = cd::set_niche_lds_limit(J->P, J->R);
    return e;
}

int create_job(const cd_job_desc *d, cd_job **out) {
    cd_job *J = new cd_job();
    Layout o;
    HostTables t;
    const int rc = size_job(J, d, Use::Job, 2 * d->N, o, t);
    if (rc != CD_OK) {
        delete J;
        return rc;
    }
    // the job's own stream does not wait for (or hold up) work on other
    // streams, such as a served tick that is running while this job is
    // admitted
    // The allocation comes from the device's stream-ordered pool: freeing it
    // (cd_job_destroy) does not wait for every stream of the device, which
    // hipFree does, so jobs can come and go while others run.
    hipError_t e = streams().take(&J->dev, &J->stream);
    if (e == hipSuccess) e = keep_pool_memory();
    if (e == hipSuccess) e = allocated([&] { return hipMallocAsync(&J->mem, o.total, J->stream); });
    if (e != hipSuccess) {
        if (J->stream) (void)hipStreamDestroy(J->stream);
        delete J;
        return fail(CD_E_NOMEM, std::string("hipMallocAsync: ") + hipGetErrorString(e));
    }
    J->mem_bytes = o.total;
    char *base = (char *)J->mem;
    std::vector<char> image(o.head, 0);
    describe_job(J, d, Use::Job, o, t, base, image.data());
    e = hipMemsetAsync(base + o.head, 0, o.total - o.head, J->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(base, image.data(), o.head, hipMemcpyHostToDevice, J->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(J->stream);  // the image is released below
    if (e == hipSuccess) e = job_lds_limits(J, true);
    if (e != hipSuccess) {
        (void)hipFreeAsync(J->mem, J->stream);
        (void)hipStreamSynchronize(J->stream);
        (void)hipStreamDestroy(J->stream);
        delete J;
        return fail(CD_E_DEVICE, std::string("job setup: ") + hipGetErrorString(e));
    }
    *out = J;
    return CD_OK;
}

// A stream with a device and a pinned host buffer for the calls that hold
// nothing from one to the next (cd_eval_batch, cd_nds, cd_select; cd_job_read
// takes the pinned buffer and the events).  A call
// takes one for its duration -- an idle one of its device, else a new one -- so
// calls of several threads run side by side; at most SHOTS_IDLE idle ones and
// buffers of at most SHOT_KEEP bytes are kept, the rest is freed with the
// call, and the idle ones too when an allocation fails (allocated).  With them,
// one launch that fetches the set-up and one synchronisation an evaluation of 16
// designs takes 49 us, a selection of 1024 from 2048 89; with a job allocated,
// filled by ten transfers and freed for each, 294 and 288.
constexpr size_t EVAL_CHUNK = (size_t)1 << 20, READ_CHUNK = (size_t)4 << 20,  // bytes of packed rows
                 EVAL_WINDOW = (size_t)32 << 20;
constexpr size_t SHOTS_IDLE = 4, SHOT_KEEP = (size_t)64 << 20;
struct Shot {
    int dev = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    char *mem = nullptr, *host = nullptr;
    size_t mem_cap = 0, host_cap = 0;
    hipError_t reserve(size_t mem_bytes, size_t host_bytes) {
        hipError_t e = hipSuccess;
        if (mem_bytes > mem_cap) {
            if (mem) (void)hipFreeAsync(mem, stream);
            mem = nullptr;
            mem_cap = 0;
            e = allocated([&] { return hipMallocAsync((void **)&mem, mem_bytes + mem_bytes / 4, stream); });
            if (e == hipSuccess) mem_cap = mem_bytes + mem_bytes / 4;
        }
        if (e == hipSuccess && host_bytes > host_cap) {
            if (host) (void)hipHostFree(host);
            host = nullptr;
            host_cap = 0;
            e = allocated([&] { return hipHostMalloc((void **)&host, host_bytes + host_bytes / 4, hipHostMallocDefault); });
            if (e == hipSuccess) host_cap = host_bytes + host_bytes / 4;
        }
        return e;
    }
    void free() {
        if (mem) (void)hipFreeAsync(mem, stream);
        if (stream) {
            (void)hipStreamSynchronize(stream);
            (void)hipStreamDestroy(stream);
        }
        if (host) (void)hipHostFree(host);
        for (hipEvent_t x : ev)
            if (x) (void)hipEventDestroy(x);
    }
};
struct Shots {
    std::mutex mu;
    std::vector<Shot> idle;
    hipError_t take(Shot &s) {
        hipError_t e = hipGetDevice(&s.dev);
        if (e != hipSuccess) return e;
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t i = idle.size(); i-- > 0;)
                if (idle[i].dev == s.dev) {
                    s = idle[i];
                    idle.erase(idle.begin() + (ptrdiff_t)i);
                    return hipSuccess;
                }
        }
        e = hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking);
        for (hipEvent_t &x : s.ev)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
        if (e == hipSuccess) e = keep_pool_memory();
        return e;
    }
    // ok: the call's work has ended without an error
    void give(Shot &s, bool ok) {
        if (ok) {
            if (s.mem_cap > SHOT_KEEP) {
                (void)hipFreeAsync(s.mem, s.stream);
                s.mem = nullptr;
                s.mem_cap = 0;
            }
            if (s.host_cap > SHOT_KEEP) {
                (void)hipHostFree(s.host);
                s.host = nullptr;
                s.host_cap = 0;
            }
            std::lock_guard<std::mutex> lk(mu);
            if (idle.size() < SHOTS_IDLE) {
                idle.push_back(s);
                return;
            }
        }
        s.free();
    }
    void drop_idle() {
        std::vector<Shot> all;
        {
            std::lock_guard<std::mutex> lk(mu);
            all.swap(idle);
        }
        for (Shot &s : all) s.free();
    }
};
Shots &shots() {  // (never destroyed: the runtime may be gone by then)
    static Shots *p = new Shots();
    return *p;
}
void drop_idle_shots() { shots().drop_idle(); }

// Initialisation of the children's work list `w.off` (offspring generations go
// through enqueue_generation): the designs, the stem of every CDS, objective 5.
// fresh: the pool has not been written before.
hipError_t enqueue_init(const Launch &w, hipStream_t s, bool fresh) {
    hipError_t e = cd::launch_design(cd::MODE_INIT, w.jobs, w.off, w.n_off, w.lds, s, nullptr, nullptr,
                                     cd::StemList{0, 0, 0}, fresh ? 1 : 0);
    if (e == hipSuccess) e = cd::launch_stem(w.jobs, w.off, w.n_off, w.mg, w.stem_lds, s);
    if (e == hipSuccess) e = cd::launch_stem_finish(w.jobs, w.off, w.n_off, s);
    return e;
}

}  // namespace

namespace cdhost {

hipError_t enqueue_generation(const Launch &w, hipStream_t s, hipEvent_t *ev) {
    // ev (optional): CD_PROFILE_KERNELS + 1 events recorded around the six
    // phases -- offspring (both k_design launch classes), stem list,
    // dominance, fronts, association, niching
    auto mark = [&](int k) { return ev ? hipEventRecord(ev[k], s) : hipSuccess; };
    hipError_t e = mark(0);
    const cd::StemList sl = cd::stem_list_plan(w.n_off, w.mg);
    if (e == hipSuccess) {
        const int ns = w.n_small > 0 && w.n_small < w.n_off ? w.n_small : 0;
        if (ns)
            e = cd::launch_design(cd::MODE_OFFSPRING, w.jobs, w.off, ns, w.lds_small, s, w.stem_list, w.stem_ctl, sl, 0);
        if (e == hipSuccess)
            e = cd::launch_design(cd::MODE_OFFSPRING, w.jobs, w.off + ns, w.n_off - ns, w.lds, s, w.stem_list,
                                  w.stem_ctl, sl, ns, w.sh.design_threads);
    }
    if (e == hipSuccess) e = mark(1);
    if (e == hipSuccess)
        e = cd::launch_stem_list(w.jobs, w.off, w.n_off, w.mg, w.longest, w.stem_list, w.stem_ctl, sl, w.sh.stem_waves, w.stem_lds, s);
    if (e == hipSuccess) e = mark(2);
    if (e == hipSuccess)
        e = cd::launch_dominance(w.jobs, w.dom, w.n_dom, true, w.stem_ctl, sl.groups, w.sh.dom_rows, s);
    if (e == hipSuccess) e = mark(3);
    const bool fused = cd::fuse_fronts(w.max_pool, w.pool);
    if (e == hipSuccess && !fused) e = cd::launch_fronts(w.jobs, w.njobs, w.max_pool, w.sh.fronts_threads, s);
    if (e == hipSuccess) e = mark(4);
    if (e == hipSuccess)
        e = fused ? cd::launch_front_associate(w.jobs, w.asc, w.n_asc, w.sh.assoc_designs, s)
                  : cd::launch_associate(w.jobs, w.asc, w.n_asc, w.sh.assoc_designs, s);
    if (e == hipSuccess) e = mark(5);
    if (e == hipSuccess) e = cd::launch_niche(w.jobs, w.njobs, w.max_pool, w.max_refs, w.sh.niche_threads, s);
    if (e == hipSuccess) e = mark(6);
    return e;
}

void build_lists(cd_job *const *jobs, int count, const cd::Shapes &sh, WorkLists &wl) {
    wl = WorkLists();
    // children of the jobs whose k_design LDS is at most sh.design_split
    // first (a launch of its own, so that more of them share a CU); within
    // each class the jobs with the most codons per child (L * m) first, so
    // that the longest workgroups start early and short ones fill the end of
    // the launch
    std::vector<int> order(count);
    for (int j = 0; j < count; ++j) order[j] = j;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return (int64_t)jobs[a]->L * jobs[a]->m > (int64_t)jobs[b]->L * jobs[b]->m;
    });
    for (int pass = 0; pass < 2; ++pass)
        for (int j : order) {
            cd_job *J = jobs[j];
            if ((J->lds <= (size_t)sh.design_split) != (pass == 0)) continue;
            for (int c = 0; c < J->N; ++c) wl.off.push_back(make_int2(j, c));
            if (pass == 0) {
                wl.n_small += J->N;
                wl.lds_small = std::max(wl.lds_small, J->lds);
            }
        }
    for (int j = 0; j < count; ++j) {
        cd_job *J = jobs[j];
        wl.descs.push_back(J->h);
        wl.n_cds += J->N * J->m;
        job_lists(J->P, J->W, sh, wl.dom, wl.asc, j);
        wl.lds = std::max(wl.lds, J->lds);
        wl.stem_lds = std::max(wl.stem_lds, J->stem_lds);
        wl.max_pool = std::max(wl.max_pool, J->P);
        wl.pool += J->P;
        wl.max_refs = std::max(wl.max_refs, J->R);
        wl.mg = std::max(wl.mg, J->m);
        wl.longest = std::max(wl.longest, J->L);
    }
}

hipError_t set_lds_limits(const WorkLists &wl) {
    hipError_t e = hipSuccess;
    if (wl.lds > 48 * 1024) e = cd::set_design_lds_limit(wl.lds);
    if (e == hipSuccess && cd::stem_list_lds(wl.stem_lds) > 48 * 1024)
        e = cd::set_stem_lds_limit(cd::stem_list_lds(wl.stem_lds));
    if (e == hipSuccess) e = cd::set_niche_lds_limit(wl.max_pool, wl.max_refs);
    return e;
}

}  // namespace cdhost

using cdhost::enqueue_generation;

namespace {

int capture(hipStream_t s, hipGraph_t *g, hipGraphExec_t *ge, const Launch &w, int generations) {
    HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    hipError_t e = hipSuccess;
    for (int k = 0; k < generations && e == hipSuccess; ++k) e = enqueue_generation(w, s, nullptr);
    hipGraph_t graph = nullptr;
    hipError_t e2 = hipStreamEndCapture(s, &graph);
    if (e != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        return fail(CD_E_DEVICE, std::string("capture: ") + hipGetErrorString(e));
    }
    if (e2 != hipSuccess) return fail(CD_E_DEVICE, std::string("end capture: ") + hipGetErrorString(e2));
    e = hipGraphInstantiate(ge, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(graph);
        return fail(CD_E_DEVICE, std::string("graph instantiation: ") + hipGetErrorString(e));
    }
    *g = graph;
    return CD_OK;
}

// Enqueue `generations` generations: blocks of GRAPH_BLOCK as graph launches,
// the others kernel by kernel.  The first GRAPH_AFTER generations of a graph's
// life go kernel by kernel too, so that the device has work while the host
// captures the graph, and short runs need none.
int step_graphs(StepGraphs &G, hipStream_t s, const Launch &w, int generations) {
    int g = generations;
    for (; g > 0 && !G.exec && G.direct < GRAPH_AFTER; --g, ++G.direct) HIPCHK(enqueue_generation(w, s, nullptr));
    if (g >= GRAPH_BLOCK && !G.exec) {
        const int rc = capture(s, &G.graph, &G.exec, w, GRAPH_BLOCK);
        if (rc != CD_OK) return rc;
    }
    for (; g >= GRAPH_BLOCK; g -= GRAPH_BLOCK) HIPCHK(hipGraphLaunch(G.exec, s));
    for (; g > 0; --g) HIPCHK(enqueue_generation(w, s, nullptr));
    return CD_OK;
}

Launch job_launch(cd_job *J) {
    return Launch{J->d_self, 1,          J->d_off,     J->N,          J->d_dom,   J->n_dom,   J->d_asc,
                  J->n_asc,  J->lds,     J->stem_lds,  J->P,          J->R,       J->m,   J->L,
                  J->d_slist,
                  J->d_sctl, J->N * J->m, 0,           0,             J->P,          J->shapes};
}

// The calling thread's device is `dev` while it lives: a job is stepped and read
// whichever device is current, and its kernels, and the events recorded on its
// stream, have to be of the stream's device.
class OnDevice {
  public:
    explicit OnDevice(int dev) {
        int now = dev;
        if (hipGetDevice(&now) == hipSuccess && now != dev && hipSetDevice(dev) == hipSuccess) was_ = now;
    }
    ~OnDevice() {
        if (was_ >= 0) (void)hipSetDevice(was_);
    }
    OnDevice(const OnDevice &) = delete;
    OnDevice &operator=(const OnDevice &) = delete;

  private:
    int was_ = -1;
};

// Wait for the job's own stream and for the streams of the batches that hold it.
hipError_t sync_job(cd_job *J) {
    for (cd_batch *B : J->batches) {
        const hipError_t e = hipStreamSynchronize(B->stream);
        if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(J->stream);
}

// Run `generations` generations of `w` launching every kernel apart, with
// HIP events on stream s around each phase; kernel_ms receives the mean
// duration of each phase (CD_PROFILE_KERNELS values).
int profile_generations(const Launch &w, hipStream_t s, int generations, float *kernel_ms) {
    constexpr int NK = CD_PROFILE_KERNELS;
    hipEvent_t ev[NK + 1];
    for (auto &e : ev) HIPCHK(hipEventCreate(&e));
    double acc[NK] = {0};
    for (int g = 0; g < generations; ++g) {
        HIPCHK(cdhost::enqueue_generation(w, s, ev));
        HIPCHK(hipEventSynchronize(ev[NK]));
        for (int k = 0; k < NK; ++k) {
            float t = 0.f;
            HIPCHK(hipEventElapsedTime(&t, ev[k], ev[k + 1]));
            acc[k] += t;
        }
    }
    for (int k = 0; k < NK; ++k) kernel_ms[k] = generations > 0 ? (float)(acc[k] / generations) : 0.f;
    for (auto &e : ev) HIPCHK(hipEventDestroy(e));
    return CD_OK;
}

// Coordinate search over the launch shapes.  Every candidate runs `gens`
// ordinary generations of the work (all shapes give the same results, so
// the job's trajectory does not depend on the search); a candidate's cost is
// the mean time of the phases its parameter changes, from HIP events around
// each phase.  Parameters are settled one after another, each from the best
// shapes so far; `apply` installs shapes and returns the launch description.
template <class Apply>
int tune_shapes(const cd::Shapes &start, int njobs, int gens, hipStream_t s, Apply apply, cd::Shapes *best,
                int *run) {
    struct Param {
        int cd::Shapes::*field;
        std::vector<int> values;
        unsigned phases;  // bit k: phase k of the generation profile
    };
    const std::vector<Param> params = {
        {&cd::Shapes::design_split, {0, 6000, 8500, 11000}, 0x3u},
        {&cd::Shapes::design_threads, {256, 512}, 0x1u},
        {&cd::Shapes::stem_waves, {5, 6, 7, 8}, 0x2u},
        {&cd::Shapes::dom_rows, {64, 128, 256}, 0x4u},
        {&cd::Shapes::fronts_threads, {256, 512, 1024}, 0x8u},
        {&cd::Shapes::assoc_designs, {4, 8, 16, 32, 64}, 0x10u},
        {&cd::Shapes::niche_threads, {256, 512, 1024}, 0x20u},
    };
    // the parameters of kernels that this work does not launch keep their values:
    // their candidates differ by chance alone
    auto used = [](const Param &p, const Launch &w) {
        if (p.field == &cd::Shapes::stem_waves) return cd::stem_path(w.n_off, w.mg, w.longest) != cd::STEM_PATH_EACH;
        if (p.field == &cd::Shapes::fronts_threads) return !cd::fuse_fronts(w.max_pool, w.pool);
        return true;
    };
    cd::Shapes cur = start;
    *run = 0;
    for (const Param &p : params) {
        if (p.field == &cd::Shapes::design_split && njobs == 1) continue;  // one job is one launch class
        double best_cost = 1e30;
        int best_v = cur.*(p.field);
        for (int v : p.values) {
            cd::Shapes cand = cur;
            cand.*(p.field) = v;
            Launch w{};
            int rc = apply(cand, &w);
            if (rc != CD_OK) return rc;
            float ms[CD_PROFILE_KERNELS];
            rc = profile_generations(w, s, gens, ms);
            if (rc != CD_OK) return rc;
            *run += gens;
            double cost = 0.0;
            for (int k = 0; k < CD_PROFILE_KERNELS; ++k)
                if (p.phases >> k & 1u) cost += ms[k];
            if (cost < best_cost && used(p, w)) {
                best_cost = cost;
                best_v = v;
            }
        }
        cur.*(p.field) = best_v;
    }
    Launch w{};
    const int rc = apply(cur, &w);
    if (rc != CD_OK) return rc;
    *best = cur;
    return CD_OK;
}

}  // namespace

namespace cdhost {

namespace {
std::mutex g_tune_mu;
std::map<std::string, cd::Shapes> g_tuned;

int log2_bucket(int64_t x) {
    int b = 0;
    while (x > 1) {
        x >>= 1;
        ++b;
    }
    return b;
}
}  // namespace

// (with the kernels that its launches take: within one bucket of sizes they
// differ, and with them what a shape means)
std::string work_signature(cd_job *const *jobs, int count) {
    int64_t children = 0, lm = 0, pool = 0, pools = 0;
    int mg = 0, longest = 0, refs = 0;
    for (int j = 0; j < count; ++j) {
        children += jobs[j]->N;
        lm = std::max(lm, (int64_t)jobs[j]->L * jobs[j]->m);
        pool = std::max(pool, (int64_t)jobs[j]->P);
        pools += jobs[j]->P;
        mg = std::max(mg, jobs[j]->m);
        longest = std::max(longest, jobs[j]->L);
        refs = std::max(refs, jobs[j]->R);
    }
    const int path = (int)cd::stem_path((int)children, mg, longest) + 4 * (int)cd::fuse_fronts((int)pool, (int)pools) +
                     8 * (int)cd::takes_place_niche((int)pool, refs) + 16 * (int)(children > cd::DESIGN_MANY);
    int dev = 0;
    (void)hipGetDevice(&dev);
    return "dev" + std::to_string(dev) + "/jobs" + std::to_string(log2_bucket(count)) + "/children" +
           std::to_string(log2_bucket(children)) + "/codons" + std::to_string(log2_bucket(lm)) + "/pool" +
           std::to_string(log2_bucket(pool)) + "/path" + std::to_string(path);
}

// The shapes of untuned work.  Association: a wave a design while the waves
// fit the chip (pool <= 12000 designs in all), eight lanes a design above;
// few designs a workgroup where a generation is a chain of latencies (4 up to
// 512 designs, 8 up to FUSED_TOTAL, where k_front_associate runs), more
// where it is throughput.  Measured, microseconds a generation of batches of
// the 50..2000-residue mix with 4 / 8 / 16 / 64 designs a workgroup: pool 2048
// 140.1 / 137.6 / 138.7 / 142.5, pool 8192 206.7 / 204.3 / 202.9 / 205.1, pool
// 28160 557.5 / 557.1 / 557.7 / 553.6, pool 84480 1244 / 1245 / - / 1226; the
// 100-residue job (pool 256) 50.4 / 50.9.
cd::Shapes untuned_shapes(cd_job *const *jobs, int count) {
    cd::Shapes sh = count == 1 ? cd::SHAPES_JOB : cd::SHAPES_BATCH;
    int64_t pool = 0;
    for (int j = 0; j < count; ++j) pool += jobs[j]->P;
    // k_design in one launch, 512 threads a child while the workgroups are
    // resident together -- three a CU -- and longer the more codons a child has.
    // Microseconds with 256 / 512 threads: 2004 codons, 700 children 20.7 /
    // 19.8, 900 24.3 / 25.3; 6190 codons, 900 35.3 / 33.2, 2048 49.7 / 53.9;
    // 20008 codons, 1200 77.8 / 68.8, 2048 98.9 / 92.1; up to 700 codons equal
    // below 768 children and 256 faster above.  Launch classes by LDS do not pay
    // any more (a second launch's tail against a few more resident workgroups):
    // ticks of 24 / 48 / 64 jobs 454 / 797 / 1004 us in one launch, 478 / 790 /
    // 971 split at 8500 bytes, the other way round for other mixes.
    int64_t children = 0, codons = 0, tiles = 0;
    for (int j = 0; j < count; ++j) {
        tiles += (int64_t)jobs[j]->W * (jobs[j]->W + 1) / 2;
        children += jobs[j]->N;
        codons += (int64_t)jobs[j]->N * jobs[j]->L * jobs[j]->m;
    }
    sh.design_split = 0;
    sh.design_threads = children <= 640 + codons / children / 16 ? 512 : 256;
    // Domination tiles a workgroup: one while a tile's latency counts, four when
    // the chip is full of them.  Microseconds a generation with 64 / 128 / 256
    // rows: batches of 72 tiles 39.1 / 40.2 / 42.2, 544 56.8 / 57.4 / 59.0, 1056
    // 64.8 / 65.4 / 64.7, 3168 104 / 103 / 102, 6336 178 / 174 / 173, the 64-job
    // mix (17 700) 817 / 808 / 802; lone jobs of 202 codons, 528 tiles 51.3 / 52.7 /
    // 52.2, 2850 81.5 / 82.2 / 80.1, 4095 88.4 / 89.5 / 89.1, 5253 96.3 / 97.2 / 95.3,
    // 6105 101.8 / 100.2 / 99.6, 8256 113.2 / 110.6 / 112.1, 12 403 138 / 131 / 131,
    // 32 896 224 / 209 / 203.
    sh.dom_rows = tiles <= (count > 1 ? 1024 : 6000) ? 64 : 256;
    sh.assoc_designs = pool <= 512 ? 4 : pool <= cd::FUSED_TOTAL ? 8 : pool <= 12000 ? 16 : 64;
    return sh;
}

bool cached_shapes(const std::string &sig, cd::Shapes *out) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(sig);
    if (it == g_tuned.end()) return false;
    *out = it->second;
    return true;
}

void store_shapes(const std::string &sig, const cd::Shapes &sh) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[sig] = sh;
}

}  // namespace cdhost

extern "C" {

const char *cd_last_error(void) { return cdhost::g_err.c_str(); }

int64_t cd_job_device_bytes(int32_t L, int32_t m, int32_t N, int32_t H) {
    if (L < 3 || m < 2 || N < 1 || H < 1) return -1;
    const int P = 2 * N, W = (P + 63) / 64;
    int n_dom, n_asc;
    work_counts(P, W, &n_dom, &n_asc);
    return (int64_t)layout(L, m, N, P, (int)n_ref(H), W, n_dom, n_asc, Use::Job).total;
}

int cd_job_create(const cd_job_desc *desc, cd_job **out) {
    if (!out) return fail(CD_E_INVALID, "null output handle");
    int rc = validate(desc);
    if (rc != CD_OK) return rc;
    return create_job(desc, out);
}

int cd_job_init(cd_job *J) {
    if (!J || J->selection_only) return fail(CD_E_INVALID, "null job");
    // the offspring work list doubles as the (job, design) list of the init launch
    HIPCHK(enqueue_init(job_launch(J), J->stream, !J->inited));
    HIPCHK(cd::launch_init_state(J->d_self, 1, J->stream));
    J->inited = true;
    return CD_OK;
}

int cd_job_step(cd_job *J, int32_t generations) {
    if (!J || J->selection_only) return fail(CD_E_INVALID, "null job");
    if (!J->inited) return fail(CD_E_STATE, "cd_job_step before cd_job_init");
    if (!J->batches.empty()) return fail(CD_E_STATE, "the job is held by a batch: advance it through the batch");
    if (generations < 0) return fail(CD_E_INVALID, "negative generation count");
    const OnDevice on(J->dev);
    return step_graphs(J->graphs, J->stream, job_launch(J), generations);
}

int cd_job_step_timed(cd_job *J, int32_t generations, float *ms) {
    if (!J) return fail(CD_E_INVALID, "null job");
    hipEvent_t a, b;
    HIPCHK(hipEventCreate(&a));
    HIPCHK(hipEventCreate(&b));
    HIPCHK(hipEventRecord(a, J->stream));
    int rc = cd_job_step(J, generations);
    if (rc != CD_OK) return rc;
    HIPCHK(hipEventRecord(b, J->stream));
    HIPCHK(hipEventSynchronize(b));
    float t = 0.f;
    HIPCHK(hipEventElapsedTime(&t, a, b));
    if (ms) *ms = t;
    HIPCHK(hipEventDestroy(a));
    HIPCHK(hipEventDestroy(b));
    return CD_OK;
}

int cd_job_sync(cd_job *J) {
    if (!J) return fail(CD_E_INVALID, "null job");
    HIPCHK(sync_job(J));
    return CD_OK;
}

// The survivors in ascending pool index: the first N set bits of the
// survivor mask.
static void survivors_of(const std::vector<uint64_t> &mask, int N, int32_t *out) {
    int k = 0;
    for (size_t w = 0; w < mask.size() && k < N; ++w)
        for (uint64_t x = mask[w]; x && k < N; x &= x - 1) out[k++] = (int32_t)(64 * w + __builtin_ctzll(x));
    for (; k < N; ++k) out[k] = -1;
}

// Reads of a job's device state go through its own (non-blocking) stream,
// never the legacy null stream, so that they do not wait for other streams -- for
// instance a server's ticks.
static hipError_t read_state(cd_job *J, cd::SelState &st) {
    hipError_t e = sync_job(J);
    if (e == hipSuccess) e = hipMemcpyAsync(&st, J->h.st, sizeof(st), hipMemcpyDeviceToHost, J->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(J->stream);
    return e;
}

int cd_job_generation(cd_job *J, int32_t *generation) {
    if (!J || !generation) return fail(CD_E_INVALID, "null argument");
    cd::SelState st;
    HIPCHK(read_state(J, st));
    *generation = (int32_t)st.gen;
    return CD_OK;
}

int cd_job_read(cd_job *J, int8_t *genome, float *obj, int8_t *idx, int32_t *pql, int32_t *sorted, int32_t *front_of,
                float *state) {
    if (!J || J->selection_only) return fail(CD_E_INVALID, "null job");
    if (!J->inited) return fail(CD_E_STATE, "cd_job_read before cd_job_init");
    const OnDevice on(J->dev);
    const int P = J->P;
    const cd::ReadRest at(P, J->W);
    const size_t total = genome ? (size_t)P * J->m * J->L : 0, chunk = std::min(total, READ_CHUNK);
    const size_t head = (at.bytes + 255) & ~(size_t)255, room = (chunk + 255) & ~(size_t)255;
    Shot w;
    hipError_t e = shots().take(w);
    if (e == hipSuccess) e = w.reserve(0, head + 2 * room);
    for (cd_batch *B : J->batches)
        if (e == hipSuccess) e = hipStreamSynchronize(B->stream);
    // a chunk is copied out while the next one is on its way
    uint8_t *const half[2] = {(uint8_t *)w.host + head, (uint8_t *)w.host + head + room};
    auto send = [&](size_t first, int k, bool rest) {
        if (e == hipSuccess)
            e = cd::launch_read(J->d_self, half[k], rest ? w.host : nullptr, at.bytes, first, std::min(chunk, total - first), J->stream);
        if (e == hipSuccess) e = hipEventRecord(w.ev[k], J->stream);
    };
    send(0, 0, true);
    for (size_t first = 0, k = 0; first < total; first += chunk, k ^= 1) {
        if (first + chunk < total) send(first + chunk, (int)(k ^ 1), false);
        if (e == hipSuccess) e = hipEventSynchronize(w.ev[k]);
        if (e == hipSuccess) std::memcpy(genome + first, half[k], std::min(chunk, total - first));
    }
    const hipError_t es = hipStreamSynchronize(J->stream);
    if (e == hipSuccess) e = es;
    cd::SelState st;
    if (e == hipSuccess) {
        std::memcpy(&st, w.host, sizeof(st));
        if (obj) std::memcpy(obj, w.host + at.obj, (size_t)P * 24);
        if (idx) std::memcpy(idx, w.host + at.idx, (size_t)P * 12);
        if (front_of) std::memcpy(front_of, w.host + at.front, (size_t)P * 4);
        if (sorted) {
            std::vector<uint64_t> mask(J->W);
            std::memcpy(mask.data(), w.host + at.selm, (size_t)J->W * 8);
            survivors_of(mask, J->N, sorted);
        }
        const int32_t *q = (const int32_t *)(w.host + at.pql);
        if (pql)
            for (int i = 0; i < P; ++i)
                for (int k = 0; k < 3; ++k) pql[i * 3 + k] = q[(size_t)i * 4 + k];
    }
    shots().give(w, e == hipSuccess);
    HIPCHK(e);
    const int b = (int)(st.gen & 1u);
    if (state) {
        const cd::SelRes &r = st.res[b];
        std::memcpy(state, r.ext, sizeof(r.ext));
        std::memcpy(state + 36, r.ideal, sizeof(r.ideal));
        std::memcpy(state + 42, r.worst, sizeof(r.worst));
        std::memcpy(state + 48, r.nadir, sizeof(r.nadir));
    }
    return CD_OK;
}

int cd_job_profile(cd_job *J, int32_t generations, float *kernel_ms) {
    if (!J || J->selection_only || !kernel_ms) return fail(CD_E_INVALID, "null argument");
    if (!J->inited) return fail(CD_E_STATE, "cd_job_profile before cd_job_init");
    if (!J->batches.empty()) return fail(CD_E_STATE, "the job is held by a batch: advance it through the batch");
    return profile_generations(job_launch(J), J->stream, generations, kernel_ms);
}

int cd_job_cds_scanned(cd_job *J, int64_t *count) {
    if (!J || !count) return fail(CD_E_INVALID, "null argument");
    cd::SelState st;
    HIPCHK(read_state(J, st));
    *count = (int64_t)st.cds_scanned;
    return CD_OK;
}

int cd_job_destroy(cd_job *J) {
    if (!J) return CD_OK;
    if (!J->batches.empty()) return fail(CD_E_STATE, "the job is held by a batch: destroy the batch first");
    if (J->stream) (void)hipStreamSynchronize(J->stream);
    J->graphs.reset();
    if (J->mem) (void)hipFreeAsync(J->mem, J->stream);  // back to the pool, after the job's last work
    if (J->stream) {
        // the memory is free with the call: a server hands its bytes to the next
        // job, which would otherwise be allocated beside it
        if (hipStreamSynchronize(J->stream) == hipSuccess)
            streams().give(J->dev, J->stream);
        else
            (void)hipStreamDestroy(J->stream);
    }
    delete J;
    return CD_OK;
}

// One evaluation of `count` designs with a validated description.
static int evaluate(const cd_job_desc &d, const int8_t *genome, int32_t count, float *obj, int8_t *idx, int32_t *pql) {
    cd_job job;
    cd_job *J = &job;
    Layout o;
    HostTables t;
    const int rc = size_job(J, &d, Use::Evaluate, count, o, t);
    if (rc != CD_OK) return rc;
    const size_t row = (size_t)J->m * J->L, bytes = row * count;
    // pinned: the image, the packed rows (a word past them is read), the results
    const size_t r_obj = o.head + a256(bytes + 8), r_idx = r_obj + a256((size_t)count * 24), r_pql = r_idx + a256((size_t)count * 12);
    Shot w;
    hipError_t e = shots().take(w);
    if (e == hipSuccess) e = w.reserve(o.total, r_pql + (size_t)count * 16);
    if (e != hipSuccess) {
        shots().give(w, false);
        return fail(CD_E_NOMEM, std::string("eval buffers: ") + hipGetErrorString(e));
    }
    std::memset(w.host, 0, o.head);
    describe_job(J, &d, Use::Evaluate, o, t, w.mem, w.host);
    J->h.genome[0] = (int8_t *)w.host + o.head;
    J->h.obj[0] = (float *)(w.host + r_obj);
    J->h.oidx[0] = (int8_t *)w.host + r_idx;
    J->h.pql[0] = (int32_t *)(w.host + r_pql);
    std::memcpy(w.host + o.self, &J->h, sizeof(J->h));
    e = job_lds_limits(J, false);
    if (e == hipSuccess) e = cd::launch_fetch(w.mem, w.host, o.head, w.stream);
    // The rows are copied into pinned memory packed as the caller holds them,
    // EVAL_CHUNK bytes at a time, and k_design reads them from there bytewise,
    // each once: the copies overlap the kernel of the chunk before.  The stems
    // follow in one launch, and the kernels store the results to pinned memory
    // too.  2048 designs of 2004 codons, 4 MB: 206 us; with transfers by the
    // copy engine 304, with the stems chunk by chunk 232, with chunks of half the
    // size 238.
    const int per = std::max(1, (int)std::min<size_t>(EVAL_CHUNK / row, (size_t)count));
    for (int i = 0; i < count && e == hipSuccess; i += per) {
        const int n = std::min(per, count - i);
        std::memcpy(w.host + o.head + i * row, genome + i * row, n * row);
        e = cd::launch_design(cd::MODE_EVAL, J->d_self, J->d_off + i, n, J->lds, w.stream);
    }
    if (e == hipSuccess) e = cd::launch_stem(J->d_self, J->d_off, count, J->m, J->stem_lds, w.stream);
    if (e == hipSuccess) e = cd::launch_stem_finish(J->d_self, J->d_off, count, w.stream);
    const hipError_t es = hipStreamSynchronize(w.stream);
    if (e == hipSuccess) e = es;
    if (e == hipSuccess) {
        if (obj) std::memcpy(obj, w.host + r_obj, (size_t)count * 24);
        if (idx) std::memcpy(idx, w.host + r_idx, (size_t)count * 12);
        const int32_t *q = (const int32_t *)(w.host + r_pql);
        if (pql)
            for (int i = 0; i < count; ++i)
                for (int k = 0; k < 3; ++k) pql[i * 3 + k] = q[(size_t)i * 4 + k];
    }
    shots().give(w, e == hipSuccess);
    if (e != hipSuccess) return fail(CD_E_DEVICE, std::string("eval: ") + hipGetErrorString(e));
    return CD_OK;
}

int cd_eval_batch(const cd_job_desc *desc, const int8_t *genome, int32_t count, float *obj, int8_t *idx,
                  int32_t *pql) {
    if (!desc || !genome || count <= 0) return fail(CD_E_INVALID, "bad eval arguments");
    cd_job_desc d = *desc;
    d.N = (int32_t)(((int64_t)count + 1) / 2);
    d.H = 1;
    d.Pm = 0.f;
    int rc = validate(&d);
    // EVAL_WINDOW bytes of rows at a time, so that the pinned buffer is one
    // that is kept
    const size_t row = rc == CD_OK ? (size_t)d.m * d.L : 1;
    const int per = std::max(1, (int)std::min<size_t>(EVAL_WINDOW / row, (size_t)count));
    for (int i = 0; i < count && rc == CD_OK; i += per)
        rc = evaluate(d, genome + i * row, std::min(per, count - i), obj ? obj + (size_t)i * 6 : nullptr,
                      idx ? idx + (size_t)i * 12 : nullptr, pql ? pql + (size_t)i * 3 : nullptr);
    return rc;
}

// One selection (full) or sort of P objective vectors.  On success *st, mask
// (J.W words) and front (P) hold its state, survivor mask and fronts.
static int run_selection(const float *obj, int32_t P, int32_t N, int32_t H, uint32_t gen, uint64_t seed,
                         const float *extremes, bool full, cd::SelState *st, std::vector<uint64_t> *mask, int32_t *front) {
    if (!obj || P <= 0 || N <= 0 || N > P || P > 64 * cd::MAX_W || H < 1)
        return fail(CD_E_INVALID, "bad selection arguments");
    cd_job_desc d{};
    d.N = N;
    d.H = H;
    d.seed = seed;
    cd_job job;
    cd_job *J = &job;
    Layout o;
    HostTables t;
    int rc = size_job(J, &d, Use::Select, P, o, t);
    if (rc != CD_OK) return rc;
    const size_t out_bytes = o.front + (size_t)P * 4 - o.st;
    Shot w;
    hipError_t e = shots().take(w);
    if (e == hipSuccess) e = w.reserve(o.total, o.head + out_bytes);
    if (e != hipSuccess) {
        shots().give(w, false);
        return fail(CD_E_NOMEM, std::string("selection buffers: ") + hipGetErrorString(e));
    }
    std::memset(w.host, 0, o.head);
    describe_job(J, &d, Use::Select, o, t, w.mem, w.host);
    std::memcpy(w.host + o.obj[0], obj, (size_t)P * 24);
    cd::SelState *s0 = (cd::SelState *)(w.host + o.st);
    s0->gen = gen;
    if (extremes) std::memcpy(s0->res[gen & 1u].ext, extremes, sizeof(s0->res[0].ext));
    e = job_lds_limits(J, true);
    if (e == hipSuccess) e = hipMemsetAsync(w.mem + o.head, 0, o.total - o.head, w.stream);
    if (e == hipSuccess) e = cd::launch_fetch(w.mem, w.host, o.head, w.stream);
    if (e == hipSuccess) e = cd::launch_zero_np(J->d_self, 1, w.stream);
    const cd::Shapes &sh = J->shapes;
    if (e == hipSuccess) e = cd::launch_dominance(J->d_self, J->d_dom, J->n_dom, false, nullptr, 0, sh.dom_rows, w.stream);
    const bool fused = full && cd::fuse_fronts(P, P);
    if (e == hipSuccess && !fused) e = cd::launch_fronts(J->d_self, 1, P, sh.fronts_threads, w.stream);
    if (e == hipSuccess && full)
        e = fused ? cd::launch_front_associate(J->d_self, J->d_asc, J->n_asc, sh.assoc_designs, w.stream)
                  : cd::launch_associate(J->d_self, J->d_asc, J->n_asc, sh.assoc_designs, w.stream);
    if (e == hipSuccess && full) e = cd::launch_niche(J->d_self, 1, P, J->R, sh.niche_threads, w.stream);
    char *const res = w.host + o.head;
    if (e == hipSuccess) e = hipMemcpyAsync(res, w.mem + o.st, out_bytes, hipMemcpyDeviceToHost, w.stream);
    const hipError_t es = hipStreamSynchronize(w.stream);
    if (e == hipSuccess) e = es;
    if (e == hipSuccess) {
        std::memcpy(st, res, sizeof(*st));
        if (mask) {
            mask->resize(J->W);
            std::memcpy(mask->data(), res + (o.selm - o.st), (size_t)J->W * 8);
        }
        if (front) std::memcpy(front, res + (o.front - o.st), (size_t)P * 4);
    }
    shots().give(w, e == hipSuccess);
    if (e != hipSuccess) return fail(CD_E_DEVICE, std::string("selection: ") + hipGetErrorString(e));
    return CD_OK;
}

int cd_nds(const float *obj, int32_t P, int32_t N, int32_t *front_of, int32_t *n_fronts) {
    cd::SelState st;
    const int rc = run_selection(obj, P, N, 1, 0, 0, nullptr, false, &st, nullptr, front_of);
    if (rc == CD_OK && n_fronts) *n_fronts = st.res[1].last + 1;  // (the sort ran as generation 0)
    return rc;
}

int cd_select(const float *obj, int32_t N, int32_t H, uint32_t gen, uint64_t seed, float *extremes, int32_t *sorted,
              int32_t *front_of, float *norm, int32_t *flags) {
    cd::SelState st;
    std::vector<uint64_t> mask;
    const int rc = run_selection(obj, 2 * N, N, H, gen, seed, extremes, true, &st, &mask, front_of);
    if (rc != CD_OK) return rc;
    if (sorted) survivors_of(mask, N, sorted);
    const cd::SelRes &r = st.res[(gen + 1u) & 1u];
    if (extremes) std::memcpy(extremes, r.ext, sizeof(r.ext));
    if (norm) {
        std::memcpy(norm, r.ideal, 24);
        std::memcpy(norm + 6, r.worst, 24);
        std::memcpy(norm + 12, r.nadir, 24);
    }
    if (flags) {
        flags[0] = r.n_cut;
        flags[1] = r.hyp;
    }
    return CD_OK;
}

// ---------------------------------------------------------------------------
// Batched form
// ---------------------------------------------------------------------------
int cd_batch_create(cd_job *const *jobs, int32_t count, cd_batch **out) {
    if (!jobs || count <= 0 || !out) return fail(CD_E_INVALID, "bad batch arguments");
    for (int j = 0; j < count; ++j) {
        cd_job *J = jobs[j];
        if (!J || J->selection_only || !J->inited) return fail(CD_E_STATE, "batch jobs must be created and initialised");
        for (int k = 0; k < j; ++k)
            if (jobs[k] == J) return fail(CD_E_INVALID, "a job appears twice in the batch");
    }
    cd_batch *B = new cd_batch();
    for (int j = 0; j < count; ++j) {
        (void)hipStreamSynchronize(jobs[j]->stream);
        B->jobs.push_back(jobs[j]);
    }
    cd::Shapes sh;
    B->shapes = cdhost::untuned_shapes(jobs, count);
    if (cdhost::cached_shapes(cdhost::work_signature(jobs, count), &sh)) B->shapes = sh;
    cdhost::WorkLists wl;
    cdhost::build_lists(jobs, count, B->shapes, wl);
    // room for the lists in any shape: 64-row tiles and 4-design groups give the most items
    size_t cap_dom = 0, cap_asc = 0;
    for (int j = 0; j < count; ++j) {
        int nd = 0, na = 0;
        work_counts(jobs[j]->P, jobs[j]->W, &nd, &na);
        cap_dom += nd;
        cap_asc += na;
    }
    B->lds = wl.lds;
    B->stem_lds = wl.stem_lds;
    B->max_pool = wl.max_pool;
    B->pool = wl.pool;
    B->max_refs = wl.max_refs;
    B->mg = wl.mg;
    B->longest = wl.longest;
    B->n_cds = wl.n_cds;
    B->n_small = wl.n_small;
    B->lds_small = wl.lds_small;
    B->n_off = (int)wl.off.size();
    B->n_dom = (int)wl.dom.size();
    B->n_asc = (int)wl.asc.size();
    hipError_t e = hipMalloc(&B->d_jobs, sizeof(cd::DevJob) * count);
    if (e == hipSuccess) e = hipMalloc(&B->d_off, sizeof(int2) * wl.off.size());
    if (e == hipSuccess) e = hipMalloc(&B->d_dom, sizeof(int4) * cap_dom);
    if (e == hipSuccess) e = hipMalloc(&B->d_asc, sizeof(int2) * cap_asc);
    if (e == hipSuccess) e = hipMalloc(&B->d_slist, sizeof(uint2) * cd::stem_list_entries((int)wl.off.size(), wl.mg));
    if (e == hipSuccess) e = hipMalloc(&B->d_sctl, sizeof(int32_t) * cd::STEM_MAX_GROUPS);
    if (e == hipSuccess) e = hipMemset(B->d_sctl, 0, sizeof(int32_t) * cd::STEM_MAX_GROUPS);
    if (e == hipSuccess) e = hipMemcpy(B->d_jobs, wl.descs.data(), sizeof(cd::DevJob) * count, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(B->d_off, wl.off.data(), sizeof(int2) * wl.off.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(B->d_dom, wl.dom.data(), sizeof(int4) * wl.dom.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(B->d_asc, wl.asc.data(), sizeof(int2) * wl.asc.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipStreamCreate(&B->stream);
    if (e == hipSuccess) e = cdhost::set_lds_limits(wl);
    if (e != hipSuccess) {
        cd_batch_destroy(B);
        return fail(CD_E_DEVICE, std::string("batch setup: ") + hipGetErrorString(e));
    }
    for (cd_job *J : B->jobs) J->batches.push_back(B);
    *out = B;
    return CD_OK;
}

static Launch batch_launch(cd_batch *B) {
    return Launch{B->d_jobs,    (int)B->jobs.size(), B->d_off,      B->n_off,   B->d_dom,
                  B->n_dom,     B->d_asc,            B->n_asc,      B->lds,     B->stem_lds,
                  B->max_pool,  B->max_refs,         B->mg,         B->longest, B->d_slist, B->d_sctl,
                  B->n_cds,     B->n_small,          B->lds_small,  B->pool,      B->shapes};
}

int cd_batch_profile(cd_batch *B, int32_t generations, float *kernel_ms) {
    if (!B || !kernel_ms) return fail(CD_E_INVALID, "null argument");
    return profile_generations(batch_launch(B), B->stream, generations, kernel_ms);
}

int cd_batch_step(cd_batch *B, int32_t generations) {
    if (!B) return fail(CD_E_INVALID, "null batch");
    if (generations < 0) return fail(CD_E_INVALID, "negative generation count");
    const OnDevice on(B->jobs[0]->dev);
    return step_graphs(B->graphs, B->stream, batch_launch(B), generations);
}

int cd_batch_sync(cd_batch *B) {
    if (!B) return fail(CD_E_INVALID, "null batch");
    HIPCHK(hipStreamSynchronize(B->stream));
    return CD_OK;
}

int cd_batch_step_timed(cd_batch *B, int32_t generations, float *ms) {
    if (!B) return fail(CD_E_INVALID, "null batch");
    hipEvent_t a, b;
    HIPCHK(hipEventCreate(&a));
    HIPCHK(hipEventCreate(&b));
    HIPCHK(hipEventRecord(a, B->stream));
    int rc = cd_batch_step(B, generations);
    if (rc != CD_OK) return rc;
    HIPCHK(hipEventRecord(b, B->stream));
    HIPCHK(hipEventSynchronize(b));
    float t = 0.f;
    HIPCHK(hipEventElapsedTime(&t, a, b));
    if (ms) *ms = t;
    HIPCHK(hipEventDestroy(a));
    HIPCHK(hipEventDestroy(b));
    return CD_OK;
}

// Install shapes on a batch: its work lists in that shape, the captured
// graph dropped (the next step captures the new launches).
static int batch_apply_shapes(cd_batch *B, const cd::Shapes &sh) {
    cdhost::WorkLists wl;
    cdhost::build_lists(B->jobs.data(), (int)B->jobs.size(), sh, wl);
    HIPCHK(hipStreamSynchronize(B->stream));
    HIPCHK(hipMemcpy(B->d_off, wl.off.data(), sizeof(int2) * wl.off.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(B->d_dom, wl.dom.data(), sizeof(int4) * wl.dom.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(B->d_asc, wl.asc.data(), sizeof(int2) * wl.asc.size(), hipMemcpyHostToDevice));
    B->n_dom = (int)wl.dom.size();
    B->n_asc = (int)wl.asc.size();
    B->n_small = wl.n_small;
    B->lds_small = wl.lds_small;
    B->shapes = sh;
    B->graphs.reset();
    return CD_OK;
}

static int job_apply_shapes(cd_job *J, const cd::Shapes &sh) {
    std::vector<int4> dom;
    std::vector<int2> asc;
    job_lists(J->P, J->W, sh, dom, asc);
    HIPCHK(hipStreamSynchronize(J->stream));
    HIPCHK(hipMemcpy(J->d_dom, dom.data(), sizeof(int4) * dom.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(J->d_asc, asc.data(), sizeof(int2) * asc.size(), hipMemcpyHostToDevice));
    J->n_dom = (int)dom.size();
    J->n_asc = (int)asc.size();
    J->shapes = sh;
    J->graphs.reset();
    return CD_OK;
}

static_assert(sizeof(cd_shapes) == sizeof(cd::Shapes), "cd_shapes mirrors cd::Shapes");
static cd_shapes to_abi(const cd::Shapes &s) {
    cd_shapes o;
    std::memcpy(&o, &s, sizeof(o));
    return o;
}
static cd::Shapes from_abi(const cd_shapes &s) {
    cd::Shapes o;
    std::memcpy(&o, &s, sizeof(o));
    return o;
}

int cd_batch_shapes(cd_batch *B, cd_shapes *get, const cd_shapes *set) {
    if (!B) return fail(CD_E_INVALID, "null batch");
    if (set) {
        const cd::Shapes sh = from_abi(*set);
        if (!cd::shapes_valid(sh)) return fail(CD_E_INVALID, "invalid launch shapes");
        const int rc = batch_apply_shapes(B, sh);
        if (rc != CD_OK) return rc;
    }
    if (get) *get = to_abi(B->shapes);
    return CD_OK;
}

int cd_job_shapes(cd_job *J, cd_shapes *get, const cd_shapes *set) {
    if (!J || J->selection_only) return fail(CD_E_INVALID, "null job");
    if (set) {
        const cd::Shapes sh = from_abi(*set);
        if (!cd::shapes_valid(sh)) return fail(CD_E_INVALID, "invalid launch shapes");
        if (!J->batches.empty()) return fail(CD_E_STATE, "the job is held by a batch");
        const int rc = job_apply_shapes(J, sh);
        if (rc != CD_OK) return rc;
    }
    if (get) *get = to_abi(J->shapes);
    return CD_OK;
}

int cd_batch_tune(cd_batch *B, int32_t gens, cd_shapes *chosen, int32_t *generations_run) {
    if (!B || gens < 1) return fail(CD_E_INVALID, "bad tune arguments");
    cd::Shapes best;
    int run = 0;
    const int rc = tune_shapes(
        B->shapes, (int)B->jobs.size(), gens, B->stream,
        [&](const cd::Shapes &sh, Launch *w) {
            const int r = batch_apply_shapes(B, sh);
            *w = batch_launch(B);
            return r;
        },
        &best, &run);
    if (generations_run) *generations_run = run;
    if (rc != CD_OK) return rc;
    cdhost::store_shapes(cdhost::work_signature(B->jobs.data(), (int)B->jobs.size()), best);
    if (chosen) *chosen = to_abi(best);
    return CD_OK;
}

int cd_job_tune(cd_job *J, int32_t gens, cd_shapes *chosen, int32_t *generations_run) {
    if (!J || J->selection_only || gens < 1) return fail(CD_E_INVALID, "bad tune arguments");
    if (!J->inited) return fail(CD_E_STATE, "cd_job_tune before cd_job_init");
    if (!J->batches.empty()) return fail(CD_E_STATE, "the job is held by a batch: tune the batch");
    cd::Shapes best;
    int run = 0;
    const int rc = tune_shapes(
        J->shapes, 1, gens, J->stream,
        [&](const cd::Shapes &sh, Launch *w) {
            const int r = job_apply_shapes(J, sh);
            *w = job_launch(J);
            return r;
        },
        &best, &run);
    if (generations_run) *generations_run = run;
    if (rc != CD_OK) return rc;
    cd_job *self = J;
    cdhost::store_shapes(cdhost::work_signature(&self, 1), best);
    if (chosen) *chosen = to_abi(best);
    return CD_OK;
}

int cd_batch_destroy(cd_batch *B) {
    if (!B) return CD_OK;
    if (B->stream) (void)hipStreamSynchronize(B->stream);
    for (cd_job *J : B->jobs) J->batches.erase(std::remove(J->batches.begin(), J->batches.end(), B), J->batches.end());
    B->graphs.reset();
    if (B->stream) (void)hipStreamDestroy(B->stream);
    if (B->d_jobs) (void)hipFree(B->d_jobs);
    if (B->d_off) (void)hipFree(B->d_off);
    if (B->d_dom) (void)hipFree(B->d_dom);
    if (B->d_asc) (void)hipFree(B->d_asc);
    if (B->d_slist) (void)hipFree(B->d_slist);
    if (B->d_sctl) (void)hipFree(B->d_sctl);
    delete B;
    return CD_OK;
}

}  // extern "C"
