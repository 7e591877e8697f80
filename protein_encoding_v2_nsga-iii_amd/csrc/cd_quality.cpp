// cd_quality.cpp -- quality indicators of a final pool, on the host.
//
// The reference prints the hypervolume of its normalised pool by running a
// prebuilt `hv` program (src/main.cu:839-858) and the minimum distance to the
// ideal point (MinEuclid, utils.cuh:42-58); its experiment script adds the
// maximum spread (auto_execution_experiments.py:119-134).  This file computes
// them itself: the hypervolume exactly, with the WFG algorithm (While,
// Bradstreet and Barone, IEEE TEVC 16(1), 2012), for minimisation against a
// reference point.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <utility>
#include <vector>

#include "codon_nsga3.h"

namespace {

// Points are rows of d doubles in one array.  Sets shrink quickly from level
// to level, so most of the time goes into small sets: they need no allocation,
// each level has one coordinate less, three coordinates are swept, and the
// number of coordinates is a constant of the code.  400 points in six
// dimensions, a run's final pool: 51 ms with a vector per point and every level in
// all six dimensions, 3.7 ms so; 100 points on a sphere 34.8 and 1.8 ms.

// Points of one level of the recursion, and the order they are taken in.
struct Level {
    std::vector<double> pts;
    std::vector<int> order;
};

// The hypervolume of points given by rows of D doubles against the reference
// point at the origin: a coordinate is its distance to the reference point,
// so a box is a product and larger is better.
class Wfg {
  public:
    Wfg(int n, int d) : levels_((size_t)d + 1) {
        for (int k = 0; k <= d; ++k) {
            levels_[k].pts.resize((size_t)n * (size_t)k);
            levels_[k].order.resize(n);
        }
        stair_.resize(2 * ((size_t)n + 2));
    }

    // Keeps the rows of a[n][d] not weakly dominated by another (one of equal
    // ones): their number.
    template <int d>
    static int nondominated(double *a, int n) {
        int kept = 0;
        for (int i = 0; i < n; ++i) {
            const double *p = a + (size_t)i * d;
            bool out = false;
            for (int k = 0; k < kept && !out; ++k) {
                double *q = a + (size_t)k * d;
                bool ge = true, le = true;  // q >= p, q <= p
                for (int c = 0; c < d; ++c) {
                    ge &= q[c] >= p[c];
                    le &= q[c] <= p[c];
                }
                out = ge;
                if (le && !ge) {  // q goes: the last kept row takes its place
                    --kept;
                    if (k != kept) std::memcpy(q, a + (size_t)kept * d, sizeof(double) * d);
                    --k;
                }
            }
            if (!out) {
                if (kept != i) std::memmove(a + (size_t)kept * d, p, sizeof(double) * d);
                ++kept;
            }
        }
        return kept;
    }

    // Hypervolume of a[n][d], no row weakly dominated by another.  The rows
    // are taken from the worst last coordinate to the best: each adds its box
    // less what the rows after it cover of it, and as those are at least as
    // good in the last coordinate, that is its extent there times a
    // hypervolume of the other d - 1 coordinates.
    template <int d>
    double volume(const double *a, int n) {
        if (n == 0) return 0.0;
        if (n == 1) return box<d>(a);
        if constexpr (d == 1) {
            return *std::max_element(a, a + n);
        } else {
            if (n == 2) {
                double both = 1.0;
                for (int c = 0; c < d; ++c) both *= std::min(a[c], a[d + c]);
                return box<d>(a) + box<d>(a + d) - both;
            }
            int *o = levels_[d].order.data();
            for (int i = 0; i < n; ++i) o[i] = i;
            std::sort(o, o + n, [a](int x, int y) { return a[(size_t)x * d + d - 1] < a[(size_t)y * d + d - 1]; });
            if constexpr (d == 2) return volume2(a, o, n);
            else if constexpr (d == 3) return volume3(a, o, n);
            else return slices<d>(a, o, n);
        }
    }

  private:
    template <int d>
    static double box(const double *p) {
        double v = 1.0;
        for (int c = 0; c < d; ++c) v *= p[c];
        return v;
    }

    template <int d>
    double slices(const double *a, const int *o, int n) {
        double *lim = levels_[d].pts.data();
        double v = 0.0;
        for (int i = 0; i < n; ++i) {
            const double *p = a + (size_t)o[i] * d;
            int m = 0;
            bool covered = false;
            for (int j = i + 1; j < n && !covered; ++j, ++m) {
                const double *q = a + (size_t)o[j] * d;
                double *r = lim + (size_t)m * (d - 1);
                covered = true;
                for (int c = 0; c < d - 1; ++c) {
                    r[c] = std::min(p[c], q[c]);
                    covered &= q[c] >= p[c];
                }
            }
            if (covered) continue;
            m = nondominated<d - 1>(lim, m);
            v += p[d - 1] * (box<d - 1>(p) - volume<d - 1>(lim, m));
        }
        return v;
    }

    // Two coordinates: the first falls as the last rises.
    static double volume2(const double *a, const int *o, int n) {
        double v = 0.0, below = 0.0;
        for (int i = 0; i < n; ++i) {
            const double *p = a + 2 * (size_t)o[i];
            v += p[0] * (p[1] - below);
            below = p[1];
        }
        return v;
    }

    // Three coordinates: a sweep from the best last coordinate down, with the
    // staircase of the rows passed so far in the first two (x rising, y
    // falling) and its area.
    double volume3(const double *a, const int *o, int n) {
        double *x = stair_.data(), *y = x + stair_.size() / 2;
        int m = 0;
        double area = 0.0, v = 0.0;
        for (int i = n - 1; i >= 0; --i) {
            const double *p = a + 3 * (size_t)o[i];
            int k = m;  // the steps from k on have x >= p[0]
            while (k > 0 && x[k - 1] >= p[0]) --k;
            if (k == m || y[k] < p[1]) {
                // steps e .. k-1 lie under p (and step k if its x is equal)
                const int to = k < m && x[k] == p[0] ? k + 1 : k;
                int e = k;
                double left = p[0], add = 0.0;
                double low = k < m ? y[k] : 0.0;  // the staircase's height from `left` down
                while (e > 0 && y[e - 1] <= p[1]) {
                    add += (left - x[e - 1]) * (p[1] - low);
                    left = x[e - 1];
                    low = y[e - 1];
                    --e;
                }
                add += (left - (e > 0 ? x[e - 1] : 0.0)) * (p[1] - low);
                area += add;
                // p replaces steps e .. to-1
                if (to - e != 1) {
                    std::memmove(x + e + 1, x + to, sizeof(double) * (m - to));
                    std::memmove(y + e + 1, y + to, sizeof(double) * (m - to));
                }
                x[e] = p[0];
                y[e] = p[1];
                m += 1 - (to - e);
            }
            // (an area without bound times no extent would not be a number)
            const double extent = p[2] - (i > 0 ? a[3 * (size_t)o[i - 1] + 2] : 0.0);
            if (extent > 0.0) v += area * extent;
        }
        return v;
    }

    std::vector<Level> levels_;
    std::vector<double> stair_;
};

template <int d>
double volume_of(double *s, int n) {
    n = Wfg::nondominated<d>(s, n);
    return Wfg(n, d).volume<d>(s, n);
}
template <int... d>
double volume_of(double *s, int n, int dims, std::integer_sequence<int, d...>) {
    double (*const f[])(double *, int) = {volume_of<d + 1>...};
    return f[dims - 1](s, n);
}

}  // namespace

extern "C" {

/* Exact hypervolume (minimisation) of n points in d dimensions against ref;
 * points outside the reference box contribute nothing. */
int cd_hypervolume(const double *pts, int32_t n, int32_t d, const double *ref, double *out) {
    if (!pts || !ref || !out || n < 0 || d < 1 || d > 16) return CD_E_INVALID;
    std::vector<double> s;
    s.reserve((size_t)n * d);
    int kept = 0;
    for (int i = 0; i < n; ++i) {
        const double *p = pts + (size_t)i * d;
        bool inside = true;
        for (int k = 0; k < d; ++k)
            if (!(p[k] < ref[k])) inside = false;
        if (!inside) continue;
        for (int k = 0; k < d; ++k) s.push_back(ref[k] - p[k]);
        ++kept;
    }
    *out = volume_of(s.data(), kept, d, std::make_integer_sequence<int, 16>());
    return CD_OK;
}

/* Normalise raw objective records as src/main.cu:789-835 does before its
 * quality output: objectives 0-3 are stored negated and are flipped back,
 * every objective becomes (x - ideal) / (nadir - ideal) with the reference's
 * fixed ideal {1, 0.2, 0.4, 0.5, 0, 0} and nadir {0, -0.15, 0, 0, 0.6, 1},
 * then values >= 1 become 0.999999 and negative values 0.  out [n][6]. */
int cd_normalize(const float *obj, int32_t n, float *out) {
    if (!obj || !out || n < 0) return CD_E_INVALID;
    static const float ideal[6] = {1.f, 0.2f, 0.4f, 0.5f, 0.f, 0.f};
    static const float nadir[6] = {0.f, -0.15f, 0.f, 0.f, 0.6f, 1.f};
    for (int i = 0; i < n; ++i)
        for (int k = 0; k < 6; ++k) {
            float v = obj[(size_t)i * 6 + k];
            if (k < 4) v = -v;
            v = (v - ideal[k]) / (nadir[k] - ideal[k]);
            if (v >= 1.f) v = 0.999999f;
            if (v < 0.f) v = 0.f;
            out[(size_t)i * 6 + k] = v;
        }
    return CD_OK;
}

/* Minimum Euclidean distance to the origin (MinEuclid, utils.cuh:42-58) and
 * maximum spread sqrt(sum_k (max_k - min_k)^2)
 * (auto_execution_experiments.py:119-134) of n normalised points. */
int cd_min_distance_spread(const float *pts, int32_t n, float *min_dist, float *spread) {
    if (!pts || n <= 0) return CD_E_INVALID;
    double best = 1e300, sp = 0.0;
    double lo[6], hi[6];
    for (int k = 0; k < 6; ++k) {
        lo[k] = 1e300;
        hi[k] = -1e300;
    }
    for (int i = 0; i < n; ++i) {
        double s = 0.0;
        for (int k = 0; k < 6; ++k) {
            const double v = pts[(size_t)i * 6 + k];
            s += v * v;
            lo[k] = std::min(lo[k], v);
            hi[k] = std::max(hi[k], v);
        }
        best = std::min(best, std::sqrt(s));
    }
    for (int k = 0; k < 6; ++k) sp += (hi[k] - lo[k]) * (hi[k] - lo[k]);
    if (min_dist) *min_dist = (float)best;
    if (spread) *spread = (float)std::sqrt(sp);
    return CD_OK;
}

}  // extern "C"
