// Statistics on the state plan (tsg_states.h; gfx950).
//
//   k_state_stage    the run's host arrays from pinned memory, the sample
//                    rows cleared
//   k_state_seed     each (sample, column) pair into its sample's row; each
//                    tile's first window
//   k_state_count    one launch per level: every state's row is the sum of
//                    at most 8 earlier rows (bound by those gathers, which
//                    mostly hit the XCD's L2: a level is numbered along the
//                    genome and each XCD takes a contiguous run of it)
//   k_state_eval     per tile of events (branch) or rows (site), the counts
//                    of its states gathered into LDS by column; then every
//                    wave takes every fourth output: a lane evaluates the
//                    summary of 8 (4) events and the wave adds them up.  In a
//                    tile of many windows a thread takes a (window, output)
//                    and loops over the window's events
//   k_state_windows  the segment sums of each window added up (where there
//                    are many), k_state_finish: the running branch sum along
//                    the windows, normalisation
//
// A branch statistic's running sum R changes at each event by b F (b the
// change of branch length, F the summary of the event's counts), so window
// [l, r) has  R(l) (r - l) + sum over its events at x of b F (r - x),  and
// R(l) is the sum of b F over the earlier windows (trees.c:1352-1523 keeps
// the same R event by event).  Every sum has a fixed order that depends on
// the tree sequence and the query's own windows alone, so a query's results
// are the same bits alone and fused with others.
//
// Summaries: trees.c:3934-5291, the unpolarised wrapper f(x) + f(total - x)
// (trees.c:1944-1972) folded in.  Integer counts are exact in FP64 and the
// numerators are summed before the one division by the denominator.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tsg_common.h"
#include "tsg_finals.h"
#include "tsg_kernels.h"
#include "tsg_launch.h"
#include "tsg_states.h"

#define WAVE 64
#define EVAL_THREADS 256
#define FINISH_THREADS 1024

namespace {

// workgroup b of nb, each XCD (workgroups go to the 8 in turn) taking a
// contiguous run; nb or more: none
__device__ __forceinline__ int xcd_block(int b, int nb) {
    const int per = (nb + 7) / 8;
    return (b % 8) * per + b / 8;
}
unsigned xcd_grid(int64_t nb) { return 8u * (unsigned) ((nb + 7) / 8); }

// --- counts -------------------------------------------------------------------

__device__ __forceinline__ void stage(const TsgStateArgs &a, int64_t b) {
    int64_t i = b * 256 + threadIdx.x;
    if (i < a.stage_words) {
        a.stage_dst[i] = a.stage_src[i];
        return;
    }
    i -= a.stage_words;
    if (i < (int64_t) (a.num_samples + 1) * a.RW) a.x[i] = 0u;
}
int64_t stage_blocks(const TsgStateArgs &a) {
    return (a.stage_words + (int64_t) (a.num_samples + 1) * a.RW + 255) / 256;
}

// last window w of 0 .. W - 1 with win[w] <= x (0 where there is none)
__device__ __forceinline__ int window_of(const double *win, int W, double x) {
    int lo = 0, hi = W - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (win[mid] <= x) {
            lo = mid;
        } else {
            hi = mid - 1;
        }
    }
    return lo;
}

template <int TYPE>
__device__ __forceinline__ void seed(const TsgStateArgs &a, int64_t b) {
    const int64_t i = b * 256 + threadIdx.x;
    if (i < a.npairs) {
        uint32_t *row = a.x + (int64_t) (1 + a.pair_sample[i]) * a.RW;
        const int k = a.pair_col[i];
        if constexpr (TYPE == TSG_ROW_U16) {
            reinterpret_cast<uint16_t *>(row)[k] = 1;
        } else if constexpr (TYPE == TSG_ROW_I32) {
            row[k] = 1u;
        } else {
            reinterpret_cast<double *>(row)[k] = a.pair_w[i];
        }
        return;
    }
    // tile t's first window: 0 for the first tile, the last one past the last
    const int64_t j = i - a.npairs;
    if (j >= a.ntile_w) return;
    int q = 0;
    for (int p = 1; p < a.Q; p++) {
        if (a.queries[p].new_windows && a.queries[p].tw <= j) q = p;
    }
    const TsgStateQuery &Q = a.queries[q];
    const int t = (int) (j - Q.tw);
    const int tiles = Q.branch ? a.btiles : a.stiles;
    const double *tpos = Q.branch ? a.btile_pos : a.stile_pos;
    a.tile_w[j] = t == 0 ? 0
                  : t >= tiles ? Q.W - 1
                               : window_of(a.windows + Q.win_off, Q.W, tpos[t]);
}
int64_t seed_blocks(const TsgStateArgs &a) {
    return ((int64_t) a.npairs + a.ntile_w + 255) / 256;
}

template <int V>
struct Words {
    uint32_t w[V];
};
template <int V>
__device__ __forceinline__ Words<V> load_words(const uint32_t *p) {
    Words<V> r;
    if constexpr (V == 4) {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        r.w[0] = v.x, r.w[1] = v.y, r.w[2] = v.z, r.w[3] = v.w;
    } else if constexpr (V == 2) {
        const uint2 v = *reinterpret_cast<const uint2 *>(p);
        r.w[0] = v.x, r.w[1] = v.y;
    } else {
        r.w[0] = *p;
    }
    return r;
}
template <int V>
__device__ __forceinline__ void store_words(uint32_t *p, const Words<V> &r) {
    if constexpr (V == 4) {
        *reinterpret_cast<uint4 *>(p) = make_uint4(r.w[0], r.w[1], r.w[2], r.w[3]);
    } else if constexpr (V == 2) {
        *reinterpret_cast<uint2 *>(p) = make_uint2(r.w[0], r.w[1]);
    } else {
        *p = r.w[0];
    }
}

// States s0 .. s1 - 1 of a level, V words a thread.  16-bit counts are added
// two to a word: no count exceeds its column's total, so none carries over.
template <int V, bool F64>
__device__ __forceinline__ void count(const TsgStateArgs &a, int s0, int s1, int64_t b) {
    const int parts = a.RW / V;
    const int64_t i = b * 256 + threadIdx.x;
    const int64_t s = s0 + i / parts;
    const int p = (int) (i % parts) * V;
    if (s >= s1) return;
    const int4 *in =
        reinterpret_cast<const int4 *>(a.in + (s - 1 - a.num_samples) * TSG_STATE_IN);
    const int4 u = in[0], v = in[1];
    const int id[TSG_STATE_IN] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    Words<V> r[TSG_STATE_IN];
#pragma unroll
    for (int j = 0; j < TSG_STATE_IN; j++) r[j] = load_words<V>(a.x + (int64_t) id[j] * a.RW + p);
#pragma unroll
    for (int j = 1; j < TSG_STATE_IN; j++) {
        if constexpr (F64) {
#pragma unroll
            for (int w = 0; w < V; w += 2) {
                const double t = __hiloint2double(r[0].w[w + 1], r[0].w[w]) +
                                 __hiloint2double(r[j].w[w + 1], r[j].w[w]);
                r[0].w[w] = __double2loint(t);
                r[0].w[w + 1] = __double2hiint(t);
            }
        } else {
#pragma unroll
            for (int w = 0; w < V; w++) r[0].w[w] += r[j].w[w];
        }
    }
    store_words<V>(a.x + s * a.RW + p, r[0]);
}
int words_per_thread(int RW) { return RW < 4 ? RW : 4; }
int64_t count_blocks(const TsgStateArgs &a, int64_t states) {
    return (states * (a.RW / words_per_thread(a.RW)) + 255) / 256;
}

template <bool F64>
__device__ __forceinline__ void count_rw(const TsgStateArgs &a, int s0, int s1, int64_t b) {
    if (a.RW >= 4) {
        count<4, F64>(a, s0, s1, b);
    } else if (a.RW == 2) {
        count<2, F64>(a, s0, s1, b);
    } else if constexpr (!F64) {
        count<1, false>(a, s0, s1, b);
    }
}

// --- evaluation ---------------------------------------------------------------

template <int TYPE>
struct RowType {
    using T = uint16_t;
};
template <>
struct RowType<TSG_ROW_I32> {
    using T = int32_t;
};
template <>
struct RowType<TSG_ROW_F64> {
    using T = double;
};
// A site row's counts are sums of additions and subtractions, so site tiles
// hold 32-bit counts whatever the rows hold.
template <int TYPE, bool BRANCH>
struct TileType {
    using T = typename std::conditional<!BRANCH && TYPE == TSG_ROW_U16, int32_t,
                                        typename RowType<TYPE>::T>::type;
};

// first index of 0 .. n with pos[index] >= x (LDS)
__device__ __forceinline__ int lower_bound(const double *pos, int n, double x) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (pos[mid] < x) {
            lo = mid + 1;
        } else {
            hi = mid;
        }
    }
    return lo;
}

template <typename T>
__device__ __forceinline__ double2 load2(const T *col, int i);
template <>
__device__ __forceinline__ double2 load2<uint16_t>(const uint16_t *col, int i) {
    const uint32_t v = reinterpret_cast<const uint32_t *>(col)[i];
    return make_double2((double) (v & 0xFFFFu), (double) (v >> 16));
}
template <>
__device__ __forceinline__ double2 load2<int32_t>(const int32_t *col, int i) {
    const int2 v = reinterpret_cast<const int2 *>(col)[i];
    return make_double2((double) v.x, (double) v.y);
}
template <>
__device__ __forceinline__ double2 load2<double>(const double *col, int i) {
    return reinterpret_cast<const double2 *>(col)[i];
}

// Summary numerators at the counts x[0..3] (columns i, j, k, l) of sets of
// n[0..3] samples: one(x) polarised, both(x) = one(x) + one(n - x).
struct Nums {
    double n[4];
};
struct Diversity {
    static constexpr int S = 1;
    Nums p;
    __device__ double one(const double *x) const { return x[0] * (p.n[0] - x[0]); }
    __device__ double both(const double *x) const { return 2.0 * one(x); }
};
struct Segregating {
    static constexpr int S = 1;
    Nums p;
    __device__ double one(const double *x) const { return x[0] > 0 ? p.n[0] - x[0] : 0.0; }
    // n for 0 < x < n
    __device__ double both(const double *x) const {
        return (x[0] > 0 ? p.n[0] - x[0] : 0.0) + (x[0] < p.n[0] ? x[0] : 0.0);
    }
};
struct Y1 {
    static constexpr int S = 1;
    Nums p;
    __device__ double one(const double *x) const {
        const double y = p.n[0] - x[0];
        return x[0] * y * (y - 1);
    }
    __device__ double both(const double *x) const {
        return x[0] * (p.n[0] - x[0]) * (p.n[0] - 2);
    }
};
struct Divergence {
    static constexpr int S = 2;
    Nums p;
    __device__ double one(const double *x) const { return x[0] * (p.n[1] - x[1]); }
    __device__ double both(const double *x) const {
        return fma(x[0], p.n[1] - x[1], (p.n[0] - x[0]) * x[1]);
    }
};
struct Product {  // non-centred relatedness
    static constexpr int S = 2;
    Nums p;
    __device__ double one(const double *x) const { return x[0] * x[1]; }
    __device__ double both(const double *x) const {
        return fma(x[0], x[1], (p.n[0] - x[0]) * (p.n[1] - x[1]));
    }
};
template <typename D, int SLOTS>
struct Complement {  // both() from one()
    static constexpr int S = SLOTS;
    Nums p;
    __device__ double one(const double *x) const { return static_cast<const D *>(this)->f(x); }
    __device__ double both(const double *x) const {
        double y[SLOTS];
#pragma unroll
        for (int i = 0; i < SLOTS; i++) y[i] = p.n[i] - x[i];
        return static_cast<const D *>(this)->f(x) + static_cast<const D *>(this)->f(y);
    }
};
struct Y2 : Complement<Y2, 2> {
    __device__ double f(const double *x) const {
        const double y = p.n[1] - x[1];
        return x[0] * y * (y - 1);
    }
};
struct F2 : Complement<F2, 2> {
    __device__ double f(const double *x) const {
        const double y = p.n[1] - x[1];
        return (x[0] * y) * fma(x[0] - 1, y - 1, -((p.n[0] - x[0]) * x[1]));
    }
};
struct Y3 : Complement<Y3, 3> {
    __device__ double f(const double *x) const {
        return x[0] * (p.n[1] - x[1]) * (p.n[2] - x[2]);
    }
};
struct F3 : Complement<F3, 3> {
    __device__ double f(const double *x) const {
        const double b = fma(x[0] - 1, p.n[2] - x[2], -((p.n[0] - x[0]) * x[2]));
        return (x[0] * (p.n[1] - x[1])) * b;
    }
};
struct F4 {
    static constexpr int S = 4;
    Nums p;
    __device__ double b(const double *x) const { return fma(p.n[3], x[2], -(p.n[2] * x[3])); }
    __device__ double one(const double *x) const { return x[0] * (p.n[1] - x[1]) * b(x); }
    __device__ double both(const double *x) const {
        return fma(p.n[1], x[0], -(p.n[0] * x[1])) * b(x);
    }
};
// centred relatedness: slot 2 is the mean over the query's columns
struct Relatedness {
    Nums p;  // 1 / set size
    __device__ double one(const double *x) const {
        return (x[0] * p.n[0] - x[2]) * (x[1] * p.n[1] - x[2]);
    }
};
// summaries of real-valued weights (p.n: the columns' totals)
struct TraitCovariance {
    static constexpr int S = 1;
    Nums p;
    __device__ double one(const double *x) const { return x[0] * x[0]; }
    __device__ double both(const double *x) const {
        const double y = p.n[0] - x[0];
        return fma(x[0], x[0], y * y);
    }
};
struct TraitCorrelation {  // slots: trait, frequency
    static constexpr int S = 2;
    Nums p;
    __device__ double f(double x, double q) const {
        return (q > 0.0 && q < 1.0) ? (x * x) / (q * (1 - q)) : 0.0;
    }
    __device__ double one(const double *x) const { return f(x[0], x[1]); }
    __device__ double both(const double *x) const {
        return f(x[0], x[1]) + f(p.n[0] - x[0], p.n[1] - x[1]);
    }
};
struct RelatednessWeighted {  // slots: i, j, frequency
    static constexpr int S = 3;
    Nums p;
    double ca, cb;
    __device__ double f(const double *x) const {
        return (x[0] - ca * x[2]) * (x[1] - cb * x[2]);
    }
    __device__ double one(const double *x) const { return f(x); }
    __device__ double both(const double *x) const {
        const double y[3] = {p.n[0] - x[0], p.n[1] - x[1], p.n[2] - x[2]};
        return f(x) + f(y);
    }
};

// A tile's events as one lane of a wave sees them: events 128 j + 2 lane and
// the next, j < N / 2, with their weights in the window's two sums.
template <int N>
struct LaneEvents {
    double wl[N], wb[N];
};

// how a row's value follows from the summary
#define VALUE_ONE 0    // polarised, every row a pair or derived
#define VALUE_BOTH 1   // unpolarised, every event or pair row
#define VALUE_MIXED 2  // site tiles with other rows

template <typename T, int TILE, bool BRANCH, int VALUE, typename F>
__device__ __forceinline__ void add_up(const F &f, const T *const *col, const int32_t *kind,
                                       bool polarised, int lane, const LaneEvents<TILE / WAVE> &ev,
                                       double &L, double &J) {
    constexpr int N = TILE / WAVE;
#pragma unroll
    for (int j = 0; j < N / 2; j++) {
        double x0[F::S], x1[F::S];
        const int i = WAVE * j + lane;
#pragma unroll
        for (int s = 0; s < F::S; s++) {
            const double2 v = load2<T>(col[s], i);
            x0[s] = v.x;
            x1[s] = v.y;
        }
        double v0, v1;
        if constexpr (VALUE == VALUE_ONE) {
            v0 = f.one(x0);
            v1 = f.one(x1);
        } else if constexpr (VALUE == VALUE_BOTH) {
            v0 = f.both(x0);
            v1 = f.both(x1);
        } else {
            const int2 k = reinterpret_cast<const int2 *>(kind)[i];
            const bool both = !polarised;
            v0 = (both && k.x == TSG_ROW_PAIR) ? f.both(x0) : f.one(x0);
            v1 = (both && k.y == TSG_ROW_PAIR) ? f.both(x1) : f.one(x1);
            if (polarised && k.x == TSG_ROW_ANCESTRAL) v0 = 0.0;
            if (polarised && k.y == TSG_ROW_ANCESTRAL) v1 = 0.0;
        }
        L = fma(v0, ev.wl[2 * j], L);
        L = fma(v1, ev.wl[2 * j + 1], L);
        if constexpr (BRANCH) {
            J = fma(v0, ev.wb[2 * j], J);
            J = fma(v1, ev.wb[2 * j + 1], J);
        }
    }
}

template <typename T, int TILE, bool BRANCH, typename F>
__device__ __forceinline__ void add_value(const F &f, const T *const *col, const int32_t *kind,
                                          bool mixed, bool polarised, int lane,
                                          const LaneEvents<TILE / WAVE> &ev, double &L, double &J) {
    if (!BRANCH && mixed) {
        add_up<T, TILE, BRANCH, VALUE_MIXED>(f, col, kind, polarised, lane, ev, L, J);
    } else if (polarised) {
        add_up<T, TILE, BRANCH, VALUE_ONE>(f, col, kind, true, lane, ev, L, J);
    } else {
        add_up<T, TILE, BRANCH, VALUE_BOTH>(f, col, kind, false, lane, ev, L, J);
    }
}

// The trait regression's summary (trees.c:4108-4152) of event e, or of its
// complement: covariates cbase .. with their row of V, the sample count x_l.
template <int TILE>
__device__ __forceinline__ double regression(const TsgStateArgs &a, const TsgOut &o,
                                             const double *cols, int e, bool comp) {
    const double *v = a.opar + o.par;
    const double *tot = a.col_total_w;
    auto X = [&](int c) {
        const double x = cols[c * TILE + e];
        return comp ? tot[c] - x : x;
    };
    const double m = X(o.l), n = (double) o.ni;
    if (!(m > 0.0 && m < n)) return 0.0;
    double r = X(o.i), denom = m;
    for (int c = 0; c < o.ccount; c++) {
        const double z = X(o.cbase + c);
        r -= z * v[c];
        denom -= z * z;
    }
    return denom < 1e-8 ? 0.0 : (r * r) / (2 * denom * denom);
}

template <int TILE, bool BRANCH>
__device__ void add_regression(const TsgStateArgs &a, const TsgOut &o, const double *cols,
                               const int32_t *kind, bool mixed, bool polarised, int lane,
                               const LaneEvents<TILE / WAVE> &ev, double &L, double &J) {
    constexpr int N = TILE / WAVE;
    for (int j = 0; j < N; j++) {
        const int e = 2 * WAVE * (j / 2) + 2 * lane + (j & 1);
        const int k = (!BRANCH && mixed) ? kind[e] : TSG_ROW_PAIR;
        double f = (polarised && k == TSG_ROW_ANCESTRAL) ? 0.0
                                                         : regression<TILE>(a, o, cols, e, false);
        if (!polarised && k == TSG_ROW_PAIR) f = f + regression<TILE>(a, o, cols, e, true);
        double wl = 0, wb = 0;
#pragma unroll
        for (int r = 0; r < N; r++) {
            if (r == j) {
                wl = ev.wl[r];
                wb = ev.wb[r];
            }
        }
        L = fma(f, wl, L);
        if constexpr (BRANCH) J = fma(f, wb, J);
    }
}

// Output o's two sums over this lane's events, before the denominator.
template <int TYPE, int TILE, bool BRANCH>
__device__ __forceinline__ void add_output(const TsgStateArgs &a, const TsgOut &o,
                                           const typename TileType<TYPE, BRANCH>::T *cols,
                                           const double *mean, const int32_t *kind, bool mixed,
                                           int lane, const LaneEvents<TILE / WAVE> &ev, double &L,
                                           double &J) {
    using T = typename TileType<TYPE, BRANCH>::T;
    const bool pol = (o.flags & 1) != 0;
    if constexpr (TYPE == TSG_ROW_F64) {
        const double *col[4] = {cols + o.i * TILE, cols + o.j * TILE, nullptr, nullptr};
        const double *tot = a.col_total_w;
        switch (o.stat) {
        case TSG_STAT_TRAIT_COVARIANCE:
            add_value<T, TILE, BRANCH>(TraitCovariance{{{tot[o.i]}}}, col, kind, mixed, pol, lane,
                                       ev, L, J);
            break;
        case TSG_STAT_TRAIT_CORRELATION:
            col[1] = cols + o.l * TILE;
            add_value<T, TILE, BRANCH>(TraitCorrelation{{{tot[o.i], tot[o.l]}}}, col, kind, mixed,
                                       pol, lane, ev, L, J);
            break;
        case TSG_STAT_TRAIT_LINEAR_MODEL:
            add_regression<TILE, BRANCH>(a, o, cols, kind, mixed, pol, lane, ev, L, J);
            break;
        case TSG_STAT_RELATEDNESS_WEIGHTED:
            col[2] = cols + o.l * TILE;
            add_value<T, TILE, BRANCH>(
                RelatednessWeighted{
                    {{tot[o.i], tot[o.j], tot[o.l]}}, a.opar[o.par], a.opar[o.par + 1]},
                col, kind, mixed, pol, lane, ev, L, J);
            break;
        case TSG_STAT_RELATEDNESS_WEIGHTED_NONCENTRED:
            add_value<T, TILE, BRANCH>(Product{{{tot[o.i], tot[o.j]}}}, col, kind, mixed, pol,
                                       lane, ev, L, J);
            break;
        default:
            break;
        }
    } else {
        const T *col[4] = {cols + o.i * TILE, cols + o.j * TILE, cols + o.k * TILE,
                           cols + o.l * TILE};
        const Nums n = {{(double) o.ni, (double) o.nj, (double) o.nk, (double) o.nl}};
#define SUMMARY(F)                                                                             \
    {                                                                                          \
        F f;                                                                                   \
        f.p = n;                                                                               \
        add_value<T, TILE, BRANCH>(f, col, kind, mixed, pol, lane, ev, L, J);                  \
        break;                                                                                 \
    }
        switch (o.stat) {
        case TSG_STAT_DIVERSITY:
            SUMMARY(Diversity)
        case TSG_STAT_SEGREGATING_SITES:
            SUMMARY(Segregating)
        case TSG_STAT_Y1:
            SUMMARY(Y1)
        case TSG_STAT_DIVERGENCE:
            SUMMARY(Divergence)
        case TSG_STAT_RELATEDNESS_NONCENTRED:
            SUMMARY(Product)
        case TSG_STAT_Y2:
            SUMMARY(Y2)
        case TSG_STAT_F2:
            SUMMARY(F2)
        case TSG_STAT_Y3:
            SUMMARY(Y3)
        case TSG_STAT_F3:
            SUMMARY(F3)
        case TSG_STAT_F4:
            SUMMARY(F4)
#undef SUMMARY
        case TSG_STAT_RELATEDNESS: {
            constexpr int N = TILE / WAVE;
            Relatedness f;
            f.p = Nums{{1.0 / n.n[0], 1.0 / n.n[1], 0.0, 0.0}};
#pragma unroll
            for (int j = 0; j < N / 2; j++) {
                const int i = WAVE * j + lane;
                const double2 xi = load2<T>(col[0], i), xj = load2<T>(col[1], i);
                const double2 mu = load2<double>(mean, i);
                const double a0[3] = {xi.x, xj.x, mu.x}, a1[3] = {xi.y, xj.y, mu.y};
                double v0 = f.one(a0), v1 = f.one(a1);
                int2 k = make_int2(TSG_ROW_PAIR, TSG_ROW_PAIR);
                if (!BRANCH && mixed) k = reinterpret_cast<const int2 *>(kind)[i];
                if (pol) {
                    v0 = k.x == TSG_ROW_ANCESTRAL ? 0.0 : v0;
                    v1 = k.y == TSG_ROW_ANCESTRAL ? 0.0 : v1;
                } else {
                    v0 = k.x == TSG_ROW_PAIR ? 2.0 * v0 : v0;
                    v1 = k.y == TSG_ROW_PAIR ? 2.0 * v1 : v1;
                }
                L = fma(v0, ev.wl[2 * j], L);
                L = fma(v1, ev.wl[2 * j + 1], L);
                if constexpr (BRANCH) {
                    J = fma(v0, ev.wb[2 * j], J);
                    J = fma(v1, ev.wb[2 * j + 1], J);
                }
            }
            break;
        }
        default:
            break;
        }
    }
}

// Output o's summary of event e alone, before the denominator.
template <int TYPE, int TILE, bool BRANCH>
__device__ __forceinline__ double value_of(const TsgStateArgs &a, const TsgOut &o,
                                           const typename TileType<TYPE, BRANCH>::T *cols,
                                           const double *mean, const int32_t *kind, int e) {
    const bool pol = (o.flags & 1) != 0;
    const int k = BRANCH ? TSG_ROW_PAIR : kind[e];
    if (pol && k == TSG_ROW_ANCESTRAL) return 0.0;
    const bool both = !pol && k == TSG_ROW_PAIR;
    if constexpr (TYPE == TSG_ROW_F64) {
        const double *tot = a.col_total_w;
        const double x[3] = {cols[o.i * TILE + e],
                             cols[(o.stat == TSG_STAT_TRAIT_CORRELATION ? o.l : o.j) * TILE + e],
                             cols[o.l * TILE + e]};
        switch (o.stat) {
        case TSG_STAT_TRAIT_COVARIANCE: {
            const TraitCovariance f{{{tot[o.i]}}};
            return both ? f.both(x) : f.one(x);
        }
        case TSG_STAT_TRAIT_CORRELATION: {
            const TraitCorrelation f{{{tot[o.i], tot[o.l]}}};
            return both ? f.both(x) : f.one(x);
        }
        case TSG_STAT_TRAIT_LINEAR_MODEL: {
            const double v = regression<TILE>(a, o, cols, e, false);
            return both ? v + regression<TILE>(a, o, cols, e, true) : v;
        }
        case TSG_STAT_RELATEDNESS_WEIGHTED: {
            const RelatednessWeighted f{
                {{tot[o.i], tot[o.j], tot[o.l]}}, a.opar[o.par], a.opar[o.par + 1]};
            return both ? f.both(x) : f.one(x);
        }
        case TSG_STAT_RELATEDNESS_WEIGHTED_NONCENTRED: {
            const Product f{{{tot[o.i], tot[o.j]}}};
            return both ? f.both(x) : f.one(x);
        }
        default:
            return 0.0;
        }
    } else {
        const Nums n = {{(double) o.ni, (double) o.nj, (double) o.nk, (double) o.nl}};
        double x[4] = {(double) cols[o.i * TILE + e], (double) cols[o.j * TILE + e], 0.0, 0.0};
#define SUMMARY(F)                          \
    {                                       \
        F f;                                \
        f.p = n;                            \
        return both ? f.both(x) : f.one(x); \
    }
        switch (o.stat) {
        case TSG_STAT_DIVERSITY:
            SUMMARY(Diversity)
        case TSG_STAT_SEGREGATING_SITES:
            SUMMARY(Segregating)
        case TSG_STAT_Y1:
            SUMMARY(Y1)
        case TSG_STAT_DIVERGENCE:
            SUMMARY(Divergence)
        case TSG_STAT_RELATEDNESS_NONCENTRED:
            SUMMARY(Product)
        case TSG_STAT_Y2:
            SUMMARY(Y2)
        case TSG_STAT_F2:
            SUMMARY(F2)
        case TSG_STAT_RELATEDNESS: {
            x[2] = mean[e];
            const double v = Relatedness{{{1.0 / n.n[0], 1.0 / n.n[1], 0.0, 0.0}}}.one(x);
            return both ? 2.0 * v : v;
        }
        default:
            break;
        }
        x[2] = (double) cols[o.k * TILE + e];
        x[3] = (double) cols[o.l * TILE + e];
        switch (o.stat) {
        case TSG_STAT_Y3:
            SUMMARY(Y3)
        case TSG_STAT_F3:
            SUMMARY(F3)
        case TSG_STAT_F4:
            SUMMARY(F4)
        default:
            return 0.0;
        }
#undef SUMMARY
    }
}

// Four lane values a, b, c, d added up over the wave at once: lanes 0-15 get
// a's sum, 16-31 c's, 32-47 b's, 48-63 d's (each swap halves the number of
// values a lane holds: 3 swaps and 4 row rotations for 4 sums instead of 24
// steps).
__device__ __forceinline__ void swap32(double &x, double &y) {
    auto lo = __builtin_amdgcn_permlane32_swap((unsigned) __double2loint(x),
                                               (unsigned) __double2loint(y), false, false);
    auto hi = __builtin_amdgcn_permlane32_swap((unsigned) __double2hiint(x),
                                               (unsigned) __double2hiint(y), false, false);
    x = __hiloint2double((int) hi[0], (int) lo[0]);
    y = __hiloint2double((int) hi[1], (int) lo[1]);
}
__device__ __forceinline__ void swap16(double &x, double &y) {
    auto lo = __builtin_amdgcn_permlane16_swap((unsigned) __double2loint(x),
                                               (unsigned) __double2loint(y), false, false);
    auto hi = __builtin_amdgcn_permlane16_swap((unsigned) __double2hiint(x),
                                               (unsigned) __double2hiint(y), false, false);
    x = __hiloint2double((int) hi[0], (int) lo[0]);
    y = __hiloint2double((int) hi[1], (int) lo[1]);
}
template <int D>
__device__ __forceinline__ double row_rotate(double v) {  // DPP row_ror:D
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + D, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + D, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sums(double a, double b, double c, double d) {
    swap32(a, b);  // a: a's low half, b's low half; b: their high halves
    a += b;
    swap32(c, d);
    c += d;
    swap16(a, c);
    a += c;
    a += row_rotate<8>(a);
    a += row_rotate<4>(a);
    a += row_rotate<2>(a);
    a += row_rotate<1>(a);
    return a;
}

// One tile: events (BRANCH) or site rows t TILE .. of the run.
template <int TYPE, bool BRANCH>
__device__ __forceinline__ void evaluate(const TsgStateArgs &a, int t) {
    constexpr int TILE = BRANCH ? TSG_BRANCH_TILE : TSG_SITE_TILE;
    constexpr int N = TILE / WAVE;
    using T = typename TileType<TYPE, BRANCH>::T;
    extern __shared__ double smem[];
    double *spos = smem;                                       // [TILE]
    double *sb = spos + TILE;                                  // [TILE] (branch)
    double *mean = sb + (BRANCH ? TILE : 0);                   // [TILE]
    int32_t *kind = reinterpret_cast<int32_t *>(mean + TILE);  // [TILE] (site)
    T *cols = reinterpret_cast<T *>(kind + (BRANCH ? 0 : TILE));  // [K x TILE]
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    constexpr int WAVES = EVAL_THREADS / WAVE;
    const int K = a.K, RW = a.RW;
    const int total = BRANCH ? a.nev : a.nrow;
    const int e0 = t * TILE;
    const int ne = max(0, min(TILE, total - e0));
    int other = 0;
    for (int e = tid; e < TILE; e += EVAL_THREADS) {
        int ref = 0;
        double pos = 0.0, b = 0.0;
        if (e < ne) {
            if constexpr (BRANCH) {
                ref = a.ev_state[e0 + e];
                pos = a.ev_pos[e0 + e];
                b = a.ev_b[e0 + e];
            } else {
                ref = a.row_ref[e0 + e];
                pos = a.row_pos[e0 + e];
            }
        }
        spos[e] = pos;
        if constexpr (BRANCH) sb[e] = b;
        if (BRANCH || ref >= 0) {
            if constexpr (!BRANCH) kind[e] = TSG_ROW_PAIR;
            const uint32_t *row = a.x + (int64_t) ref * RW;
            auto put = [&](int w, uint32_t v) {  // word w of the row
                if constexpr (TYPE == TSG_ROW_U16) {
                    if (2 * w < K) cols[(2 * w) * TILE + e] = (T) (v & 0xFFFFu);
                    if (2 * w + 1 < K) cols[(2 * w + 1) * TILE + e] = (T) (v >> 16);
                } else if constexpr (TYPE == TSG_ROW_I32) {
                    if (w < K) cols[w * TILE + e] = (T) v;
                } else {
                    if (w < 2 * K) {
                        reinterpret_cast<uint32_t *>(cols + (w / 2) * TILE + e)[w & 1] = v;
                    }
                }
            };
            if (RW >= 4) {
                for (int w = 0; w < RW; w += 4) {
                    const uint4 v = *reinterpret_cast<const uint4 *>(row + w);
                    put(w, v.x);
                    put(w + 1, v.y);
                    put(w + 2, v.z);
                    put(w + 3, v.w);
                }
            } else {
                for (int w = 0; w < RW; w++) put(w, row[w]);
            }
        } else if constexpr (!BRANCH) {
            const int l = -1 - ref;
            const int kd = a.list_kind[l];
            kind[e] = kd;
            other = 1;
            for (int k = 0; k < K; k++) {
                T v = 0;
                if (kd == TSG_ROW_ANCESTRAL) {
                    if constexpr (TYPE == TSG_ROW_F64) {
                        v = a.col_total_w[k];
                    } else {
                        v = a.col_total[k];
                    }
                }
                for (int i = a.list_off[l]; i < a.list_off[l + 1]; i++) {
                    const int ent = a.list_ent[i];
                    const uint32_t *row = a.x + (int64_t) (ent >> 1) * RW;
                    T xv;
                    if constexpr (TYPE == TSG_ROW_U16) {
                        xv = reinterpret_cast<const uint16_t *>(row)[k];
                    } else if constexpr (TYPE == TSG_ROW_I32) {
                        xv = (T) row[k];
                    } else {
                        xv = reinterpret_cast<const double *>(row)[k];
                    }
                    v = (ent & 1) ? v - xv : v + xv;
                }
                cols[k * TILE + e] = v;
            }
        }
    }
    const bool mixed = !BRANCH && __syncthreads_or(other) != 0;
    if constexpr (BRANCH) __syncthreads();

    const int q0 = BRANCH ? 0 : a.QB, q1 = BRANCH ? a.QB : a.Q;
    constexpr int PER = BRANCH ? 2 : 1;
    for (int q = q0; q < q1; q++) {
        const TsgStateQuery &Q = a.queries[q];
        const double *win = a.windows + Q.win_off;
        const int M = Q.M;
        const int w0 = a.tile_w[Q.tw + t], w1 = a.tile_w[Q.tw + t + 1];
        if (Q.rel_cn > 0) {
            if constexpr (TYPE != TSG_ROW_F64) {
                __syncthreads();
                for (int e = tid; e < TILE; e += EVAL_THREADS) {
                    double s = 0;
                    for (int c = Q.rel_c0; c < Q.rel_c0 + Q.rel_cn; c++) {
                        s += (double) cols[c * TILE + e] / (double) a.col_total[c];
                    }
                    mean[e] = s / (double) Q.rel_cn;
                }
                __syncthreads();
            }
        }
        const int nw = w1 - w0 + 1;
        // A wave adds up an output's whole tile for each of its windows (about
        // 400 cycles); a thread a (window, output) pair's events one by one
        // (about 150 cycles each, 256 threads): whichever is less.  (Measured
        // on 500 windows over 250 sites: 1634 -> 28 us.)
        if ((int64_t) nw * nw * ((M + 3) / 4) * 8 >
            (int64_t) TILE * 3 * (((int64_t) nw * M + EVAL_THREADS - 1) / EVAL_THREADS)) {
            for (int64_t i = tid; i < (int64_t) nw * M; i += EVAL_THREADS) {
                const int w = w0 + (int) (i / M), m = (int) (i % M);
                const int ea = w == w0 ? 0 : lower_bound(spos, ne, win[w]);
                const int eb = w == w1 ? ne : lower_bound(spos, ne, win[w + 1]);
                const double wr = win[w + 1];
                const TsgOut o = a.outs[Q.mbase + m];
                double L = 0, J = 0;
                for (int e = ea; e < eb; e++) {
                    const double v = value_of<TYPE, TILE, BRANCH>(a, o, cols, mean, kind, e);
                    if constexpr (BRANCH) {
                        const double b = sb[e];
                        L = fma(v, b * (wr - spos[e]), L);
                        J = fma(v, b, J);
                    } else {
                        L += v;
                    }
                }
                if (isfinite(o.inv)) {
                    L *= o.inv;
                    J *= o.inv;
                } else {
                    L = J = eb > ea ? NAN : 0.0;
                }
                double *dst = a.partial + Q.pbase + ((int64_t) (t + w) * M + m) * PER;
                dst[0] = L;
                if constexpr (BRANCH) dst[1] = J;
            }
            continue;
        }
        for (int w = w0; w <= w1; w++) {
            const int ea = w == w0 ? 0 : lower_bound(spos, ne, win[w]);
            const int eb = w == w1 ? ne : lower_bound(spos, ne, win[w + 1]);
            const double wr = win[w + 1];
            LaneEvents<N> ev;
#pragma unroll
            for (int r = 0; r < N; r++) {
                const int e = 2 * WAVE * (r / 2) + 2 * lane + (r & 1);
                const bool on = e >= ea && e < eb;
                if constexpr (BRANCH) {
                    const double b = on ? sb[e] : 0.0;
                    ev.wb[r] = b;
                    ev.wl[r] = b * (wr - spos[e]);
                } else {
                    ev.wl[r] = on ? 1.0 : 0.0;
                    ev.wb[r] = 0.0;
                }
            }
            // outputs wave, wave + 4, ...: two (branch: sums L and J) or four
            // (site) of them a round
            constexpr int ROUND = BRANCH ? 2 : 4;
            double *dst = a.partial + Q.pbase + (int64_t) (t + w) * M * PER;
            for (int m0 = wave; m0 < M; m0 += WAVES * ROUND) {
                double acc[4] = {0, 0, 0, 0};
                double unused = 0;
#pragma unroll
                for (int i = 0; i < ROUND; i++) {
                    const int m = m0 + i * WAVES;
                    if (m >= M) break;
                    add_output<TYPE, TILE, BRANCH>(a, a.outs[Q.mbase + m], cols, mean, kind, mixed,
                                                   lane, ev, acc[BRANCH ? 2 * i : i],
                                                   BRANCH ? acc[2 * i + 1] : unused);
                }
                const double v = wave_sums(acc[0], acc[1], acc[2], acc[3]);
                // lanes 0, 16, 32, 48 hold acc 0, 2, 1, 3
                const int row = lane / 16;
                const int at = row == 1 ? 2 : (row == 2 ? 1 : row);
                const int m = m0 + (BRANCH ? at / 2 : at) * WAVES;
                if (lane % 16 == 0 && m < M) {
                    // a zero denominator: NaN at every state (trees.c:2097-2220
                    // lets it through), none where there is no event
                    const double inv = a.outs[Q.mbase + m].inv;
                    const double r = isfinite(inv) ? v * inv : (eb > ea ? NAN : 0.0);
                    dst[BRANCH ? 2 * m + (at & 1) : m] = r;
                }
            }
        }
    }
}

// --- window sums ----------------------------------------------------------------

// first tile whose successor starts at x or later (or the last tile)
__device__ __forceinline__ int first_tile(const double *tpos, int tiles, double x) {
    int lo = 0, hi = tiles - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (tpos[mid + 1] >= x) {
            hi = mid;
        } else {
            lo = mid + 1;
        }
    }
    return lo;
}

__device__ __forceinline__ int pow2_at_least(int m, int most) {
    int p = 1;
    while (p < m && p < most) p <<= 1;
    return p;
}

// Workgroup (query, window): its segments' sums, tile lanes of outputs.
__device__ __forceinline__ void window_sums(const TsgStateArgs &a, int b) {
    __shared__ double red[2][256];
    int q = 0;
    while (q + 1 < a.Q && a.queries[q + 1].wbase <= b) q++;
    const TsgStateQuery &Q = a.queries[q];
    const int w = b - Q.wbase;
    const double *win = a.windows + Q.win_off;
    const double *tpos = Q.branch ? a.btile_pos : a.stile_pos;
    const int tiles = Q.branch ? a.btiles : a.stiles;
    const int M = Q.M, per = Q.branch ? 2 : 1;
    const int tlo = first_tile(tpos, tiles, win[w]);
    const double wr = win[w + 1];
    const int mb = pow2_at_least(M, 64), tl = 256 / mb;
    const int mi = threadIdx.x & (mb - 1), ti = threadIdx.x / mb;
    for (int m0 = 0; m0 < M; m0 += mb) {
        const int m = m0 + mi;
        double L = 0, J = 0;
        if (m < M) {
            for (int t = tlo + ti; t == tlo || (t < tiles && tpos[t] < wr); t += tl) {
                const double *src = a.partial + Q.pbase + ((int64_t) (t + w) * M + m) * per;
                L += src[0];
                if (per == 2) J += src[1];
            }
        }
        red[0][threadIdx.x] = L;
        red[1][threadIdx.x] = J;
        __syncthreads();
        for (int h = tl / 2; h > 0; h >>= 1) {
            if (ti < h) {
                red[0][threadIdx.x] += red[0][threadIdx.x + h * mb];
                red[1][threadIdx.x] += red[1][threadIdx.x + h * mb];
            }
            __syncthreads();
        }
        if (ti == 0 && m < M) {
            double *dst = a.wsum + Q.cbase + ((int64_t) w * M + m) * per;
            dst[0] = red[0][threadIdx.x];
            if (per == 2) dst[1] = red[1][threadIdx.x];
        }
        __syncthreads();
    }
}

// Workgroup (query, block of 8 outputs): runs of windows per thread, the
// running branch sum's change over each run scanned, then the results.  (8
// outputs, 128 runs: blocks of 64 outputs left one workgroup a query, 104 us
// for 2000 windows of 64 outputs.)
__device__ __forceinline__ void finish(const TsgStateArgs &a, int b) {
    __shared__ double scan[FINISH_THREADS];
    int q = 0;
    while (q + 1 < a.Q && a.queries[q + 1].bbase <= b) q++;
    const TsgStateQuery &Q = a.queries[q];
    const double *win = a.windows + Q.win_off;
    const double *tpos = Q.branch ? a.btile_pos : a.stile_pos;
    const int tiles = Q.branch ? a.btiles : a.stiles;
    const int M = Q.M, W = Q.W, per = Q.branch ? 2 : 1;
    const int mb = pow2_at_least(M, TSG_FINISH_OUTPUTS), S = FINISH_THREADS / mb;
    const int mi = threadIdx.x & (mb - 1), seg = threadIdx.x / mb;
    const int m = (b - Q.bbase) * TSG_FINISH_OUTPUTS + mi;
    const bool on = m < M;
    const int wa = (int) ((int64_t) W * seg / S), wb = (int) ((int64_t) W * (seg + 1) / S);
    int t = 0;
    // window w's two sums; with the segments, tile t moves along
    auto sums = [&](int w, double &L, double &J) {
        L = J = 0;
        if (Q.by_window) {
            const double *src = a.wsum + Q.cbase + ((int64_t) w * M + m) * per;
            L = src[0];
            if (per == 2) J = src[1];
            return;
        }
        const double wr = win[w + 1];
        for (;;) {
            const double *src = a.partial + Q.pbase + ((int64_t) (t + w) * M + m) * per;
            L += src[0];
            if (per == 2) J += src[1];
            if (t + 1 < tiles && tpos[t + 1] < wr) {
                t++;
            } else {
                break;
            }
        }
    };
    double R = 0;
    if (per == 2) {
        double acc = 0;
        if (on && wa < wb) {
            t = Q.by_window ? 0 : first_tile(tpos, tiles, win[wa]);
            for (int w = wa; w < wb; w++) {
                double L, J;
                sums(w, L, J);
                acc += J;
            }
        }
        scan[threadIdx.x] = acc;
        __syncthreads();
        // inclusive scan over the runs, log steps
        for (int h = 1; h < S; h <<= 1) {
            const double v = seg >= h ? scan[threadIdx.x - h * mb] : 0.0;
            __syncthreads();
            scan[threadIdx.x] += v;
            __syncthreads();
        }
        R = seg > 0 ? scan[threadIdx.x - mb] : 0.0;
    }
    if (!on || wa >= wb) return;
    t = Q.by_window ? 0 : first_tile(tpos, tiles, win[wa]);
    double *dst = (Q.to_out ? a.out : a.raw) + Q.obase;
    for (int w = wa; w < wb; w++) {
        double L, J;
        sums(w, L, J);
        const double span = win[w + 1] - win[w];
        double v = L + R * span;
        if (Q.flags & TSG_F_SPAN_NORMALISE) v /= span;
        dst[(int64_t) w * M + m] = v;
        R += J;
    }
}

}  // namespace

// --- one run ----------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_state_stage(const TsgStateArgs a) {
    stage(a, blockIdx.x);
}
template <int TYPE>
__global__ void __launch_bounds__(256) k_state_seed(const TsgStateArgs a) {
    seed<TYPE>(a, blockIdx.x);
}
template <bool F64>
__global__ void __launch_bounds__(256) k_state_count(const TsgStateArgs a, int s0, int s1, int nb) {
    const int b = xcd_block(blockIdx.x, nb);
    if (b < nb) count_rw<F64>(a, s0, s1, b);
}
template <int TYPE, bool BRANCH>
__global__ void __launch_bounds__(EVAL_THREADS) k_state_eval(const TsgStateArgs a) {
    const int tiles = BRANCH ? a.btiles : a.stiles;
    const int t = xcd_block(blockIdx.x, tiles);
    if (t < tiles) evaluate<TYPE, BRANCH>(a, t);
}
__global__ void __launch_bounds__(256) k_state_windows(const TsgStateArgs a) {
    window_sums(a, blockIdx.x);
}
__global__ void __launch_bounds__(FINISH_THREADS) k_state_finish(const TsgStateArgs a) {
    finish(a, blockIdx.x);
}

// --- many runs: run r has the blocks pre[r] .. pre[r + 1] of a phase ---------------

namespace {
__device__ __forceinline__ int run_at(const int32_t *pre, int nrun, int b) {
    int lo = 0, hi = nrun - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= b) {
            lo = mid;
        } else {
            hi = mid - 1;
        }
    }
    return lo;
}
}  // namespace

__global__ void __launch_bounds__(256) k_states_stage(const TsgStateArgs *args, const int32_t *pre,
                                                      int nrun) {
    const int r = run_at(pre, nrun, blockIdx.x);
    stage(args[r], blockIdx.x - pre[r]);
}
template <int TYPE>
__global__ void __launch_bounds__(256) k_states_seed(const TsgStateArgs *args, const int32_t *pre,
                                                     int nrun) {
    const int r = run_at(pre, nrun, blockIdx.x);
    seed<TYPE>(args[r], blockIdx.x - pre[r]);
}
// lev: each run's level bounds [2 x nrun] of this level
template <bool F64>
__global__ void __launch_bounds__(256) k_states_count(const TsgStateArgs *args, const int32_t *pre,
                                                      const int32_t *lev, int nrun, int nb) {
    const int b = xcd_block(blockIdx.x, nb);
    if (b >= nb) return;
    const int r = run_at(pre, nrun, b);
    count_rw<F64>(args[r], lev[2 * r], lev[2 * r + 1], b - pre[r]);
}
template <int TYPE, bool BRANCH>
__global__ void __launch_bounds__(EVAL_THREADS) k_states_eval(const TsgStateArgs *args,
                                                              const int32_t *pre, int nrun,
                                                              int nb) {
    const int b = xcd_block(blockIdx.x, nb);
    if (b >= nb) return;
    const int r = run_at(pre, nrun, b);
    evaluate<TYPE, BRANCH>(args[r], b - pre[r]);
}
__global__ void __launch_bounds__(256) k_states_windows(const TsgStateArgs *args,
                                                        const int32_t *pre, int nrun) {
    const int r = run_at(pre, nrun, blockIdx.x);
    window_sums(args[r], blockIdx.x - pre[r]);
}
__global__ void __launch_bounds__(FINISH_THREADS) k_states_finish(const TsgStateArgs *args,
                                                                  const int32_t *pre, int nrun) {
    const int r = run_at(pre, nrun, blockIdx.x);
    finish(args[r], blockIdx.x - pre[r]);
}

__global__ void __launch_bounds__(256) k_states_finals(const TsgStateArgs *args,
                                                       const int32_t *pre, int nrun) {
    const int r = run_at(pre, nrun, blockIdx.x);
    const TsgStateArgs &a = args[r];
    finals(reinterpret_cast<const TsgFinal *>(a.fin), a.nfin, a.raw, a.ipar, a.dpar, a.out,
           a.fincount, blockIdx.x - pre[r]);
}

// --- launchers ----------------------------------------------------------------------

size_t tsg_state_shmem(int K, int type, bool branch) {
    const size_t tile = branch ? TSG_BRANCH_TILE : TSG_SITE_TILE;
    const size_t el = type == TSG_ROW_F64 ? 8 : (type == TSG_ROW_U16 && branch) ? 2 : 4;
    return tile * (8 + 8 + (branch ? 8 : 4) + el * (size_t) K);
}

namespace {
template <typename F>
hipError_t allow(F *fn, size_t shmem) {
    if (shmem <= 65536) return hipSuccess;
    // (one value for every launch: threads launching at once never undo each
    // other's; the kernels hold under 1 KiB of static LDS besides)
    const int most = tsg_lds_max() - 1024;
    if ((int) shmem > most) return hipErrorInvalidValue;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(fn),
                               hipFuncAttributeMaxDynamicSharedMemorySize, most);
}

template <int TYPE, bool BRANCH>
hipError_t launch_eval(const TsgStateArgs &a, hipStream_t s) {
    const size_t sh = tsg_state_shmem(a.K, TYPE, BRANCH);
    hipError_t e = allow(&k_state_eval<TYPE, BRANCH>, sh);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_state_eval<TYPE, BRANCH>), dim3(xcd_grid(BRANCH ? a.btiles : a.stiles)),
                       dim3(EVAL_THREADS), sh, s, a);
    return hipGetLastError();
}

template <int TYPE>
hipError_t launch_run(const TsgStateLaunch &r, hipEvent_t begin, hipEvent_t mid, hipEvent_t end,
                      hipStream_t s) {
    const TsgStateArgs &a = r.a;
    constexpr bool F64 = TYPE == TSG_ROW_F64;
    hipLaunchKernelGGL(k_state_stage, dim3((unsigned) stage_blocks(a)), dim3(256), 0, s, a);
    hipError_t e;
    if (begin != nullptr && (e = hipEventRecord(begin, s)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_state_seed<TYPE>), dim3((unsigned) seed_blocks(a)), dim3(256), 0, s, a);
    for (int l = 1; l < r.levels; l++) {
        const int s0 = r.level0[l], s1 = r.level0[l + 1];
        const int64_t nb = count_blocks(a, s1 - s0);
        if (nb <= 0) continue;
        if (nb > INT32_MAX / 2) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_state_count<F64>), dim3(xcd_grid(nb)), dim3(256), 0, s, a, s0, s1,
                           (int) nb);
    }
    if (a.QB > 0 && (e = launch_eval<TYPE, true>(a, s)) != hipSuccess) return e;
    if (mid != nullptr && (e = hipEventRecord(mid, s)) != hipSuccess) return e;
    if (a.Q > a.QB && (e = launch_eval<TYPE, false>(a, s)) != hipSuccess) return e;
    if (end != nullptr && (e = hipEventRecord(end, s)) != hipSuccess) return e;
    if (r.wgroups > 0) {
        hipLaunchKernelGGL(k_state_windows, dim3((unsigned) r.wgroups), dim3(256), 0, s, a);
    }
    hipLaunchKernelGGL(k_state_finish, dim3((unsigned) r.fgroups), dim3(FINISH_THREADS), 0, s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (a.nfin > 0) {
        return tsg_launch_finals(a.fin, a.nfin, a.raw, a.ipar, a.dpar, a.out, a.fincount, s);
    }
    return hipSuccess;
}

// phases of a many-run launch: stage, seed, branch and site evaluation,
// windows, finish, composites, then one per level
enum { PH_STAGE, PH_SEED, PH_BRANCH, PH_SITE, PH_WINDOWS, PH_FINISH, PH_FINALS, PH_LEVEL };

int levels_of(const TsgStateLaunch *runs, int nrun) {
    int l = 1;
    for (int r = 0; r < nrun; r++) l = std::max(l, runs[r].levels);
    return l;
}
}  // namespace

hipError_t tsg_launch_states(const TsgStateLaunch &r, hipEvent_t begin, hipEvent_t mid,
                             hipEvent_t end, hipStream_t s) {
    switch (r.type) {
    case TSG_ROW_U16:
        return launch_run<TSG_ROW_U16>(r, begin, mid, end, s);
    case TSG_ROW_I32:
        return launch_run<TSG_ROW_I32>(r, begin, mid, end, s);
    default:
        return launch_run<TSG_ROW_F64>(r, begin, mid, end, s);
    }
}

int tsg_state_prefixes(const TsgStateLaunch *runs, int nrun, std::vector<int32_t> &pre) {
    const int levels = levels_of(runs, nrun);
    pre.clear();
    auto phase = [&](auto blocks) {
        int64_t at = 0;
        pre.push_back(0);
        for (int r = 0; r < nrun; r++) {
            at += blocks(runs[r]);
            if (at > INT32_MAX / 2) return false;
            pre.push_back((int32_t) at);
        }
        return true;
    };
    bool ok = phase([](const TsgStateLaunch &r) { return stage_blocks(r.a); }) &&
              phase([](const TsgStateLaunch &r) { return seed_blocks(r.a); }) &&
              phase([](const TsgStateLaunch &r) { return (int64_t) (r.a.QB > 0 ? r.a.btiles : 0); }) &&
              phase([](const TsgStateLaunch &r) {
                  return (int64_t) (r.a.Q > r.a.QB ? r.a.stiles : 0);
              }) &&
              phase([](const TsgStateLaunch &r) { return (int64_t) r.wgroups; }) &&
              phase([](const TsgStateLaunch &r) { return (int64_t) r.fgroups; }) &&
              phase([](const TsgStateLaunch &r) { return (r.a.fincount + 255) / 256; });
    for (int l = 1; ok && l < levels; l++) {
        ok = phase([l](const TsgStateLaunch &r) {
            return l < r.levels ? count_blocks(r.a, r.level0[l + 1] - r.level0[l]) : (int64_t) 0;
        });
    }
    if (!ok) return -1;
    for (int l = 1; l < levels; l++) {
        for (int r = 0; r < nrun; r++) {
            const bool in = l < runs[r].levels;
            pre.push_back(in ? runs[r].level0[l] : 0);
            pre.push_back(in ? runs[r].level0[l + 1] : 0);
        }
    }
    return 0;
}

namespace {
template <int TYPE>
hipError_t launch_multi(const TsgStateLaunch *runs, const TsgStateArgs *args, int nrun,
                        const std::vector<int32_t> &pre_h, const int32_t *pre, hipStream_t s) {
    constexpr bool F64 = TYPE == TSG_ROW_F64;
    const int levels = levels_of(runs, nrun);
    const int stride = nrun + 1;
    auto total = [&](int ph) { return pre_h[(size_t) ph * stride + nrun]; };
    auto at = [&](int ph) { return pre + (size_t) ph * stride; };
    hipLaunchKernelGGL(k_states_stage, dim3(total(PH_STAGE)), dim3(256), 0, s, args, at(PH_STAGE),
                       nrun);
    if (total(PH_SEED) > 0) {
        hipLaunchKernelGGL((k_states_seed<TYPE>), dim3(total(PH_SEED)), dim3(256), 0, s, args,
                           at(PH_SEED), nrun);
    }
    const int32_t *lev = at(PH_LEVEL + levels - 1);
    for (int l = 1; l < levels; l++) {
        const int nb = total(PH_LEVEL + l - 1);
        if (nb <= 0) continue;
        hipLaunchKernelGGL((k_states_count<F64>), dim3(xcd_grid(nb)), dim3(256), 0, s, args,
                           at(PH_LEVEL + l - 1), lev + (size_t) (l - 1) * 2 * nrun, nrun, nb);
    }
    size_t sb = 0, ss = 0;
    for (int r = 0; r < nrun; r++) {
        sb = std::max(sb, tsg_state_shmem(runs[r].a.K, TYPE, true));
        ss = std::max(ss, tsg_state_shmem(runs[r].a.K, TYPE, false));
    }
    hipError_t e;
    if (total(PH_BRANCH) > 0) {
        if ((e = allow(&k_states_eval<TYPE, true>, sb)) != hipSuccess) return e;
        hipLaunchKernelGGL((k_states_eval<TYPE, true>), dim3(xcd_grid(total(PH_BRANCH))),
                           dim3(EVAL_THREADS), sb, s, args, at(PH_BRANCH), nrun,
                           total(PH_BRANCH));
    }
    if (total(PH_SITE) > 0) {
        if ((e = allow(&k_states_eval<TYPE, false>, ss)) != hipSuccess) return e;
        hipLaunchKernelGGL((k_states_eval<TYPE, false>), dim3(xcd_grid(total(PH_SITE))),
                           dim3(EVAL_THREADS), ss, s, args, at(PH_SITE), nrun, total(PH_SITE));
    }
    if (total(PH_WINDOWS) > 0) {
        hipLaunchKernelGGL(k_states_windows, dim3(total(PH_WINDOWS)), dim3(256), 0, s, args,
                           at(PH_WINDOWS), nrun);
    }
    hipLaunchKernelGGL(k_states_finish, dim3(total(PH_FINISH)), dim3(FINISH_THREADS), 0, s, args,
                       at(PH_FINISH), nrun);
    if (total(PH_FINALS) > 0) {
        hipLaunchKernelGGL(k_states_finals, dim3(total(PH_FINALS)), dim3(256), 0, s, args,
                           at(PH_FINALS), nrun);
    }
    return hipGetLastError();
}
}  // namespace

hipError_t tsg_launch_states_multi(const TsgStateLaunch *runs, const TsgStateArgs *args, int nrun,
                                   const std::vector<int32_t> &pre_h, const int32_t *pre,
                                   hipStream_t s) {
    switch (runs[0].type) {
    case TSG_ROW_U16:
        return launch_multi<TSG_ROW_U16>(runs, args, nrun, pre_h, pre, s);
    case TSG_ROW_I32:
        return launch_multi<TSG_ROW_I32>(runs, args, nrun, pre_h, pre, s);
    default:
        return launch_multi<TSG_ROW_F64>(runs, args, nrun, pre_h, pre, s);
    }
}
