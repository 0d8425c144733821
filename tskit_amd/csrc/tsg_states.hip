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
#define SPECTRUM_SLOTS 1024
// windows whose first events a tile keeps at a time
#define EDGES 256

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
    const double *win = a.windows + Q.win_off;
    if (t <= tiles) {
        a.tile_w[j] = t == 0 ? 0 : t >= tiles ? Q.W - 1 : window_of(win, Q.W, tpos[t]);
    } else {
        const int w = t - (tiles + 1);
        a.tile_w[j] = w >= Q.W ? tiles - 1 : first_tile(tpos, tiles, win[w]);
    }
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

// States order[s0 .. s1 - 1] of a level, V words a thread.  16-bit counts are added
// two to a word: no count exceeds its column's total, so none carries over.
template <int V, bool F64>
__device__ __forceinline__ void count(const TsgStateArgs &a, int s0, int s1, int64_t b) {
    const int parts = a.RW / V;
    const int64_t i = b * 256 + threadIdx.x;
    int64_t s = s0 + i / parts;
    const int p = (int) (i % parts) * V;
    if (s >= s1) return;
    if (a.order != nullptr) s = a.order[s];
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

// What a tile holds a column as.  A site row's counts are sums of additions
// and subtractions, so site tiles of counts hold 32 bits whatever the rows do.
template <int TYPE, bool BRANCH, bool WIDE>
struct TileType {
    using T = double;
};
template <>
struct TileType<TSG_ROW_U16, true, true> {
    using T = uint16_t;
};
template <>
struct TileType<TSG_ROW_U16, false, true> {
    using T = int32_t;
};
template <bool BRANCH>
struct TileType<TSG_ROW_I32, BRANCH, true> {
    using T = int32_t;
};

// Elements from one column of a tile to the next: a few more than its
// events, so that threads reading one event of different columns read
// different banks (without: 20 conflict cycles per LDS instruction on 64
// columns), and aligned for the paired loads.
template <typename T>
constexpr int stride_of(int tile) {
    return tile + 2;
}

// A record at an address that is the same for the whole wave, written by no
// kernel at the same time (k_state_stage, before this kernel, wrote it: the
// scalar caches are clean at a kernel's start): scalar loads.
template <typename R>
__device__ __forceinline__ R uniform(const R *p) {
    typedef const __attribute__((address_space(4))) int32_t *Const;
    static_assert(sizeof(R) % 4 == 0, "whole words");
    Const q = (Const) (uintptr_t) p;
    int32_t w[sizeof(R) / 4];
#pragma unroll
    for (size_t i = 0; i < sizeof(R) / 4; i++) w[i] = q[i];
    R r;
    __builtin_memcpy(&r, w, sizeof(R));
    return r;
}

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

// Summary numerators at the counts x[0..3] (columns c[0..3]) of sets of
// n[0..3] samples: one(x) polarised; both(x) = one(x) + one(n - x), an event
// or a pair row of an unpolarised output; lone(x): a single allele of one.
// Where one(x) = one(n - x), both(x) is one(x) and the output's scale has
// the factor 2.
struct Nums {
    double n[4];
};
struct Diversity {
    static constexpr int S = 1;
    Nums p;
    __device__ double one(const double *x) const { return x[0] * (p.n[0] - x[0]); }
    __device__ double both(const double *x) const { return one(x); }
    __device__ double lone(const double *x) const { return 0.5 * one(x); }
};
struct Segregating {
    static constexpr int S = 1;
    Nums p;
    __device__ double one(const double *x) const { return x[0] > 0 ? p.n[0] - x[0] : 0.0; }
    // n for 0 < x < n
    __device__ double both(const double *x) const {
        return (x[0] > 0 ? p.n[0] - x[0] : 0.0) + (x[0] < p.n[0] ? x[0] : 0.0);
    }
    __device__ double lone(const double *x) const { return one(x); }
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
    __device__ double lone(const double *x) const { return one(x); }
};
struct Divergence {
    static constexpr int S = 2;
    Nums p;
    __device__ double one(const double *x) const { return x[0] * (p.n[1] - x[1]); }
    __device__ double both(const double *x) const {
        return fma(x[0], p.n[1] - x[1], (p.n[0] - x[0]) * x[1]);
    }
    __device__ double lone(const double *x) const { return one(x); }
};
struct Product {  // non-centred relatedness, also of weights
    static constexpr int S = 2;
    Nums p;
    __device__ double one(const double *x) const { return x[0] * x[1]; }
    __device__ double both(const double *x) const {
        return fma(x[0], x[1], (p.n[0] - x[0]) * (p.n[1] - x[1]));
    }
    __device__ double lone(const double *x) const { return one(x); }
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
    __device__ double lone(const double *x) const { return one(x); }
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
    __device__ double lone(const double *x) const { return one(x); }
};
// centred relatedness: slot 2 is the mean over the query's columns
struct Relatedness {
    static constexpr int S = 3;
    double ri, rj;  // 1 / set size
    __device__ double one(const double *x) const {
        return (x[0] * ri - x[2]) * (x[1] * rj - x[2]);
    }
    __device__ double both(const double *x) const { return one(x); }
    __device__ double lone(const double *x) const { return 0.5 * one(x); }
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
    __device__ double lone(const double *x) const { return one(x); }
};
struct TraitCorrelation : Complement<TraitCorrelation, 2> {  // slots: trait, frequency
    __device__ double f(const double *x) const {
        const double q = x[1];
        return (q > 0.0 && q < 1.0) ? (x[0] * x[0]) / (q * (1 - q)) : 0.0;
    }
};
struct RelatednessWeighted : Complement<RelatednessWeighted, 3> {  // slots: i, j, frequency
    double ca, cb;
    __device__ double f(const double *x) const {
        return (x[0] - ca * x[2]) * (x[1] - cb * x[2]);
    }
};

// A tile's events as one lane of a wave sees them: events 128 j + 2 lane and
// the next, j < N / 2, with their weights in the window's two sums (zero for
// the others' events) and, bit by bit, which are the window's.
template <int N>
struct LaneEvents {
    double wl[N], wb[N];
    uint32_t on;
};

// The tile of one workgroup (LDS).
template <typename T>
struct Tile {
    const double *mean;   // centred relatedness: the query's mean
    const int32_t *kind;  // site rows
    bool mixed;           // some row is not a pair
    const T *cols;        // [K x TILE]
};

// how a row's value follows from the summary
#define VALUE_ONE 0    // polarised, every row a pair or derived
#define VALUE_BOTH 1   // unpolarised, every event or pair row
#define VALUE_MIXED 2  // site tiles with other rows

// Summaries of counts are finite, so a weight of zero leaves an event out; of
// weights (REAL) they may be infinite or NaN, and 0 x NaN would reach every
// window of the tile.
template <typename T, int TILE, bool BRANCH, bool REAL, int VALUE, typename F, typename C2>
__device__ __forceinline__ void add_up(const F &f, const T *c0, const T *c1, const C2 *c2,
                                       const T *c3, const int32_t *kind, bool polarised, int lane,
                                       const LaneEvents<TILE / WAVE> &ev, double &L, double &J) {
    constexpr int N = TILE / WAVE;
#pragma unroll
    for (int j = 0; j < N / 2; j++) {
        double x0[4], x1[4];
        const int i = WAVE * j + lane;
        double2 v = load2<T>(c0, i);
        x0[0] = v.x, x1[0] = v.y;
        if constexpr (F::S > 1) v = load2<T>(c1, i), x0[1] = v.x, x1[1] = v.y;
        if constexpr (F::S > 2) v = load2<C2>(c2, i), x0[2] = v.x, x1[2] = v.y;
        if constexpr (F::S > 3) v = load2<T>(c3, i), x0[3] = v.x, x1[3] = v.y;
        double v0, v1;
        if constexpr (VALUE == VALUE_ONE) {
            v0 = f.one(x0);
            v1 = f.one(x1);
        } else if constexpr (VALUE == VALUE_BOTH) {
            v0 = f.both(x0);
            v1 = f.both(x1);
        } else {
            const int2 k = reinterpret_cast<const int2 *>(kind)[i];
            if (polarised) {
                v0 = k.x == TSG_ROW_ANCESTRAL ? 0.0 : f.one(x0);
                v1 = k.y == TSG_ROW_ANCESTRAL ? 0.0 : f.one(x1);
            } else {
                v0 = k.x == TSG_ROW_PAIR ? f.both(x0) : f.lone(x0);
                v1 = k.y == TSG_ROW_PAIR ? f.both(x1) : f.lone(x1);
            }
        }
        if constexpr (REAL) {
            v0 = (ev.on >> (2 * j)) & 1 ? v0 : 0.0;
            v1 = (ev.on >> (2 * j + 1)) & 1 ? v1 : 0.0;
        }
        L = fma(v0, ev.wl[2 * j], L);
        L = fma(v1, ev.wl[2 * j + 1], L);
        if constexpr (BRANCH) {
            J = fma(v0, ev.wb[2 * j], J);
            J = fma(v1, ev.wb[2 * j + 1], J);
        }
    }
}

// The trait regression's summary (trees.c:4108-4152) of event e, or of its
// complement: covariates cbase .. with their row of V, the sample count in
// column c[3].
template <int TILE>
__device__ __forceinline__ double regression(const TsgStateArgs &a, const TsgStateOut &o,
                                             const double *cols, int e, bool comp) {
    const double *v = a.opar + o.par;
    const double *tot = a.col_total_w;
    auto X = [&](int c) {
        const double x = cols[c * stride_of<double>(TILE) + e];
        return comp ? tot[c] - x : x;
    };
    const double m = X(o.c[3]);
    if (!(m > 0.0 && m < (double) o.samples)) return 0.0;
    double r = X(o.c[0]), denom = m;
    for (int c = 0; c < o.ccount; c++) {
        const double z = X(o.cbase + c);
        r -= z * v[c];
        denom -= z * z;
    }
    return denom < 1e-8 ? 0.0 : (r * r) / (2 * denom * denom);
}

// Calls use(make) for the summary `stat`, make(o) being the summary of output
// o of that kind.
template <int TYPE, typename U>
__device__ __forceinline__ void with_summary(int stat, U use) {
#define SUMMARY(ID, F)                                                  \
    case ID:                                                            \
        use([](const TsgStateOut &o) {                                  \
            F f;                                                        \
            f.p = Nums{{o.n[0], o.n[1], o.n[2], o.n[3]}};               \
            return f;                                                   \
        });                                                             \
        break;
    if constexpr (TYPE == TSG_ROW_F64) {
        switch (stat) {
            SUMMARY(TSG_STAT_TRAIT_COVARIANCE, TraitCovariance)
            SUMMARY(TSG_STAT_TRAIT_CORRELATION, TraitCorrelation)
            SUMMARY(TSG_STAT_RELATEDNESS_WEIGHTED_NONCENTRED, Product)
        case TSG_STAT_RELATEDNESS_WEIGHTED:
            use([](const TsgStateOut &o) {
                RelatednessWeighted f;
                f.p = Nums{{o.n[0], o.n[1], o.n[2], o.n[3]}};
                f.ca = o.coef[0];
                f.cb = o.coef[1];
                return f;
            });
            break;
        default:
            break;
        }
    } else {
        switch (stat) {
            SUMMARY(TSG_STAT_DIVERSITY, Diversity)
            SUMMARY(TSG_STAT_SEGREGATING_SITES, Segregating)
            SUMMARY(TSG_STAT_Y1, Y1)
            SUMMARY(TSG_STAT_DIVERGENCE, Divergence)
            SUMMARY(TSG_STAT_RELATEDNESS_NONCENTRED, Product)
            SUMMARY(TSG_STAT_Y2, Y2)
            SUMMARY(TSG_STAT_F2, F2)
            SUMMARY(TSG_STAT_Y3, Y3)
            SUMMARY(TSG_STAT_F3, F3)
            SUMMARY(TSG_STAT_F4, F4)
        case TSG_STAT_RELATEDNESS:
            use([](const TsgStateOut &o) { return Relatedness{o.coef[0], o.coef[1]}; });
            break;
        default:
            break;
        }
    }
#undef SUMMARY
}
// its slot 2 is the query's mean, not a column
template <typename F>
constexpr bool reads_mean = std::is_same<F, Relatedness>::value;

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

// A round's sums of a wave into the segment: two outputs (branch: sums L and
// J) or four (site); lanes 0, 16, 32, 48 hold acc 0, 2, 1, 3.
template <bool BRANCH, int WAVES>
__device__ __forceinline__ void store_round(const double (&acc)[4], const double (&scale)[4],
                                            int m0, int count, int lane, bool any, double *dst) {
    constexpr int PER = BRANCH ? 2 : 1;
    const double v = wave_sums(acc[0], acc[1], acc[2], acc[3]);
    const int row = lane / 16;
    const int at = row == 1 ? 2 : (row == 2 ? 1 : row);
    const int i = BRANCH ? at / 2 : at;
    if (lane % 16 == 0 && m0 + i * WAVES < count) {
        const double sc = i == 0 ? scale[0] : i == 1 ? scale[1] : i == 2 ? scale[2] : scale[3];
        // (a zero denominator: 0 x inf is the reference's NaN at every state,
        // but a window without events has 0)
        dst[(m0 + i * WAVES) * PER + (BRANCH ? (at & 1) : 0)] = any ? v * sc : 0.0;
    }
}

// `count` outputs of one summary over the window's events: this wave's are
// wave, wave + 4, ...; the next round's records are read while a round is
// summed.
template <typename T, int TILE, bool BRANCH, bool REAL, int VALUE, typename Make>
__device__ __forceinline__ void add_run(Make make, const TsgStateOut *outs, int count,
                                        const Tile<T> &tile, bool polarised, int wave, int lane,
                                        const LaneEvents<TILE / WAVE> &ev, bool any, double *dst) {
    constexpr int WAVES = EVAL_THREADS / WAVE, ROUND = BRANCH ? 2 : 4, STRIDE = stride_of<T>(TILE);
    if (wave >= count) return;
    TsgStateOut o[ROUND];
#pragma unroll
    for (int i = 0; i < ROUND; i++) o[i] = uniform(outs + min(wave + i * WAVES, count - 1));
    for (int m0 = wave; m0 < count; m0 += WAVES * ROUND) {
        double acc[4] = {0, 0, 0, 0}, scale[4] = {0, 0, 0, 0}, unused = 0;
#pragma unroll
        for (int i = 0; i < ROUND; i++) {
            const auto f = make(o[i]);
            using F = typename std::decay<decltype(f)>::type;
            scale[i] = o[i].scale;
            const T *c0 = tile.cols + o[i].c[0] * STRIDE, *c1 = tile.cols + o[i].c[1] * STRIDE;
            const T *c2 = tile.cols + o[i].c[2] * STRIDE, *c3 = tile.cols + o[i].c[3] * STRIDE;
            o[i] = uniform(outs + min(m0 + (i + ROUND) * WAVES, count - 1));
            if (i > 0 && m0 + i * WAVES >= count) continue;
            double &L = acc[BRANCH ? 2 * i : i], &J = BRANCH ? acc[(2 * i + 1) & 3] : unused;
            if constexpr (reads_mean<F>) {
                add_up<T, TILE, BRANCH, REAL, VALUE>(f, c0, c1, tile.mean, c3, tile.kind, polarised,
                                                     lane, ev, L, J);
            } else {
                add_up<T, TILE, BRANCH, REAL, VALUE>(f, c0, c1, c2, c3, tile.kind, polarised, lane,
                                                     ev, L, J);
            }
        }
        store_round<BRANCH, WAVES>(acc, scale, m0, count, lane, any, dst);
    }
}

template <int TILE, bool BRANCH>
__device__ __forceinline__ void add_regressions(const TsgStateArgs &a, const TsgStateOut *outs,
                                                int count, const Tile<double> &tile, int wave,
                                                int lane, const LaneEvents<TILE / WAVE> &ev,
                                                bool any, double *dst) {
    constexpr int WAVES = EVAL_THREADS / WAVE, N = TILE / WAVE;
    for (int m = wave; m < count; m += WAVES) {
        const TsgStateOut o = uniform(outs + m);
        const bool pol = o.polarised != 0;
        double L = 0, J = 0;
#pragma unroll
        for (int r = 0; r < N; r++) {
            const int e = 2 * WAVE * (r / 2) + 2 * lane + (r & 1);
            const int k = (!BRANCH && tile.mixed) ? tile.kind[e] : TSG_ROW_PAIR;
            double f = (pol && k == TSG_ROW_ANCESTRAL)
                           ? 0.0
                           : regression<TILE>(a, o, tile.cols, e, false);
            if (!pol && k == TSG_ROW_PAIR) f = f + regression<TILE>(a, o, tile.cols, e, true);
            f = (ev.on >> r) & 1 ? f : 0.0;
            L = fma(f, ev.wl[r], L);
            if constexpr (BRANCH) J = fma(f, ev.wb[r], J);
        }
        const double acc[4] = {L, J, 0, 0}, scale[4] = {o.scale, 0, 0, 0};
        store_round<BRANCH, WAVES>(acc, scale, m, m + 1, lane, any, dst);
    }
}

// `count` outputs of one summary over cn windows of a tile: a thread adds up
// the events of a (window, output) pair one by one.  Window i has the events
// edge[i] .. edge[i + 1] and ends at wend[i]; its sums go to dst, windows M
// outputs apart.
template <int TYPE, int TILE, bool BRANCH, typename T>
__device__ __forceinline__ void add_items(const TsgStateArgs &a, const TsgStateOut *outs,
                                          const TsgStateOut &first, int count, const Tile<T> &tile,
                                          const double *spos, const double *sb,
                                          const int32_t *edge, const double *wend, int cn,
                                          double *dst, int M) {
    constexpr int STRIDE = stride_of<T>(TILE), PER = BRANCH ? 2 : 1;
    const bool pol = first.polarised != 0;
    auto items = [&](auto prepare) {
        // a thread keeps its output while there is room for them all
        for (int mc = 0; mc < count; mc += EVAL_THREADS) {
            const int mn = min(EVAL_THREADS, count - mc), groups = EVAL_THREADS / mn;
            const int m = mc + (int) threadIdx.x % mn;
            if ((int) threadIdx.x >= groups * mn) continue;
            const TsgStateOut o = outs[m];
            const auto value = prepare(o);
            for (int i = (int) threadIdx.x / mn; i < cn; i += groups) {
                const int ea = edge[i], eb = edge[i + 1];
                const double wr = wend[i];
                double L = 0, J = 0;
                for (int e = ea; e < eb; e++) {
                    const double v = value(e);
                    if constexpr (BRANCH) {
                        const double b = sb[e];
                        L = fma(v, b * (wr - spos[e]), L);
                        J = fma(v, b, J);
                    } else {
                        L += v;
                    }
                }
                // (a zero denominator: 0 x inf is the reference's NaN at every
                // state, but a window without events has 0)
                double *to = dst + ((int64_t) i * M + m) * PER;
                to[0] = eb > ea ? L * o.scale : 0.0;
                if constexpr (BRANCH) to[1] = eb > ea ? J * o.scale : 0.0;
            }
        }
    };
    if constexpr (TYPE == TSG_ROW_F64) {
        if (first.stat == TSG_STAT_TRAIT_LINEAR_MODEL) {
            items([&](const TsgStateOut &o) {
                return [&](int e) {
                    const int k = (!BRANCH && tile.mixed) ? tile.kind[e] : TSG_ROW_PAIR;
                    if (pol && k == TSG_ROW_ANCESTRAL) return 0.0;
                    double v = regression<TILE>(a, o, tile.cols, e, false);
                    if (!pol && k == TSG_ROW_PAIR) v = v + regression<TILE>(a, o, tile.cols, e, true);
                    return v;
                };
            });
            return;
        }
    }
    with_summary<TYPE>(first.stat, [&](auto make) {
        items([&](const TsgStateOut &o) {
            const auto f = make(o);
            using F = typename std::decay<decltype(f)>::type;
            const T *c0 = tile.cols + o.c[0] * STRIDE, *c1 = tile.cols + o.c[1] * STRIDE;
            const T *c2 = tile.cols + o.c[2] * STRIDE, *c3 = tile.cols + o.c[3] * STRIDE;
            return [=, &tile](int e) {
                double x[4] = {(double) c0[e], 0.0, 0.0, 0.0};
                if constexpr (F::S > 1) x[1] = (double) c1[e];
                if constexpr (reads_mean<F>) {
                    x[2] = tile.mean[e];
                } else if constexpr (F::S > 2) {
                    x[2] = (double) c2[e];
                }
                if constexpr (F::S > 3) x[3] = (double) c3[e];
                const int k = (!BRANCH && tile.mixed) ? tile.kind[e] : TSG_ROW_PAIR;
                if (pol) return k == TSG_ROW_ANCESTRAL ? 0.0 : f.one(x);
                return k == TSG_ROW_PAIR ? f.both(x) : f.lone(x);
            };
        });
    });
}

// One tile: events (BRANCH) or site rows t TILE .. of the run.  WIDE: more
// columns than an FP64 tile takes.
template <int TYPE, bool BRANCH, bool WIDE>
__device__ __forceinline__ void evaluate(const TsgStateArgs &a, int t) {
    constexpr int TILE = BRANCH ? TSG_BRANCH_TILE : TSG_SITE_TILE;
    constexpr int N = TILE / WAVE;
    constexpr bool REAL = TYPE == TSG_ROW_F64;
    using T = typename TileType<TYPE, BRANCH, WIDE>::T;
    constexpr int STRIDE = stride_of<T>(TILE);
    extern __shared__ double smem[];
    double *spos = smem;                                       // [TILE]
    double *sb = spos + TILE;                                  // [TILE] (branch)
    double *mean = sb + (BRANCH ? TILE : 0);                   // [TILE]
    int32_t *kind = reinterpret_cast<int32_t *>(mean + TILE);  // [TILE] (site)
    double *wend = reinterpret_cast<double *>(kind + (BRANCH ? 0 : TILE));  // [EDGES]
    int32_t *edge = reinterpret_cast<int32_t *>(wend + EDGES);              // [EDGES + 4]
    T *cols = reinterpret_cast<T *>(edge + EDGES + 4);                      // [K x STRIDE]
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
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
                    if (2 * w < K) cols[(2 * w) * STRIDE + e] = (T) (v & 0xFFFFu);
                    if (2 * w + 1 < K) cols[(2 * w + 1) * STRIDE + e] = (T) (v >> 16);
                } else if constexpr (TYPE == TSG_ROW_I32) {
                    if (w < K) cols[w * STRIDE + e] = (T) (int32_t) v;
                } else {
                    if (w < 2 * K) {
                        reinterpret_cast<uint32_t *>(cols + (w / 2) * STRIDE + e)[w & 1] = v;
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
                        v = (T) a.col_total[k];
                    }
                }
                for (int i = a.list_off[l]; i < a.list_off[l + 1]; i++) {
                    const int ent = a.list_ent[i];
                    const uint32_t *row = a.x + (int64_t) (ent >> 1) * RW;
                    T xv;
                    if constexpr (TYPE == TSG_ROW_U16) {
                        xv = (T) reinterpret_cast<const uint16_t *>(row)[k];
                    } else if constexpr (TYPE == TSG_ROW_I32) {
                        xv = (T) (int32_t) row[k];
                    } else {
                        xv = reinterpret_cast<const double *>(row)[k];
                    }
                    v = (ent & 1) ? v - xv : v + xv;
                }
                cols[k * STRIDE + e] = v;
            }
        }
    }
    const bool mixed = !BRANCH && __syncthreads_or(other) != 0;
    if constexpr (BRANCH) __syncthreads();
    const Tile<T> tile{mean, kind, mixed, cols};

    const int q0 = BRANCH ? 0 : a.QB, q1 = BRANCH ? a.QB : a.Q;
    constexpr int PER = BRANCH ? 2 : 1;
    for (int q = q0; q < q1; q++) {
        const TsgStateQuery Q = uniform(a.queries + q);
        const double *win = a.windows + Q.win_off;
        const int M = Q.M;
        const int w0 = a.tile_w[Q.tw + t], w1 = a.tile_w[Q.tw + t + 1];
        if (Q.rel_cn > 0) {
            if constexpr (TYPE != TSG_ROW_F64) {
                __syncthreads();
                for (int e = tid; e < TILE; e += EVAL_THREADS) {
                    double s = 0;
                    for (int c = Q.rel_c0; c < Q.rel_c0 + Q.rel_cn; c++) {
                        s += (double) cols[c * STRIDE + e] / (double) a.col_total[c];
                    }
                    mean[e] = s / (double) Q.rel_cn;
                }
                __syncthreads();
            }
        }
        const int nw = w1 - w0 + 1;
        // A wave adds up an output's whole tile for each of its windows (about
        // 400 cycles); a thread a (window, output) pair's events one by one
        // (about 50 cycles an event, 150 a row, 256 threads): whichever is
        // less.  (Branch tiles of 5 windows, 64 outputs: 107 us, 40 in pairs;
        // of 20 windows, 31 outputs: 91 in pairs; site tiles of 2 or 3
        // windows, 60 outputs: 40 us, 100 in pairs.)
        if ((int64_t) nw * nw * ((M + 3) / 4) * 8 >
            (int64_t) TILE * (BRANCH ? 1 : 3) *
                (((int64_t) nw * M + EVAL_THREADS - 1) / EVAL_THREADS)) {
            for (int c0 = w0; c0 <= w1; c0 += EDGES) {
                const int cn = min(EDGES, w1 - c0 + 1);
                // the windows' first events, found once for all outputs
                __syncthreads();
                for (int i = tid; i <= cn; i += EVAL_THREADS) {
                    const int w = c0 + i;
                    edge[i] = w == w0 ? 0 : w > w1 ? ne : lower_bound(spos, ne, win[w]);
                    if (i < cn) wend[i] = win[w + 1];
                }
                __syncthreads();
                for (int m = 0; m < M;) {
                    const TsgStateOut first = uniform(a.outs + Q.mbase + m);
                    const int count = min(first.run, M - m);
                    double *dst = a.partial + Q.pbase + ((int64_t) (t + c0) * M + m) * PER;
                    add_items<TYPE, TILE, BRANCH>(a, a.outs + Q.mbase + m, first, count, tile, spos,
                                                  sb, edge, wend, cn, dst, M);
                    m += count;
                }
            }
            continue;
        }
        for (int w = w0; w <= w1; w++) {
            const int ea = w == w0 ? 0 : lower_bound(spos, ne, win[w]);
            const int eb = w == w1 ? ne : lower_bound(spos, ne, win[w + 1]);
            const double wr = win[w + 1];
            LaneEvents<N> ev;
            ev.on = 0;
#pragma unroll
            for (int r = 0; r < N; r++) {
                const int e = 2 * WAVE * (r / 2) + 2 * lane + (r & 1);
                const bool on = e >= ea && e < eb;
                if constexpr (REAL) ev.on |= (uint32_t) on << r;
                if constexpr (BRANCH) {
                    const double b = on ? sb[e] : 0.0;
                    ev.wb[r] = b;
                    ev.wl[r] = b * (wr - spos[e]);
                } else {
                    ev.wl[r] = on ? 1.0 : 0.0;
                    ev.wb[r] = 0.0;
                }
            }
            double *dst = a.partial + Q.pbase + (int64_t) (t + w) * M * PER;
            for (int m = 0; m < M;) {
                // a run of outputs of one summary, polarised or not
                const TsgStateOut first = uniform(a.outs + Q.mbase + m);
                const TsgStateOut *outs = a.outs + Q.mbase + m;
                const int count = min(first.run, M - m);
                if constexpr (TYPE == TSG_ROW_F64) {
                    if (first.stat == TSG_STAT_TRAIT_LINEAR_MODEL) {
                        add_regressions<TILE, BRANCH>(a, outs, count, tile, wave, lane, ev, eb > ea,
                                                      dst + m * PER);
                    }
                }
                with_summary<TYPE>(first.stat, [&](auto make) {
                    if (!BRANCH && mixed) {
                        add_run<T, TILE, BRANCH, REAL, VALUE_MIXED>(
                            make, outs, count, tile, first.polarised != 0, wave, lane, ev, eb > ea,
                            dst + m * PER);
                    } else if (first.polarised) {
                        add_run<T, TILE, BRANCH, REAL, VALUE_ONE>(make, outs, count, tile, true,
                                                                  wave, lane, ev, eb > ea,
                                                                  dst + m * PER);
                    } else {
                        add_run<T, TILE, BRANCH, REAL, VALUE_BOTH>(make, outs, count, tile, false,
                                                                   wave, lane, ev, eb > ea,
                                                                   dst + m * PER);
                    }
                });
                m += count;
            }
        }
    }
}

// --- window sums ----------------------------------------------------------------

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
    const int tiles = Q.branch ? a.btiles : a.stiles;
    const int M = Q.M, per = Q.branch ? 2 : 1;
    const int32_t *first = a.tile_w + Q.tw + tiles + 1;
    const int tlo = first[w], thi = first[w + 1];
    const int mb = pow2_at_least(M, 64), tl = 256 / mb;
    const int mi = threadIdx.x & (mb - 1), ti = threadIdx.x / mb;
    for (int m0 = 0; m0 < M; m0 += mb) {
        const int m = m0 + mi;
        double L = 0, J = 0;
        if (m < M) {
            for (int t = tlo + ti; t <= thi; t += tl) {
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
    __shared__ double scan[TSG_FINISH_THREADS];
    int q = 0;
    while (q + 1 < a.Q && a.queries[q + 1].bbase <= b) q++;
    const TsgStateQuery &Q = a.queries[q];
    const double *win = a.windows + Q.win_off;
    const int tiles = Q.branch ? a.btiles : a.stiles;
    const int M = Q.M, W = Q.W, per = Q.branch ? 2 : 1;
    const int mb = pow2_at_least(M, TSG_FINISH_OUTPUTS), S = TSG_FINISH_THREADS / mb;
    const int mi = threadIdx.x & (mb - 1), seg = threadIdx.x / mb;
    const int m = (b - Q.bbase) * TSG_FINISH_OUTPUTS + mi;
    const bool on = m < M;
    const int wa = (int) ((int64_t) W * seg / S), wb = (int) ((int64_t) W * (seg + 1) / S);
    const int32_t *first = a.tile_w + Q.tw + tiles + 1;
    // window w's two sums
    auto sums = [&](int w, double &L, double &J) {
        L = J = 0;
        if (Q.by_window) {
            const double *src = a.wsum + Q.cbase + ((int64_t) w * M + m) * per;
            L = src[0];
            if (per == 2) J = src[1];
            return;
        }
        const int thi = first[w + 1];
        for (int t = first[w]; t <= thi; t++) {
            const double *src = a.partial + Q.pbase + ((int64_t) (t + w) * M + m) * per;
            L += src[0];
            if (per == 2) J += src[1];
        }
    };
    // a run's first windows stay in registers between the two passes
    constexpr int KEEP = 8;
    double Lk[KEEP], Jk[KEEP];
    const int n = on ? wb - wa : 0;
#pragma unroll
    for (int i = 0; i < KEEP; i++) {
        Lk[i] = Jk[i] = 0;
        if (i < n) sums(wa + i, Lk[i], Jk[i]);
    }
    double R = 0;
    if (per == 2) {
        double acc = 0;
#pragma unroll
        for (int i = 0; i < KEEP; i++) acc += Jk[i];
        for (int i = KEEP; i < n; i++) {
            double L, J;
            sums(wa + i, L, J);
            acc += J;
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
    double *dst = (Q.to_out ? a.out : a.raw) + Q.obase;
    auto put = [&](int w, double L, double J) {
        const double span = win[w + 1] - win[w];
        double v = L + R * span;
        if (Q.flags & TSG_F_SPAN_NORMALISE) v /= span;
        dst[(int64_t) w * M + m] = v;
        R += J;
    };
#pragma unroll
    for (int i = 0; i < KEEP; i++) {
        if (i < n) put(wa + i, Lk[i], Jk[i]);
    }
    for (int i = KEEP; i < n; i++) {
        double L, J;
        sums(wa + i, L, J);
        put(wa + i, L, J);
    }
}

}  // namespace

// --- node statistics --------------------------------------------------------------

// Column k of state s.
template <int TYPE>
__device__ __forceinline__ double row_value(const TsgStateArgs &a, int s, int k) {
    const uint32_t *row = a.x + (int64_t) s * a.RW;
    return TYPE == TSG_ROW_U16 ? (double) reinterpret_cast<const uint16_t *>(row)[k]
                               : (double) (int32_t) row[k];
}

// Output o's summary at state s, before the scale.
template <int TYPE>
__device__ __forceinline__ double state_value(const TsgStateArgs &a, const TsgStateOut &o,
                                              const TsgStateQuery &Q, int s) {
    double mean = 0;
    if (Q.rel_cn > 0) {
        for (int c = Q.rel_c0; c < Q.rel_c0 + Q.rel_cn; c++) {
            mean += row_value<TYPE>(a, s, c) / (double) a.col_total[c];
        }
        mean /= (double) Q.rel_cn;
    }
    double x[4] = {row_value<TYPE>(a, s, o.c[0]), row_value<TYPE>(a, s, o.c[1]), 0.0, 0.0};
    double v = 0.0;
    with_summary<TYPE>(o.stat, [&](auto make) {
        const auto f = make(o);
        using F = typename std::decay<decltype(f)>::type;
        if constexpr (reads_mean<F>) {
            x[2] = mean;
        } else {
            if constexpr (F::S > 2) x[2] = row_value<TYPE>(a, s, o.c[2]);
            if constexpr (F::S > 3) x[3] = row_value<TYPE>(a, s, o.c[3]);
        }
        v = o.polarised ? f.one(x) : f.both(x);
    });
    return v;
}

// Thread (run, output): a run of one node's states along the genome, each
// the summary times its span in every window it crosses, added to
// res[(window x N + node) x M + output] once per run and window (FP64 atomic
// adds: a node's runs meet there in any order).  A chunk sweep added at
// every event of a node's path: on 8000 samples, 8 sets, 347 us; this, 22 us.
template <int TYPE>
__global__ void __launch_bounds__(256) k_state_nodes(const TsgStateArgs a, const TsgNodeArgs g,
                                                     int64_t b0) {
    const int64_t i = (b0 + blockIdx.x) * 256 + threadIdx.x;
    const TsgStateQuery &Q = a.queries[0];
    const int M = Q.M, W = Q.W;
    const int64_t r = i / M;
    const int m = (int) (i % M);
    if (r >= g.runs) return;
    const TsgStateOut o = a.outs[m];
    const double *win = a.windows;
    const int node = g.run_node[r];
    const int p0 = g.run_piece0[r], p1 = g.run_piece0[r + 1];
    const bool last = r + 1 == g.runs || g.run_node[r + 1] != node;
    int w = W > 1 ? window_of(win, W, g.run_from[p0]) : 0;
    double acc = 0;
    auto add = [&]() {
        double *dst = g.res + ((int64_t) w * g.num_nodes + node) * M + m;
        atomicAdd(dst, acc * o.scale);
        acc = 0;
    };
    for (int p = p0; p < p1; p++) {
        double from = g.run_from[p];
        const double to = (p + 1 < p1 || !last) ? g.run_from[p + 1] : g.length;
        const double f = state_value<TYPE>(a, o, Q, g.run_state[p]);
        while (w + 1 < W && win[w + 1] <= to) {
            acc = fma(f, win[w + 1] - from, acc);
            add();
            from = win[++w];
        }
        acc = fma(f, to - from, acc);
    }
    add();
}

// --- allele frequency spectrum ------------------------------------------------------
// Columns are the sample sets; which alleles and branches cover some samples
// and not all is in the plan (row_all, the pieces left out).

namespace {

// Index of counts c[0 .. K) in the spectrum of the sets' sizes; folded
// (unpolarised): complemented where the allele is the minor one, ties broken
// on the trailing sets (trees.c:3469-3496).
__device__ __forceinline__ int64_t spectrum_index(const TsgSpectrumArgs &g, int K, int32_t *c) {
    if (!g.polarised) {
        double half = 0;
        int sum = 0;
        for (int k = 0; k < K; k++) {
            half += (double) g.dims[k] - 1;
            sum += c[k];
        }
        half /= 2;
        int k = K;
        while (sum == half && k > 0) {
            k--;
            half -= ((double) (g.dims[k] - 1)) / 2;
            sum -= c[k];
        }
        if (sum > half) {
            for (k = 0; k < K; k++) c[k] = (int32_t) g.dims[k] - 1 - c[k];
        }
    }
    int64_t at = 0;
    for (int k = 0; k < K; k++) at = at * g.dims[k] + c[k];
    return at;
}

template <int TYPE>
__device__ __forceinline__ int32_t row_count(const TsgStateArgs &a, int s, int k) {
    const uint32_t *row = a.x + (int64_t) s * a.RW;
    return TYPE == TSG_ROW_U16 ? (int32_t) reinterpret_cast<const uint16_t *>(row)[k]
                               : (int32_t) row[k];
}

}  // namespace

// Thread per site row: one (polarised) or a half (folded) per allele that is
// not fixed, in half-units (integers: exact, whatever the order).
template <int TYPE>
__global__ void __launch_bounds__(256) k_spectrum_site(const TsgStateArgs a,
                                                       const TsgSpectrumArgs g) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.nrow) return;
    const int all = g.row_all[i];
    if (all <= 0 || all >= a.num_samples) return;
    const int ref = a.row_ref[i];
    const int K = a.K;
    unsigned long long *hist = g.hist_u + window_of(g.windows, g.W, a.row_pos[i]) * g.size;
    int32_t c[TSG_SPECTRUM_SETS];
    if (ref >= 0) {
        for (int k = 0; k < K; k++) c[k] = row_count<TYPE>(a, ref, k);
        if (g.polarised) {
            atomicAdd(&hist[spectrum_index(g, K, c)], 2ull);
            return;
        }
        atomicAdd(&hist[spectrum_index(g, K, c)], 1ull);
        for (int k = 0; k < K; k++) c[k] = a.col_total[k] - row_count<TYPE>(a, ref, k);
        atomicAdd(&hist[spectrum_index(g, K, c)], 1ull);
        return;
    }
    const int l = -1 - ref;
    const bool ancestral = a.list_kind[l] == TSG_ROW_ANCESTRAL;
    if (ancestral && g.polarised) return;
    for (int k = 0; k < K; k++) {
        int32_t v = ancestral ? a.col_total[k] : 0;
        for (int e = a.list_off[l]; e < a.list_off[l + 1]; e++) {
            const int32_t x = row_count<TYPE>(a, a.list_ent[e] >> 1, k);
            v += (a.list_ent[e] & 1) ? -x : x;
        }
        c[k] = v;
    }
    atomicAdd(&hist[spectrum_index(g, K, c)], g.polarised ? 2ull : 1ull);
}

// Thread per branch piece: its span times the branch's length in each time
// window, cut at the windows it crosses; a piece that ends at a window's end
// counts where the edge was there before it (trees.c:3650-3690).
//
// Bound by adds to one address: most branches lie above one or two samples,
// so a few cells of each window take most of them.  The pieces are in order
// of their ends, so those of a workgroup fall into one or two windows; it
// adds into SPECTRUM_SLOTS cells of LDS, a cell to the first index that
// claims it, and sends each on once; other indexes go to memory directly.
template <int TYPE>
__global__ void __launch_bounds__(256) k_spectrum_branch(const TsgStateArgs a,
                                                         const TsgSpectrumArgs g, int per) {
    __shared__ unsigned long long cell[SPECTRUM_SLOTS];  // index + 1, 0: free
    __shared__ double sum[SPECTRUM_SLOTS];
    for (int i = threadIdx.x; i < SPECTRUM_SLOTS; i += 256) {
        cell[i] = 0;
        sum[i] = 0;
    }
    __syncthreads();
    const int64_t first = (int64_t) blockIdx.x * per;
    const int last = (int) min(first + per, (int64_t) g.npieces);
    for (int i = (int) first + threadIdx.x; i < last; i += 256) {
        const TsgBranchPiece p = g.pieces[i];
        int32_t c[TSG_SPECTRUM_SETS];
        for (int k = 0; k < a.K; k++) c[k] = row_count<TYPE>(a, p.state, k);
        const int64_t at = spectrum_index(g, a.K, c);
        auto add = [&](int w, double span) {
            for (int tw = 0; tw < g.TW && g.time_windows[tw] < p.tp; tw++) {
                const double length = fmax(0.0, fmin(g.time_windows[tw + 1], p.tp) -
                                                    fmax(g.time_windows[tw], p.tu));
                const int64_t to = ((int64_t) w * g.TW + tw) * g.size + at;
                const int slot = (int) (((uint64_t) to * 0x9e3779b97f4a7c15ull) >> 54);
                static_assert(SPECTRUM_SLOTS == 1 << (64 - 54), "slot bits");
                const unsigned long long key = (unsigned long long) to + 1;
                const unsigned long long was = atomicCAS(&cell[slot], 0ull, key);
                if (was == 0 || was == key) {
                    unsafeAtomicAdd(&sum[slot], span * length);
                } else {
                    unsafeAtomicAdd(&g.hist_d[to], span * length);
                }
            }
        };
        int w = window_of(g.windows, g.W, p.from);
        double from = p.from;
        while (w < g.W && g.windows[w + 1] <= p.to) {
            const double end = g.windows[w + 1];
            if (p.ins < end) add(w, end - from);
            from = end;
            w++;
        }
        if (w < g.W && p.to > from) add(w, p.to - from);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < SPECTRUM_SLOTS; i += 256) {
        if (cell[i] != 0) unsafeAtomicAdd(&g.hist_d[cell[i] - 1], sum[i]);
    }
}

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
template <int TYPE, bool BRANCH, bool WIDE>
__global__ void __launch_bounds__(EVAL_THREADS) k_state_eval(const TsgStateArgs a) {
    const int tiles = BRANCH ? a.btiles : a.stiles;
    const int t = xcd_block(blockIdx.x, tiles);
    if (t < tiles) evaluate<TYPE, BRANCH, WIDE>(a, t);
}
__global__ void __launch_bounds__(256) k_state_windows(const TsgStateArgs a) {
    window_sums(a, blockIdx.x);
}
__global__ void __launch_bounds__(TSG_FINISH_THREADS) k_state_finish(const TsgStateArgs a) {
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
template <int TYPE, bool BRANCH, bool WIDE>
__global__ void __launch_bounds__(EVAL_THREADS) k_states_eval(const TsgStateArgs *args,
                                                              const int32_t *pre, int nrun,
                                                              int nb) {
    const int b = xcd_block(blockIdx.x, nb);
    if (b >= nb) return;
    const int r = run_at(pre, nrun, b);
    evaluate<TYPE, BRANCH, WIDE>(args[r], b - pre[r]);
}
__global__ void __launch_bounds__(256) k_states_windows(const TsgStateArgs *args,
                                                        const int32_t *pre, int nrun) {
    const int r = run_at(pre, nrun, blockIdx.x);
    window_sums(args[r], blockIdx.x - pre[r]);
}
__global__ void __launch_bounds__(TSG_FINISH_THREADS) k_states_finish(const TsgStateArgs *args,
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
    const size_t el = (type == TSG_ROW_F64 || K <= TSG_STATE_F64_COLUMNS) ? 8
                      : (type == TSG_ROW_U16 && branch)                   ? 2
                                                                          : 4;
    return tile * (8 + 8 + (branch ? 8 : 4)) + EDGES * 8 + (EDGES + 4) * 4 +
           el * (tile + 2) * (size_t) K + 16;
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

template <int TYPE, bool BRANCH, bool WIDE>
hipError_t launch_eval_as(const TsgStateArgs &a, hipStream_t s) {
    const size_t sh = tsg_state_shmem(a.K, TYPE, BRANCH);
    hipError_t e = allow(&k_state_eval<TYPE, BRANCH, WIDE>, sh);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_state_eval<TYPE, BRANCH, WIDE>),
                       dim3(xcd_grid(BRANCH ? a.btiles : a.stiles)), dim3(EVAL_THREADS), sh, s, a);
    return hipGetLastError();
}
template <int TYPE, bool BRANCH>
hipError_t launch_eval(const TsgStateArgs &a, hipStream_t s) {
    if (TYPE == TSG_ROW_F64 || a.K <= TSG_STATE_F64_COLUMNS) {
        return launch_eval_as<TYPE, BRANCH, false>(a, s);
    }
    return launch_eval_as<TYPE, BRANCH, TYPE != TSG_ROW_F64>(a, s);
}

template <bool F64>
hipError_t launch_levels(const TsgStateLaunch &r, hipStream_t s) {
    const TsgStateArgs &a = r.a;
    for (int l = 1; l < r.levels; l++) {
        const int s0 = r.level0[l], s1 = r.level0[l + 1];
        const int64_t nb = count_blocks(a, s1 - s0);
        if (nb <= 0) continue;
        if (nb > INT32_MAX / 2) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_state_count<F64>), dim3(xcd_grid(nb)), dim3(256), 0, s, a, s0, s1,
                           (int) nb);
    }
    return hipGetLastError();
}

template <int TYPE>
hipError_t launch_counts(const TsgStateLaunch &r, hipEvent_t begin, hipStream_t s) {
    const TsgStateArgs &a = r.a;
    constexpr bool F64 = TYPE == TSG_ROW_F64;
    hipLaunchKernelGGL(k_state_stage, dim3((unsigned) stage_blocks(a)), dim3(256), 0, s, a);
    hipError_t e;
    if (begin != nullptr && (e = hipEventRecord(begin, s)) != hipSuccess) return e;
    hipLaunchKernelGGL((k_state_seed<TYPE>), dim3((unsigned) seed_blocks(a)), dim3(256), 0, s, a);
    return launch_levels<F64>(r, s);
}

template <int TYPE>
hipError_t launch_run(const TsgStateLaunch &r, hipEvent_t begin, hipEvent_t mid, hipEvent_t end,
                      hipStream_t s) {
    const TsgStateArgs &a = r.a;
    hipError_t e = launch_counts<TYPE>(r, begin, s);
    if (e != hipSuccess) return e;
    if (a.QB > 0 && (e = launch_eval<TYPE, true>(a, s)) != hipSuccess) return e;
    if (mid != nullptr && (e = hipEventRecord(mid, s)) != hipSuccess) return e;
    if (a.Q > a.QB && (e = launch_eval<TYPE, false>(a, s)) != hipSuccess) return e;
    if (end != nullptr && (e = hipEventRecord(end, s)) != hipSuccess) return e;
    if (r.wgroups > 0) {
        hipLaunchKernelGGL(k_state_windows, dim3((unsigned) r.wgroups), dim3(256), 0, s, a);
    }
    hipLaunchKernelGGL(k_state_finish, dim3((unsigned) r.fgroups), dim3(TSG_FINISH_THREADS), 0, s, a);
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

hipError_t tsg_launch_state_counts(const TsgStateLaunch &r, hipEvent_t begin, hipStream_t s) {
    switch (r.type) {
    case TSG_ROW_U16:
        return launch_counts<TSG_ROW_U16>(r, begin, s);
    case TSG_ROW_I32:
        return launch_counts<TSG_ROW_I32>(r, begin, s);
    default:
        return launch_counts<TSG_ROW_F64>(r, begin, s);
    }
}

hipError_t tsg_launch_state_levels(const TsgStateLaunch &r, hipStream_t s) {
    return launch_levels<false>(r, s);
}

hipError_t tsg_launch_state_nodes(const TsgStateLaunch &r, const TsgNodeArgs &g, int M,
                                  hipStream_t s) {
    return tsg_in_launches(((int64_t) g.runs * M + 255) / 256, [&](int64_t b, unsigned count) {
        if (r.type == TSG_ROW_U16) {
            hipLaunchKernelGGL((k_state_nodes<TSG_ROW_U16>), dim3(count), dim3(256), 0, s, r.a, g, b);
        } else {
            hipLaunchKernelGGL((k_state_nodes<TSG_ROW_I32>), dim3(count), dim3(256), 0, s, r.a, g, b);
        }
    });
}

hipError_t tsg_launch_spectrum(const TsgStateLaunch &r, const TsgSpectrumArgs &g, bool branch,
                               hipStream_t s) {
    const int64_t n = branch ? g.npieces : r.a.nrow;
    if (n == 0) return hipSuccess;
    // (branch: at most 1024 workgroups, so that each adds up more of them)
    const int per = branch ? 256 * (int) ((n + 256 * 1024 - 1) / (256 * 1024)) : 256;
    const unsigned nb = (unsigned) ((n + per - 1) / per);
    if (branch && r.type == TSG_ROW_U16) {
        hipLaunchKernelGGL((k_spectrum_branch<TSG_ROW_U16>), dim3(nb), dim3(256), 0, s, r.a, g, per);
    } else if (branch) {
        hipLaunchKernelGGL((k_spectrum_branch<TSG_ROW_I32>), dim3(nb), dim3(256), 0, s, r.a, g, per);
    } else if (r.type == TSG_ROW_U16) {
        hipLaunchKernelGGL((k_spectrum_site<TSG_ROW_U16>), dim3(nb), dim3(256), 0, s, r.a, g);
    } else {
        hipLaunchKernelGGL((k_spectrum_site<TSG_ROW_I32>), dim3(nb), dim3(256), 0, s, r.a, g);
    }
    return hipGetLastError();
}

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
    auto phase = [&](auto blocks, int threads = 256) {
        int64_t at = 0;
        pre.push_back(0);
        for (int r = 0; r < nrun; r++) {
            at += blocks(runs[r]);
            // (with what rounding up to the 8 XCDs adds)
            if ((at + 8) * threads > TSG_LAUNCH_THREADS) return false;
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
              phase([](const TsgStateLaunch &r) { return (int64_t) r.fgroups; }, TSG_FINISH_THREADS) &&
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
template <int TYPE, bool WIDE>
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
        if ((e = allow(&k_states_eval<TYPE, true, WIDE>, sb)) != hipSuccess) return e;
        hipLaunchKernelGGL((k_states_eval<TYPE, true, WIDE>), dim3(xcd_grid(total(PH_BRANCH))),
                           dim3(EVAL_THREADS), sb, s, args, at(PH_BRANCH), nrun,
                           total(PH_BRANCH));
    }
    if (total(PH_SITE) > 0) {
        if ((e = allow(&k_states_eval<TYPE, false, WIDE>, ss)) != hipSuccess) return e;
        hipLaunchKernelGGL((k_states_eval<TYPE, false, WIDE>), dim3(xcd_grid(total(PH_SITE))),
                           dim3(EVAL_THREADS), ss, s, args, at(PH_SITE), nrun, total(PH_SITE));
    }
    if (total(PH_WINDOWS) > 0) {
        hipLaunchKernelGGL(k_states_windows, dim3(total(PH_WINDOWS)), dim3(256), 0, s, args,
                           at(PH_WINDOWS), nrun);
    }
    hipLaunchKernelGGL(k_states_finish, dim3(total(PH_FINISH)), dim3(TSG_FINISH_THREADS), 0, s, args,
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
    const bool wide = runs[0].a.K > TSG_STATE_F64_COLUMNS;
    switch (runs[0].type) {
    case TSG_ROW_U16:
        return wide ? launch_multi<TSG_ROW_U16, true>(runs, args, nrun, pre_h, pre, s)
                    : launch_multi<TSG_ROW_U16, false>(runs, args, nrun, pre_h, pre, s);
    case TSG_ROW_I32:
        return wide ? launch_multi<TSG_ROW_I32, true>(runs, args, nrun, pre_h, pre, s)
                    : launch_multi<TSG_ROW_I32, false>(runs, args, nrun, pre_h, pre, s);
    default:
        return launch_multi<TSG_ROW_F64, false>(runs, args, nrun, pre_h, pre, s);
    }
}
