// The composites evaluated after the window sums, shared by the kernels of
// every plan.
#pragma once
#include <hip/hip_runtime.h>

#include "tsg_common.h"

// FP64 composites of the reference's Python layer.
struct TsgFinal {
    int32_t kind;       // tsg_final_id
    int32_t Kq;         // number of sample sets (TajD: sets; Fst: sets)
    int32_t P;          // number of final outputs per window
    int32_t W;
    int64_t rawbase, outbase;
    int64_t pbase;      // params: Fst -> index pairs (int32 pairs); TajD -> per-set (n,h,g)
    int32_t Mraw;
};

__device__ __forceinline__ void finals(const TsgFinal *fin, int nq, const double *raw,
                                       const int32_t *ipar, const double *dpar, double *out,
                                       int64_t total, int64_t bx) {
    const int64_t gid = bx * 256 + threadIdx.x;
    if (gid >= total) return;
    int q = 0;
    int64_t rem = gid;
    while (q < nq) {
        const int64_t n = (int64_t) fin[q].W * fin[q].P;
        if (rem < n) break;
        rem -= n;
        q++;
    }
    const TsgFinal &F = fin[q];
    const int w = (int) (rem / F.P);
    const int p = (int) (rem % F.P);
    const double *r = raw + F.rawbase + (int64_t) w * F.Mraw;
    double v;
    switch (F.kind) {
    case TSG_FINAL_FST: {  // trees.py:10113-10125
        const int u = ipar[F.pbase + 2 * p], x = ipar[F.pbase + 2 * p + 1];
        const double du = r[u], dv = r[x], duv = r[F.Kq + p];
        const double denom = du + dv + 2 * duv;
        v = 1.0 - 2 * (du + dv) / denom;
        break;
    }
    case TSG_FINAL_TAJIMAS_D: {  // trees.py:10008-10018
        const double n = dpar[F.pbase + 3 * p], h = dpar[F.pbase + 3 * p + 1];
        const double g = dpar[F.pbase + 3 * p + 2];
        const double T = r[p], S = r[F.Kq + p];
        const double aa = (n + 1) / (3 * (n - 1) * h) - 1 / (h * h);
        const double bb = 2 * (n * n + n + 3) / (9 * n * (n - 1)) - (n + 2) / (h * n) + g / (h * h);
        v = (T - S / h) / sqrt(aa * S + (bb / (h * h + g)) * S * (S - 1));
        break;
    }
    case TSG_FINAL_PROPORTION:  // trees.py:8958-8974
        v = r[p] / r[F.P];
        break;
    default:
        v = r[p];
    }
    out[F.outbase + (int64_t) w * F.P + p] = v;
}
