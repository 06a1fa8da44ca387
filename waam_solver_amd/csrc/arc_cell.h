/*
 * arc_cell.h — arc heat-source weights (reference kernels.py:406-622) and the compensated block
 * reduction used for the weight total; shared by the standalone and fused arc kernels.
 */
#pragma once

#include "thermal_cell.h"

namespace waam {

struct ArcParams {
    int kind;  // 0 Gaussian (Gaussian2D / ConicalVolume), 1 Goldak
    float arc_i, arc_j, arc_k;
    float inv2s2;                                  // Gaussian
    float sgn, ff, fr, af, ar, b, cax;             // Goldak
    float pen;
    int enable;
};

/* the shape weight of cell (i, j, k): Gaussian exp or Goldak pdf */
__device__ __forceinline__ float arc_shape(const ArcParams &p, int i, int j, int k)
{
    float di = (float)i - p.arc_i, dj = (float)j - p.arc_j, dk = (float)k - p.arc_k;
    if (p.kind == 0) {
        float r2 = di * di + dj * dj + dk * dk * 0.25f;
        return waam_expf(-r2 * p.inv2s2);
    }
    const float eps = 1e-6f;
    float x = di * p.sgn;
    bool front = x >= 0.0f;
    float a = front ? p.af : p.ar;
    float frac = front ? p.ff : p.fr;
    return frac * waam_expf(-3.0f * ((x * x) / (a * a + eps) + (dj * dj) / (p.b * p.b + eps) +
                                     (dk * dk) / (p.cax * p.cax + eps)));
}

/* Returns false for cells the reference skips (w_dep < 1e-6); otherwise the shape weight wg and
 * the surface weight wdep, whose product is the pass-1 term and (epw*wg)*wdep the pass-2
 * increment. */
__device__ __forceinline__ bool arc_cell_weights(const ArcParams &p, int i, int j, int k, float fl,
                                                 float &wg, float &wdep)
{
    wdep = arc_deposition_weight(k, p.arc_k, fl, p.pen, p.enable);
    if (wdep < 1e-6f) return false;
    wg = arc_shape(p, i, j, k);
    return true;
}

__device__ __forceinline__ double shfl_down64(double v, int off)
{
    return __hiloint2double(__shfl_down(__double2hiint(v), off),
                            __shfl_down(__double2loint(v), off));
}

/* The block's total of its threads' compensated pairs, in thread 0 (blocks of a power of two of at
 * least 64 threads; every thread calls it): halves added pairwise, between wavefronts through
 * LDS, then within the first by shuffles. The same additions as a tree in LDS all the way, whose
 * eight barriers cost a 256-thread block 2 us. */
__device__ __forceinline__ void block_reduce_pair(double &s, double &c, double *sh_s, double *sh_c)
{
    const int t = (int)(threadIdx.y * blockDim.x + threadIdx.x);
    sh_s[t] = s;
    sh_c[t] = c;
    __syncthreads();
    for (int off = (int)(blockDim.x * blockDim.y) / 2; off >= 64; off >>= 1) {
        if (t < off) {
            double ss, e;
            two_sum(s, sh_s[t + off], ss, e);
            c = c + sh_c[t + off] + e;
            s = ss;
            sh_s[t] = s;
            sh_c[t] = c;
        }
        __syncthreads();
    }
    if (t < 64) {
        for (int off = 32; off > 0; off >>= 1) {
            const double os = shfl_down64(s, off), oc = shfl_down64(c, off);
            double ss, e;
            two_sum(s, os, ss, e);
            c = c + oc + e;
            s = ss;
        }
    }
}

}  // namespace waam
