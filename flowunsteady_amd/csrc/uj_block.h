// uj_block.h -- one workgroup's share of the all-pairs U and J: a block of
// consecutive targets against a contiguous range of sources, staged through
// LDS one tile of BLK sources at a time.  The single-field kernels call these
// with the whole field as the source range; the batched kernels call them with
// the range of the target's own field (fields never interact).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_math.h"

namespace vpmx {

// ---------------------------------------------------------------------------
// FP64.  Source records (x, y, z, Gx) (Gy, Gz, sigma, 1/sigma).  The 15 sums
// of a target are kept without the -1/(4 pi) factor:
// d = (u 0..2, w = sum A Gamma 0..2, radial J 0..8 (k + 3 l)).

// One pair with radial coefficients A, B added to the sums.
__device__ __forceinline__ void f64_accumulate(const double4 a, const double4 b, double dx,
                                               double dy, double dz, double A, double B,
                                               double d[15])
{
    const double G1 = a.w, G2 = b.x, G3 = b.y;
    const double c1 = fma(dy, G3, -dz * G2), c2 = fma(dz, G1, -dx * G3), c3 = fma(dx, G2, -dy * G1);
    d[0] = fma(A, c1, d[0]); d[1] = fma(A, c2, d[1]); d[2] = fma(A, c3, d[2]);
    d[3] = fma(A, G1, d[3]); d[4] = fma(A, G2, d[4]); d[5] = fma(A, G3, d[5]);
    const double ex = B * dx, ey = B * dy, ez = B * dz;
    d[6] = fma(c1, ex, d[6]); d[7] = fma(c2, ex, d[7]); d[8] = fma(c3, ex, d[8]);
    d[9] = fma(c1, ey, d[9]); d[10] = fma(c2, ey, d[10]); d[11] = fma(c3, ey, d[11]);
    d[12] = fma(c1, ez, d[12]); d[13] = fma(c2, ez, d[13]); d[14] = fma(c3, ez, d[14]);
}

// A pair known to be the singular one: for the gaussian kernels 1 - g(rho) <
// 3e-19 and rho g'(rho) < 2e-17 at rho >= 9.5, so g = 1 and g' = 0 to FP64
// rounding (no exp, no division).
__device__ __forceinline__ void f64_pair_far(const double4 a, const double4 b, double xi,
                                             double yi, double zi, double d[15])
{
    const double dx = xi - a.x, dy = yi - a.y, dz = zi - a.z;
    const double rinv = rsq_f64(fma(dx, dx, fma(dy, dy, dz * dz)));
    const double ri2 = rinv * rinv, A = ri2 * rinv;
    f64_accumulate(a, b, dx, dy, dz, A, -3.0 * A * ri2, d);
}

// Any pair: the far form while every lane of the wave has rho^2 >= 90.25,
// else the full evaluation; coincident pairs skipped
// (src/FLOWUnsteady_processing_force.jl:895).  b.z holds pair_const_f64 here.
// DS: the core-size derivatives D[U], D[J] in the same sums, zero beyond
// rho^2 = X_CORE for the gaussian kernels.
template <int K, bool DS>
__device__ __forceinline__ void f64_pair(const double4 a, const double4 b, double xi, double yi,
                                         double zi, double d[15])
{
    const double dx = xi - a.x, dy = yi - a.y, dz = zi - a.z;
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double x = r2 * (b.w * b.w);
    if constexpr (K == GAUSSIANERF || K == GAUSSIAN) {
        if (__all(x >= (DS ? X_CORE : X_FAR))) {
            if constexpr (!DS) {
                const double rinv = rsq_f64(r2), ri2 = rinv * rinv, A = ri2 * rinv;
                f64_accumulate(a, b, dx, dy, dz, A, -3.0 * A * ri2, d);
            }
            return;
        }
    }
    if (!(r2 > 0.0)) return;
    double A, B;
    if constexpr (DS) {
        radial_dsig_f64<K>(r2, x, b.w, b.z, A, B);
    } else {
        const double rinv = K == WINCKELMANS ? 0.0 : rsq_f64(r2);
        radial_f64<K>(r2, x, rinv, rinv * rinv, b.w, b.z, A, B);
    }
    f64_accumulate(a, b, dx, dy, dz, A, B, d);
}

// The 15 sums of TG targets (thread t of the workgroup holds target
// t % TG at (xi, yi, zi)) against source slots [s0, s1), staged through LDS NT
// records at a time, the next tile loading while one computes.  With TG < NT
// the workgroup's NT / TG waves of a target share each tile: slice t / TG takes
// its NT / TG-th run of the records, and the slices are added in order at the
// end (slice 0's threads hold the totals).  A field of n particles gives n / TG
// workgroups that way, and with the split source ranges of small launches
// enough of them to fill the 256 CUs from a few hundred particles on: with one
// target per thread of 256 and segments of 1024 a field of 8,000 ran as 256
// workgroups, one wave per SIMD (RK3 step with relaxation 2.90 -> 1.24 ms
// together with the shorter pair; 601 particles, 0.50 -> 0.18 ms per UJ_gpu).
//
// With tile bounds `tb` (per 64 slots from slot 0: (centre, radius), (largest
// sigma, -, -, -); TG = 64, s0 a multiple of 64) a run whose gap to the targets'
// box is >= 9.5 sigma_max (> 0 for the singular kernel) takes f64_pair_far for
// every pair without the per-pair test.
template <int K, int NT, int TG, bool DS>
__device__ __forceinline__ void uj_f64_sums(const double4 *__restrict__ src, int64_t s0,
                                            int64_t s1, double xi, double yi, double zi,
                                            const double4 *__restrict__ tb, double4 *tile,
                                            double d[15])
{
    constexpr int SL = NT / TG;
    static_assert(NT % TG == 0 && TG % 64 == 0, "whole waves per slice");
    const int t = threadIdx.x, sl = t / TG;
    double cx = 0.0, cy = 0.0, cz = 0.0, rad = 0.0;
    if (tb) {   // box of the wave's 64 targets
        double lo[3] = {xi, yi, zi}, hi[3] = {xi, yi, zi};
        for (int o = 32; o > 0; o >>= 1)
            for (int k = 0; k < 3; ++k) {
                lo[k] = fmin(lo[k], __shfl_xor(lo[k], o));
                hi[k] = fmax(hi[k], __shfl_xor(hi[k], o));
            }
        const double hx = 0.5 * (hi[0] - lo[0]), hy = 0.5 * (hi[1] - lo[1]), hz = 0.5 * (hi[2] - lo[2]);
        cx = lo[0] + hx;
        cy = lo[1] + hy;
        cz = lo[2] + hz;
        rad = sqrt(hx * hx + hy * hy + hz * hz);
    }
    for (int k = 0; k < 15; ++k) d[k] = 0.0;
    double4 ra = make_double4(0.0, 0.0, 0.0, 0.0), rb = make_double4(0.0, 0.0, 1.0, 1.0);
    if (s0 + t < s1) {
        ra = src[2 * (s0 + t)];
        rb = src[2 * (s0 + t) + 1];
    }
    for (int64_t base = s0; base < s1; base += NT) {
        __syncthreads();
        tile[2 * t] = ra;
        tile[2 * t + 1] = make_double4(rb.x, rb.y, pair_const_f64<K>(rb.z, rb.w), rb.w);
        __syncthreads();
        const int64_t js = base + NT + t;
        if (js < s1) {
            ra = src[2 * js];
            rb = src[2 * js + 1];
        }
        // this slice's run of the tile: TG records, or its share of a partial tile
        const int have = (int)(s1 - base < NT ? s1 - base : NT);
        const int run = have == NT ? TG : (have + SL - 1) / SL;
        const int j0 = sl * run, cnt = min(run, have - j0);   // may be <= 0
        bool far = false;
        if constexpr (!DS && TG == 64 && K != WINCKELMANS) {
            if (tb && have == NT) {
                const int64_t ts = (base + j0) / TG;
                const double4 S = tb[2 * ts];
                const double ex = S.x - cx, ey = S.y - cy, ez = S.z - cz;
                const double gap = sqrt(ex * ex + ey * ey + ez * ez) - S.w - rad;
                far = K == SINGULAR ? gap > 0.0 : gap >= RHO_FAR * tb[2 * ts + 1].x;
            }
        }
        const double4 *tj = tile + 2 * j0;
        if (far) {
#pragma unroll 2
            for (int jj = 0; jj < TG; ++jj) f64_pair_far(tj[2 * jj], tj[2 * jj + 1], xi, yi, zi, d);
        } else {
            for (int jj = 0; jj < cnt; ++jj)
                f64_pair<K, DS>(tj[2 * jj], tj[2 * jj + 1], xi, yi, zi, d);
        }
    }
    if constexpr (SL > 1) {   // the slices of a target, added in slice order
        double *red = reinterpret_cast<double *>(tile);
        static_assert(15 * TG <= 8 * NT, "a slice's sums fit the tile");
        for (int s = 1; s < SL; ++s) {
            __syncthreads();
            if (sl == s)
                for (int k = 0; k < 15; ++k) red[k * TG + t % TG] = d[k];
            __syncthreads();
            if (sl == 0)
                for (int k = 0; k < 15; ++k) d[k] += red[k * TG + t];
        }
    }
}

// The 12 values (U, J column-major) of a target from its 15 sums.
__device__ __forceinline__ void uj_f64_values(const double d[15], double v[12])
{
    const double k = -INV4PI;
    v[0] = k * d[0]; v[1] = k * d[1]; v[2] = k * d[2];
    v[3] = k * d[6];
    v[4] = k * (d[7] - d[5]);
    v[5] = k * (d[8] + d[4]);
    v[6] = k * (d[9] + d[5]);
    v[7] = k * d[10];
    v[8] = k * (d[11] - d[3]);
    v[9] = k * (d[12] - d[4]);
    v[10] = k * (d[13] + d[3]);
    v[11] = k * d[14];
}

// U and J of target i (stride ldo) from its 12 values.
__device__ __forceinline__ void uj_f64_store(const double v[12], int64_t i, int64_t ldo,
                                             double *__restrict__ U, double *__restrict__ J,
                                             int reset)
{
    for (int k = 0; k < 3; ++k) U[k * ldo + i] = reset ? v[k] : U[k * ldo + i] + v[k];
    for (int k = 0; k < 9; ++k) J[k * ldo + i] = reset ? v[3 + k] : J[k * ldo + i] + v[3 + k];
}

// Mixed precision: the 14 FP64 sums of one target block against sources
// [s0, s1).  Targets are the sorted slots [t0, t1) of `tgt`; sources the
// sorted slots of (spos, sgam).  Coordinates are taken relative to the block's
// first target in FP64 and rounded to FP32; FP32 partials are folded into
// FP64 every MIXED_FOLD pairs (once per tile for far tiles).  d = (U0..2, W0..2, J0..7) before the -1/(4 pi) factor.
//
// A far pair is 34 instructions, about 74 cycles of its SIMD at the rate of two per
// four cycles, and takes 105: the vector units are 71 % busy, and the four waves
// per SIMD that 112 registers allow do not cover the rest (cube of 1,048,576:
// 749-765 ms per UJ).  Two targets per thread halve the LDS reads but leave two
// or three waves: 925-1036 ms; five waves spill: 843 ms.  The
// unroll counts keep the near loop at 112 VGPRs, four waves (4 and 4 in place of
// 8 and 2: 753 ms; a batch of 24 fields 45.0 against 43.5).
//
// With tile bounds `tb` (per BLK-slot tile counted from slot `torg`: (centre,
// radius), (largest sigma, -, -, -); the block's own targets are tile
// (t0 - torg)/BLK), a tile whose every pair is in the far field -- gap >=
// 7.001 sigma_max for the gaussian kernels, gap > 0 for the singular one --
// runs mixed_pair_far without per-pair tests, the same arithmetic the per-pair
// path takes for such pairs.  t0 - torg and s0 - torg must then be multiples
// of BLK.
//
// DS: the core-size derivatives D[U], D[J] in the same 14 sums
// (mixed_pair_dsig); far tiles are skipped, their pairs being beyond the
// cores (e^{-24.5} of the core value for the gaussian kernels).
template <int K, int BLK, bool DS = false>
__device__ __forceinline__ void uj_mixed_sums(const double4 *__restrict__ tgt, int64_t t0,
                                              int64_t t1, const double4 *__restrict__ spos,
                                              const float4 *__restrict__ sgam, int64_t s0,
                                              int64_t s1, const double4 *__restrict__ tb,
                                              int64_t torg, float4 *tpos, float4 *tgam,
                                              float4 *tlo, double d[14])
{
    static_assert(BLK % MIXED_FOLD == 0, "tiles hold whole fold groups");
    const int t = threadIdx.x;
    const int64_t s = t0 + t;
    const bool active = s < t1;
    const double4 o = tgt[t0];
    float xi = 0.f, yi = 0.f, zi = 0.f, xl = 0.f, yl = 0.f, zl = 0.f;
    if (active) {
        const double4 p = tgt[s];
        const double ox = p.x - o.x, oy = p.y - o.y, oz = p.z - o.z;
        xi = (float)ox;
        yi = (float)oy;
        zi = (float)oz;
        xl = (float)(ox - (double)xi);
        yl = (float)(oy - (double)yi);
        zl = (float)(oz - (double)zi);
    }
    double4 T = make_double4(0.0, 0.0, 0.0, 0.0);
    if (tb) T = tb[2 * ((t0 - torg) / BLK)];
    for (int k = 0; k < 14; ++k) d[k] = 0.0;

    for (int64_t base = s0; base < s1; base += BLK) {
        __syncthreads();
        const int64_t js = base + t;
        if (js < s1) {
            const double4 p = spos[js];
            const double ox = p.x - o.x, oy = p.y - o.y, oz = p.z - o.z;
            const float hx = (float)ox, hy = (float)oy, hz = (float)oz;
            tpos[t] = make_float4(hx, hy, hz, (float)p.w);
            tlo[t] = make_float4((float)(ox - (double)hx), (float)(oy - (double)hy),
                                 (float)(oz - (double)hz), 0.f);
            tgam[t] = sgam[js];
        }
        __syncthreads();
        const int cnt = (int)((s1 - base) < BLK ? (s1 - base) : BLK);
        bool far = false;
        if constexpr (K == GAUSSIANERF || K == GAUSSIAN || K == SINGULAR) {
            if (tb && cnt == BLK) {
                const int64_t ts = (base - torg) / BLK;
                const double4 S = tb[2 * ts];
                const double ex = S.x - T.x, ey = S.y - T.y, ez = S.z - T.z;
                const double gap = sqrt(ex * ex + ey * ey + ez * ez) - S.w - T.w;
                if constexpr (K == SINGULAR)
                    far = gap > 0.0;
                else
                    far = gap >= 7.001 * tb[2 * ts + 1].x;
            }
        }
        MixedAcc acc;
        if constexpr (DS) {
            if (!far) {
                if (cnt == BLK) {
                    for (int jb = 0; jb < BLK; jb += MIXED_FOLD) {
#pragma unroll 2
                        for (int jj = jb; jj < jb + MIXED_FOLD; ++jj)
                            mixed_pair_dsig_hl<K>(tpos[jj], tlo[jj], tgam[jj], xi, yi, zi, xl,
                                                  yl, zl, acc);
                        mixed_fold(d, acc);
                    }
                } else {
                    for (int jj = 0; jj < cnt; ++jj) {
                        mixed_pair_dsig_hl<K>(tpos[jj], tlo[jj], tgam[jj], xi, yi, zi, xl, yl,
                                              zl, acc);
                        if ((jj & (MIXED_FOLD - 1)) == MIXED_FOLD - 1) mixed_fold(d, acc);
                    }
                }
            }
        } else if (far) {
            // far pairs are at least 7 core sizes (or a gap) away: their terms
            // stay small and one partial per tile suffices
#pragma unroll 8
            for (int jj = 0; jj < BLK; ++jj)
                mixed_pair_far<K>(tpos[jj], tgam[jj], xi, yi, zi, acc);
        } else if (cnt == BLK) {
            for (int jb = 0; jb < BLK; jb += MIXED_FOLD) {
#pragma unroll 2
                for (int jj = jb; jj < jb + MIXED_FOLD; ++jj)
                    mixed_pair_hl<K>(tpos[jj], &tlo[jj], tgam[jj], xi, yi, zi, xl, yl, zl, acc);
                mixed_fold(d, acc);
            }
        } else {
            for (int jj = 0; jj < cnt; ++jj) {
                mixed_pair_hl<K>(tpos[jj], &tlo[jj], tgam[jj], xi, yi, zi, xl, yl, zl, acc);
                if ((jj & (MIXED_FOLD - 1)) == MIXED_FOLD - 1) mixed_fold(d, acc);
            }
        }
        mixed_fold(d, acc);
    }
}

// U and J of target i from the 14 sums: J = -1/(4 pi) (radial + eps_klm W_m),
// J22 from the zero trace; reset = 0 adds to what U, J hold.
__device__ __forceinline__ void uj_mixed_store(const double d[14], int64_t i, int64_t ldo,
                                               double *__restrict__ U, double *__restrict__ J,
                                               int reset)
{
    const double k = -INV4PI;
    double u0 = k * d[0], u1 = k * d[1], u2 = k * d[2];
    double j0 = k * d[6], j1 = k * (d[7] - d[5]), j2 = k * (d[8] + d[4]);
    double j3 = k * (d[9] + d[5]), j4 = k * d[10], j5 = k * (d[11] - d[3]);
    double j6 = k * (d[12] - d[4]), j7 = k * (d[13] + d[3]), j8 = -k * (d[6] + d[10]);
    if (!reset) {
        u0 += U[i]; u1 += U[ldo + i]; u2 += U[2 * ldo + i];
        j0 += J[i]; j1 += J[ldo + i]; j2 += J[2 * ldo + i];
        j3 += J[3 * ldo + i]; j4 += J[4 * ldo + i]; j5 += J[5 * ldo + i];
        j6 += J[6 * ldo + i]; j7 += J[7 * ldo + i]; j8 += J[8 * ldo + i];
    }
    U[i] = u0; U[ldo + i] = u1; U[2 * ldo + i] = u2;
    J[i] = j0; J[ldo + i] = j1; J[2 * ldo + i] = j2;
    J[3 * ldo + i] = j3; J[4 * ldo + i] = j4; J[5 * ldo + i] = j5;
    J[6 * ldo + i] = j6; J[7 * ldo + i] = j7; J[8 * ldo + i] = j8;
}

// One block: sums over [s0, s1) and the store through perm (stride ldo).
template <int K, int BLK, bool DS = false>
__device__ __forceinline__ void uj_mixed_block(const double4 *__restrict__ tgt, int64_t t0,
                                               int64_t t1, const int32_t *__restrict__ perm,
                                               const double4 *__restrict__ spos,
                                               const float4 *__restrict__ sgam, int64_t s0,
                                               int64_t s1, int64_t ldo,
                                               double *__restrict__ U, double *__restrict__ J,
                                               int reset, float4 *tpos, float4 *tgam,
                                               float4 *tlo,
                                               const double4 *__restrict__ tb = nullptr,
                                               int64_t torg = 0)
{
    double d[14];
    uj_mixed_sums<K, BLK, DS>(tgt, t0, t1, spos, sgam, s0, s1, tb, torg, tpos, tgam, tlo, d);
    const int64_t s = t0 + threadIdx.x;
    if (s < t1) uj_mixed_store(d, perm[s], ldo, U, J, reset);
}

}  // namespace vpmx
