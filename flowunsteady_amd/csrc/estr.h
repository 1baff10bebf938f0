// estr.h -- FP64 SFS stretching (docs/src/theory/rvpm.md:251-262)
//   E_i = sum_j zeta_j S(J_i - J_j, Gamma_j),  zeta_j = zeta(|x_i - x_j|/sigma_j)/sigma_j^3,
// and for the dynamic procedure its core-size derivative
//   D[E]_i = sum_j zD_j S(J_i - J_j, Gamma_j) + zeta_j S(DJ_i - DJ_j, Gamma_j),
// as the direct and the near-field kernels share it.
//
// S is linear in both arguments, so with J, DJ taken relative to a reference
//   E_i = S(J_i, sum_j zeta_j Gamma_j) - sum_j zeta_j S(J_j, Gamma_j):
// the stretching of a source is formed once when its record enters LDS, and a
// pair adds 6 products (15 with D[E]) in place of 21 (45).  The reference is the
// J (and the DJ) of least norm among the workgroup's targets (estr_least): then
// |J_i - J_ref| <= 2 |J_i|, so that the two parts round no coarser than the J_i and
// J_j they are made of, also where the workgroup holds a far stronger vortex, and
// near the size of J's variation where J is smooth.  (With the first target as the
// reference a weak cluster in a strong vortex's workgroup lost the digits of their
// ratio.)  A particle's own term, zero, is left out by index, so that an
// isolated particle gets E = 0 and no rounding of its own stretching.
#pragma once
#include <hip/hip_runtime.h>

#include "device_math.h"

namespace vpmx {

// Source record of NR double4: (x, y, z, 1/sigma) (Gamma, 0) (J0..3) (J4..7)
// (J8, 0, 0, 0); DYN: the last is (J8, DJ0..2) followed by (DJ3..6) (DJ7, DJ8, 0, 0).
template <bool DYN>
constexpr int ESTR_NR = DYN ? 7 : 5;
// LDS record of NL double2: (x, y) (z, 1/sigma^2) (w G0, w G1) (w G2, s0) (s1, s2),
// DYN: (t0, t1) (t2, 0), with w zeta's constant over sigma^3, s = S(J_j, w Gamma_j),
// t = S(DJ_j, w Gamma_j).
template <bool DYN>
constexpr int ESTR_NL = DYN ? 7 : 5;

// The nine J (and with DYN DJ) entries of a source record.
template <bool DYN>
__device__ __forceinline__ void estr_rec_j(const double4 *r, double *Jv, double *DJv)
{
    const double4 q2 = r[2], q3 = r[3], q4 = r[4];
    Jv[0] = q2.x; Jv[1] = q2.y; Jv[2] = q2.z; Jv[3] = q2.w;
    Jv[4] = q3.x; Jv[5] = q3.y; Jv[6] = q3.z; Jv[7] = q3.w; Jv[8] = q4.x;
    if constexpr (DYN) {
        const double4 q5 = r[5], q6 = r[6];
        DJv[0] = q4.y; DJv[1] = q4.z; DJv[2] = q4.w;
        DJv[3] = q5.x; DJv[4] = q5.y; DJv[5] = q5.z; DJv[6] = q5.w;
        DJv[7] = q6.x; DJv[8] = q6.y;
    }
}

// The index, over the wave's lanes, whose J has the least norm (to 20 bits; NaN
// last, ties to the lowest index): the same in every lane.
__device__ __forceinline__ int estr_least(const double J[9], int index)
{
    double q = 0.0;
    for (int k = 0; k < 9; ++k) q += fabs(J[k]);
    uint64_t key = (uint64_t)(uint32_t)__double2hiint(q) << 32 | (uint32_t)index;
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t other = __shfl_xor((unsigned long long)key, o);
        key = other < key ? other : key;
    }
    return __builtin_amdgcn_readfirstlane((int)(uint32_t)key);
}

// J and DJ of the references among the records rec[NR index], index = the lane's own.
template <bool DYN>
__device__ __forceinline__ void estr_reference(const double4 *rec, int index, double Jr[9],
                                               double DJr[9])
{
    constexpr int NR = ESTR_NR<DYN>;
    double J[9], DJ[9], other[9];
    estr_rec_j<DYN>(rec + NR * index, J, DJ);
    const int ij = estr_least(J, index);
    estr_rec_j<DYN>(rec + NR * ij, Jr, other);
    if constexpr (DYN) {
        const int id = estr_least(DJ, index);
        estr_rec_j<DYN>(rec + NR * id, other, DJr);
    }
}

// S_k = sum_l J[l,k] g_l (transposed) or sum_l J[k,l] g_l (classic).
template <bool TRANSPOSED>
__device__ __forceinline__ void stretch_of(const double J[9], const double g[3], double S[3])
{
    for (int k = 0; k < 3; ++k)
        if constexpr (TRANSPOSED)
            S[k] = fma(J[3 * k], g[0], fma(J[3 * k + 1], g[1], J[3 * k + 2] * g[2]));
        else
            S[k] = fma(J[k], g[0], fma(J[k + 3], g[1], J[k + 6] * g[2]));
}

// zeta and zD = -(3 zeta + rho zeta') over zeta's constant, at x = rho^2.
template <int K>
constexpr double ESTR_W = K == GAUSSIANERF ? 0.06349363593424097     // (2 pi)^-3/2
                          : K == GAUSSIAN  ? 0.238732414637843      // 3/(4 pi)
                                           : 0.5968310365946075;    // 15/(8 pi), Winckelmans
template <int K, bool DYN>
__device__ __forceinline__ void estr_shape(double x, double &z, double &zD)
{
    if constexpr (K == GAUSSIANERF) {
        z = exp_mhalf(x);
        if constexpr (DYN) zD = (x - 3.0) * z;
    } else if constexpr (K == GAUSSIAN) {
        const double r3 = x * sqrt(x);
        z = exp_mhalf(2.0 * r3);
        if constexpr (DYN) zD = 3.0 * (r3 - 1.0) * z;
    } else {
        const double si = rsq_f64(x + 1.0), si2 = si * si;
        z = si2 * si2 * si2 * si;
        if constexpr (DYN) zD = fma(-7.0, si2, 4.0) * z;
    }
}

// LDS record o of the source record r, J and DJ relative to (Jr, DJr).
template <int K, bool TRANSPOSED, bool DYN>
__device__ __forceinline__ void estr_stage(const double4 *r, const double Jr[9],
                                           const double DJr[9], double2 *o)
{
    const double4 p = r[0], gm = r[1];
    const double w = ESTR_W<K> * (p.w * p.w * p.w);
    const double g[3] = {w * gm.x, w * gm.y, w * gm.z};
    double Jv[9], DJv[9], s[3];
    estr_rec_j<DYN>(r, Jv, DJv);
    for (int k = 0; k < 9; ++k) Jv[k] -= Jr[k];
    stretch_of<TRANSPOSED>(Jv, g, s);
    o[0] = make_double2(p.x, p.y);
    o[1] = make_double2(p.z, p.w * p.w);
    o[2] = make_double2(g[0], g[1]);
    o[3] = make_double2(g[2], s[0]);
    o[4] = make_double2(s[1], s[2]);
    if constexpr (DYN) {
        for (int k = 0; k < 9; ++k) DJv[k] -= DJr[k];
        stretch_of<TRANSPOSED>(DJv, g, s);
        o[5] = make_double2(s[0], s[1]);
        o[6] = make_double2(s[2], 0.0);
    }
}

// Sums of a target: a = zeta Gamma, b = zeta s, c = zD Gamma, d = zD s + zeta t.
struct EstrAcc {
    double a[3] = {0.0, 0.0, 0.0}, b[3] = {0.0, 0.0, 0.0}, c[3] = {0.0, 0.0, 0.0},
           d[3] = {0.0, 0.0, 0.0};
};

// One pair (self: the target itself).  e^{-x/2} is zero from x = 1490 on, so a
// pair beyond 1500 in every lane is left out for the gaussian kernels.
template <int K, bool DYN>
__device__ __forceinline__ void estr_pair(const double2 *q, double xi, double yi, double zi,
                                          bool self, EstrAcc &e)
{
    const double2 p = q[0], ps = q[1];
    const double dx = xi - p.x, dy = yi - p.y, dz = zi - ps.x;
    const double x = fma(dx, dx, fma(dy, dy, dz * dz)) * ps.y;
    if constexpr (K != WINCKELMANS)
        if (__all(x >= X_CORE)) return;
    double z, zD = 0.0;
    estr_shape<K, DYN>(x, z, zD);
    z = self ? 0.0 : z;
    const double2 q2 = q[2], q3 = q[3], q4 = q[4];
    const double g[3] = {q2.x, q2.y, q3.x}, s[3] = {q3.y, q4.x, q4.y};
    for (int k = 0; k < 3; ++k) {
        e.a[k] = fma(z, g[k], e.a[k]);
        e.b[k] = fma(z, s[k], e.b[k]);
    }
    if constexpr (DYN) {
        zD = self ? 0.0 : zD;
        const double2 q5 = q[5], q6 = q[6];
        const double t[3] = {q5.x, q5.y, q6.x};
        for (int k = 0; k < 3; ++k) {
            e.c[k] = fma(zD, g[k], e.c[k]);
            e.d[k] = fma(zD, s[k], fma(z, t[k], e.d[k]));
        }
    }
}

// E (and D[E]) of a target from its sums and its record r.
template <bool TRANSPOSED, bool DYN>
__device__ __forceinline__ void estr_values(const EstrAcc &e, const double4 *r, const double Jr[9],
                                            const double DJr[9], double v[DYN ? 6 : 3])
{
    double Jv[9], DJv[9], s[3];
    estr_rec_j<DYN>(r, Jv, DJv);
    for (int k = 0; k < 9; ++k) Jv[k] -= Jr[k];
    stretch_of<TRANSPOSED>(Jv, e.a, s);
    for (int k = 0; k < 3; ++k) v[k] = s[k] - e.b[k];
    if constexpr (DYN) {
        double t[3];
        for (int k = 0; k < 9; ++k) DJv[k] -= DJr[k];
        stretch_of<TRANSPOSED>(Jv, e.c, s);
        stretch_of<TRANSPOSED>(DJv, e.a, t);
        for (int k = 0; k < 3; ++k) v[3 + k] = (s[k] - e.d[k]) + t[k];
    }
}

}  // namespace vpmx
