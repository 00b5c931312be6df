// vlct_physics.hpp -- per-face / per-cell device functions of the VL+CT step.
//
// Templated on the arithmetic type T (double for the reference-parity path,
// float for the FP32 reconstruction/Riemann stage of the mixed path).  The
// expression trees keep the reference's parenthesisation and left-to-right
// association; the library is built with -ffp-contract=off so the FP64 path
// rounds exactly like the reference's CPU build.  The FP32 solves' fused
// multiply-adds are written out (mad and the others below).
#pragma once

#include <hip/hip_runtime.h>

// The namespace of the device code and of its launch templates: `enzoe` in
// the default build; a unit that compiles the same templates under other
// floating-point flags (the contracted FP64 step) names another one before
// including, so that the two sets of instantiations never share a symbol.
#ifndef ENZOE_KNS
#define ENZOE_KNS enzoe
#endif

namespace ENZOE_KNS {

// field slots used for cell-centred state, primitives and fluxes
enum : int {
  S_RHO = 0, S_VX = 1, S_VY = 2, S_VZ = 3, S_E = 4, S_BX = 5, S_BY = 6,
  S_BZ = 7, S_N = 8
};
// Riemann LUT order, MHD (EnzoRiemannImpl.hpp:40-56)
enum : int { L_D = 0, L_BI, L_BJ, L_BK, L_VI, L_VJ, L_VK, L_E };
// Riemann LUT order, hydro (EnzoRiemannImpl.hpp:21-36)
enum : int { H_D = 0, H_VI, H_VJ, H_VK, H_E };

enum : int { RS_HLLE = 0, RS_HLLC = 1, RS_HLLD = 2 };
enum : int { RC_NN = 0, RC_PLM = 1, RC_PLM_ATHENA = 2 };

// Division and square root: correctly rounded in FP64 (reference parity);
// hardware reciprocal / square root (about 1 ulp) in FP32, where the
// mixed-precision path is judged by its L1 error instead.
//
// The FP64 division without the operand scaling that covers the ends of the
// exponent range: the hardware's reciprocal (24 good bits), two Newton
// steps, the product and one correction by the exact residual; 1 / b takes
// one cubic step and the correction (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990).  The hardware's
// fix-up puts zeros, infinities and NaN right.  9 and 7 instructions instead
// of 11, and none of the wait states that the scaled form's flag costs.
// Rounded as IEEE division for 2^-1000 < |b| < 2^1000 and quotients and
// residuals in the normal range.  (For a mantissa of all ones the last
// correction of 1 / b is a tie that the sign of the seed's error decides; on
// gfx950 it comes out right: compared with IEEE division over both ends of
// the mantissas of every binade from 2^-1021 to 2^1021, no difference.)  A
// subnormal divisor or a quotient that overflows gives NaN where IEEE
// division gives a large number or infinity: no state gets there whose
// densities and pressures stay above floors of normal size (1e-200 unless
// set), speeds and sums of roots included.  With the shared reciprocals (qdiv_inv) and
// the roots below the FP64 flux kernels, bound by their instruction issue,
// take 1.51 and 2.11 ms on a 256^3 block (nearest neighbour, PLM) instead
// of 1.67 and 2.23.
__device__ __forceinline__ double qrcp(double b) {
  const double y0 = __builtin_amdgcn_rcp(b);
  const double e = __builtin_fma(-b, y0, 1.0);
  const double y = __builtin_fma(__builtin_fma(e, e, e), y0, y0);
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, y, 1.0), y, y), b, 1.0);
}
__device__ __forceinline__ float qrcp(float b) { return __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double qdiv(double a, double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
  y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
  const double q = a * y;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), y, q), b, a);
}
__device__ __forceinline__ float qdiv(float a, float b) {
  return a * __builtin_amdgcn_rcpf(b);
}
// The FP64 square root without the scaling steps that a general one needs:
// from the hardware's reciprocal root, one Goldschmidt step and two
// corrections of g by the exact residual x - g g (Markstein, "IA-64 and
// Elementary Functions", 2000), 10 instructions, for 2^-767 <= x < 2^769;
// sqrt() outside (zeros, negatives, NaN among them).  Correctly rounded
// either way.  The pair form takes two roots side by side, so that their
// dependent chains overlap, behind one test.
__device__ __forceinline__ double root_tame(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
__device__ __forceinline__ unsigned root_key(double x) {
  return (unsigned)(__double2hiint(x) - 0x10000000);
}
constexpr unsigned ROOT_KEYS = 0x60000000u;  // keys of the tame range lie below
__device__ __forceinline__ double qsqrt(double x) {
  double g = root_tame(x);
  if (__builtin_expect(root_key(x) >= ROOT_KEYS, 0)) g = sqrt(x);
  return g;
}
__device__ __forceinline__ void qsqrt2(double a, double b, double &ra, double &rb) {
  ra = root_tame(a);
  rb = root_tame(b);
  const unsigned ka = root_key(a), kb = root_key(b);
  if (__builtin_expect((ka > kb ? ka : kb) >= ROOT_KEYS, 0)) {
    ra = sqrt(a);
    rb = sqrt(b);
  }
}
__device__ __forceinline__ void qsqrt2(float a, float b, float &ra, float &rb) {
  ra = __builtin_amdgcn_sqrtf(a);
  rb = __builtin_amdgcn_sqrtf(b);
}
__device__ __forceinline__ float qsqrt(float a) {
  return __builtin_amdgcn_sqrtf(a);
}
// a / b where inv = 1 / b is at hand: in FP64 the product and one correction
// by the exact residual, which rounds as the division does when inv is the
// correctly rounded reciprocal: 4 instructions.
__device__ __forceinline__ double qdiv_inv(double a, double b, double inv) {
  const double q = a * inv;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), inv, q), b, a);
}
__device__ __forceinline__ float qdiv_inv(float a, float, float inv) { return a * inv; }

// Multiply-adds of the Riemann solves.  FP32 (the mixed path): one rounding,
// written out here and never left to the compiler.  The FP32 HLLD solve
// divides by differences that can cancel down to their rounding (and HLLE
// takes the root of one), so a multiply-add that is fused in one kernel and
// not in another can change a cell by as much as it holds; like this every
// kernel that runs a solve rounds alike.  FP64: the product and the sum
// rounded in turn, as the reference does (the contracted build's compiler
// fuses them).
__device__ __forceinline__ double mad(double a, double b, double c) { return a * b + c; }
__device__ __forceinline__ float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// a b - c
__device__ __forceinline__ double msub(double a, double b, double c) { return a * b - c; }
__device__ __forceinline__ float msub(float a, float b, float c) {
  return __builtin_fmaf(a, b, -c);
}
// c + a b, c - a b
__device__ __forceinline__ double add_mul(double c, double a, double b) { return c + a * b; }
__device__ __forceinline__ float add_mul(float c, float a, float b) {
  return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double sub_mul(double c, double a, double b) { return c - a * b; }
__device__ __forceinline__ float sub_mul(float c, float a, float b) {
  return __builtin_fmaf(-a, b, c);
}
// c + a / b, c - a / b, where inv = 1 / b is at hand
__device__ __forceinline__ double add_div(double c, double a, double b, double inv) {
  return c + qdiv_inv(a, b, inv);
}
__device__ __forceinline__ float add_div(float c, float a, float, float inv) {
  return __builtin_fmaf(a, inv, c);
}
__device__ __forceinline__ double sub_div(double c, double a, double b, double inv) {
  return c - qdiv_inv(a, b, inv);
}
__device__ __forceinline__ float sub_div(float c, float a, float, float inv) {
  return __builtin_fmaf(-a, inv, c);
}
// ... and where it is not (c - a / b, c + a / b)
__device__ __forceinline__ double add_div(double c, double a, double b) { return c + qdiv(a, b); }
__device__ __forceinline__ float add_div(float c, float a, float b) {
  return __builtin_fmaf(a, __builtin_amdgcn_rcpf(b), c);
}
__device__ __forceinline__ double sub_div(double c, double a, double b) { return c - qdiv(a, b); }
__device__ __forceinline__ float sub_div(float c, float a, float b) {
  return __builtin_fmaf(-a, __builtin_amdgcn_rcpf(b), c);
}

// a1 b1 + a2 b2.  FP32: the first product is fused onto the second, with SWAP
// the second onto the first.
template <bool SWAP>
__device__ __forceinline__ double dot2(double a1, double b1, double a2, double b2) {
  return a1 * b1 + a2 * b2;
}
template <bool SWAP>
__device__ __forceinline__ float dot2(float a1, float b1, float a2, float b2) {
  return SWAP ? __builtin_fmaf(a2, b2, a1 * b1) : __builtin_fmaf(a1, b1, a2 * b2);
}
// Where the FP32 solves fuse the second product of such a sum.  Either order
// is as good; these are the ones that the path's results have always been
// formed with, which the ill-conditioned faces hold it to.  D: the face's
// axis; RECON: reconstructed states (not the nearest-neighbour ones); HALF:
// states from the half-step primitives (the pressure at hand).  The rules
// follow the fields: of two transverse components the earlier of x, y, z is
// fused, of a left and a right value the one whose operands come first.
template <int D, bool RECON, bool HALF>
struct SumOrder {
  static constexpr bool kj = D == 1;              // transverse components j, k
  static constexpr bool kj_roe = kj && !RECON;    // ... of the Roe average
  static constexpr bool ji_roe = D == 2 && !RECON;  // normal and first transverse velocity
  static constexpr bool rl = RECON && HALF;       // sqrt(rho) weighted left and right values
  static constexpr bool energy = !HALF;           // internal and kinetic energy
};
// Internal plus kinetic energy density p / (gamma - 1) + (rho / 2) v^2, where
// inv = 1 / (gamma - 1).
template <bool SWAP>
__device__ __forceinline__ double energy_density(double p, double gm1, double inv, double half_rho,
                                                 double v2) {
  return qdiv_inv(p, gm1, inv) + half_rho * v2;
}
template <bool SWAP>
__device__ __forceinline__ float energy_density(float p, float, float inv, float half_rho,
                                                float v2) {
  return dot2<SWAP>(p, inv, half_rho, v2);
}
// a quotient a / b that sums are formed with
template <typename T> struct Quotient;
template <> struct Quotient<double> {
  double q;
  __device__ __forceinline__ Quotient(double a, double b) : q(qdiv(a, b)) {}
  __device__ __forceinline__ double minus(double c) const { return q - c; }  // a / b - c
  __device__ __forceinline__ double from(double c) const { return c - q; }   // c - a / b
};
template <> struct Quotient<float> {
  float a, inv, q;
  __device__ __forceinline__ Quotient(float num, float b)
      : a(num), inv(__builtin_amdgcn_rcpf(b)), q(num * inv) {}
  __device__ __forceinline__ float minus(float c) const { return __builtin_fmaf(a, inv, -c); }
  __device__ __forceinline__ float from(float c) const { return __builtin_fmaf(-a, inv, c); }
};

template <typename T> __device__ __forceinline__ T dmin(T a, T b) {
  return (b < a) ? b : a;  // std::min
}
template <typename T> __device__ __forceinline__ T dmax(T a, T b) {
  return (a < b) ? b : a;  // std::max
}
// enzo_utils::min of three values (src/Enzo/utils/utils.hpp:82-89)
template <typename T> __device__ __forceinline__ T dmin3(T a, T b, T c) {
  if (a < b) return (c < a) ? c : a;
  return (c < b) ? c : b;
}
// The same minimum of the magnitudes |a|, |b|, |c| with the hardware
// minimum (IEEE minNum): the two agree on every input, NaN included, except
// where |b| is NaN (the reference's comparisons then return |b|, minNum
// would drop it), which the final select restores.  Used by the PLM limiter,
// whose arguments are differences (never signalling NaNs).
template <typename T> __device__ __forceinline__ T dmin3_abs(T a, T b, T c) {
  const T m = __builtin_fmin(__builtin_fmin(fabs(a), fabs(b)), fabs(c));
  return (b == b) ? m : fabs(b);
}
template <typename T> __device__ __forceinline__ T dsign(T v) {
  return (T)((T(0) < v) - (v < T(0)));
}

// PLM_EnzoRKLimiter (EnzoReconstructorPLM.hpp:287-302)
template <typename T>
__device__ __forceinline__ T limiter_enzo(T vm1, T v, T vp1, T theta) {
  T dv_c = T(0.5) * (vp1 - vm1);
  T dv_l = (v - vm1) * theta;
  T dv_r = (vp1 - v) * theta;
  return (T(0.5) * (dsign(dv_l) + dsign(dv_r))) * dmin3_abs(dv_l, dv_r, dv_c);
}
// The same limiter in FP32 (the mixed path, judged by its L1 distance to
// the FP64 result, not bit for bit), with the sign factor taken from the
// sign bits: equal signs give copysign(m, dv_l), unequal ones 0, and where
// a difference is zero m is 0 as well.  The result equals the form above
// but for the sign of a zero and for how a NaN difference spreads; it
// takes about 12 instructions instead of 20 in the issue-bound FP32 flux
// kernel.
__device__ __forceinline__ float limiter_enzo(float vm1, float v, float vp1, float theta) {
  const float dv_c = 0.5f * (vp1 - vm1);
  const float dv_l = (v - vm1) * theta;
  const float dv_r = (vp1 - v) * theta;
  const float m = __builtin_fminf(__builtin_fminf(fabsf(dv_l), fabsf(dv_r)), fabsf(dv_c));
  const bool same = ((__float_as_uint(dv_l) ^ __float_as_uint(dv_r)) & 0x80000000u) == 0u;
  return same ? copysignf(m, dv_l) : 0.0f;
}

// PLM_AthenaLimiter (EnzoReconstructorPLM.hpp:337-345)
template <typename T>
__device__ __forceinline__ T limiter_athena(T vm1, T v, T vp1) {
  T dv_l = (v - vm1);
  T dv_r = (vp1 - v);
  T temp = dv_l * dv_r;
  if (temp <= T(0)) return T(0);
  return qdiv(T(2) * temp, dv_l + dv_r);
}

// EnzoEOSIdeal::fast_magnetosonic_speed<-1> (EnzoEOSIdeal.hpp:111-140) of
// the two states of a face, side by side; std::pow(x, 2) == x*x exactly.
// w in the MHD LUT order.
template <class O, typename T>
__device__ __forceinline__ void fast_ms_speeds(const T wl[8], const T wr[8], T gamma, T &cl,
                                               T &cr) {
  const T *w[2] = {wl, wr};
  T sum[2], rad[2], rt[2];
#pragma unroll
  for (int s = 0; s < 2; s++) {
    const T d = w[s][L_D], bi = w[s][L_BI], bj = w[s][L_BJ], bk = w[s][L_BK];
    const T B2 = mad(bi, bi, dot2<O::kj>(bj, bj, bk, bk));
    const T inv_density = qrcp(d);
    const T cs2 = qdiv_inv(gamma * w[s][L_E], d, inv_density);
    const T va2_cos2 = (bi * bi) * inv_density;
    sum[s] = mad(B2, inv_density, cs2);  // va2 + cs2
    rad[s] = msub(sum[s], sum[s], T(4) * cs2 * va2_cos2);
  }
  qsqrt2(rad[0], rad[1], rt[0], rt[1]);
  qsqrt2(T(0.5) * (sum[0] + rt[0]), T(0.5) * (sum[1] + rt[1]), cl, cr);
}

template <typename T> struct Cons1D { T d, mx, my, mz, e, by, bz; };

// enzo_riemann_utils::passive_eint_flux (EnzoRiemannUtils.hpp:224-249),
// dual-energy formalism: the specific internal energy p / ((gamma-1) rho)
// of the side the density flux comes from, selected branch-free as the
// reference writes it, times the density flux.  Split in two: the specific
// energies (EnzoEOSIdeal::specific_eint, EnzoEOSIdeal.hpp:79-82) depend on
// the face states only, so the flux kernel evaluates them before the solve
// and keeps two values live through it instead of four.
template <typename T>
__device__ __forceinline__ T specific_eint(T density, T pressure, T gamma) {
  return qdiv(pressure, (gamma - T(1)) * density);
}
template <typename T>
__device__ __forceinline__ T upwind_eint_flux(T eint_l, T eint_r, T density_flux) {
  const T upwind = T(density_flux > T(0)) * eint_l + T(density_flux <= T(0)) * eint_r;
  return upwind * density_flux;
}

// HLLD (Miyoshi & Kusano 2005) following HLLDKernel::operator()
// (src/Enzo/hydro-mhd/riemann/EnzoRiemannHLLD.hpp:40-404).  In/out in the
// MHD LUT order; flux[L_BI] is 0.  vbar (dual energy, may be null): the
// interface velocity of :418-447 -- the left/right normal velocity outside
// the fan, else the contact speed scaled by the outer state's coefficient.
// igm1: 1 / (gamma - 1), the same for every face of a launch.
template <class O = SumOrder<0, false, false>, typename T>
__device__ __forceinline__ void hlld(const T wli[8], const T wri[8], T gamma, T igm1,
                                     T flx[8], T *vbar = nullptr) {
  const T SMALL_NUMBER = T(1.0e-8);
  T spd[5];
  Cons1D<T> ul, ur, ulst, uldst, urdst, urst, fl, fr;
  // the outer states' physical fluxes are formed where the fan region is
  // selected: held from the start they would stay live through the whole
  // solve

  const T pressure_l = wli[L_E];
  const T pressure_r = wri[L_E];
  const T bxi = wli[L_BI];

  T bxsq = bxi * bxi;
  const T bsql = mad(bxi, bxi, dot2<O::kj>(wli[L_BJ], wli[L_BJ], wli[L_BK], wli[L_BK]));
  const T bsqr = mad(bxi, bxi, dot2<O::kj>(wri[L_BJ], wri[L_BJ], wri[L_BK], wri[L_BK]));
  T pbl = T(0.5) * bsql;
  T pbr = T(0.5) * bsqr;
  const T v2l = mad(wli[L_VI], wli[L_VI], dot2<O::kj>(wli[L_VJ], wli[L_VJ], wli[L_VK], wli[L_VK]));
  const T v2r = mad(wri[L_VI], wri[L_VI], dot2<O::kj>(wri[L_VJ], wri[L_VJ], wri[L_VK], wri[L_VK]));

  ul.d = wli[L_D];
  ul.mx = wli[L_VI] * ul.d;
  ul.my = wli[L_VJ] * ul.d;
  ul.mz = wli[L_VK] * ul.d;
  ul.e = dot2<O::energy>(pressure_l, igm1, T(0.5) * wli[L_D], v2l) + pbl;
  ul.by = wli[L_BJ];
  ul.bz = wli[L_BK];

  ur.d = wri[L_D];
  ur.mx = wri[L_VI] * ur.d;
  ur.my = wri[L_VJ] * ur.d;
  ur.mz = wri[L_VK] * ur.d;
  ur.e = dot2<O::energy>(pressure_r, igm1, T(0.5) * wri[L_D], v2r) + pbr;
  ur.by = wri[L_BJ];
  ur.bz = wri[L_BK];

  T cfl, cfr;
  fast_ms_speeds<O>(wli, wri, gamma, cfl, cfr);

  spd[0] = dmin(wli[L_VI] - cfl, wri[L_VI] - cfr);
  spd[4] = dmax(wli[L_VI] + cfl, wri[L_VI] + cfr);

  T ptl = add_mul(pressure_l, T(0.5), bsql);
  T ptr = add_mul(pressure_r, T(0.5), bsqr);

  T sdl = spd[0] - wli[L_VI];
  T sdr = spd[4] - wri[L_VI];
  const Quotient<T> sm(msub(sdr, ur.mx, sdl * ul.mx) + (ptl - ptr),
                       msub(sdr, ur.d, sdl * ul.d));
  spd[2] = sm.q;

  T sdml = sm.from(spd[0]);
  T sdmr = spd[4] - spd[2];
  T sdml_inv = qrcp(sdml);
  T sdmr_inv = qrcp(sdmr);
  if (vbar) {
    // as soon as the outer and contact speeds are known (fewer live
    // registers through the rest of the solve): l_coef = (S_l - vx_L) /
    // (S_l - S_M) = sdl / sdml, r_coef = sdr / sdmr
    const T l_coef = qdiv_inv(sdl, sdml, sdml_inv);
    const T r_coef = qdiv_inv(sdr, sdmr, sdmr_inv);
    if (spd[0] > T(0)) {
      *vbar = wli[L_VI];
    } else if (spd[4] < T(0)) {
      *vbar = wri[L_VI];
    } else if (spd[2] >= T(0)) {
      *vbar = spd[2] * l_coef;
    } else {
      *vbar = spd[2] * r_coef;
    }
  }
  ulst.d = ul.d * sdl * sdml_inv;
  urst.d = ur.d * sdr * sdmr_inv;
  T ulst_d_inv = qrcp(ulst.d);
  T urst_d_inv = qrcp(urst.d);
  T sqrtdl, sqrtdr;
  qsqrt2(ulst.d, urst.d, sqrtdl, sqrtdr);

  spd[1] = sub_div(spd[2], fabs(bxi), sqrtdl);
  spd[3] = add_div(spd[2], fabs(bxi), sqrtdr);

  T ptstl = add_mul(ptl, ul.d * sdl, sm.minus(wli[L_VI]));
  T ptstr = add_mul(ptr, ur.d * sdr, sm.minus(wri[L_VI]));
  T ptst = T(0.5) * (ptstr + ptstl);

  // the transverse star states of both sides, side by side, then the rare
  // side whose Alfven wave sits on the outer one
  ulst.mx = ulst.d * spd[2];
  urst.mx = urst.d * spd[2];
  {
    const T denl = msub(ul.d * sdl, sdml, bxsq), denr = msub(ur.d * sdr, sdmr, bxsq);
    const T denl_inv = qrcp(denl), denr_inv = qrcp(denr);
    T tmpl = qdiv_inv(bxi * (sdl - sdml), denl, denl_inv);
    T tmpr = qdiv_inv(bxi * (sdr - sdmr), denr, denr_inv);
    ulst.my = ulst.d * sub_mul(wli[L_VJ], ul.by, tmpl);
    ulst.mz = ulst.d * sub_mul(wli[L_VK], ul.bz, tmpl);
    urst.my = urst.d * sub_mul(wri[L_VJ], ur.by, tmpr);
    urst.mz = urst.d * sub_mul(wri[L_VK], ur.bz, tmpr);
    tmpl = qdiv_inv(msub(ul.d, sdl * sdl, bxsq), denl, denl_inv);
    tmpr = qdiv_inv(msub(ur.d, sdr * sdr, bxsq), denr, denr_inv);
    ulst.by = ul.by * tmpl;
    ulst.bz = ul.bz * tmpl;
    urst.by = ur.by * tmpr;
    urst.bz = ur.bz * tmpr;
    const bool flat_l = fabs(denl) < (SMALL_NUMBER)*ptst;
    const bool flat_r = fabs(denr) < (SMALL_NUMBER)*ptst;
    if (__builtin_expect(flat_l || flat_r, 0)) {
      if (flat_l) {
        ulst.my = ulst.d * wli[L_VJ];
        ulst.mz = ulst.d * wli[L_VK];
        ulst.by = ul.by;
        ulst.bz = ul.bz;
      }
      if (flat_r) {
        urst.my = urst.d * wri[L_VJ];
        urst.mz = urst.d * wri[L_VK];
        urst.by = ur.by;
        urst.bz = ur.bz;
      }
    }
  }
  const T mbstl = mad(ulst.mx, bxi, mad(ulst.my, ulst.by, ulst.mz * ulst.bz));
  T vbstl = mbstl * ulst_d_inv;
  const T vbl = dot2<O::kj>(wli[L_VJ], ul.by, wli[L_VK], ul.bz);
  ulst.e = add_mul(add_mul(msub(sdl, ul.e, ptl * wli[L_VI]), ptst, spd[2]), bxi,
                   sub_mul(mad(wli[L_VI], bxi, vbl), mbstl, ulst_d_inv)) *
           sdml_inv;
  const T mbstr = mad(urst.mx, bxi, mad(urst.my, urst.by, urst.mz * urst.bz));
  T vbstr = mbstr * urst_d_inv;
  const T vbr = dot2<O::kj>(wri[L_VJ], ur.by, wri[L_VK], ur.bz);
  urst.e = add_mul(add_mul(msub(sdr, ur.e, ptr * wri[L_VI]), ptst, spd[2]), bxi,
                   sub_mul(mad(wri[L_VI], bxi, vbr), mbstr, urst_d_inv)) *
           sdmr_inv;

  if (T(0.5) * bxsq < (SMALL_NUMBER)*ptst) {
    uldst = ulst;
    urdst = urst;
  } else {
    T invsumd = qrcp(sqrtdl + sqrtdr);
    T bxsig = (bxi > T(0) ? T(1) : T(-1));
    uldst.d = ulst.d;
    urdst.d = urst.d;
    uldst.mx = ulst.mx;
    urdst.mx = urst.mx;

    T tmp = invsumd * add_mul(mad(sqrtdl, ulst.my * ulst_d_inv, sqrtdr * (urst.my * urst_d_inv)),
                              bxsig, urst.by - ulst.by);
    uldst.my = uldst.d * tmp;
    urdst.my = urdst.d * tmp;

    tmp = invsumd * add_mul(mad(sqrtdl, ulst.mz * ulst_d_inv, sqrtdr * (urst.mz * urst_d_inv)),
                            bxsig, urst.bz - ulst.bz);
    uldst.mz = uldst.d * tmp;
    urdst.mz = urdst.d * tmp;

    tmp = invsumd * add_mul(add_mul(sqrtdl * urst.by, sqrtdr, ulst.by),
                            bxsig * sqrtdl * sqrtdr,
                            msub(urst.my, urst_d_inv, ulst.my * ulst_d_inv));
    uldst.by = urdst.by = tmp;

    tmp = invsumd * add_mul(add_mul(sqrtdl * urst.bz, sqrtdr, ulst.bz),
                            bxsig * sqrtdl * sqrtdr,
                            msub(urst.mz, urst_d_inv, ulst.mz * ulst_d_inv));
    uldst.bz = urdst.bz = tmp;

    tmp = mad(spd[2], bxi,
              qdiv_inv(mad(uldst.my, uldst.by, uldst.mz * uldst.bz), uldst.d, ulst_d_inv));
    uldst.e = sub_mul(ulst.e, sqrtdl * bxsig, vbstl - tmp);
    urdst.e = add_mul(urst.e, sqrtdr * bxsig, vbstr - tmp);
  }

  auto flux_l = [&]() {
    fl.d = ul.mx;
    fl.mx = mad(ul.mx, wli[L_VI], ptl) - bxsq;
    fl.my = msub(ul.my, wli[L_VI], bxi * ul.by);
    fl.mz = msub(ul.mz, wli[L_VI], bxi * ul.bz);
    fl.e = msub(wli[L_VI], ul.e + ptl - bxsq, bxi * vbl);
    fl.by = msub(ul.by, wli[L_VI], bxi * wli[L_VJ]);
    fl.bz = msub(ul.bz, wli[L_VI], bxi * wli[L_VK]);
  };
  auto flux_r = [&]() {
    fr.d = ur.mx;
    fr.mx = mad(ur.mx, wri[L_VI], ptr) - bxsq;
    fr.my = msub(ur.my, wri[L_VI], bxi * ur.by);
    fr.mz = msub(ur.mz, wri[L_VI], bxi * ur.bz);
    fr.e = msub(wri[L_VI], ur.e + ptr - bxsq, bxi * vbr);
    fr.by = msub(ur.by, wri[L_VI], bxi * wri[L_VJ]);
    fr.bz = msub(ur.bz, wri[L_VI], bxi * wri[L_VK]);
  };
  // Select the region of the fan containing the interface; the state
  // differences of each wave are formed lazily (only the ones used).
  if (spd[0] >= T(0)) {
    flux_l();
    flx[L_D] = fl.d; flx[L_VI] = fl.mx; flx[L_VJ] = fl.my; flx[L_VK] = fl.mz;
    flx[L_E] = fl.e; flx[L_BJ] = fl.by; flx[L_BK] = fl.bz;
  } else if (spd[4] <= T(0)) {
    flux_r();
    flx[L_D] = fr.d; flx[L_VI] = fr.mx; flx[L_VJ] = fr.my; flx[L_VK] = fr.mz;
    flx[L_E] = fr.e; flx[L_BJ] = fr.by; flx[L_BK] = fr.bz;
  } else if (spd[1] >= T(0)) {
    flux_l();
    flx[L_D] = add_mul(fl.d, spd[0], ulst.d - ul.d);
    flx[L_VI] = add_mul(fl.mx, spd[0], ulst.mx - ul.mx);
    flx[L_VJ] = add_mul(fl.my, spd[0], ulst.my - ul.my);
    flx[L_VK] = add_mul(fl.mz, spd[0], ulst.mz - ul.mz);
    flx[L_E] = add_mul(fl.e, spd[0], ulst.e - ul.e);
    flx[L_BJ] = add_mul(fl.by, spd[0], ulst.by - ul.by);
    flx[L_BK] = add_mul(fl.bz, spd[0], ulst.bz - ul.bz);
  } else if (spd[2] >= T(0)) {
    flux_l();
    flx[L_D] = add_mul(add_mul(fl.d, spd[0], ulst.d - ul.d), spd[1], uldst.d - ulst.d);
    flx[L_VI] = add_mul(add_mul(fl.mx, spd[0], ulst.mx - ul.mx), spd[1], uldst.mx - ulst.mx);
    flx[L_VJ] = add_mul(add_mul(fl.my, spd[0], ulst.my - ul.my), spd[1], uldst.my - ulst.my);
    flx[L_VK] = add_mul(add_mul(fl.mz, spd[0], ulst.mz - ul.mz), spd[1], uldst.mz - ulst.mz);
    flx[L_E] = add_mul(add_mul(fl.e, spd[0], ulst.e - ul.e), spd[1], uldst.e - ulst.e);
    flx[L_BJ] = add_mul(add_mul(fl.by, spd[0], ulst.by - ul.by), spd[1], uldst.by - ulst.by);
    flx[L_BK] = add_mul(add_mul(fl.bz, spd[0], ulst.bz - ul.bz), spd[1], uldst.bz - ulst.bz);
  } else if (spd[3] > T(0)) {
    flux_r();
    flx[L_D] = add_mul(add_mul(fr.d, spd[4], urst.d - ur.d), spd[3], urdst.d - urst.d);
    flx[L_VI] = add_mul(add_mul(fr.mx, spd[4], urst.mx - ur.mx), spd[3], urdst.mx - urst.mx);
    flx[L_VJ] = add_mul(add_mul(fr.my, spd[4], urst.my - ur.my), spd[3], urdst.my - urst.my);
    flx[L_VK] = add_mul(add_mul(fr.mz, spd[4], urst.mz - ur.mz), spd[3], urdst.mz - urst.mz);
    flx[L_E] = add_mul(add_mul(fr.e, spd[4], urst.e - ur.e), spd[3], urdst.e - urst.e);
    flx[L_BJ] = add_mul(add_mul(fr.by, spd[4], urst.by - ur.by), spd[3], urdst.by - urst.by);
    flx[L_BK] = add_mul(add_mul(fr.bz, spd[4], urst.bz - ur.bz), spd[3], urdst.bz - urst.bz);
  } else {
    flux_r();
    flx[L_D] = add_mul(fr.d, spd[4], urst.d - ur.d);
    flx[L_VI] = add_mul(fr.mx, spd[4], urst.mx - ur.mx);
    flx[L_VJ] = add_mul(fr.my, spd[4], urst.my - ur.my);
    flx[L_VK] = add_mul(fr.mz, spd[4], urst.mz - ur.mz);
    flx[L_E] = add_mul(fr.e, spd[4], urst.e - ur.e);
    flx[L_BJ] = add_mul(fr.by, spd[4], urst.by - ur.by);
    flx[L_BK] = add_mul(fr.bz, spd[4], urst.bz - ur.bz);
  }
  flx[L_BI] = T(0);
}

// conserved state + physical flux, MHD LUT (EnzoRiemannUtils.hpp:48-149)
template <class O, typename T>
__device__ __forceinline__ void mhd_cons_flux(const T w[8], T gamma, T cons[8],
                                              T flux[8]) {
  for (int i = 0; i < 4; i++) cons[i] = w[i];
  for (int i = 4; i < 8; i++) cons[i] = w[i] * w[L_D];
  {
    T density = w[L_D];
    const T vi = w[L_VI], vj = w[L_VJ], vk = w[L_VK];
    const T v2 = mad(vi, vi, dot2<O::kj>(vj, vj, vk, vk));
    const T gm1 = gamma - T(1);
    // with the magnetic energy density
    cons[L_E] = add_mul(energy_density<O::energy>(w[L_E], gm1, qrcp(gm1), T(0.5) * density, v2),
                        T(0.5),
                        mad(w[L_BI], w[L_BI], dot2<O::kj>(w[L_BJ], w[L_BJ], w[L_BK], w[L_BK])));
  }
  const T vi = w[L_VI], vj = w[L_VJ], vk = w[L_VK];
  const T Bi = w[L_BI], Bj = w[L_BJ], Bk = w[L_BK];
  const T etot = cons[L_E];
  const T ptot = add_mul(w[L_E], T(0.5), mad(Bi, Bi, dot2<O::kj>(Bj, Bj, Bk, Bk)));
  const T mom_i = cons[L_VI];
  flux[L_D] = mom_i;
  flux[L_VI] = msub(mom_i, vi, Bi * Bi) + ptot;
  flux[L_VJ] = msub(mom_i, vj, Bj * Bi);
  flux[L_VK] = msub(mom_i, vk, Bk * Bi);
  flux[L_E] = msub(etot + ptot, vi, mad(Bi, vi, dot2<O::kj>(Bj, vj, Bk, vk)) * Bi);
  flux[L_BI] = T(0);
  flux[L_BJ] = msub(Bj, vi, Bi * vj);
  flux[L_BK] = msub(Bk, vi, Bi * vk);
}

// HLLE for MHD: HLLKernel<EinfeldtWavespeed<MHDLUT>>
// (EnzoRiemannHLL.hpp:44-172, 238-320); vbar (dual energy, may be null):
// the normal velocity interpolated between the outer speeds (:330-340)
template <class O = SumOrder<0, false, false>, typename T>
__device__ __forceinline__ void hlle_mhd(const T wl[8], const T wr[8],
                                         T gamma, T flux[8],
                                         T *vbar = nullptr) {
  T cl[8], cr[8], fl[8], fr[8];
  mhd_cons_flux<O>(wl, gamma, cl, fl);
  mhd_cons_flux<O>(wr, gamma, cr, fr);
  T c_l, c_r;
  fast_ms_speeds<O>(wl, wr, gamma, c_l, c_r);
  T left_speed = (wl[L_VI] - c_l);
  T right_speed = (wr[L_VI] + c_r);
  T sqrtrho_l, sqrtrho_r;
  qsqrt2(wl[L_D], wr[L_D], sqrtrho_l, sqrtrho_r);
  T inv_sqrtrho_tot = qrcp(sqrtrho_l + sqrtrho_r);
  const T vi_sum = dot2<O::rl>(sqrtrho_l, wl[L_VI], sqrtrho_r, wr[L_VI]);
  T vi_roe = vi_sum * inv_sqrtrho_tot;
  T vj_roe = dot2<O::rl>(sqrtrho_l, wl[L_VJ], sqrtrho_r, wr[L_VJ]) * inv_sqrtrho_tot;
  T vk_roe = dot2<O::rl>(sqrtrho_l, wl[L_VK], sqrtrho_r, wr[L_VK]) * inv_sqrtrho_tot;
  T v_roe2 = add_mul(dot2<O::ji_roe>(vi_roe, vi_roe, vj_roe, vj_roe), vk_roe, vk_roe);
  const T ptot_l = add_mul(wl[L_E], T(0.5),
                           mad(wl[L_BI], wl[L_BI], dot2<O::kj>(wl[L_BJ], wl[L_BJ], wl[L_BK], wl[L_BK])));
  const T ptot_r = add_mul(wr[L_E], T(0.5),
                           mad(wr[L_BI], wr[L_BI], dot2<O::kj>(wr[L_BJ], wr[L_BJ], wr[L_BK], wr[L_BK])));
  T h_l = qdiv_inv(cl[L_E] + ptot_l, wl[L_D], qrcp(wl[L_D]));
  T h_r = qdiv_inv(cr[L_E] + ptot_r, wr[L_D], qrcp(wr[L_D]));
  const T h_sum = mad(sqrtrho_l, h_l, sqrtrho_r * h_r);
  // roe_cfast_
  T rho_roe = sqrtrho_l * sqrtrho_r;
  T rho_roe_inv = qrcp(rho_roe);
  T bi_roe = wl[L_BI];
  T bj_roe = add_mul(sqrtrho_l * wr[L_BJ], sqrtrho_r, wl[L_BJ]) * inv_sqrtrho_tot;
  T bk_roe = add_mul(sqrtrho_l * wr[L_BK], sqrtrho_r, wl[L_BK]) * inv_sqrtrho_tot;
  T b_roe2 = add_mul(add_mul(bi_roe * bi_roe, bj_roe, bj_roe), bk_roe, bk_roe);
  T gamma_prime = gamma - T(1);
  T dbj = wl[L_BJ] - wr[L_BJ];
  T dbk = wl[L_BK] - wr[L_BK];
  T x_prime =
      (dot2<O::kj>(dbj, dbj, dbk, dbk) * T(0.5) * (gamma_prime - T(1)) * inv_sqrtrho_tot);
  // gamma_prime - y_prime
  const T gy = sub_div(gamma_prime, (gamma_prime - T(1)) * (wl[L_D] + wr[L_D]) * T(0.5), rho_roe,
                       rho_roe_inv);
  // (h_roe - v_roe2 / 2 first)
  T tilde_a2 = msub(gamma_prime,
                    sub_div(msub(h_sum, inv_sqrtrho_tot, T(0.5) * v_roe2), b_roe2, rho_roe,
                            rho_roe_inv),
                    x_prime);
  T tilde_vai2 = qdiv_inv(bi_roe * bi_roe, rho_roe, rho_roe_inv);
  T tilde_va2 = add_div(tilde_vai2, gy * dot2<O::kj_roe>(bj_roe, bj_roe, bk_roe, bk_roe), rho_roe,
                        rho_roe_inv);
  T s = tilde_a2 + tilde_va2;
  T c_roe = qsqrt(T(0.5) * (s + qsqrt(msub(s, s, T(4) * tilde_a2 * tilde_vai2))));
  T bp = fmax(mad(vi_sum, inv_sqrtrho_tot, c_roe), right_speed);
  T bm = fmin(msub(vi_sum, inv_sqrtrho_tot, c_roe), left_speed);
  bp = fmax(bp, T(0));
  bm = fmin(bm, T(0));
  T inv_speed_diff = qrcp(bp - bm);
#pragma unroll
  for (int f = 0; f < 8; f++) {
    const bool mom = f == L_VI || f == L_VJ || f == L_VK;
    const T diff = mom ? msub(wr[f], wr[L_D], cl[f]) : cr[f] - cl[f];
    flux[f] = add_mul(msub(bp, fl[f], bm * fr[f]), diff * bp, bm) * inv_speed_diff;
  }
  if (vbar) *vbar = (bp * wl[L_VI] - bm * wr[L_VI]) * inv_speed_diff;
}

// HLLC (HLLCKernel::operator(), EnzoRiemannHLLC.hpp:34-172) with
// EinfeldtWavespeed<HydroLUT> (EnzoRiemannHLL.hpp:44-130).  Hydro LUT.
// vbar (dual energy, may be null): the weighted outer velocities of :166-170
template <class O = SumOrder<0, false, false>, typename T>
__device__ __forceinline__ void hllc(const T wl[5], const T wr[5], T gamma,
                                     T flux[5], T *vbar = nullptr) {
  const T pressure_l = wl[H_E];
  const T pressure_r = wr[H_E];
  T cons_l[5], cons_r[5];
  {
    const T *w[2] = {wl, wr};
    T *c[2] = {cons_l, cons_r};
#pragma unroll
    for (int s = 0; s < 2; s++) {
      c[s][H_D] = w[s][H_D];
      for (int i = 1; i < 5; i++) c[s][i] = w[s][i] * w[s][H_D];
      T density = w[s][H_D];
      const T vi = w[s][H_VI], vj = w[s][H_VJ], vk = w[s][H_VK];
      const T gm1 = gamma - T(1);
      c[s][H_E] = energy_density<O::energy>(w[s][H_E], gm1, qrcp(gm1), T(0.5) * density,
                                            mad(vi, vi, dot2<O::kj>(vj, vj, vk, vk))) + T(0);
    }
  }
  T cs_l, cs_r;
  {
    const T inv_l = qrcp(wl[H_D]), inv_r = qrcp(wr[H_D]);
    T c_l, c_r;
    qsqrt2(qdiv_inv(gamma * pressure_l, wl[H_D], inv_l),
           qdiv_inv(gamma * pressure_r, wr[H_D], inv_r), c_l, c_r);
    T left_speed = (wl[H_VI] - c_l);
    T right_speed = (wr[H_VI] + c_r);
    T sqrtrho_l, sqrtrho_r;
    qsqrt2(wl[H_D], wr[H_D], sqrtrho_l, sqrtrho_r);
    T inv_sqrtrho_tot = qrcp(sqrtrho_l + sqrtrho_r);
    const T vi_sum = dot2<O::rl>(sqrtrho_l, wl[H_VI], sqrtrho_r, wr[H_VI]);
    T vi_roe = vi_sum * inv_sqrtrho_tot;
    T vj_roe = dot2<O::rl>(sqrtrho_l, wl[H_VJ], sqrtrho_r, wr[H_VJ]) * inv_sqrtrho_tot;
    T vk_roe = dot2<O::rl>(sqrtrho_l, wl[H_VK], sqrtrho_r, wr[H_VK]) * inv_sqrtrho_tot;
    T v_roe2 = add_mul(dot2<O::ji_roe>(vi_roe, vi_roe, vj_roe, vj_roe), vk_roe, vk_roe);
    T h_l = qdiv_inv(cons_l[H_E] + pressure_l, wl[H_D], inv_l);
    T h_r = qdiv_inv(cons_r[H_E] + pressure_r, wr[H_D], inv_r);
    // h_roe - v_roe2 / 2
    T temp = msub(dot2<O::rl>(sqrtrho_l, h_l, sqrtrho_r, h_r), inv_sqrtrho_tot, T(0.5) * v_roe2);
    T c_roe = qsqrt((gamma - T(1)) * dmax(temp, T(0)));
    cs_r = fmax(mad(vi_sum, inv_sqrtrho_tot, c_roe), right_speed);
    cs_l = fmin(msub(vi_sum, inv_sqrtrho_tot, c_roe), left_speed);
  }
  T bm = fmin(cs_l, T(0));
  T bp = fmax(cs_r, T(0));
  T tl = sub_mul(pressure_l, (cs_l - wl[H_VI]) * wl[H_D], wl[H_VI]);
  T tr = sub_mul(pressure_r, (cs_r - wr[H_VI]) * wr[H_D], wr[H_VI]);
  T dl = wl[H_D] * (cs_l - wl[H_VI]);
  T dr = -wr[H_D] * (cs_r - wr[H_VI]);
  T q1 = qrcp(add_mul(dl, -wr[H_D], cs_r - wr[H_VI]));  // 1 / (dl + dr)
  T cw = (tr - tl) * q1;
  T cp = mad(dl, tr, dr * tl) * q1;
  T sl, sr, sm;
  {
    // the contact's side: its share of the outer flux, |cw| / (its distance
    // to the outer speed), and the middle state's
    const bool left = cw >= T(0);
    const T den = left ? cw - bm : bp - cw, den_inv = qrcp(den);
    const T share = qdiv_inv(left ? cw : -cw, den, den_inv);
    sl = left ? share : T(0);
    sr = left ? T(0) : share;
    sm = qdiv_inv(left ? -bm : bp, den, den_inv);
  }
  if (vbar) *vbar = (sl * (wl[H_VI] - bm) + sr * (wr[H_VI] - bp));
  cp = dmax(cp, T(0));
  T momentumi_l = cons_l[H_VI];
  T momentumi_r = cons_r[H_VI];
  T dfl = sub_mul(momentumi_l, bm, wl[H_D]);
  T dfr = sub_mul(momentumi_r, bp, wr[H_D]);
  T ufl = mad(momentumi_l, wl[H_VI] - bm, pressure_l);
  T ufr = mad(momentumi_r, wr[H_VI] - bp, pressure_r);
  T vfl = (wl[H_D] * wl[H_VJ] * (wl[H_VI] - bm));
  T vfr = (wr[H_D] * wr[H_VJ] * (wr[H_VI] - bp));
  T wfl = (wl[H_D] * wl[H_VK] * (wl[H_VI] - bm));
  T wfr = (wr[H_D] * wr[H_VK] * (wr[H_VI] - bp));
  T efl = add_mul(cons_l[H_E] * (wl[H_VI] - bm), pressure_l, wl[H_VI]);
  T efr = add_mul(cons_r[H_E] * (wr[H_VI] - bp), pressure_r, wr[H_VI]);
  flux[H_D] = add_mul(sl * dfl, sr, dfr);
  flux[H_VI] = add_mul(add_mul(sl * ufl, sr, ufr), sm, cp);
  flux[H_VJ] = add_mul(sl * vfl, sr, vfr);
  flux[H_VK] = add_mul(sl * wfl, sr, wfr);
  flux[H_E] = add_mul(add_mul(sl * efl, sr, efr), sm * cp, cw);
}

}  // namespace ENZOE_KNS
