// tt06_exact.hpp -- configuration A of the TT06Dev reaction on gfx950: the
// exact TT06 voltage functions instead of rational fits.
//
// REACTION_FACTORY(TT06Dev) defaults to tolerance = 0 (elec/TT06Dev_Reaction.cc:600-602);
// then padeApprox keeps each function itself (elec/pade.cc:237-268), the
// reaction runs the generic gate update TT06Func::updateGate
// (elec/TT06Func.cc:64-161: Rush-Larsen with exp for m, dt*(mhu - g)*tauR for
// the others, every cell of the group) and the generic non-gate update with
// fv0..fv6 (elec/TT06NonGates.c:319-364).  mod = 1 (jhTauSmooth) swaps the h
// and j rates for their smoothed forms (TauRecipMod, elec/TT06Tau.cc:131-151):
// a cubic Hermite bridge on [x0, x1], whose coefficients the host computes.
//
// Every expression keeps the reference's operation order and the including
// translation unit is compiled without contraction, so results differ from
// the reference's x86 build only where the exponentials here and the device's
// log and sqrt round differently from glibc's (a few ulps).
#pragma once

#include <hip/hip_runtime.h>

#include "tt06_f64.hpp"

namespace cdh {

// The functions' exponents and quotients.
//
// An exponential takes 19 instructions here: n = rint(x / ln 2), the rest r
// by two FMAs (Cody and Waite), exp(r) = 1 + r (1 + r q(r)) with q of degree
// 10 (its interpolation at the Chebyshev nodes of [-ln 2 / 2, ln 2 / 2];
// 3e-19 relative), and the scaling by 2^n, which gives infinity or 0 past the
// range.  Against quadruple precision it is off by 0.257 ulp in the mean and
// 0.856 at most (20 million arguments drawn from [-30, 30]); the device
// library's mean is 0.258.  The library's takes some 25, six of them to catch arguments past the range
// one by one.  Here the voltage is clamped once per cell instead, to +-1e7,
// where every one of the functions below has long reached the value it has at
// infinity; NaN stays NaN.
//
// A quotient by a literal multiplies by the literal's reciprocal and corrects
// once (Markstein): 3 instructions, correctly rounded, for finite dividends.
//
// With these and div64 the drop-in reaction with the exact functions takes 31
// us for 300,007 cells (39 before) and 556 for 6.7 million (679), the fused
// step of 512,000 cells 48.8 us (59.7).
template <class ET>
struct ExactMath {
   ET *E;
   // |x| < 1e12 or NaN
   __device__ __forceinline__ double ex(double x) const
   {
      const double n = rint(mul_vs(x, E->ex[0]));
      double r = __builtin_fma(n, E->ex[1], x);
      r = __builtin_fma(n, E->ex[2], r);
      const double q = horner64<3, 13, true>(E->ex, r);
      return ldexp(__builtin_fma(r, __builtin_fma(r, q, 1.0), 1.0), exponent(n));
   }
   // n as an integer, the nearest one past an int's range (n reaches 6e11) and 0
   // for NaN, as the instruction converts; the language leaves those undefined
   __device__ __forceinline__ static int exponent(double n)
   {
      int i;
      asm("v_cvt_i32_f64 %0, %1" : "=v"(i) : "v"(n));
      return i;
   }
   __device__ __forceinline__ static double clamp(double V)
   {
      V = V > 1e7 ? 1e7 : V;
      return V < -1e7 ? -1e7 : V;
   }
};

// a / c for a literal c
__device__ __forceinline__ double over(double a, double c)
{
   const double rc = 1.0 / c;
   const double q = a * rc;
   return __builtin_fma(__builtin_fma(-c, q, a), rc, q);
}

// Gate steady states and rates, elec/TT06Func.cc:261-417, at a clamped V.
template <class ET>
struct ExactGates : ExactMath<ET> {
   using ExactMath<ET>::ex;
   __device__ __forceinline__ static double inv(double x) { return div64(1.0, x); }
   __device__ __forceinline__ static double sq(double x) { return x * x; }

   __device__ __forceinline__ double mMhu(double V) const { return inv(sq(1.0 + ex(over(-56.8600 - V, 9.03000)))); }
   __device__ __forceinline__ double mTauR(double V) const
   {
      const double t1 = inv(1.0 + ex(over(-60.0 - V, 5.0)));
      const double t2 = div64(0.10000, 1.0 + ex(over(V + 35.0, 5.0))) +
                        div64(0.100000, 1.0 + ex(over(V - 50.0, 200.0)));
      return inv(t1 * t2);
   }
   __device__ __forceinline__ double hjMhu(double V) const { return inv(sq(1.0 + ex(over(V + 71.5500, 7.43000)))); }
   __device__ __forceinline__ double hTauR(double V) const
   {
      const double t1 = (V < -40.0 ? 0.0570000 * ex(over(-(V + 80.0), 6.80000)) : 0.0);
      const double t2 = (V < -40.0 ? 2.70000 * ex(0.0790000 * V) + 310000. * ex(0.348500 * V)
                                   : div64(0.770000, 0.130000 * (1.0 + ex(over(V + 10.6600, -11.1000)))));
      return t1 + t2;
   }
   __device__ __forceinline__ double jTauR(double V) const
   {
      const double t1 = (V < -40.0 ? div64((-25428.0 * ex(0.244400 * V) - 6.94800e-06 * ex(-0.0439100 * V)) *
                                               (V + 37.7800),
                                           1.0 + ex(0.311000 * (V + 79.2300)))
                                   : 0.0);
      const double t2 = (V < -40.0 ? div64(0.0242400 * ex(-0.0105200 * V), 1.0 + ex(-0.137800 * (V + 40.1400)))
                                   : div64(0.600000 * ex(0.0570000 * V), 1.0 + ex(-0.100000 * (V + 32.0))));
      return t1 + t2;
   }
   __device__ __forceinline__ double Xr1Mhu(double V) const { return inv(1.0 + ex(over(-26.0 - V, 7.0))); }
   __device__ __forceinline__ double Xr1TauR(double V) const
   {
      const double t1 = div64(1.0 + ex(over(-45.0 - V, 10.0)), 450.0);
      const double t2 = div64(1.0 + ex(over(V + 30.0, 11.5000)), 6.0);
      return t1 * t2;
   }
   __device__ __forceinline__ double Xr2Mhu(double V) const { return inv(1.0 + ex(over(V + 88.0, 24.0))); }
   __device__ __forceinline__ double Xr2TauR(double V) const
   {
      const double t1 = div64(1.0 + ex(over(-60.0 - V, 20.0)), 3.0);
      const double t2 = div64(1.0 + ex(over(V - 60.0, 20.0)), 1.120);
      return t1 * t2;
   }
   __device__ __forceinline__ double XsMhu(double V) const { return inv(1.0 + ex(over(-5.0 - V, 14.0))); }
   __device__ __forceinline__ double XsTauR(double V) const
   {
      const double t1 = div64(1400.00, sqrt(1.0 + ex(over(5.0 - V, 6.0))));
      const double t2 = inv(1.0 + ex(over(V - 35.0, 15.0)));
      return inv(t1 * t2 + 80.0);
   }
   __device__ __forceinline__ double rMhu(double V) const { return inv(1.0 + ex(over(20.0 - V, 6.0))); }
   __device__ __forceinline__ double rTauR(double V) const
   {
      return inv(9.50000 * ex(over(-sq(V + 40.0), 1800.00)) + 0.800000);
   }
   __device__ __forceinline__ double dMhu(double V) const { return inv(1.0 + ex(over(-8.0 - V, 7.50000))); }
   __device__ __forceinline__ double dTauR(double V) const
   {
      const double t1 = div64(1.40000, 1.0 + ex(over(-35.0 - V, 13.0))) + 0.250000;
      const double t2 = div64(1.40000, 1.0 + ex(over(V + 5.0, 5.0)));
      const double t3 = inv(1.0 + ex(over(50.0 - V, 20.0)));
      return inv(t1 * t2 + t3);
   }
   __device__ __forceinline__ double fMhu(double V) const { return inv(1.0 + ex(over(V + 20.0, 7.0))); }
   __device__ __forceinline__ double fTauR(double V) const
   {
      return inv(1102.50 * ex(over(-sq(V + 27.0), 225.0)) + div64(200.0, 1.0 + ex(over(13.0 - V, 10.0))) +
                 div64(180.0, 1.0 + ex(over(V + 30.0, 10.0))) + 20.0);
   }
   __device__ __forceinline__ double f2Mhu(double V) const { return div64(0.670000, 1.0 + ex(over(V + 35.0, 7.0))) + 0.330000; }
   __device__ __forceinline__ double f2TauR(double V) const
   {
      return inv(562.0 * ex(over(-sq(V + 27.0), 240.0)) + div64(31.0, 1.0 + ex(over(25.0 - V, 10.0))) +
                 div64(80.0, 1.0 + ex(over(V + 30.0, 10.0))));
   }
   __device__ __forceinline__ double jLMhu(double V) const { return ex(over(-(V + 91.0) * 2, 6.1)); }
   __device__ __forceinline__ double jLTauR(double) const { return 1.0 / 670.0; }
   __device__ __forceinline__ double sMhu0(double V) const { return inv(1.0 + ex(over(V + 28.0, 5.0))); }
   __device__ __forceinline__ double sMhu1(double V) const { return inv(1.00000 + ex(over(V + 20.0000, 5.00000))); }
   __device__ __forceinline__ double sTauR0(double V) const
   {
      return inv(1000.0 * ex(over(-sq(V + 67.0), 1000.0)) + 8.0);
   }
   __device__ __forceinline__ double sTauR1(double V) const
   {
      return inv(85.0000 * ex(over(-sq(V + 45.0000), 320.000)) +
                 div64(5.00000, 1.00000 + ex(over(V - 20.0000, 5.00000))) + 3.00000);
   }
};

// TauRecipMod with the host's cubic {x0, x1, c0..c3}: the cubic inside
// [x0, x1], the raw rate outside (elec/TT06Tau.cc:131-151)
template <class C>
__device__ __forceinline__ double smoothed(C h, double V, double raw)
{
   if (V < h[0] || V > h[1]) return raw;
   const double x = V - h[0];
   return h[2] + x * (h[3] + x * (h[4] + x * h[5]));
}

// fv0..fv6 exactly (elec/TT06NonGates.c:319-364)
template <class ET, class KT>
struct ExactVoltageFns : ExactMath<ET> {
   using ExactMath<ET>::E, ExactMath<ET>::ex, ExactMath<ET>::clamp;
   KT *K;
   __device__ __forceinline__ ExactVoltageFns(ET *e, KT *k) : ExactMath<ET>{e}, K(k) {}
   __device__ __forceinline__ void fv05(double V, double fv[6]) const
   {
      const double f1 = E->f1, Vc = clamp(V);
      const double expV1 = ex(-f1 * Vc);
      fv[0] = div64(E->f2, 1.0 + 0.1245 * ex(-0.1 * Vc * f1) + 0.0353 * expV1);
      {
         const double expV5 = ex(E->f5 * Vc);
         const double expV = expV5 * expV1;
         const double fva = div64(1.0, E->f3 + E->f4 * expV);
         fv[1] = expV5 * fva;
         fv[2] = expV * fva * E->f6;
      }
      {
         const double x = 2.0 * f1 * (V - 15.0), xc = 2.0 * f1 * (Vc - 15.0);
         const double x2 = x * x;
         fv[3] = x2 < 1e-4 ? (1 + 0.5 * x + x2 / 12.0 - x2 * x2 / 720) * E->f7a
                           : div64(E->f7a * x, 1.0 - ex(-xc));
         fv[4] = x2 < 1e-4 ? (1 - 0.5 * x + x2 / 12.0 - x2 * x2 / 720) * E->f9a
                           : div64(E->f9a * x, ex(xc) - 1.0);
      }
      fv[5] = div64(E->f10, 1.0 + ex(over(25.0 - Vc, 5.98)));
   }
   __device__ __forceinline__ double fv6(double dV0) const
   {
      const double d = clamp(dV0);
      const double xx = div64(3.0 * ex(0.0002 * d + 0.02) + ex(0.1 * d - 1.0), 1.0 + ex(-0.5 * d)) *
                        (10.0 + 10 * ex(0.06 * d - 12.0));
      return div64(K->c12, 1.0 + xx);
   }
};

template <class ET, class KT>
__device__ __forceinline__ ExactVoltageFns<ET, KT> exact_voltage_fns(ET *E, KT *K)
{
   return ExactVoltageFns<ET, KT>(E, K);
}

// TT06Func::updateGate (elec/TT06Func.cc:64-161) with the exact functions:
// every cell, m by Rush-Larsen, the others by g += dt*(mhu - g)*tauR.
// `gmask` (every bit set) puts each gate in a basic block of its own, as in
// gates64.
template <class ET>
__device__ __forceinline__ void gates_exact64(const ET &E, int s_switch, double dt,
                                              double V, double *st, uint32_t gmask)
{
   const ExactGates<const ET> g{&E};
   const double Vc = g.clamp(V);
   if (gmask & (1u << 0)) st[S_M] += (g.mMhu(Vc) - st[S_M]) * (1 - exp(-dt * g.mTauR(Vc)));
   if (gmask & (1u << 1)) {
      const double mhu = g.hjMhu(Vc);
      const double raw = g.hTauR(Vc);
      const double tauR = E.mod ? smoothed(E.hmod, V, raw) : raw;
      st[S_H] += dt * (mhu - st[S_H]) * tauR;
   }
   if (gmask & (1u << 2)) {
      const double mhu = g.hjMhu(Vc);
      const double raw = g.jTauR(Vc);
      const double tauR = E.mod ? smoothed(E.jmod, V, raw) : raw;
      st[S_J] += dt * (mhu - st[S_J]) * tauR;
   }
   if (gmask & (1u << 3)) st[S_XR1] += dt * (g.Xr1Mhu(Vc) - st[S_XR1]) * g.Xr1TauR(Vc);
   if (gmask & (1u << 4)) st[S_XR2] += dt * (g.Xr2Mhu(Vc) - st[S_XR2]) * g.Xr2TauR(Vc);
   if (gmask & (1u << 5)) st[S_XS] += dt * (g.XsMhu(Vc) - st[S_XS]) * g.XsTauR(Vc);
   if (gmask & (1u << 6)) st[S_R] += dt * (g.rMhu(Vc) - st[S_R]) * g.rTauR(Vc);
   if (gmask & (1u << 7)) st[S_D] += dt * (g.dMhu(Vc) - st[S_D]) * g.dTauR(Vc);
   if (gmask & (1u << 8)) st[S_F] += dt * (g.fMhu(Vc) - st[S_F]) * g.fTauR(Vc);
   if (gmask & (1u << 9)) st[S_F2] += dt * (g.f2Mhu(Vc) - st[S_F2]) * g.f2TauR(Vc);
   if (gmask & (1u << 10)) st[S_JL] += dt * (g.jLMhu(Vc) - st[S_JL]) * g.jLTauR(Vc);
   if (gmask & (1u << 11)) {
      if (s_switch) st[S_S] += dt * (g.sMhu1(Vc) - st[S_S]) * g.sTauR1(Vc);
      else          st[S_S] += dt * (g.sMhu0(Vc) - st[S_S]) * g.sTauR0(Vc);
   }
}

}  // namespace cdh
