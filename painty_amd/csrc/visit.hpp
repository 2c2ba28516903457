// The arithmetic of one imprint visit, shared by every stamp kernel.
//
// pickupPaint (renderer/FootprintBrush.hxx:349-384), then depositPaint
// (:393-431), with blend() (:331-340).  Storage is reached through an accessor
// so the kernels that keep the pickup map in global memory and the persistent
// one (map in LDS) execute the same instructions and produce the same bits.
#pragma once

#include <hip/hip_runtime.h>

namespace pnt {

// MinVolume = 0.001 (FootprintBrush.hxx:26).
constexpr double kMinVolume = 0.001;

// The arithmetic runs in FP64, as the reference's does (vec3 is Eigen's
// double vector): loads widen the stored FP32 values, every volume and
// threshold test is the reference's own expression in double precision, and
// each K/S result is rounded to FP32 once, when it is stored (canvas and
// snapshot volumes are stored in FP64).  Over the hundreds of dependent visits
// a pixel and a pickup cell take in a long stamp list, only that storage
// rounding accumulates (an FP32 chain would add the rounding of every
// intermediate step as well).
//
// blend(va, a, vb, b) = vt > MinVolume ? (va*a + vb*b) / vt : a with
// vt = va + vb (FootprintBrush.hxx:331-340) is not rounded step by step as
// there: its channels share the weights va/vt and vb/vt, through one
// reciprocal, two operations a channel (a product and a fused multiply-add).
// The result is within 5e-16 relative of the quotient, before it is rounded to
// FP32 for storage, and no volume or test depends on it.

// 1/v for a normal v > MinVolume: the hardware's estimate (2^-23 or better)
// and two Newton steps, within an ulp; no scaling for denormals or infinities.
__device__ __forceinline__ double rcpd(double v) {
  double r = __builtin_amdgcn_rcp(v);
  r = __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
}

__device__ __forceinline__ float rcpf(float x) { return __builtin_amdgcn_rcpf(x); }

// Accessor interface:
//   float pick(int c) / void set_pick(int c, float)   c = 0..2 K, 3..5 S, 6 V
//   float src(int c) (c < 6) / double src_v() / void set_src_v(double)
//                                                      pickup source (snapshot or canvas)
//   float canvas(int c) (c < 6) / double canvas_v()
//   void set_canvas(int c, float) (c < 6) / void set_canvas_v(double)
// Canvas and source volumes are FP64 in memory, so every volume that a
// MinVolume test sees is the reference's own number; contraction is off so
// that the volumes' products and sums round as the reference's do.
template <class Acc>
__device__ __forceinline__ void paint_visit_math(Acc& a, float fh_f, double pickup_rate,
                                                 double dep_rate, double cap, const float pK[3],
                                                 const float pS[3]) {
#pragma clang fp contract(off)
  const double fh = fh_f;
  {  // pickupPaint (FootprintBrush.hxx:349-384)
    const double vP = a.pick(6);
    const double vC = a.src_v();
    const double vLeave = (pickup_rate * vC) * fh;
    if (vLeave > kMinVolume) {
      a.set_src_v(vC - vLeave);
      const double vt = vP + vLeave;
      if (vt > kMinVolume) {
        const double iv = rcpd(vt), wP = vP * iv, wL = vLeave * iv;
        double nv[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) nv[c] = __builtin_fma(wP, a.pick(c), wL * a.src(c));
#pragma unroll
        for (int c = 0; c < 6; ++c) a.set_pick(c, (float)nv[c]);
      }
      a.set_pick(6, (float)(vP + vLeave));
    }
  }
  {  // depositPaint (FootprintBrush.hxx:393-431)
    const double vP = a.pick(6);
    const double vFree = fmax(0.0, cap - vP);
    double src[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) src[c] = a.pick(c);
    const double vt = vP + vFree;
    if (vt > kMinVolume) {
      const double iv = rcpd(vt), wP = vP * iv, wF = vFree * iv;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        src[c] = __builtin_fma(wP, src[c], wF * (double)pK[c]);
        src[3 + c] = __builtin_fma(wP, src[3 + c], wF * (double)pS[c]);
      }
    }
    a.set_pick(6, (float)(vP - (dep_rate * vP) * fh));
    const double vC = a.canvas_v();
    const double vB = cap * fh;
    const double vt2 = vB + vC;
    if (vt2 > kMinVolume) {
      const double iv = rcpd(vt2), wB = vB * iv, wC = vC * iv;
      double nv[6];
#pragma unroll
      for (int c = 0; c < 6; ++c) nv[c] = __builtin_fma(wB, src[c], wC * a.canvas(c));
#pragma unroll
      for (int c = 0; c < 6; ++c) a.set_canvas(c, (float)nv[c]);
    } else {
#pragma unroll
      for (int c = 0; c < 6; ++c) a.set_canvas(c, (float)src[c]);
    }
    a.set_canvas_v(vB + vC);
  }
}

}  // namespace pnt
