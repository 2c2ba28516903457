// Display output: Renderer::render (renderer/Renderer.hxx:60-156) -- the
// composite lit by a point light with a Beckmann / Cook-Torrance specular
// term over the height field of the wet layer's thickness V -- and the pixel
// transform of io::imSave (io/src/ImageIO.cxx:158-183): linear -> sRGB and
// quantisation to 8 or 16 bits.
//
// Both are per-pixel.  render reads K, S, V, R0 (44 B) and writes R (12 B);
// the four V neighbours come from the caches.  It is bound by its FP32
// arithmetic beside those bytes: 42 us at 1920 x 1080 with a 64-bit division
// for the pixel's row, three IEEE divisions per normalisation and the
// identities below left in, 23 without (23 us of bytes at copy rate).
// encode reads 12 B and writes 3 or 6 B per pixel: 41 us with FP64 pow and
// single-byte stores, 13 (6 us of bytes) with the root below, four pixels
// a thread.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.hpp"
#include "km.hpp"

namespace pnt {
namespace {

constexpr int kBlock = 256;
constexpr float kPiF = 3.14159265358979323846f;  // Math.hxx:21-22

// cv::borderInterpolate(p, len, BORDER_REFLECT) for p in [-1, len] (the
// default border of Interpolate, image/Mat.hxx:69-71); at integer positions
// Interpolate returns the bordered pixel itself.
__device__ __forceinline__ int reflect_index(int p, int len) {
  if (len == 1) return 0;
  if (p < 0) return -p - 1;
  if (p >= len) return 2 * len - p - 1;
  return p;
}

struct F3 {
  float x, y, z;
};
__device__ __forceinline__ float dot3(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
// 1/x and 1/sqrt(x) of normal x > 0: the hardware's estimate and one Newton
// step, within an ulp.
__device__ __forceinline__ float rcp1(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ float rsq1(float x) {
  const float r = __builtin_amdgcn_rsqf(x);
  return __builtin_fmaf(0.5f * r, __builtin_fmaf(-x * r, r, 1.0f), r);
}
// Eigen's normalized() of a nonzero vector.
__device__ __forceinline__ F3 unit3(F3 a) {
  const float r = rsq1(dot3(a, a));
  return F3{a.x * r, a.y * r, a.z * r};
}

struct RenderArgs {
  Layer7 L;
  Rgb3 R0, out;
  int rows, cols;
  Divisor by_cols;
};

// One thread per pixel, in linear order: no lane idles, whatever the canvas'
// width.  Blocks of 64 columns by four rows, which need no division, took 25 us
// at 1920 x 1080 against 23, and 918 against 20 on two million rows of one
// pixel; with a 64-bit division the linear order took 42 and 38.  Renderer.hxx:97-152,
// evaluated in FP32.  The Beckmann exponent tan(acos(x))^2 is evaluated as
// (1 - x^2) / x^2 (the same value; FP32 acos loses the digits near 1 that this
// form keeps; x = 0 gives +inf and a zero term, as tan(acos(0))^2 ~ 2.7e32
// does in FP64).  With a = s21 - s01 and b = s12 - s10 the normal
// normalized(va x vb), va = normalized(2, 0, a), vb = normalized(0, 2, b), is
// (-a, -b, 2) / |.|; the light direction is normalised once, and its squared
// length in the attenuation is 1; the Fresnel term Ks + (1 - Ks) q^5 is 1 for
// the renderer's Ks = 1.
__device__ __forceinline__ void render_pixel(const RenderArgs& a, int i, int j) {
  const int64_t row = (int64_t)i * a.cols, p = row + j;
  float K[3], S[3], Kd[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    K[c] = a.L.ks[c][p];
    S[c] = a.L.ks[3 + c][p];
    Kd[c] = a.R0.p[c][p];
  }
  const double* V = a.L.v;  // thickness, evaluated in FP32 below
  const float s11 = (float)V[p];
  const float s01 = (float)V[row + reflect_index(j - 1, a.cols)];
  const float s21 = (float)V[row + reflect_index(j + 1, a.cols)];
  const float s10 = (float)V[(int64_t)reflect_index(i - 1, a.rows) * a.cols + j];
  const float s12 = (float)V[(int64_t)reflect_index(i + 1, a.rows) * a.cols + j];
  km_pixel(K, S, Kd, s11);  // compR = compose(canvas)
  // normal with z negated (Renderer.hxx:113-121)
  const F3 nrm = unit3(F3{s01 - s21, s10 - s12, -2.0f});
  // light at (-200, -1500, -2000), eye at (cols/2, rows/2, -100)
  const float px = (float)j, py = (float)i;
  const F3 l = unit3(F3{-200.0f - px, -1500.0f - py, -2000.0f - s11});
  const F3 v = unit3(F3{0.5f * (float)a.cols - px, 0.5f * (float)a.rows - py, -100.0f - s11});
  const F3 hv = F3{v.x + l.x, v.y + l.y, v.z + l.z};
  const float hh = dot3(hv, hv);
  const float hr = hh > 0.0f ? rsq1(hh) : 1.0f;
  const F3 h = F3{hv.x * hr, hv.y * hr, hv.z * hr};
  const float NdotH = fmaxf(0.0f, dot3(nrm, h));
  const float VdotH = fmaxf(0.0f, dot3(v, h));
  const float NdotV = fmaxf(0.0f, dot3(nrm, v));
  const float NdotL = fmaxf(0.0f, dot3(nrm, l));
  constexpr float m = 0.5f, s = 0.2f, lightPower = 15.0f;
  float spec = 0.0f;
  if (NdotL > 0.0f && NdotV > 0.0f) {
    const float x2 = NdotH * NdotH;
    const float A = rcp1(m * m + x2 * x2 * kPiF);
    const float B = expf(-((1.0f - x2) / x2) * (1.0f / (m * m)));
    const float g = 2.0f * NdotH * fminf(NdotV, NdotL) / VdotH;  // std::min(G1, G2)
    const float G = g < 1.0f ? g : 1.0f;  // std::min(1.0, g)
    spec = (A * B * G) * rcp1(NdotL * NdotV);
  }
  // a volume that is no number has no light direction: as its squared length
  // would, it makes the pixel NaN, which the clamp below makes 0
  const float beta = __builtin_isfinite(s11) ? lightPower * (1.0f / (4.0f * kPiF)) : NAN;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float r = (beta * NdotL) * ((1.0f - s) * Kd[c] + s * spec) + (Kd[c] * 0.2f) * Kd[c];
    a.out.p[c][p] = fminf(fmaxf(r, 0.0f), 1.0f);
  }
}

__global__ __launch_bounds__(kBlock) void k_render(RenderArgs a) {
  const uint32_t p = blockIdx.x * kBlock + threadIdx.x;  // a canvas has < 2^31 pixels
  if (p >= (uint32_t)a.rows * (uint32_t)a.cols) return;
  const uint32_t i = a.by_cols.div(p);
  render_pixel(a, (int)i, (int)(p - i * (uint32_t)a.cols));
}

// ColorConverter::rgb2srgb (core/Color.hxx:197-205) and Mat::convertTo's
// saturate_cast (round half to even), so that the integer result is that of
// FP64 pow on the same float input.
__device__ __forceinline__ double srgb_exact(double x) {
  return x <= 0.00313066844250063 ? x * 12.92 : 1.055 * pow(x, 1.0 / 2.4) - 0.055;
}
__device__ __forceinline__ double encode_clamp(double r, double scale) {
  return r < 0.0 ? 0.0 : (r > scale ? scale : r);
}
__device__ double encode_exact(float xf, int to_srgb, double scale) {
  const double x = (double)xf;
  return encode_clamp(rint((to_srgb ? srgb_exact(x) : x) * scale), scale);
}
// y = x^(1/2.4) solves y^12 = x^5: from the FP32 power (3e-7 or better) one
// FP64 Newton step leaves 1e-12.  *sure is cleared where that is not enough: a
// value within 1e-6 of a rounding edge of the scaled result, and anything but
// 0.0031 < x < 1.
__device__ __forceinline__ double encode_fast(float xf, int to_srgb, double scale, bool* sure) {
  const double x = (double)xf;
  if (!to_srgb) {
    *sure = true;
    return encode_clamp(rint(x * scale), scale);
  }
  const float y0 = __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(xf) * (1.0f / 2.4f));
  const double y = (double)y0, x2 = x * x, x5 = x2 * x2 * x;
  const double y2 = y * y, y4 = y2 * y2, y8 = y4 * y4, y11 = y8 * y2 * y;
  const double y1 = y - __builtin_fma(y11, y, -x5) * (double)__builtin_amdgcn_rcpf(12.0f * (float)y11);
  const double t = __builtin_fma(1.055, y1, -0.055) * scale;
  const double r = rint(t);
  *sure = xf > 0.0031307f && xf < 1.0f && fabs(t - r) < 0.5 - 1e-6;
  return r;
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_encode(int64_t n, Rgb3 in, int to_srgb, double scale,
                                                   T* out) {
  const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (p >= n) return;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    bool sure;
    double r = encode_fast(in.p[c][p], to_srgb, scale, &sure);
    if (!sure) r = encode_exact(in.p[c][p], to_srgb, scale);
    out[3 * p + c] = (T)r;
  }
}

// Four pixels a thread: 16-byte loads of the planes (a plane of odd size
// leaves the next one on a 4-byte boundary, which these loads allow), and
// their twelve values in three words.  The last n % 4 pixels go one a thread,
// behind the fours (a launch of their own took 3 us more).
template <class T>
__global__ __launch_bounds__(kBlock) void k_encode_vec(int64_t n, Rgb3 in, int to_srgb,
                                                       double scale, T* out) {
  using Word = typename std::conditional<sizeof(T) == 1, uint32_t, uint64_t>::type;
  const int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x, n4 = n / 4;
  if (q >= n4) {
    const int64_t p = 3 * n4 + q;
    if (p < n)
#pragma unroll 1
      for (int c = 0; c < 3; ++c) {
        const float* plane = c == 0 ? in.p[0] : (c == 1 ? in.p[1] : in.p[2]);
        out[3 * p + c] = (T)encode_exact(plane[p], to_srgb, scale);
      }
    return;
  }
  typedef float Float4 __attribute__((ext_vector_type(4), aligned(4)));
  Float4 v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = *reinterpret_cast<const Float4*>(in.p[c] + 4 * q);
  Word w[3] = {0, 0, 0};
  unsigned redo = 0u;
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    const float x = v[k % 3][k / 3];
    bool sure;
    const double r = encode_fast(x, to_srgb, scale, &sure);
    w[k / 4] |= (Word)(T)(sure ? r : 0.0) << (8 * sizeof(T) * (k % 4));
    redo |= (sure ? 0u : 1u) << k;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) reinterpret_cast<Word*>(out)[3 * q + k] = w[k];
  // the few others, over what was just stored
  while (redo) {
    const int k = __ffs((int)redo) - 1;
    redo &= redo - 1;
    const int c = k % 3;
    const float* plane = c == 0 ? in.p[0] : (c == 1 ? in.p[1] : in.p[2]);
    out[12 * q + k] = (T)encode_exact(plane[4 * q + k / 3], to_srgb, scale);
  }
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// The image word-aligned: four pixels a thread; otherwise one a thread
// (single-value stores).
template <class T>
void launch_encode_t(int64_t n, const Rgb3& in, int to_srgb, double scale, T* out, hipStream_t s) {
  if (((uintptr_t)out & (4 * sizeof(T) - 1)) == 0)
    k_encode_vec<T><<<blocks_for(n / 4 + n % 4), kBlock, 0, s>>>(n, in, to_srgb, scale, out);
  else
    k_encode<T><<<blocks_for(n), kBlock, 0, s>>>(n, in, to_srgb, scale, out);
  PNT_HIP_CHECK(hipGetLastError());
}

}  // namespace

void launch_render(int rows, int cols, const Layer7& L, const Rgb3& R0, const Rgb3& out,
                   hipStream_t s) {
  if ((int64_t)rows * cols <= 0) return;
  k_render<<<blocks_for((int64_t)rows * cols), kBlock, 0, s>>>(
      RenderArgs{L, R0, out, rows, cols, Divisor::of((uint32_t)cols)});
  PNT_HIP_CHECK(hipGetLastError());
}

void launch_encode(int64_t n, const Rgb3& in, int to_srgb, int bits, void* out, hipStream_t s) {
  if (n <= 0) return;
  if (bits == 16)
    launch_encode_t(n, in, to_srgb, 65535.0, static_cast<uint16_t*>(out), s);
  else
    launch_encode_t(n, in, to_srgb, 255.0, static_cast<uint8_t*>(out), s);
}

}  // namespace pnt
