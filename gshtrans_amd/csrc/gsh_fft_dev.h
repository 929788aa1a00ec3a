// gsh_fft_dev.h -- device pieces shared by the ring FFT kernels
// (gsh_fft_wave.hip, gsh_fft_ring.hip): complex arithmetic, in-register DFTs
// of 2^k points and field element access.
#pragma once

#include "gsh_internal.h"

namespace gsh {
namespace {

// cos(pi k / 16) and sin(pi k / 16), k = 0..16.
constexpr double kCos16[17] = {
    1.0,                     0.98078528040323044913, 0.92387953251128675613,
    0.83146961230254523708,  0.70710678118654752440, 0.55557023301960222474,
    0.38268343236508977173,  0.19509032201612826785, 0.0,
    -0.19509032201612826785, -0.38268343236508977173, -0.55557023301960222474,
    -0.70710678118654752440, -0.83146961230254523708, -0.92387953251128675613,
    -0.98078528040323044913, -1.0};
constexpr double kSin16[17] = {
    0.0,                    0.19509032201612826785, 0.38268343236508977173,
    0.55557023301960222474, 0.70710678118654752440, 0.83146961230254523708,
    0.92387953251128675613, 0.98078528040323044913, 1.0,
    0.98078528040323044913, 0.92387953251128675613, 0.83146961230254523708,
    0.70710678118654752440, 0.55557023301960222474, 0.38268343236508977173,
    0.19509032201612826785, 0.0};

__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * conj(b)
__device__ __forceinline__ double2 cmulc(double2 a, double2 b) {
  return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}

// a * exp(i SIGN pi K / 16); K is a constant after unrolling.
template <int SIGN>
__device__ __forceinline__ double2 rot16(double2 a, int K) {
  if (K == 0) return a;
  if (K == 8) return SIGN > 0 ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
  // exp(i SIGN pi / 4) = h (1 + SIGN i), exp(i SIGN 3 pi / 4) = h (-1 + SIGN i)
  const double h = kCos16[4];
  if (K == 4) return make_double2(h * (a.x - SIGN * a.y), h * (a.y + SIGN * a.x));
  if (K == 12) return make_double2(h * (-a.x - SIGN * a.y), h * (SIGN * a.x - a.y));
  const double c = kCos16[K], s = SIGN * kSin16[K];
  return make_double2(a.x * c - a.y * s, a.x * s + a.y * c);
}

constexpr int bitrev(int x, int bits) {
  int r = 0;
  for (int i = 0; i < bits; i++) r |= ((x >> i) & 1) << (bits - 1 - i);
  return r;
}
constexpr int log2c(int x) { return x <= 1 ? 0 : 1 + log2c(x >> 1); }

// In-register DFT of length R (radix-2 decimation in frequency); on return
// v[bitrev(k)] holds X[k] = sum_j v_in[j] exp(i SIGN 2 pi j k / R).
template <int R, int SIGN>
__device__ __forceinline__ void dft_reg(double2* v) {
#pragma unroll
  for (int h = R / 2; h >= 1; h >>= 1) {
#pragma unroll
    for (int base = 0; base < R; base += 2 * h) {
#pragma unroll
      for (int j = 0; j < h; j++) {
        const double2 a = v[base + j], b = v[base + j + h];
        v[base + j] = cadd(a, b);
        // twiddle exp(i SIGN 2 pi j / (2h)) = exp(i SIGN pi (16 j / h) / 16)
        v[base + j + h] = rot16<SIGN>(csub(a, b), 16 * j / h);
      }
    }
  }
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Field element access for FP64 or FP32 storage (index in elements).
template <int F32>
__device__ __forceinline__ double2 ld_cplx(const void* b, long i) {
  if (F32) {
    const float2 v = static_cast<const float2*>(b)[i];
    return make_double2(v.x, v.y);
  }
  return static_cast<const double2*>(b)[i];
}
template <int F32>
__device__ __forceinline__ double ld_real(const void* b, long i) {
  if (F32) return static_cast<const float*>(b)[i];
  return static_cast<const double*>(b)[i];
}
template <int F32>
__device__ __forceinline__ void st_cplx(void* b, long i, double2 v) {
  if (F32)
    static_cast<float2*>(b)[i] = make_float2((float)v.x, (float)v.y);
  else
    static_cast<double2*>(b)[i] = v;
}
template <int F32>
__device__ __forceinline__ void st_real(void* b, long i, double v) {
  if (F32)
    static_cast<float*>(b)[i] = (float)v;
  else
    static_cast<double*>(b)[i] = v;
}

// Two consecutive real samples (elements i, i + 1) of a real field.
template <int F32>
__device__ __forceinline__ double2 ld_pair(const void* b, long i) {
  if (F32) {
    const float2 v = *reinterpret_cast<const float2*>(static_cast<const float*>(b) + i);
    return make_double2(v.x, v.y);
  }
  return *reinterpret_cast<const double2*>(static_cast<const double*>(b) + i);
}

// Re (op kExprReal) or Im (kExprImag) of a complex sample, and of the two
// consecutive complex samples i, i + 1 (FP64 storage).
__device__ __forceinline__ double cplx_part(double2 z, int op) {
  return op == kExprImag ? z.y : z.x;
}
__device__ __forceinline__ double2 cplx_part2(const void* b, long i, int op) {
  const double2 z0 = static_cast<const double2*>(b)[i];
  const double2 z1 = static_cast<const double2*>(b)[i + 1];
  return make_double2(cplx_part(z0, op), cplx_part(z1, op));
}
// A real expression of two consecutive samples of each operand.
__device__ __forceinline__ double2 expr_pair(int op, double2 a, double2 b, double s) {
  return make_double2(expr_real(op, a.x, b.x, s), expr_real(op, a.y, b.y, s));
}

}  // namespace
}  // namespace gsh
