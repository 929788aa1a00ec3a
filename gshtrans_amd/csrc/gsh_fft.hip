// gsh_fft.hip -- ring FFTs of 2049 .. 4095 points, and the lMax = 0 branches.
//
// The reference runs one FFTW plan per ring (GaussLegendreGrid.h:147-174 for
// the analysis, :266-319 for the synthesis): an unnormalised c2c/c2r backward
// transform of the order bins F_m placed at k = m (m >= 0) and k = N + m
// (m < 0), and an unnormalised c2c/r2c forward transform of each ring.
// gsh_fft_ring.hip and gsh_fft_wave.hip transform in registers every ring whose
// length is a power of two or at most 2048.  The other lengths (1024 < lMax <
// 2048) take Bluestein's chirp-z identity jk = (j^2 + k^2 - (k-j)^2)/2 through a
// convolution of 8192 points: one workgroup per ring keeps it in 128 KiB of LDS
// and runs Stockham autosort passes of radix 4 (and one of radix 2) in place,
// values going through registers between barriers.  Chirp multiply, FFT, multiply
// by the transformed chirp filter, inverse FFT, chirp multiply (Bluestein 1970).
#include "gsh_internal.h"

namespace gsh {
namespace {

constexpr int kFFTThreads = 256;
constexpr int kFFTPoints = 8192;  // of the convolution, the ring zero-padded to them

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
// multiply by s*i (s = +1 or -1)
__device__ __forceinline__ double2 cmuli(double2 a, int s) {
  return s > 0 ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// Stockham autosort passes over buf.  SIGN = -1 forward, +1 backward.
template <int SIGN>
__device__ void stockham(double2* buf, const double2* __restrict__ tw) {
  constexpr int M = kFFTPoints;
  constexpr int quarter = M / 4, half = M / 2;
  int Ns = 1;
  // radix-4 passes
  while (4 * Ns <= M) {
    constexpr int kPer = quarter / kFFTThreads;
    double2 v[kPer][4];
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      const int j = threadIdx.x + i * kFFTThreads;
      const int k = j & (Ns - 1);
      double2 a0 = buf[j], a1 = buf[j + quarter], a2 = buf[j + 2 * quarter],
              a3 = buf[j + 3 * quarter];
      if (Ns > 1) {
        const int step = M / (Ns * 4);
        double2 w1 = tw[k * step], w2 = tw[2 * k * step], w3 = tw[3 * k * step];
        if (SIGN > 0) {
          w1.y = -w1.y;
          w2.y = -w2.y;
          w3.y = -w3.y;
        }
        a1 = cmul(a1, w1);
        a2 = cmul(a2, w2);
        a3 = cmul(a3, w3);
      }
      const double2 t0 = cadd(a0, a2), t1 = csub(a0, a2);
      const double2 t2 = cadd(a1, a3), t3 = cmuli(csub(a1, a3), SIGN);
      v[i][0] = cadd(t0, t2);
      v[i][1] = cadd(t1, t3);
      v[i][2] = csub(t0, t2);
      v[i][3] = csub(t1, t3);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      const int j = threadIdx.x + i * kFFTThreads;
      double2* y = buf + (j / Ns) * Ns * 4 + (j & (Ns - 1));
      y[0] = v[i][0];
      y[Ns] = v[i][1];
      y[2 * Ns] = v[i][2];
      y[3 * Ns] = v[i][3];
    }
    __syncthreads();
    Ns *= 4;
  }
  // the last pass, radix 2: Ns = M / 2
  constexpr int kPer = half / kFFTThreads;
  double2 v[kPer][2];
#pragma unroll
  for (int i = 0; i < kPer; i++) {
    const int j = threadIdx.x + i * kFFTThreads;
    double2 w1 = tw[j];
    if (SIGN > 0) w1.y = -w1.y;
    const double2 a0 = buf[j], a1 = cmul(buf[j + half], w1);
    v[i][0] = cadd(a0, a1);
    v[i][1] = csub(a0, a1);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer; i++) {
    const int j = threadIdx.x + i * kFFTThreads;
    buf[j] = v[i][0];
    buf[j + half] = v[i][1];
  }
  __syncthreads();
}

__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }

// Unnormalised DFT of the ring in buf (N points, zero from there on).
// SIGN = -1 forward, +1 backward.
template <int SIGN>
__device__ void ring_dft(double2* buf, const FFTParams& p) {
  auto chirp = [&] {
    for (int j = threadIdx.x; j < p.N; j += kFFTThreads) {
      const double2 w = SIGN < 0 ? p.chirp[j] : cconj(p.chirp[j]);
      buf[j] = cmul(buf[j], w);
    }
    __syncthreads();
  };
  chirp();
  stockham<-1>(buf, p.tw);
  const double2* h = SIGN < 0 ? p.hf : p.hb;
  for (int j = threadIdx.x; j < kFFTPoints; j += kFFTThreads) buf[j] = cmul(buf[j], h[j]);
  __syncthreads();
  stockham<+1>(buf, p.tw);
  chirp();
}

// Synthesis of field f at colatitude theta: bins from F, backward FFT, write
// the ring.
__global__ __launch_bounds__(kFFTThreads) void fft_synth(FFTParams p) {
  __shared__ double2 buf[kFFTPoints];
  const int theta = blockIdx.x / p.nfield;
  const int f = blockIdx.x % p.nfield;
  const int N = p.N;
  const int cw = p.cw, ncg = (p.ncol + cw - 1) / cw;
  // slot s of this field at Fp[cw s]
  const double* Fp = p.F + f_index(theta, 0, 2 * f, p.nslot, ncg, cw);
  const int lf = ring_lmax(p, f);
  for (int k = threadIdx.x; k < kFFTPoints; k += kFFTThreads) {
    double2 X = make_double2(0.0, 0.0);
    if (k < N) {
      if (!p.real) {
        if (k <= lf) {
          const int s = k - p.m_first;
          X = make_double2(Fp[cw * (long)s], Fp[cw * (long)s + 1]);
        }
        if (k >= N - lf) {
          const int s = (k - N) - p.m_first;
          X = cadd(X, make_double2(Fp[cw * (long)s], Fp[cw * (long)s + 1]));
        }
      } else {
        // Hermitian spectrum from bins 0..N/2 (c2r semantics).
        const int kk = k <= N / 2 ? k : N - k;
        if (kk <= lf) {
          const int s = kk - p.m_first;
          X = make_double2(Fp[cw * (long)s], Fp[cw * (long)s + 1]);
          if (kk == 0 || kk == N / 2) X.y = 0.0;
          else if (k > N / 2) X.y = -X.y;
        }
      }
    }
    buf[k] = X;
  }
  __syncthreads();
  ring_dft<+1>(buf, p);
  const long ring = (long)(p.fmap ? p.fmap[f] : f) * p.fstride + (long)theta * N;
  for (int j = threadIdx.x; j < N; j += kFFTThreads) {
    const long o = ring + j;
    const double2 x = buf[j];
    if (p.real && p.f32)
      static_cast<float*>(p.fout)[o] = (float)x.x;
    else if (p.real)
      static_cast<double*>(p.fout)[o] = x.x;
    else if (p.f32)
      static_cast<float2*>(p.fout)[o] = make_float2((float)x.x, (float)x.y);
    else
      static_cast<double2*>(p.fout)[o] = x;
  }
}

// Analysis of field f at colatitude theta: load the ring, forward FFT, scatter
// weighted bins into F.
__global__ __launch_bounds__(kFFTThreads) void fft_anal(FFTParams p) {
  __shared__ double2 buf[kFFTPoints];
  const int theta = blockIdx.x / p.nfield;
  const int f = blockIdx.x % p.nfield;
  const int N = p.N;
  const long ring = (long)(p.fmap ? p.fmap[f] : f) * p.fstride + (long)theta * N;
  for (int j = threadIdx.x; j < kFFTPoints; j += kFFTThreads) {
    double2 x = make_double2(0.0, 0.0);
    if (j < N) {
      const long o = ring + j;
      auto load = [&](const void* b) {
        if (p.real && p.f32) return make_double2(static_cast<const float*>(b)[o], 0.0);
        if (p.real) return make_double2(static_cast<const double*>(b)[o], 0.0);
        if (p.f32) {
          const float2 y = static_cast<const float2*>(b)[o];
          return make_double2(y.x, y.y);
        }
        return static_cast<const double2*>(b)[o];
      };
      if (p.src_cplx) {  // Re or Im of a complex field, transformed as a real ring
        const double2 z = static_cast<const double2*>(p.fin)[o];
        x.x = p.op == kExprImag ? z.y : z.x;
      } else {
        x = load(p.fin);
        if (p.op) {  // pointwise expression of the fields
          const double2 y = expr_binary(p.op) ? load(p.fin2) : make_double2(0.0, 0.0);
          x = p.real ? make_double2(expr_real(p.op, x.x, y.x, p.scalar.x), 0.0)
                     : expr_cplx(p.op, x, y, p.scalar);
        }
      }
    }
    buf[j] = x;
  }
  __syncthreads();
  ring_dft<-1>(buf, p);
  const double w = p.wq[theta];
  const int lf = ring_lmax(p, f);
  for (int s = threadIdx.x; s < p.nslot; s += kFFTThreads) {
    const int m = s + p.m_first;
    if (abs(m) > lf) continue;
    const int k = m >= 0 ? m : N + m;
    double2 X = buf[k];
    if (p.adjoint && p.real) {
      // c2r bin weights: 2 for 0 < k < N/2, real part only at k = 0, N/2
      if (k == 0 || 2 * k == N) X.y = 0.0;
      else X = make_double2(2.0 * X.x, 2.0 * X.y);
    }
    const long fi = fa_index(s, 2 * f, theta, p.n_cg, p.nquad, p.cw);
    if (p.fa32) {
      float* Fp = reinterpret_cast<float*>(p.F) + fi;
      Fp[0] = (float)(X.x * w);
      Fp[1] = (float)(X.y * w);
    } else {
      p.F[fi] = X.x * w;
      p.F[fi + 1] = X.y * w;
    }
    // The last ring also zeroes the padding rows of the last colatitude
    // quad, which the Legendre contraction reads as B operands.
    for (int tp = theta + 1; p.zero_pad && theta == p.ntheta - 1 && tp < 4 * p.nquad; tp++) {
      const long zi = fa_index(s, 2 * f, tp, p.n_cg, p.nquad, p.cw);
      if (p.fa32) {
        reinterpret_cast<float*>(p.F)[zi] = 0.0f;
        reinterpret_cast<float*>(p.F)[zi + 1] = 0.0f;
      } else {
        p.F[zi] = 0.0;
        p.F[zi + 1] = 0.0;
      }
    }
  }
}

// lmax == 0 branches of the reference act on element 0 only
// (GaussLegendreGrid.h:137-140 and :251-260): the synthesis writes
// out[0] = c[0] 2 sqrt(pi), the analysis assigns c[0] = f[0] / (2 sqrt(pi))
// (even though its general branch accumulates).  mode 2 is the adjoint of
// that synthesis: c[0] = 2 sqrt(pi) f[0] (real part only for real fields).
__global__ void lmax0_kernel(int mode, int real, int nfield, const double* in, long istride,
                             double* out, long ostride) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nfield) return;
  const double inv_sqrtpi = 0.56418958354775628695;  // 1/sqrt(pi)
  if (mode == 1) {
    // in: complex coefficients; out: real or complex field
    const double* c = in + 2 * (long)f * istride;
    if (real) {
      out[(long)f * ostride] = c[0] * 2.0 / inv_sqrtpi;
    } else {
      out[2 * (long)f * ostride] = c[0] * 2.0 / inv_sqrtpi;
      out[2 * (long)f * ostride + 1] = c[1] * 2.0 / inv_sqrtpi;
    }
  } else {
    // in: field; out: complex coefficients
    double re, im;
    if (real) {
      re = in[(long)f * istride];
      im = 0.0;
    } else {
      re = in[2 * (long)f * istride];
      im = in[2 * (long)f * istride + 1];
    }
    const double sc = mode == 2 ? 2.0 / inv_sqrtpi : inv_sqrtpi / 2.0;
    double* c = out + 2 * (long)f * ostride;
    c[0] = re * sc;
    c[1] = im * sc;
  }
}

}  // namespace

hipError_t launch_fft_synth(const FFTParams& p, hipStream_t s) {
  if (p.M != kFFTPoints || p.N > p.M / 2) return hipErrorInvalidValue;
  if (p.fa32) return hipErrorInvalidValue;  // FP32 bins: wavefront kernels only
  hipLaunchKernelGGL(fft_synth, dim3((long)p.ntheta * p.nfield), dim3(kFFTThreads), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_fft_anal(const FFTParams& p0, hipStream_t s) {
  FFTParams p = p0;
  p.n_cg = (p.ncol + p.cw - 1) / p.cw;
  p.nquad = (p.ntheta + 3) / 4;
  if (p.M != kFFTPoints || p.N > p.M / 2) return hipErrorInvalidValue;
  hipLaunchKernelGGL(fft_anal, dim3((long)p.ntheta * p.nfield), dim3(kFFTThreads), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_lmax0(int mode, int real, int nfield, const double* in, long istride,
                        double* out, long ostride, hipStream_t s) {
  hipLaunchKernelGGL(lmax0_kernel, dim3((nfield + 255) / 256), dim3(256), 0, s, mode, real,
                     nfield, in, istride, out, ostride);
  return hipGetLastError();
}

}  // namespace gsh
