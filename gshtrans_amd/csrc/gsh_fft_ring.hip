// gsh_fft_ring.hip -- ring FFTs of any length: M / 16 threads per ring, 16
// complex values per thread in registers.
//
// Same transforms as gsh_fft_wave.hip (GaussLegendreGrid.h:147-174, 266-319)
// for the ring lengths it has no kernel for, and for calls of few fields,
// whose wavefront kernel would run mostly empty.  A power of two N in 64 ..
// 4096 is transformed directly (M = N), any other N <= 2048 through
// Bluestein's identity jk = (j^2 + k^2 - (k - j)^2) / 2 as a cyclic
// convolution of M points, M the smallest power of two >= 2 N - 1 (Bluestein
// 1970).
//
// What bounds it: the chain of LDS exchanges of a ring, then HBM.  Stockham
// passes of radix 16, 8 and 4 (three for M >= 512, two below) keep a thread's
// values at x[t + (M / 16) e], e < 16, before and after every pass, so
//  - the first pass reads, and the last pass writes, global memory directly,
//  - the filter multiplication of Bluestein's convolution and the inverse
//    transform's first pass follow the forward transform's last in registers:
//    four exchanges for the two transforms.
// Rings of M <= 1024 live in one wavefront (no workgroup barrier); the LDS
// rows are padded by one value in 16, which spreads every 16-lane phase of the
// exchanges over all banks.  Twiddles are powers of one table entry per pass.
// lMax=360 (720-point rings, M = 2048), 20 complex fields: 382 -> 97 us
// synthesis, 381 -> 92 us analysis against a whole workgroup per ring with every
// pass in LDS.
// Rings of at most 32 points are summed directly (direct_dft): a convolution of
// 64 points rounds up to twice as much as the transform of the ring itself
// (lMax = 2: 3.7e-16 in place of 1.5e-16 relative to extended precision).
// Real fields go two rings at a time as x_a + i x_b, two colatitudes of one
// field (a field's Inf or NaN reaches no other field).
#include "gsh_fft_dev.h"
#include "gsh_internal.h"

namespace gsh {
namespace {

// Radix of pass i of an M-point transform (0: none).
constexpr int radix(int M, int i) {
  const int a[3] = {M == 512 ? 8 : 16, M == 64 ? 4 : M == 128 || M == 512 || M == 1024 ? 8 : 16,
                    M < 512 ? 0 : M <= 2048 ? 8 : 16};
  return a[i];
}
constexpr int npass(int M) { return M < 512 ? 2 : 3; }
// Pass i of the inverse transform: the radices in reverse, so that it starts
// from the values a thread ends the forward transform with.
constexpr int radix_rev(int M, int i) { return radix(M, npass(M) - 1 - i); }

__device__ __forceinline__ int pad(int p) { return p + (p >> 4); }

template <int M>
struct Ring {
  static constexpr int T = M / 16;                       // threads per ring
  static constexpr int kThreads = T < 64 ? 64 : T;       // threads per workgroup
  static constexpr int kRings = kThreads / T;            // rings per workgroup
  static constexpr int kStride = M + M / 16;             // padded ring in LDS
  static __device__ __forceinline__ void sync() {
    if (kThreads > 64)
      __syncthreads();
    else
      wave_sync();
  }
};

// DFT of length R over v[q + (16 / R) i], i < R, whose upper half is zero.
template <int R, int SIGN>
__device__ __forceinline__ void dft_half(double2* u) {
#pragma unroll
  for (int j = 0; j < R / 2; j++) u[j + R / 2] = rot16<SIGN>(u[j], 16 * j / (R / 2));
#pragma unroll
  for (int h = R / 4; h >= 1; h >>= 1)
#pragma unroll
    for (int base = 0; base < R; base += 2 * h)
#pragma unroll
      for (int j = 0; j < h; j++) {
        const double2 a = u[base + j], b = u[base + j + h];
        u[base + j] = cadd(a, b);
        u[base + j + h] = rot16<SIGN>(csub(a, b), 16 * j / h);
      }
}

// The table entries that the passes of one transform start their twiddle
// powers from, loaded before anything waits (a load inside a pass would add
// its latency to the chain of exchanges): entry q of pass i >= 1 is
// exp(-2 pi i (j % Ns) / (Ns R)), j = t + T q.
template <int M, bool REV>
struct Twiddles {
  double2 w[2][4];
  __device__ __forceinline__ Twiddles(const double2* tw, int t) {
    int ns = REV ? radix_rev(M, 0) : radix(M, 0);
#pragma unroll
    for (int i = 1; i < npass(M); i++) {
      const int R = REV ? radix_rev(M, i) : radix(M, i);
#pragma unroll
      for (int q = 0; q < 16 / R; q++)
        w[i - 1][q] = tw[((t + M / 16 * q) & (ns - 1)) * (M / (ns * R))];
      ns *= R;
    }
  }
};

// One Stockham pass of radix R after Ns points are done: butterflies j = t +
// T q, q < 16 / R, each over v[q + (16 / R) i].  LAST passes leave the result
// in place; the others go through LDS.
template <int M, int SIGN, int R, int NS, bool LAST, bool HALF>
__device__ __forceinline__ void pass(double2 (&v)[16], double2* lds, const double2* w1, int t) {
  constexpr int T = M / 16, Q = 16 / R, LR = log2c(R);
#pragma unroll
  for (int q = 0; q < Q; q++) {
    double2 u[R];
#pragma unroll
    for (int i = 0; i < R; i++) u[i] = v[q + Q * i];
    if (NS > 1) {
      double2 w[R];
      w[1] = w1[q];
#pragma unroll
      for (int i = 2; i < R; i++) w[i] = cmul(w[i / 2], w[i - i / 2]);
#pragma unroll
      for (int i = 1; i < R; i++) u[i] = SIGN < 0 ? cmul(u[i], w[i]) : cmulc(u[i], w[i]);
    }
    if (HALF)
      dft_half<R, SIGN>(u);
    else
      dft_reg<R, SIGN>(u);
#pragma unroll
    for (int i = 0; i < R; i++) v[q + Q * i] = u[bitrev(i, LR)];
  }
  if (!LAST) {
    Ring<M>::sync();
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int j = t + T * q;
      const int p = (j / NS) * (NS * R) + (j & (NS - 1));
#pragma unroll
      for (int i = 0; i < R; i++) lds[pad(p + i * NS)] = v[q + Q * i];
    }
    Ring<M>::sync();
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = lds[pad(t + T * e)];
  }
}

// M-point transform of v[e] = x[t + T e]; on return v[e] = X[t + T e].  REV
// runs the radices in reverse order; HALF: x[k] = 0 for k >= M / 2.
template <int M, int SIGN, bool REV, bool HALF>
__device__ __forceinline__ void ring_fft(double2 (&v)[16], double2* lds,
                                         const Twiddles<M, REV>& tw, int t) {
  constexpr int R0 = REV ? radix_rev(M, 0) : radix(M, 0);
  constexpr int R1 = REV ? radix_rev(M, 1) : radix(M, 1);
  pass<M, SIGN, R0, 1, false, HALF>(v, lds, nullptr, t);
  if constexpr (npass(M) == 2) {
    pass<M, SIGN, R1, R0, true, false>(v, lds, tw.w[0], t);
  } else {
    constexpr int R2 = REV ? radix_rev(M, 2) : radix(M, 2);
    pass<M, SIGN, R1, R0, false, false>(v, lds, tw.w[0], t);
    pass<M, SIGN, R2, R0 * R1, true, false>(v, lds, tw.w[1], t);
  }
}

// Unnormalised DFT of a ring of N <= 32 points (N even) held by 4 threads as
// v[e] = x[t + 4 e], e < 8, with one root of unity per term: p.tw[j] = exp(-2 pi
// i j / N).  The outputs k = t + 4 e of a thread are of one class modulo 4 (modulo
// 2), so the N / 4 (N / 2) terms left after a radix-4 (radix-2) butterfly are the
// same for all of them.  Four partial sums per output: less rounding than one
// chain, and independent multiply-adds.
template <int SIGN>
__device__ __forceinline__ void direct_dft(double2 (&v)[16], double2* lds, const FFTParams& p,
                                           int t) {
  constexpr int E = 8, ROOT = 34;  // outputs per thread; the roots' place in LDS
  static_assert(ROOT + 4 * E <= Ring<64>::kStride, "ring and roots share a row");
  const int N = p.N, four = N % 4 == 0, H = four ? N / 4 : N / 2;
#pragma unroll
  for (int e = 0; e < E; e++) {
    lds[t + 4 * e] = v[e];  // zero from N on
    lds[ROOT + t + 4 * e] = p.tw[t + 4 * e];
  }
  Ring<64>::sync();
  double2 a[E][4];
  int j[E], dj[E];  // root of the next term, its step
#pragma unroll
  for (int e = 0; e < E; e++) {
    j[e] = 0;
    dj[e] = t + 4 * e < N ? t + 4 * e : 0;
#pragma unroll
    for (int r = 0; r < 4; r++) a[e][r] = make_double2(0.0, 0.0);
  }
  for (int n0 = 0; n0 < H; n0 += 4) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int n = n0 + r;
      double2 x = make_double2(0.0, 0.0);
      if (n < H) {
        const double2 x0 = lds[n], x1 = lds[n + H];
        if (four) {
          const double2 x2 = lds[n + 2 * H], x3 = lds[n + 3 * H];
          const double2 s = t & 1 ? csub(x0, x2) : cadd(x0, x2);
          const double2 d = t & 1 ? rot16<SIGN>(csub(x1, x3), 8) : cadd(x1, x3);
          x = t & 2 ? csub(s, d) : cadd(s, d);
        } else {
          x = t & 1 ? csub(x0, x1) : cadd(x0, x1);
        }
      }
#pragma unroll
      for (int e = 0; e < E; e++) {
        double2 w = lds[ROOT + j[e]];
        if (SIGN > 0) w.y = -w.y;
        a[e][r].x = fma(x.x, w.x, fma(-x.y, w.y, a[e][r].x));
        a[e][r].y = fma(x.x, w.y, fma(x.y, w.x, a[e][r].y));
        j[e] += dj[e];
        j[e] -= j[e] >= N ? N : 0;
      }
    }
  }
#pragma unroll
  for (int e = 0; e < E; e++) v[e] = cadd(cadd(a[e][0], a[e][2]), cadd(a[e][1], a[e][3]));
}

// Unnormalised N-point DFT of the ring held as v[e] = x[t + T e] (zero from N
// on): direct (BLUE 0, M = N), or Bluestein's, or for rings of at most 32 points
// (M = 64 and N < M) the sums themselves.
template <int M, int BLUE, int SIGN>
__device__ __forceinline__ void ring_dft(double2 (&v)[16], double2* lds, const FFTParams& p,
                                         const Twiddles<M, false>& tw, int t) {
  if constexpr (!BLUE) {
    ring_fft<M, SIGN, false, false>(v, lds, tw, t);
  } else if constexpr (M == 64) {
    direct_dft<SIGN>(v, lds, p, t);
  } else {
    constexpr int T = M / 16;
    auto chirp = [&](int e) {
      const double2 c = p.chirp[min(t + T * e, p.N - 1)];
      v[e] = SIGN < 0 ? cmul(v[e], c) : cmulc(v[e], c);
    };
#pragma unroll
    for (int e = 0; e < 8; e++) chirp(e);
    ring_fft<M, -1, false, true>(v, lds, tw, t);
    const double2* h = SIGN < 0 ? p.hf : p.hb;
    const Twiddles<M, true> rev(p.tw, t);
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = cmul(v[e], h[t + T * e]);
    ring_fft<M, +1, true, false>(v, lds, rev, t);
#pragma unroll
    for (int e = 0; e < 8; e++) chirp(e);
  }
}

// The ring (complex) or pair of rings (real) of this thread.
struct RingId {
  bool a, b;        // present
  int ta, fa, tb, fb;  // colatitude and field
};
__device__ __forceinline__ RingId ring_id(const FFTParams& p, int r) {
  RingId d;
  if (!p.real) {
    d.ta = r / p.nfield;
    d.fa = r - d.ta * p.nfield;
    d.a = d.ta < p.ntheta;
    d.b = false;
    d.tb = d.ta;
    d.fb = d.fa;
  } else {
    const int q = r / p.nfield;
    d.ta = 2 * q;
    d.tb = 2 * q + 1;
    d.fa = d.fb = r - q * p.nfield;
    d.a = d.ta < p.ntheta;
    d.b = d.tb < p.ntheta;
  }
  return d;
}

// Ring of this thread: consecutive workgroups of an XCD take consecutive
// rings, whose bins share lines of F / FA.
template <int M>
__device__ __forceinline__ int my_ring() {
  const int per = gridDim.x >> 3;
  const int b = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  return b * Ring<M>::kRings + threadIdx.x / Ring<M>::T;
}

__device__ __forceinline__ double2 ld_bin(const FFTParams& p, long i) {
  if (p.fa32) {
    const float2 x = *reinterpret_cast<const float2*>(reinterpret_cast<const float*>(p.F) + i);
    return make_double2(x.x, x.y);
  }
  return *reinterpret_cast<const double2*>(p.F + i);
}
__device__ __forceinline__ void st_bin(const FFTParams& p, long i, double2 x) {
  if (p.fa32)
    *reinterpret_cast<float2*>(reinterpret_cast<float*>(p.F) + i) =
        make_float2((float)x.x, (float)x.y);
  else
    *reinterpret_cast<double2*>(p.F + i) = x;
}

// Synthesis: order bins of F -> backward DFT -> field ring.
template <int M, int BLUE>
__global__ __launch_bounds__(Ring<M>::kThreads) void fft_synth_r(FFTParams p) {
  constexpr int T = Ring<M>::T;
  constexpr int EN = BLUE ? 8 : 16;  // N <= M / 2 with Bluestein
  __shared__ double2 lds_all[Ring<M>::kRings * Ring<M>::kStride];
  double2* lds = lds_all + (threadIdx.x / T) * Ring<M>::kStride;
  const int t = threadIdx.x % T;
  const RingId d = ring_id(p, my_ring<M>());
  const int N = p.N, cw = p.cw, ncg = (p.ncol + cw - 1) / cw;
  const Twiddles<M, false> tw(p.tw, t);
  double2 v[16];
#pragma unroll
  for (int e = 0; e < 16; e++) v[e] = make_double2(0.0, 0.0);
  if (d.a) {
    const long ba = f_index(d.ta, 0, 2 * d.fa, p.nslot, ncg, cw);
    const int la = ring_lmax(p, d.fa);
    if (!p.real) {
#pragma unroll
      for (int e = 0; e < EN; e++) {
        const int k = t + T * e;
        const bool lo = k <= la, hi = k >= N - la && k < N;
        // absent bins read slot 0 and are zeroed
        const double2 x = ld_bin(p, ba + (long)cw * (lo ? k - p.m_first : hi ? k - N - p.m_first
                                                                             : -p.m_first));
        if (lo || hi) v[e] = x;
      }
      // Bin N/2 holds orders N/2 and -N/2 when lmax = N/2.
      if (2 * la >= N && t == (N / 2) % T) {
        const double2 x = ld_bin(p, ba + (long)cw * (-N / 2 - p.m_first));
#pragma unroll
        for (int e = 0; e < EN; e++)
          if (t + T * e == N / 2) v[e] = cadd(v[e], x);
      }
    } else {
      const long bb = d.b ? f_index(d.tb, 0, 2 * d.fb, p.nslot, ncg, cw) : ba;
      const int lb = d.b ? ring_lmax(p, d.fb) : -1;
      // Hermitian spectra from bins 0 .. N/2 (c2r: Im of bins 0 and N/2 is
      // ignored): Z = X_a + i X_b.
#pragma unroll
      for (int e = 0; e < EN; e++) {
        const int k = t + T * e;
        const int kk = 2 * k <= N ? k : N - k;
        const bool oa = k < N && kk <= la, ob = k < N && kk <= lb;
        const double2 xa = ld_bin(p, ba + (oa ? (long)cw * kk : 0));
        const double2 xb = ld_bin(p, bb + (ob ? (long)cw * kk : 0));
        const double s = kk == 0 || 2 * kk == N ? 0.0 : 2 * k > N ? -1.0 : 1.0;
        // a select, not a product: the ignored parts may hold anything
        const double ya = oa && s != 0.0 ? s * xa.y : 0.0, yb = ob && s != 0.0 ? s * xb.y : 0.0;
        v[e] = make_double2((oa ? xa.x : 0.0) - yb, ya + (ob ? xb.x : 0.0));
      }
    }
  }
  ring_dft<M, BLUE, +1>(v, lds, p, tw, t);
  if (!d.a) return;
  const long oa = (long)field_index(p.fmap, d.fa) * p.fstride + (long)d.ta * N;
  if (!p.real) {
#pragma unroll
    for (int e = 0; e < EN; e++) {
      const int n = t + T * e;
      if (BLUE && n >= N) continue;
      if (p.f32)
        st_cplx<1>(p.fout, oa + n, v[e]);
      else
        st_cplx<0>(p.fout, oa + n, v[e]);
    }
  } else {
    const long ob = (long)field_index(p.fmap, d.fb) * p.fstride + (long)d.tb * N;
#pragma unroll
    for (int e = 0; e < EN; e++) {
      const int n = t + T * e;
      if (BLUE && n >= N) continue;
      if (p.f32) {
        st_real<1>(p.fout, oa + n, v[e].x);
        if (d.b) st_real<1>(p.fout, ob + n, v[e].y);
      } else {
        st_real<0>(p.fout, oa + n, v[e].x);
        if (d.b) st_real<0>(p.fout, ob + n, v[e].y);
      }
    }
  }
}

// One sample of the analysed ring: the field's, or the pointwise expression of
// the fields.
__device__ __forceinline__ double2 ld_sample(const FFTParams& p, long i) {
  if (p.src_cplx) return make_double2(cplx_part(ld_cplx<0>(p.fin, i), p.op), 0.0);
  auto load = [&](const void* b) {
    if (p.real) return make_double2(p.f32 ? ld_real<1>(b, i) : ld_real<0>(b, i), 0.0);
    return p.f32 ? ld_cplx<1>(b, i) : ld_cplx<0>(b, i);
  };
  const double2 x = load(p.fin);
  const double2 y = expr_binary(p.op) ? load(p.fin2) : make_double2(0.0, 0.0);
  return p.real ? make_double2(expr_real(p.op, x.x, y.x, p.scalar.x), 0.0)
                : expr_cplx(p.op, x, y, p.scalar);
}

// Analysis: field ring -> forward DFT -> weighted bins into FA.
template <int M, int BLUE>
__global__ __launch_bounds__(Ring<M>::kThreads) void fft_anal_r(FFTParams p) {
  constexpr int T = Ring<M>::T;
  constexpr int EN = BLUE ? 8 : 16;
  __shared__ double2 lds_all[Ring<M>::kRings * Ring<M>::kStride];
  double2* lds = lds_all + (threadIdx.x / T) * Ring<M>::kStride;
  const int t = threadIdx.x % T;
  const RingId d = ring_id(p, my_ring<M>());
  const int N = p.N, cw = p.cw;
  const Twiddles<M, false> tw(p.tw, t);
  const double wa = d.a ? p.wq[d.ta] : 0.0, wb = d.b ? p.wq[d.tb] : 0.0;
  double2 v[16];
#pragma unroll
  for (int e = 0; e < 16; e++) v[e] = make_double2(0.0, 0.0);
  if (d.a) {
    const long oa = (long)field_index(p.fmap, d.fa) * p.fstride + (long)d.ta * N;
    const long ob = d.b ? (long)field_index(p.fmap, d.fb) * p.fstride + (long)d.tb * N : oa;
    // Plain fields first: every load issued before the first use, samples past
    // the ring clamped and zeroed.
    if (!p.op && !p.src_cplx && !p.f32) {
#pragma unroll
      for (int e = 0; e < EN; e++) {
        const int n = BLUE ? min(t + T * e, N - 1) : t + T * e;
        if (!p.real)
          v[e] = ld_cplx<0>(p.fin, oa + n);
        else
          v[e] = make_double2(ld_real<0>(p.fin, oa + n), ld_real<0>(p.fin, ob + n));
      }
    } else {
#pragma unroll
      for (int e = 0; e < EN; e++) {
        const int n = BLUE ? min(t + T * e, N - 1) : t + T * e;
        v[e] = ld_sample(p, oa + n);
        if (p.real) v[e].y = ld_sample(p, ob + n).x;
      }
    }
#pragma unroll
    for (int e = 0; e < EN; e++) {
      if (p.real && !d.b) v[e].y = 0.0;
      if (BLUE && t + T * e >= N) v[e] = make_double2(0.0, 0.0);
    }
  }
  ring_dft<M, BLUE, -1>(v, lds, p, tw, t);
  const int n_cg = p.n_cg, nquad = p.nquad;
  if (!p.real) {
    if (d.a) {
      const int la = ring_lmax(p, d.fa);
      const long b0 = fa_index(-p.m_first, 2 * d.fa, d.ta, n_cg, nquad, cw);  // order 0
      const long sst = fa_index(1, 0, 0, n_cg, nquad, cw);
#pragma unroll
      for (int e = 0; e < EN; e++) {
        const int k = t + T * e;
        const bool lo = k <= la;
        if (lo || (k >= N - la && k < N))
          st_bin(p, b0 + (lo ? k : k - N) * sst, make_double2(v[e].x * wa, v[e].y * wa));
      }
      // Bin N/2 belongs to orders N/2 and -N/2 when lmax = N/2.
      if (2 * la >= N && t == (N / 2) % T) {
#pragma unroll
        for (int e = 0; e < EN; e++)
          if (t + T * e == N / 2)
            st_bin(p, b0 - N / 2 * sst, make_double2(v[e].x * wa, v[e].y * wa));
      }
    }
  } else {
    // X_a[k] = (Z[k] + conj Z[N - k]) / 2, X_b[k] = (Z[k] - conj Z[N - k]) / (2 i).
    Ring<M>::sync();
#pragma unroll
    for (int e = 0; e < EN; e++) {
      const int k = t + T * e;
      if (k < N) lds[pad(k)] = v[e];
    }
    Ring<M>::sync();
    if (d.a) {
      const int la = ring_lmax(p, d.fa), lb = d.b ? ring_lmax(p, d.fb) : -1;
      const long b0 = fa_index(0, 2 * d.fa, d.ta, n_cg, nquad, cw);
      const long b1 = fa_index(0, 2 * d.fb, d.tb, n_cg, nquad, cw);
      const long sst = fa_index(1, 0, 0, n_cg, nquad, cw);
      for (int k = t; k <= max(la, lb); k += T) {
        const double2 z = lds[pad(k)], zp = lds[pad(k == 0 ? 0 : N - k)];
        // Adjoint of the c2r synthesis: weight 2 for 0 < k < N/2, real part
        // only at k = 0 and N/2.
        const bool edge = k == 0 || 2 * k == N;
        const double hw = p.adjoint && !edge ? 1.0 : 0.5;
        double2 xa = make_double2((z.x + zp.x) * hw * wa, (z.y - zp.y) * hw * wa);
        double2 xb = make_double2((z.y + zp.y) * hw * wb, (zp.x - z.x) * hw * wb);
        if (p.adjoint && edge) xa.y = xb.y = 0.0;
        if (k <= la) st_bin(p, b0 + k * sst, xa);
        if (k <= lb) st_bin(p, b1 + k * sst, xb);
      }
    }
  }
  // The ring of the last colatitude zeroes the padding rows of its quad.
  const bool za = p.zero_pad && d.a && d.ta == p.ntheta - 1;
  const bool zb = p.zero_pad && d.b && d.tb == p.ntheta - 1;
  if (za || zb)
    for (int tp = p.ntheta; tp < 4 * nquad; tp++)
      for (int s = t; s < p.nslot; s += T) {
        if (za) st_bin(p, fa_index(s, 2 * d.fa, tp, n_cg, nquad, cw), make_double2(0.0, 0.0));
        if (zb) st_bin(p, fa_index(s, 2 * d.fb, tp, n_cg, nquad, cw), make_double2(0.0, 0.0));
      }
}

template <int M>
hipError_t go(const FFTParams& p, bool anal, hipStream_t s) {
  const long rings = (long)(p.real ? (p.ntheta + 1) / 2 : p.ntheta) * p.nfield;
  const long blocks = (rings + Ring<M>::kRings - 1) / Ring<M>::kRings;
  const dim3 grid((blocks + 7) / 8 * 8), block(Ring<M>::kThreads);
  if (p.M == p.N) {
    if (anal)
      hipLaunchKernelGGL((fft_anal_r<M, 0>), grid, block, 0, s, p);
    else
      hipLaunchKernelGGL((fft_synth_r<M, 0>), grid, block, 0, s, p);
  } else {
    if (anal)
      hipLaunchKernelGGL((fft_anal_r<M, 1>), grid, block, 0, s, p);
    else
      hipLaunchKernelGGL((fft_synth_r<M, 1>), grid, block, 0, s, p);
  }
  return hipGetLastError();
}

}  // namespace

bool ring_fft_supported(int M) { return M >= 64 && M <= 4096; }

hipError_t launch_fft_ring(const FFTParams& p0, bool anal, hipStream_t s) {
  FFTParams p = p0;
  p.n_cg = (p.ncol + p.cw - 1) / p.cw;
  p.nquad = (p.ntheta + 3) / 4;
  switch (p.M) {
    case 64: return go<64>(p, anal, s);
    case 128: return go<128>(p, anal, s);
    case 256: return go<256>(p, anal, s);
    case 512: return go<512>(p, anal, s);
    case 1024: return go<1024>(p, anal, s);
    case 2048: return go<2048>(p, anal, s);
    case 4096: return go<4096>(p, anal, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gsh
