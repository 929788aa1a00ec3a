// gsh_legendre.hip -- recurrence checkpoints, and the FP32-MFMA Legendre
// analysis, on gfx950.  (The FP64 contractions and the FP32 synthesis are in
// gsh_pair.hip.)
//
// For one order m and upper index n the reference sums, per colatitude ring,
//   analysis   c_lm = sum_i D^l_{mn}(theta_i) w_i (2 pi / N) X_m(theta_i)
//              (GaussLegendreGrid.h:181-207)
// reading D from a precomputed O(L^3) table (Wigner.h:122-130, 305-314).
// Here D is generated in registers by the three-term recurrence in l
// (Wigner.h:427-445), one lane per colatitude:
//   e_l = (a_l cos(theta) - b_l) e_{l-1} - c_l e_{l-2},   e_{l0-1} = 0,
// with e_{l0} the Ortho-normalised seed of Wigner.h:52-95 (computed on the
// host with the reference's libm expression) and (a, b, c) the recurrence
// coefficients with the Ortho factor sqrt(2l+1)/(2 sqrt(pi)) folded in.
//
// The sums over theta are dense contractions per order m: (l x theta) .
// (theta x columns), columns = (real, imaginary) x fields.  Recurrence lanes
// hold one theta each; a per-wave LDS transpose turns them into MFMA operands.
#include "gsh_internal.h"

namespace gsh {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A operand: row lane%16, k lane/16; B operand: k lane/16, column lane%16; the
// lane holding column lane%16 holds C rows 4 (lane/16) + r.
__device__ __forceinline__ f4 mma(double a, double b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32((float)a, (float)b, c, 0, 0, 0);
}

// Order handled by work index mw: complex fields take m = 0, -1, 1, -2, 2, ...
// (longest l-ranges first); real fields take m = 0, 1, 2, ...
__device__ __forceinline__ int order_of(int mw, int real) {
  return real ? mw : ((mw & 1) ? -((mw + 1) >> 1) : (mw >> 1));
}

// Coefficient index of (l, m): GSHIndices<All>(lmax, lmax, n).Index(l, m) =
// l^2 - n^2 + m + l, or GSHIndices<NonNegative>: l(l+1)/2 - |n|(|n|+1)/2 + m
// (Indexing.h:104-146).
__device__ __forceinline__ long coef_index(int l, int m, int nabs, int real) {
  return real ? (long)l * (l + 1) / 2 - (long)nabs * (nabs + 1) / 2 + m
              : (long)l * l - (long)nabs * nabs + m + l;
}

// One recurrence step with uniform coefficients q and per-lane cos.
__device__ __forceinline__ void rec_step(const d4 q, double cs, double& e0, double& e1) {
  const double t = fma(q.x, cs, -q.y);
  const double en = fma(t, e0, -(q.z * e1));
  e1 = e0;
  e0 = en;
}

// ---------------------------------------------------------------------------
// Analysis in FP32 (v_mfma_f32_16x16x4f32 on FP32-rounded operands with FP32
// accumulation; the recurrence and weights stay FP64).  Workgroup = 4 waves
// for one (order, 16-column group), covering every colatitude.  The colatitudes are cut into quads (the K=4 of one
// MFMA); each wave owns MB full blocks of 16 quads (64 lanes), wave w taking
// blocks w, w+4, ...; the leftover quads (fewer than 64) are dealt round-robin
// to the waves as a "tail" block.  Per chunk of 64 degrees each wave walks
// its blocks: the block's B operands (X'[theta][col], one per quad) sit in
// registers (the next block's are loaded while the current one runs), the
// block's recurrence advances 16 steps per 16-degree tile, an LDS transpose
// forms 16x4 A operands (16 degrees x 4 colatitudes), and MFMAs accumulate
// C[l][col].  The tail block accumulates into its own registers so the main
// accumulators never cross a branch.  The four waves' partial sums are then
// added in LDS in a fixed order.  Degrees past lmax are computed but never
// written; colatitudes past the grid have zero seeds, so their D vanish.
// ---------------------------------------------------------------------------
constexpr int kAnalLT = 4;  // 16-degree tiles per chunk

template <int MB>
__global__ __launch_bounds__(256) void leg_anal_f32(LegParams p) {
  __shared__ double tr[4][16][66];  // also holds the cross-wave reduction
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  // Work item: (order, pass, column group).
  const uint2 it = work_item(p.items, p.items_per);
  if (it.x == ~0u) return;
  const int mw = it.x;
  const int pass = it.y & 0xffff;
  const int cg = it.y >> 16;
  const int m = order_of(mw, p.real);
  const int l0 = max(abs(m), p.nabs);
  const int lmax = p.lmax;
  const int slot = m - p.m_first;
  const int krow = lane >> 4;
  const int col = cg * 16 + (lane & 15);
  const int lc = l0 + kPass * pass;  // first degree of the pass
  // Recurrence coefficients of the pass (entries lc+1 .. lc+64, 2 KiB),
  // staged in LDS.  Entries up to L + kRecPad exist.
  __shared__ uint4 rsa[128];
  const uint4* recq = reinterpret_cast<const uint4*>(p.rec + (ld_uniform(p.roff, m + p.L) - l0));
  const int tid = threadIdx.x;
  if (tid < 128) rsa[tid] = recq[2 * (lc + 1) + tid];
  __syncthreads();
  const d4* rl = reinterpret_cast<const d4*>(&rsa[0]);  // entry lc + 1 + j
  // Recurrence state at degree lc: the seed for pass 0, else the checkpoint.
  const double2* ckp = ck_rows(p, m) + ((kPass / kCk) * pass - 1) * (long)p.ntheta;
  auto state = [&](int t, double& e0_, double& e1_) {
    if (pass == 0) {
      e0_ = p.seeds[(long)(m + p.L) * p.ntheta + t];
      e1_ = 0.0;
    } else {
      const double2 s2 = ckp[t];
      e0_ = s2.x;
      e1_ = s2.y;
    }
  };
  const bool cv = col < p.ncol;
  const int lf = field_lmax(p, cv ? col >> 1 : 0);  // this column's truncation degree
  const long cbase = (long)field_index(p.fmap, cv ? col >> 1 : 0) * p.cstride;
  const int lwg = p.cg_lmax ? ld_uniform(p.cg_lmax, cg) : lmax;  // degree loop bound
  const int nt = p.ntheta;
  // B operands of this (order, column group): quad-major, 64 lanes per quad,
  // read with raw buffer loads (one lane offset register, scalar quad
  // offsets; quads past the end read as zero).
  const __amdgpu_buffer_rsrc_t fa = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.F + ((long)slot * p.n_cg + cg) * p.nquad * 64), (short)0, p.nquad * 512,
      0x00020000);
  const int voff = lane * 8;
  auto ldB = [&](int quad) -> double {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(fa, voff, quad * 512, 0));
  };

  // Full blocks: block bi of this wave starts at colatitude 64*(wave + 4*bi).
  double cs[MB > 0 ? MB : 1], e0[MB > 0 ? MB : 1], e1[MB > 0 ? MB : 1];
#pragma unroll
  for (int bi = 0; bi < MB; bi++) {
    const int t = 64 * (wave + 4 * bi) + lane;
    cs[bi] = p.cosv[t];
    state(t, e0[bi], e1[bi]);
  }
  // Tail: quads 4*w + 16*i + {0..3} after the full blocks; lane j covers
  // quad i = j/4, colatitude tail0 + 16*(j/4) + 4*wave + j%4.
  const int tail0 = 256 * MB;
  const int ntailq = (nt - tail0 + 3) >> 2;
  const int tq = (ntailq - wave + 3) >> 2;  // tail quads of this wave
  const int tt = tail0 + 16 * (lane >> 2) + 4 * wave + (lane & 3);
  const bool ttv = tt < nt;
  const int ttc = min(tt, nt - 1);
  double e0s, e1s;
  state(ttc, e0s, e1s);
  const double cs0 = p.cosv[ttc];
  double cst = ttv ? cs0 : 0.0;
  double e0t = ttv ? e0s : 0.0;
  double e1t = ttv ? e1s : 0.0;

  auto loadBlk = [&](int bi, double* Bq) {
#pragma unroll
    for (int q = 0; q < 16; q++) Bq[q] = ldB(16 * (wave + 4 * bi) + q);
  };
  // 16 recurrence steps of one block into the transpose buffer: tile lt of
  // the pass, staged coefficients rl (entry lc + 1 + j at rl[j]).
  auto steps16 = [&](const d4* rl, int lt, double cs_, double& e0_, double& e1_) {
    const d4* r = rl + 16 * lt;
#pragma unroll
    for (int k = 0; k < 16; k++) {
      tr[wave][k][lane] = e0_;
      rec_step(r[k], cs_, e0_, e1_);
    }
  };

  (void)lwg;
  {
    f4 acc[kAnalLT];
#pragma unroll
    for (int lt = 0; lt < kAnalLT; lt++) acc[lt] = f4{0.f, 0.f, 0.f, 0.f};

    double Ba[16], Bb[16];
    if (MB > 0) loadBlk(0, Ba);
#pragma unroll
    for (int bi = 0; bi < MB; bi++) {
      double* Bcur = (bi & 1) ? Bb : Ba;
      double* Bnext = (bi & 1) ? Ba : Bb;
      if (bi + 1 < MB) loadBlk(bi + 1, Bnext);
#pragma unroll
      for (int lt = 0; lt < kAnalLT; lt++) {
        steps16(rl, lt, cs[bi], e0[bi], e1[bi]);
        wave_sync();
#pragma unroll
        for (int q = 0; q < 16; q++) {
          const double A = tr[wave][lane & 15][4 * q + krow];
          acc[lt] = mma(A, Bcur[q], acc[lt]);
        }
        wave_sync();
      }
    }

    if (tq > 0) {
      f4 acct[kAnalLT];
#pragma unroll
      for (int lt = 0; lt < kAnalLT; lt++) acct[lt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int lt = 0; lt < kAnalLT; lt++) {
        steps16(rl, lt, cst, e0t, e1t);
        wave_sync();
        for (int i = 0; i < tq; i++) {
          const int q = (tail0 >> 2) + 4 * i + wave;  // global quad index
          const double Bv = ldB(q);
          const double A = tr[wave][lane & 15][4 * i + krow];
          acct[lt] = mma(A, Bv, acct[lt]);
        }
        wave_sync();
      }
#pragma unroll
      for (int lt = 0; lt < kAnalLT; lt++) acc[lt] += acct[lt];
    }

    // Cross-wave reduction in a fixed order; wave w sums degree tile w.
    double* red = &tr[0][0][0];
    __syncthreads();
#pragma unroll
    for (int lt = 0; lt < kAnalLT; lt++)
#pragma unroll
      for (int r = 0; r < 4; r++) red[((wave * kAnalLT + lt) * 4 + r) * 64 + lane] = acc[lt][r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int lt = wave;
      double s = red[((0 * kAnalLT + lt) * 4 + r) * 64 + lane];
      s += red[((1 * kAnalLT + lt) * 4 + r) * 64 + lane];
      s += red[((2 * kAnalLT + lt) * 4 + r) * 64 + lane];
      s += red[((3 * kAnalLT + lt) * 4 + r) * 64 + lane];
      const int l = lc + 16 * lt + 4 * krow + r;
      if (cv && l <= lf) {
        const long ci = (cbase + coef_index(l, m, p.nabs, p.real)) * 2 + (col & 1);
        double v = s;
        if (p.accumulate) v += p.cout[ci];
        if (p.zero_last && lf == p.L && l == lf && m == lf) v = 0.0;
        p.cout[ci] = v;
      }
    }
  }
}

template <int MB>
hipError_t launch_anal(const LegParams& p, hipStream_t s) {
  hipLaunchKernelGGL((leg_anal_f32<MB>), dim3(8 * p.items_per), dim3(256), 0, s, p);
  return hipGetLastError();
}

// Recurrence checkpoints: order m = m_first + blockIdx.y runs its recurrence
// for 256 colatitudes per workgroup from the seed at l0 and stores the state
// (e_l, e_{l-1}) at l = l0 + kCk k, k = 1 .. nck - 1, with the same
// arithmetic as the transform kernels.  The coefficients are staged in LDS
// 64 degrees at a time (all threads of the workgroup share the order).
//
// Scaling against underflow: a seed below the normal range (far from the
// turning point, high degree) starts scaled, e = sseed = seed * 2^k; the
// recurrence is linear and homogeneous, so the scaled state runs the same
// steps, and whenever |e_l| passes 2^600 both values are divided by 2^600
// (exactly) and k drops by as much, until k = 0.  The stored states are the
// unscaled ones, e * 2^-k: zero while they are below the double range, and
// accurate once the order's values rise toward significance.  Lanes with
// k = 0 take exactly the steps of the transform kernels.
__global__ __launch_bounds__(256) void rec_checkpoints(LegParams p) {
  const int m = p.m_first + blockIdx.y;
  const int mi = m + p.L;
  const int l0 = max(abs(m), p.nabs);
  const int nt = p.ntheta;
  const int t = blockIdx.x * 256 + threadIdx.x;
  const int tc = min(t, nt - 1);
  const double cs = p.cosv[tc];
  double e0 = p.seeds[(long)mi * nt + tc], e1 = 0.0;
  int kk = p.skexp ? p.skexp[(long)mi * nt + tc] : 0;
  if (kk > 0) e0 = p.sseed[(long)mi * nt + tc];
  int kfirst = kk == 0 && fabs(e0) >= kNegligible ? 0 : 0x7fff;  // first state that matters
  const int nck = (p.L - l0 + kCk) / kCk;
  __shared__ uint4 rs[128];
  const uint4* recq = reinterpret_cast<const uint4*>(p.rec + (ld_uniform(p.roff, mi) - l0));
  double2* out = const_cast<double2*>(ck_rows(p, m));
  // Entries up to L + kRecPad exist, so staging 64 entries past any
  // checkpoint's start stays in bounds.
  for (int k = 1; k < nck; k++) {
    const int lp = l0 + kCk * (k - 1);
    const int j0 = (k - 1) % (64 / kCk) * kCk;  // position in the staged 64
    if (j0 == 0) {
      __syncthreads();
      if (threadIdx.x < 128) rs[threadIdx.x] = recq[2 * (lp + 1) + threadIdx.x];
      __syncthreads();
    }
    const d4* rl = reinterpret_cast<const d4*>(rs) + j0;
#pragma unroll
    for (int j = 0; j < kCk; j++) {
      rec_step(rl[j], cs, e0, e1);
      if (kk > 0 && fabs(e0) > 0x1p+600) {
        const int r = min(kk, 600);
        e0 = ldexp(e0, -r);
        e1 = ldexp(e1, -r);
        kk -= r;
      }
    }
    const double s0 = kk > 0 ? ldexp(e0, -kk) : e0;
    const double s1 = kk > 0 ? ldexp(e1, -kk) : e1;
    if (kfirst == 0x7fff && (fabs(s0) >= kNegligible || fabs(s1) >= kNegligible)) kfirst = k;
    if (t < nt) out[(long)(k - 1) * nt + t] = make_double2(s0, s1);
  }
  // The degrees after the last state are stored nowhere, so an order whose
  // states are all negligible runs them too (entries past L are zero).
  if (kfirst == 0x7fff) {
    const d4* rl = reinterpret_cast<const d4*>(recq) + l0 + kCk * (nck - 1) + 1;
    double big = 0.0;
    for (int j = 0; j < kCk; j++) {
      rec_step(rl[j], cs, e0, e1);
      big = fmax(big, fabs(e0));
    }
    if (ldexp(big, -kk) >= kNegligible) kfirst = nck;
  }
  // kf: the checkpoint before the first state that matters at any of 16 rows
  // (the degrees up to it are negligible: below the turning point the values
  // of an order rise with the degree).
  if (t >= nt) kfirst = 0x7fff;
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) kfirst = min(kfirst, __shfl_xor(kfirst, d));
  if ((threadIdx.x & 15) == 0 && t < nt)
    p.kf_out[(long)mi * p.nrt + (t >> 4)] =
        static_cast<unsigned short>(kfirst == 0x7fff ? kfirst : max(kfirst - 1, 0));
}

}  // namespace

hipError_t launch_rec_checkpoints(const LegParams& p, int norder, hipStream_t s) {
  hipLaunchKernelGGL(rec_checkpoints, dim3((p.ntheta + 255) / 256, norder), dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_leg_anal_f32(const LegParams& p0, hipStream_t s) {
  if (!p0.ck || !p0.ckoff || (!p0.real && !p0.ckn)) return hipErrorInvalidValue;  // tables required
  LegParams p = p0;
  p.n_cg = (p.ncol + 15) / 16;
  p.nquad = (p.ntheta + 3) / 4;
  const int mb = p.nquad / 64;  // full 16-quad blocks per wave
  switch (mb) {
    case 0: return launch_anal<0>(p, s);
    case 1: return launch_anal<1>(p, s);
    case 2: return launch_anal<2>(p, s);
    case 3: return launch_anal<3>(p, s);
    case 4: return launch_anal<4>(p, s);
    case 5: return launch_anal<5>(p, s);
    case 6: return launch_anal<6>(p, s);
    case 7: return launch_anal<7>(p, s);
    case 8: return launch_anal<8>(p, s);
    case 9: return launch_anal<9>(p, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gsh
