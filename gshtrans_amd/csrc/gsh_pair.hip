// gsh_pair.hip -- FP64 Legendre contractions (and the FP32-MFMA synthesis)
// over orders m >= 0, one workgroup for both orders m and -m.
//
// The recurrence values of order m >= 0 serve order -m as well, on the
// equatorially symmetric Gauss-Legendre nodes (Wigner.h:52-95, 386-472):
//   n = 0   d^l_{-m,0}(t) = (-1)^m d^l_{m,0}(t), and the parity
//           d^l_{m,0}(pi - t) = (-1)^(l+m) d^l_{m,0}(t): the sums run over the
//           northern rows only, degrees of even and odd l + m apart (SYM = 1);
//   n != 0  d^l_{-m,n}(t) = (-1)^(l+n) d^l_{m,n}(pi - t): order -m reads or
//           writes the mirrored rows with signed coefficients (SYM = 0).
// So an item's columns are "virtual": 2 nfield columns of order m, then as
// many of order -m (complex fields, m > 0).
//
// What bounds these kernels: on this chip FP64 MFMA and FP64 vector
// instructions share one pipe (a half-and-half mix of both runs at the sum of
// their times, 61 of 68 TFLOP/s), so every recurrence step is paid in MFMA
// time.  The four waves of a workgroup therefore share the recurrence values
// through LDS: each value is computed once for up to 64 (synthesis) or 128 virtual
// columns (3 FP64 instructions against as many multiply-adds), 16 degrees at a time from
// the checkpoint table, one chunk ahead of the MFMAs that use it.
//
// Near the poles d^l_{mn} is evanescent for l < m / sin t.  Values of the 16
// degrees from a checkpoint count as zero at the 16 rows of a tile where all of
// them, and all at lower degrees, are below 2^-120: kf[order][row tile] holds the
// first checkpoint that counts, and blocks of zeros are left out of the MFMAs (at
// lMax = 1024 a fifth of the work).  So a sum over coefficients c is off by at
// most 2^-120 sum |c| of the terms left out, which is below the rounding of any
// larger term; a field of high orders only has zeros near the poles where its
// values are that small.  What is left out does not depend on how a batch is
// tiled: a synthesis that starts at an earlier degree for another of its row tiles
// multiplies by zeros, and an analysis leaves out the rows of a whole pass of 128
// degrees.  Inf and NaN of the terms left out still reach the result (added as
// 0 * value).
#include <algorithm>
#include <type_traits>

#include "gsh_internal.h"

namespace gsh {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// The matrix instruction: CT columns per tile, 16 rows, K = 4; the lane
// holding column col(lane) holds the NR rows row(lane, r).  A operand: row
// lane % 16, k lane / 16; B operand: k lane / 16, column col(lane).
//   0  v_mfma_f64_16x16x4_f64
//   1  v_mfma_f32_16x16x4_f32 on FP32-rounded operands
//   2  v_mfma_f64_4x4x4_4b_f64: four blocks of 4 rows against the same 4
//      columns, a quarter of the time of 0 (for calls of few columns)
template <int KIND>
struct Mma;
template <>
struct Mma<0> {
  typedef double elem;
  typedef d4 acc;
  static constexpr int CT = 16, NR = 4;
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
  static __device__ __forceinline__ double get(const acc& c, int r) { return c[r]; }
  static __device__ __forceinline__ void add(acc& c, double v) { c += v; }
};
template <>
struct Mma<1> {
  typedef float elem;
  typedef f4 acc;
  static constexpr int CT = 16, NR = 4;
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  static __device__ __forceinline__ double get(const acc& c, int r) { return c[r]; }
  static __device__ __forceinline__ void add(acc& c, float v) { c += v; }
};
template <>
struct Mma<2> {
  typedef double elem;
  typedef double acc;
  static constexpr int CT = 4, NR = 1;
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int) {
    return 4 * ((lane >> 2) & 3) + (lane >> 4);
  }
  static __device__ __forceinline__ double get(const acc& c, int) { return c; }
  static __device__ __forceinline__ void add(acc& c, double v) { c += v; }
};

// One recurrence step with uniform coefficients {a, b, c} and per-lane cos.
__device__ __forceinline__ void rec_step(double2 ab, double c, double cs, double& e0, double& e1) {
  const double t = fma(ab.x, cs, -ab.y);
  const double en = fma(t, e0, -(c * e1));
  e1 = e0;
  e0 = en;
}

// Coefficient index of (l, m), as in Indexing.h:104-146.
__device__ __forceinline__ int coef_index(int l, int m, int nabs, int real) {
  return real ? l * (l + 1) / 2 - nabs * (nabs + 1) / 2 + m : l * l - nabs * nabs + m + l;
}

// Work item of this workgroup: (m, sub | group << 16, first checkpoint row of
// order m, first recurrence entry of order m).  The offsets travel with the
// item, so that nothing waits for a table of them.
__device__ __forceinline__ uint4 pair_item(const LegParams& p) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  const int b = blockIdx.x;
  const u4 v = ld_uniform(reinterpret_cast<const u4*>(p.items), (long)(b & 7) * p.items_per + (b >> 3));
  return make_uint4(v.x, v.y, v.z, v.w);
}

// A virtual column of an item: order sign, column, the column's field and its
// truncation degree.  Columns past the last read column 0 and store nothing.
struct VCol {
  bool valid;
  int sgn;  // 1: order -m
  int col;  // 2 field + part
  int lf;   // truncation degree
  int field;
};
// Virtual column v of order m.  Wide launches (vint) interleave tiles of 16
// columns of order m and of order -m, so that a tile has one order sign and a
// workgroup's columns belong to few fields; narrow ones append the columns of
// order -m to those of order m.
__device__ __forceinline__ VCol vcol(const LegParams& p, int v, int m) {
  VCol c;
  const bool two = p.pair && m > 0;
  if (p.vint) {
    c.sgn = p.pair ? (v >> 4) & 1 : 0;
    c.col = p.pair ? (v >> 5) * 16 + (v & 15) : v;
    c.valid = c.col < p.ncol && (two || !c.sgn);
  } else {
    c.valid = v < (two ? 2 * p.ncol : p.ncol);
    c.sgn = v >= p.ncol ? 1 : 0;
    c.col = v - c.sgn * p.ncol;
  }
  if (!c.valid) c.col = c.sgn = 0;
  c.lf = field_lmax(p, c.col >> 1);
  c.field = field_index(p.fmap, c.col >> 1);
  return c;
}
// Largest truncation degree of the virtual columns v0 .. v0 + nv - 1, the
// first a multiple of 32 when interleaved: the fields of a batch of uneven
// truncation are ordered by descending degree.
__device__ __forceinline__ int vcol_lmax(const LegParams& p, int v0, int nv, int m) {
  int col = v0;
  if (p.vint && p.pair)
    col = (v0 >> 5) * 16;
  else if (p.pair && m > 0 && v0 < p.ncol && v0 + nv > p.ncol)
    col = 0;
  else
    col = v0 % p.ncol;
  return field_lmax(p, min(col, p.ncol - 1) >> 1);
}
// Minimum over the 16 lanes of a row (the four rows alike; wave-uniform).
__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) v = min(v, __shfl_xor(v, d));
  return __builtin_amdgcn_readfirstlane(v);
}


// Narrow tiles multiply for a few hundred cycles per chunk, which hides
// neither a load nor the barrier: they keep one D buffer (two barriers per
// chunk) and run three or four workgroups per CU instead of two.
constexpr int nbuf(int kind, int tiles) { return kind == 2 || tiles <= 2 ? 1 : 2; }
// Workgroups per CU (waves per SIMD) that the registers are cut to.
constexpr int waves(int kind, int tiles, int nj) {
  return nbuf(kind, tiles) == 2 ? 2 : kind != 2 && nj == 2 ? 3 : 4;
}
// The same for the synthesis: waves of one column tile keep one D buffer too
// (32 and 64 columns, two buffers and two workgroups: lMax=1000, n=2, 16 and 32
// real fields 817 and 1356 us, one and three 697 and 1174 us).
constexpr int synth_nbuf(int kind, int sym, int tiles, int nj) {
  return !sym && nj == 1 ? 1 : nbuf(kind, tiles);
}
constexpr int synth_waves(int kind, int sym, int tiles, int nj) {
  if (sym || nj == 2 || tiles <= 2 || kind == 2) return waves(kind, tiles, sym ? 2 : nj);
  return kind == 0 ? 3 : tiles <= 4 ? 4 : 2;
}

// ---------------------------------------------------------------------------
// Synthesis.  An item is (m, row block, group of virtual columns); the 4
// waves share the D values of (32 degrees) x (RT WR + 1 row tiles) and split
// the tile: WR row groups of RT row tiles x WC column groups of NJ column
// tiles.  Wave w produces degrees 16 (w / 2) .. + 15 of each chunk for 64
// rows (blocks of 16 row tiles: chunks of 16 degrees, 64 rows each wave); the
// last row group takes one row tile more where the block has it (ntheta = 2^k
// + 1 would otherwise leave a block of one row).  SYM: one
// column tile per wave, the even and odd degrees in accumulators of their own.
//
// Beside the MFMAs every vector instruction costs about 3 of an MFMA's 72
// cycles (measured, two waves per SIMD), so the coefficient loads step one
// byte offset per 4 degrees and mask nothing until a column's last degrees.
// A load of B operands is 32 pieces of 16 bytes (4 degrees of 8 fields), 32
// cycles of the CU's address path, so it has to serve many row tiles: waves of 4
// row tiles x 1 column tile for 32 columns and of 8 x 1 for 64, where 2 x 2 and
// 4 x 2 fetched each operand twice (lMax=1000, n=2, 16 real fields 904 -> 697 us, 32
// fields 1340 -> 1174 us; 64 fields in two groups of 64 columns take 2305 us, 2378
// in one of 8 x 2).  FP32, whose products take half the time, gains from the
// shared production of 128 columns (lMax=1000, 64 complex fields 3180 us, 3240).
// Bound: FP64 MFMA, 47 of 71 TFLOP/s of the products issued.  lMax=1024, 64
// fields: 7.21 -> 4.97 ms (complex, n=2) and 3.55 -> 1.56 ms (real, n=0) against
// a kernel that ran the recurrence of every order for every 32 columns; FP32
// 3.98 -> 2.50 ms, the mean of both.
// ---------------------------------------------------------------------------
template <int KIND, int SYM, int RT, int NJ, int WR>
__global__ __launch_bounds__(256, synth_waves(KIND, SYM, RT, NJ)) void leg_synth_p(LegParams p) {
  typedef Mma<KIND> M;
  typedef typename M::elem E;
  constexpr int WC = 4 / WR;
  constexpr int TW = RT * WR;      // row tiles of a block without the extra one
  constexpr int NH = TW <= 8 ? 2 : 1;  // 16-degree segments of a chunk
  constexpr int SC = kCk * NH;     // degrees per chunk
  constexpr int PW = 4 / NH;       // waves that produce a segment, 64 rows each
  static_assert(16 * TW <= 64 * PW, "every row of a block is produced");
  // Elements per degree row in LDS: 9 (17) row tiles, padded so that the A
  // operands of both forms spread over all banks.
  constexpr int SP = TW <= 8 ? 152 : 280;
  constexpr int NB = SYM ? 2 : NJ; // accumulators per row tile
  constexpr int NC = SYM ? 1 : NJ; // column tiles per wave
  constexpr int NBUF = synth_nbuf(KIND, SYM, RT, NJ);
  __shared__ E D[NBUF][SC * SP];
  __shared__ uint4 rs[2][2 * SC];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint4 it = pair_item(p);
  if (it.x == ~0u) return;
  const int wr = wave / WC, wc = wave % WC;
  const int m = it.x, tb = it.y & 0xffff, cg = it.y >> 16;
  const int nt = p.ntheta, nr = SYM ? (nt + 1) / 2 : nt;
  const int rtt = (nr + 15) >> 4;
  // Blocks 0 .. next - 1 have TW + 1 row tiles, the others TW.
  const int next = max(0, rtt - p.n_tsb * TW);
  const int tile0 = tb * TW + min(tb, next);
  const int ntile = min(TW + (tb < next ? 1 : 0), rtt - tile0);
  const bool ext = ntile > TW;
  const int l0 = max(m, p.nabs);
  const int krow = lane >> 4;

  // Columns of this wave.
  const int vb = cg * (WC * NC * M::CT);  // first virtual column of the block
  VCol vc[NC];
  const char* cbase[NC];  // (l, m) of order m at cbase + 16 coef_index(l, m)
  int lmin = 1 << 20, lww = -1;  // smallest and largest degree of the wave's columns
#pragma unroll
  for (int j = 0; j < NC; j++) {
    vc[j] = vcol(p, vb + (wc * NC + j) * M::CT + lane % M::CT, m);
    cbase[j] = reinterpret_cast<const char*>(p.cin + (long)vc[j].field * p.cstride * 2 +
                                             (vc[j].col & 1)) -
               (vc[j].sgn ? 32l * m : 0);
    lmin = min(lmin, vc[j].lf);
    lww = max(lww, vc[j].valid ? vc[j].lf : -1);
  }
  lmin = wave_min(lmin);
  lww = -wave_min(-lww);
  const int lwg = vcol_lmax(p, vb, WC * NC * M::CT, m);

  // First checkpoint that counts at any of the block's rows.
  const unsigned short* kfm = p.kf + (long)(m + p.L) * p.nrt;
  const int kfl = kfm[tile0 + min(lane & 31, ntile - 1)];  // lane i: row tile i
  int ks = wave_min(kfl);  // tiles 0 .. 15
  if (TW > 15) ks = min(ks, __builtin_amdgcn_readlane(kfl, 16));
  ks = min(ks, max(0, lwg - l0 + kCk) / kCk);
  const int ls = l0 + kCk * ks;
  const int nchunk = ls > lwg ? 0 : (lwg - ls + SC) / SC;

  // Coefficient loads: accumulator b reads degree l + d (d = krow, or SYM
  // 2 krow + b) of every ST-th degree l, GB loads per 16 degrees.  A group
  // of 16 degrees from l with l + 15 <= lmin is inside every column's degrees
  // (plain()); its byte offset off[b] steps by an arithmetic progression.  The
  // others clamp each load to a valid address, and operand() masks them.
  constexpr int ST = SYM ? 8 : 4;
  constexpr int GB = SYM ? 2 : 4;
  constexpr int NO = SYM ? 2 : 1;  // offsets: order -m shares order m's
  unsigned off[NO], step[NO];
  unsigned sgn[NC];  // sign bit of order -m (SYM0: the parity of l is the lane's)
#pragma unroll
  for (int b = 0; b < NO; b++) {
    const int l = l0 + (SYM ? 2 * krow + b : krow);
    off[b] = 16u * coef_index(l, m, p.nabs, p.real);
    step[b] = (SYM ? 16 * l + 72 : 8 * l + 20) * (p.real ? 8u : 16u);
  }
  const unsigned sinc = (SYM ? 128 : 32) * (p.real ? 8u : 16u);
#pragma unroll
  for (int j = 0; j < NC; j++)
    sgn[j] = vc[j].sgn && ((SYM ? m : l0 + krow + p.n) & 1) ? 0x80000000u : 0u;
  auto plain = [&](int l) { return l + kCk - 1 <= lmin; };
  auto load_group = [&](int l, double (&B)[GB][NB]) {
    if (plain(l)) {
#pragma unroll
      for (int g = 0; g < GB; g++) {
#pragma unroll
        for (int b = 0; b < NB; b++)
          B[g][b] = *reinterpret_cast<const double*>(cbase[SYM ? 0 : b] + off[SYM ? b : 0]);
#pragma unroll
        for (int b = 0; b < NO; b++) {
          off[b] += step[b];
          step[b] += sinc;
        }
      }
    } else {
#pragma unroll
      for (int g = 0; g < GB; g++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const VCol& c = vc[SYM ? 0 : b];
          const int ll = min(l + ST * g + (SYM ? 2 * krow + b : krow), c.lf);
          // A field without a degree of this order reads its element 0.
          const long o = c.lf >= l0 ? 16l * coef_index(ll, m, p.nabs, p.real) : c.sgn ? 32l * m : 0;
          B[g][b] = *reinterpret_cast<const double*>(cbase[SYM ? 0 : b] + o);
        }
    }
  };
  // Operand of accumulator b from the raw load of group g of the 16 degrees
  // from l (mask: not plain(l)).  SYM: the sign of order -m goes to the result.
  auto operand = [&](auto mask, double v, int b, int l, int g) -> E {
    if (!SYM) {
      uint2 u = __builtin_bit_cast(uint2, v);
      u.y ^= sgn[SYM ? 0 : b];
      v = __builtin_bit_cast(double, u);
    }
    if (decltype(mask)::value && l + ST * g + (SYM ? 2 * krow + b : krow) > vc[SYM ? 0 : b].lf)
      v = 0.0;
    return (E)v;
  };

  // Degrees left out: 0 * value.
  E pz[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) pz[b] = (E)0;
  for (int l = l0; l < ls; l += kCk) {
    double t[GB][NB];
    load_group(l, t);
#pragma unroll
    for (int g = 0; g < GB; g++)
#pragma unroll
      for (int b = 0; b < NB; b++) pz[b] += (E)0 * operand(std::true_type{}, t[g][b], b, l, g);
  }

  // Production: wave -> (16-degree segment, 64 rows), and for the extra row
  // tile lanes 0..15 of the segment's first wave.
  const int seg = wave / PW;
  const int prow = 64 * (wave % PW) + lane;
  const bool xprod = ext && 16 * TW == 64 * PW && wave % PW == 0;
  constexpr int XR = 16 * TW;  // first row of the extra tile
  const int t = 16 * tile0 + prow, tx = 16 * tile0 + XR + (lane & 15);
  const bool tv = t < nr, txv = xprod && lane < 16 && tx < nr;
  const double cs = tv ? p.cosv[t] : 0.0, csx = txv ? p.cosv[tx] : 0.0;
  const int nck = (p.L - l0 + kCk) / kCk;  // checkpoints 1 .. nck - 1 exist
  // First checkpoints that count at the wave's four row tiles and at the extra
  // one, in scalar registers (a per-lane copy of them costs the widest tiles 3%,
  // loads of their own 0.2 us of a small launch); from kmax on all of them count.
  int kt[5];
#pragma unroll
  for (int i = 0; i < 4; i++) kt[i] = __builtin_amdgcn_readlane(kfl, 4 * (wave % PW) + i);
  kt[4] = __builtin_amdgcn_readlane(kfl, TW);
  const int kmax = max(max(max(kt[0], kt[1]), max(kt[2], kt[3])), kt[4]);
  const unsigned long long rows = __ballot(tv), rowsx = __ballot(txv);
  const double* seedm = p.seeds + (long)(m + p.L) * nt;
  const double2* ckm = p.ck + (long)it.z * nt;
  auto state = [&](int c, bool extra, int row) -> double2 {
    const int k = ks + NH * c + seg;
    unsigned long long live = k < nck ? extra ? rowsx : rows : 0;
    if (k < kmax) {
      if (extra) {
        live = k < kt[4] ? 0 : live;
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) live &= k < kt[i] ? ~(0xffffull << (16 * i)) : ~0ull;
      }
    }
    double2 s = make_double2(0.0, 0.0);
    if (__builtin_amdgcn_inverse_ballot_w64(live)) {
      if (k == 0)
        s.x = seedm[row];
      else
        s = ckm[(long)(k - 1) * nt + row];
    }
    return s;
  };
  const uint4* recq = reinterpret_cast<const uint4*>(p.rec + ((long)it.w - l0));
  auto fetch_rec = [&](int c) {
    return tid < 2 * SC ? recq[2 * (ls + SC * c + 1) + tid] : make_uint4(0, 0, 0, 0);
  };
  auto produce = [&](int c, double2 s, double csv, int row) {
    const double2* r = reinterpret_cast<const double2*>(rs[c & 1]) + 2 * kCk * seg;
    E* d = D[NBUF == 2 ? c & 1 : 0] + (kCk * seg) * SP + row;
    double e0 = s.x, e1 = s.y;
#pragma unroll 4
    for (int j = 0; j < kCk; j++) {
      d[j * SP] = (E)e0;
      rec_step(r[2 * j], r[2 * j + 1].x, csv, e0, e1);
    }
  };

  typename M::acc acc[RT + 1][NB];
#pragma unroll
  for (int i = 0; i <= RT; i++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[i][b] = typename M::acc{};
  const bool xt = ext && wr == WR - 1;  // this wave has the extra row tile

  double B[NH][GB][NB];
  // MFMAs of the 16 degrees from l (half h of chunk c) for N row tiles: no
  // branch inside, so that the LDS reads of later steps overlap the MFMAs.
  auto mma_group = [&](auto nrow, auto mask, int c, int h, double (&Bh)[GB][NB]) {
    constexpr int N = decltype(nrow)::value;
    const int l = ls + SC * c + kCk * h;
    const E* d = D[NBUF == 2 ? c & 1 : 0] + (kCk * h) * SP + 16 * (wr * RT) + (lane & 15);
#pragma unroll
    for (int g = 0; g < GB; g++) {
      E X[NB];
#pragma unroll
      for (int j = 0; j < NB; j++) X[j] = operand(mask, Bh[g][j], j, l, g);
#pragma unroll
      for (int b = 0; b < (SYM ? 2 : 1); b++) {
        const E* dr = d + (SYM ? 8 * g + 2 * krow + b : 4 * g + krow) * SP;
#pragma unroll
        for (int i = 0; i < N; i++) {
          const E A = dr[16 * i];
          if (SYM) {
            acc[i][b] = M::mma(A, X[b], acc[i][b]);
          } else {
#pragma unroll
            for (int j = 0; j < NB; j++) acc[i][j] = M::mma(A, X[j], acc[i][j]);
          }
        }
      }
    }
  };

  if (nchunk > 0) {
#pragma unroll
    for (int h = 0; h < NH; h++) load_group(ls + kCk * h, B[h]);
    double2 st = state(0, false, t), sx = state(0, true, tx);
    if (tid < 2 * SC) rs[0][tid] = fetch_rec(0);
    uint4 rq = make_uint4(0, 0, 0, 0);
    __syncthreads();
    // Chunk c + 1 is produced (NBUF 1: chunk c) while its state and
    // recurrence coefficients for the chunk after it are on their way.
    auto advance = [&](int c) {
      produce(c, st, cs, prow);
      if (xprod && lane < 16) produce(c, sx, csx, XR + lane);
      if (c + 1 < nchunk) {
        st = state(c + 1, false, t);
        sx = state(c + 1, true, tx);
        // rs[(c + 1) & 1] was last read producing chunk c - 1, a barrier ago.
        if (tid < 2 * SC) rs[(c + 1) & 1][tid] = rq;
        if (c + 2 < nchunk) rq = fetch_rec(c + 2);
      }
    };
    if (nchunk > 1) rq = fetch_rec(1);
    if (NBUF == 2) advance(0);
    // The chunks inside every column's degrees, then the others.
    const int nplain = min(nchunk, max(0, lmin + 1 - ls) / SC);
    auto run = [&](auto nrow, auto mask, int ca, int cb) {
      for (int c = ca; c < cb; c++) {
        __syncthreads();
        if (NBUF == 2) {
          if (c + 1 < nchunk) advance(c + 1);
        } else {
          advance(c);
          __syncthreads();
        }
#pragma unroll
        for (int h = 0; h < NH; h++) {
          if (!decltype(mask)::value || ls + SC * c + kCk * h <= lww)
            mma_group(nrow, mask, c, h, B[h]);
          if (ls + SC * (c + 1) + kCk * h <= lww) load_group(ls + SC * (c + 1) + kCk * h, B[h]);
        }
      }
    };
    if (xt) {
      run(std::integral_constant<int, RT + 1>{}, std::false_type{}, 0, nplain);
      run(std::integral_constant<int, RT + 1>{}, std::true_type{}, nplain, nchunk);
    } else {
      run(std::integral_constant<int, RT>{}, std::false_type{}, 0, nplain);
      run(std::integral_constant<int, RT>{}, std::true_type{}, nplain, nchunk);
    }
  }

  // 0 * (degrees left out), summed over the operand rows of each column.
  if (ls > l0) {
#pragma unroll
    for (int b = 0; b < NB; b++) {
      E z = pz[b];
      z += __shfl_xor(z, 16);
      z += __shfl_xor(z, 32);
#pragma unroll
      for (int i = 0; i <= RT; i++) M::add(acc[i][b], z);
    }
  }

  // Store: order m at row t, order -m at the mirrored row (n != 0).
  const long frow = f_index(1, 0, 0, p.nslot, (p.ncol + p.cw - 1) / p.cw, p.cw);  // F per row
#pragma unroll
  for (int j = 0; j < NC; j++) {
    if (!vc[j].valid) continue;
    double* f = p.F + f_index(0, (vc[j].sgn ? -m : m) - p.m_first, vc[j].col, p.nslot, 0, p.cw);
    const bool mirrored = !SYM && vc[j].sgn;
#pragma unroll
    for (int i = 0; i <= RT; i++) {
      if (i == RT && !xt) continue;
#pragma unroll
      for (int r = 0; r < M::NR; r++) {
        const int tr = 16 * (wr * RT + i) + M::row(lane, r);
        const int row = 16 * tile0 + tr;
        if (tr >= 16 * ntile || row >= nr) continue;
        if (SYM) {
          double e = M::get(acc[i][0], r), o = M::get(acc[i][1], r);
          if (sgn[j]) {
            e = -e;
            o = -o;
          }
          f[row * frow] = e + o;
          if (nt - 1 - row != row) f[(nt - 1 - row) * frow] = e - o;
        } else {
          f[(mirrored ? nt - 1 - row : row) * frow] = M::get(acc[i][j], r);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Analysis.  An item is (m, pass, group of virtual columns): a pass covers up
// to 128 degrees (nu units of 32), walking the rows in chunks of 32.  Thread
// (seg, row) produces 16 degrees of the next chunk from its checkpoint.  The 4 waves
// split the pass: WR degree groups of LT tiles x WC column groups of NJ tiles.
// SYM: the rows run over the north, a degree tile holds 16 degrees of one
// parity, multiplied with X(t) +- X(nt-1-t).
// Bound: FP64 MFMA, 52 of 71 TFLOP/s of the products issued; without the bin
// loads it takes 12% less, without the stores 6%, without the recurrence 5%.
// lMax=1024, 64 fields: mean of complex n=2 and real n=0 5.58 -> 2.86 ms.
// ---------------------------------------------------------------------------
template <int KIND, int SYM, int LT, int NJ>
__global__ __launch_bounds__(256, waves(KIND, LT, NJ)) void leg_anal_p(LegParams p) {
  typedef Mma<KIND> M;
  constexpr int WR = 8 / LT, WC = 4 / WR;
  constexpr int NBUF = nbuf(KIND, LT);
  constexpr int PD = 128;             // degrees per pass
  constexpr int PU = PD / 32;         // units per pass
  constexpr int CR = 32;              // rows per chunk
  constexpr int AP = CR + 2;          // elements per degree row in LDS
  constexpr int NQ = CR / 4;          // quads per chunk
  __shared__ double D[NBUF][PD * AP];
  __shared__ uint4 rs[2 * PD];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint4 it = pair_item(p);
  if (it.x == ~0u) return;
  const int wr = wave / WC, wc = wave % WC;
  const int m = it.x, pass = it.y & 0xffff, cg = it.y >> 16;
  const int nt = p.ntheta, nr = SYM ? (nt + 1) / 2 : nt;
  const int l0 = max(m, p.nabs);
  const int krow = lane >> 4;
  const int vb = cg * (WC * NJ * M::CT);
  // B operands: row 4 q + krow (mirrored for order -m; SYM: the row and its
  // mirror) of a column of FA, whose rows are cw elements apart.
  constexpr int NL = SYM ? 2 * NJ : NJ;
  const int cw = KIND == 0 && NJ == 2 ? 16 : p.cw;  // more than 8 columns: 16
  VCol vc[NJ];
  const double* fb[NL];  // lane's row of quad 0
  int fs[NL];            // elements per quad
  int lw = -1;           // largest degree of this wave's columns
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    vc[j] = vcol(p, vb + (wc * NJ + j) * M::CT + lane % M::CT, m);
    const int slot = (vc[j].sgn ? -m : m) - p.m_first;
    const double* f0 = p.F + fa_index(slot, vc[j].col, 0, p.n_cg, p.nquad, cw);
    if (SYM) {
      fb[2 * j] = f0 + cw * krow;
      fs[2 * j] = 4 * cw;
      fb[2 * j + 1] = f0 + cw * (nt - 1 - krow);
      fs[2 * j + 1] = -4 * cw;
    } else {
      fb[j] = vc[j].sgn ? f0 + cw * (nt - 1 - krow) : f0 + cw * krow;
      fs[j] = vc[j].sgn ? -4 * cw : 4 * cw;
    }
    lw = max(lw, vc[j].valid ? vc[j].lf : -1);
  }
  lw = -wave_min(-lw);
  const int lwg = vcol_lmax(p, vb, WC * NJ * M::CT, m);
  if (l0 > lwg) return;
  // Units of 32 degrees, PU to a pass (the last pass takes what is left).
  const int U = (lwg - l0 + 32) >> 5;
  const int u0 = PU * pass, nu = min(U - u0, PU);
  if (nu <= 0) return;
  const int lp = l0 + 32 * u0;

  // Rows that count for a whole pass, whatever part of it this group's degrees
  // fill: chunks c0 .. c1 (chunks past 64 always run).
  const int nch = (nr + CR - 1) / CR;
  const int nrt = (nr + 15) >> 4;
  const unsigned short* kf = p.kf + (long)(m + p.L) * p.nrt;
  int c0, c1 = nch - 1;
  {
    const int kend = 2 * (u0 + PU);
    bool live = false;
    if (lane < nch)
#pragma unroll
      for (int i = 0; i < CR / 16; i++) live = live || kf[min(CR / 16 * lane + i, nrt - 1)] < kend;
    const unsigned long long b = __ballot(live);
    c0 = b ? __builtin_ctzll(b) : min(nch, 64);
    if (nch <= 64 && b) c1 = 63 - __builtin_clzll(b);
  }

  if (tid < 64 * nu)
    rs[tid] = reinterpret_cast<const uint4*>(p.rec + ((long)it.w - l0))[2 * (lp + 1) + tid];

  // Production: thread -> (16-degree segment, row of the chunk).
  const int seg = tid / CR, prow = tid % CR;
  const int nck = (p.L - l0 + kCk) / kCk;
  const int kk = 2 * u0 + seg;
  const bool pv = seg < 2 * nu && kk < nck;
  const double* seedm = p.seeds + (long)(m + p.L) * nt;
  const double2* ckm = p.ck + ((long)it.z + kk - 1) * nt;
  double cs = 0.0;
  auto state = [&](int c) -> double2 {
    const int row = CR * c + prow;
    double2 s = make_double2(0.0, 0.0);
    cs = 0.0;
    if (pv && row < nr) {
      cs = p.cosv[row];
      if (kk == 0)
        s.x = seedm[row];
      else
        s = ckm[row];
    }
    return s;
  };
  // Row of degree 16 seg + j of the pass in LDS: SYM keeps the two parities
  // of a unit of 32 degrees apart.
  auto produce = [&](int buf, double2 s) {
    if ((64 / CR) * wave >= 2 * nu) return;  // the wave's segments are past the pass
    const double2* r = reinterpret_cast<const double2*>(rs) + 2 * kCk * seg;
    double* d = D[buf] + (SYM ? 32 * (seg >> 1) + 8 * (seg & 1) : 16 * seg) * AP + prow;
    double e0 = s.x, e1 = s.y;
#pragma unroll 4
    for (int j = 0; j < kCk; j++) {
      d[(SYM ? 16 * (j & 1) + (j >> 1) : j) * AP] = e0;
      rec_step(r[2 * j], r[2 * j + 1].x, cs, e0, e1);
    }
  };

  // Quads q .. of full() groups lie strictly inside the rows (SYM: of the
  // north, without the equator); the last ones are clamped to valid rows (rows
  // past the last have D = 0, and SYM takes the equator once).
  const int nfull = (SYM ? nt / 2 : nt) >> 2;
  auto load_quads = [&](int q, auto& B) {
    constexpr int N = sizeof(B) / sizeof(B[0]);
    if (q + N <= nfull) {
#pragma unroll
      for (int j = 0; j < NL; j++)
#pragma unroll
        for (int g = 0; g < N; g++) B[g][j] = fb[j][(q + g) * fs[j]];
    } else {
#pragma unroll
      for (int g = 0; g < N; g++) {
        const int back = max(0, 4 * (q + g) + krow - (nt - 1));  // rows past the last
#pragma unroll
        for (int j = 0; j < NL; j++)
          B[g][j] = fb[j][(q + g) * fs[j] + (fs[j] > 0 ? -cw : cw) * back];
      }
    }
  };

  typename M::acc acc[LT][NJ];
#pragma unroll
  for (int i = 0; i < LT; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[i][j] = typename M::acc{};

  const int nq = (nr + 3) >> 2;
  // Rows left out: 0 * value.
  double pz[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) pz[j] = 0.0;
  for (int c = 0; c < nch; c++) {
    if (c == c0) c = c1 + 1;
    if (c >= nch) break;
    double b[4][NL];
#pragma unroll
    for (int h = 0; h < NQ / 4; h++) {
      load_quads(NQ * c + 4 * h, b);
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int j = 0; j < NL; j++) pz[SYM ? j >> 1 : j] += 0.0 * b[q][j];
    }
  }

  constexpr int GQ = SYM ? 2 : 4;  // quads per group of loads
  constexpr int NG = NQ / GQ;
  // This wave's units: those of its degree group, up to its columns' degrees.
  constexpr int WU = LT / 2;
  const int mine = min(min(nu, (lw - lp + 32) >> 5) - wr * WU, WU);
  double Bq[2][GQ][NL];
  // All degree tiles of the wave (whole), or those of its units: tiles past
  // the pass are skipped in pairs.
  auto run_group = [&](auto whole, auto full, int buf, int c, int h, double (&B)[GQ][NL]) {
    const double* d = D[buf] + (16 * LT * wr + (lane & 15)) * AP + 4 * GQ * h + krow;
#pragma unroll
    for (int g = 0; g < GQ; g++) {
      double X[2][NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        if (SYM) {
          const double a = B[g][2 * j];
          double b = B[g][2 * j + 1];
          if (!decltype(full)::value) {
            const int row = 4 * (NQ * c + GQ * h + g) + krow;
            b = nt - 1 - row > row ? b : 0.0;
          }
          X[0][j] = a + b;
          X[1][j] = a - b;
        } else {
          X[0][j] = B[g][j];
        }
      }
      double A[LT];
#pragma unroll
      for (int i = 0; i < LT; i++) A[i] = d[16 * i * AP + 4 * g];
#pragma unroll
      for (int u = 0; u < WU; u++)
        if (decltype(whole)::value || u < mine) {
#pragma unroll
          for (int i = 2 * u; i < 2 * u + 2; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = M::mma(A[i], X[SYM ? i & 1 : 0][j], acc[i][j]);
        }
    }
  };

  __syncthreads();
  if (c0 <= c1) {
    load_quads(NQ * c0, Bq[0]);
    double2 st = state(c0);
    if (NBUF == 2) {
      produce(0, st);
      if (c0 < c1) st = state(c0 + 1);
    }
    // The chunks whose rows lie strictly inside, then the last.
    const int cfull = min(c1 + 1, nfull / NQ);
    auto run = [&](auto whole, auto full, int ca, int cb) {
      for (int c = ca; c < cb; c++) {
        const int buf = NBUF == 2 ? (c - c0) & 1 : 0;
        __syncthreads();
        load_quads(NQ * c + GQ, Bq[1]);
        if (NBUF == 2) {
          if (c < c1) {
            produce(buf ^ 1, st);
            if (c + 1 < c1) st = state(c + 2);
          }
        } else {
          produce(0, st);
          if (c < c1) st = state(c + 1);
          __syncthreads();
        }
#pragma unroll
        for (int h = 0; h < NG; h++) {
          if (decltype(full)::value || NQ * c + GQ * h < nq)
            run_group(whole, full, buf, c, h, Bq[h & 1]);
          if (h + 2 < NG)
            load_quads(NQ * c + GQ * (h + 2), Bq[h & 1]);
          else if (h + 2 == NG && c < c1)
            load_quads(NQ * (c + 1), Bq[0]);
        }
      }
    };
    if (mine == WU) {
      run(std::true_type{}, std::true_type{}, c0, cfull);
      run(std::true_type{}, std::false_type{}, max(c0, cfull), c1 + 1);
    } else {
      run(std::false_type{}, std::true_type{}, c0, cfull);
      run(std::false_type{}, std::false_type{}, max(c0, cfull), c1 + 1);
    }
  }

#pragma unroll
  for (int j = 0; j < NJ; j++) {
    double z = pz[j];
    z += __shfl_xor(z, 16);
    z += __shfl_xor(z, 32);
#pragma unroll
    for (int i = 0; i < LT; i++) M::add(acc[i][j], z);
  }

#pragma unroll
  for (int i = 0; i < LT; i++) {
    if (i >= 2 * mine) continue;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      if (!vc[j].valid) continue;
      const int mo = vc[j].sgn ? -m : m;
      double* co = p.cout + ((long)vc[j].field * p.cstride) * 2 + (vc[j].col & 1);
#pragma unroll
      for (int r = 0; r < M::NR; r++) {
        const int tile = wr * LT + i, mr = M::row(lane, r);
        const int l = lp + (SYM ? 32 * (tile >> 1) + 2 * mr + (tile & 1) : 16 * tile + mr);
        if (l > vc[j].lf) continue;
        double v = M::get(acc[i][j], r);
        if (vc[j].sgn && ((SYM ? m : l + p.n) & 1)) v = -v;
        const long ci = 2 * (long)coef_index(l, mo, p.nabs, p.real);
        if (p.accumulate) v += co[ci];
        if (p.zero_last && vc[j].lf == p.L && l == p.L && mo == p.L) v = 0.0;
        co[ci] = v;
      }
    }
  }
}

template <int KIND, int SYM, int RT, int NJ, int WR>
hipError_t go_synth(const LegParams& p, hipStream_t s) {
  hipLaunchKernelGGL((leg_synth_p<KIND, SYM, RT, NJ, WR>), dim3(8 * p.items_per), dim3(256), 0, s, p);
  return hipGetLastError();
}
template <int KIND, int SYM, int LT, int NJ>
hipError_t go_anal(const LegParams& p, hipStream_t s) {
  hipLaunchKernelGGL((leg_anal_p<KIND, SYM, LT, NJ>), dim3(8 * p.items_per), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace

// Tile of a launch: ncol columns (twice that many virtual ones when paired),
// nr rows, norder orders, uneven: fields of different truncation degrees.
// Wider tiles share each recurrence value and each A operand among more
// columns; the narrow ones keep the matrix unit off padding columns: at most 8
// columns take the 4-column instruction, at most 16 (32) one (two) tiles of
// 16; more are interleaved by order sign.  Every tile adds a sum's terms in the
// same order, so a batch equals its fields one by one.  Uneven batches stop at 64 (32 in
// the analysis), whose fields have neighbouring degrees.  A launch of fewer than
// kFewBlocks workgroups takes narrower tiles (and no 9th row tile): a wave
// then has fewer MFMAs between two barriers, and idle CUs repeat the recurrence
// for the other columns.  lMax=256, complex: 8 fields (514 workgroups of 32
// columns) 39.2 -> 34.1 us analysis with n=1, 33.8 -> 30.1 (synthesis) and 28.1 ->
// 24.2 us with n=0; lMax=384 (1155 of them) no gain, 69.7 -> 80.7 us analysis.
constexpr int kFewBlocks = 600;
static void set_cols(PairTile& t, int cols) {
  t.cols = cols;
  t.nj = cols == 16 ? 1 : 2;
  t.rt = cols <= 32 ? 2 : cols / 16;
}
// Columns that groups of cols multiply for v of them.
static int padded(int v, int cols) { return (v + cols - 1) / cols * cols; }
static PairTile pair_tile(int ncol, int pair, bool f32m) {
  PairTile t;
  const int V = ncol * (pair ? 2 : 1);
  t.kind = f32m ? 1 : V <= 8 ? 2 : 0;
  t.vint = V > 32 ? 1 : 0;
  t.vcols = t.vint ? (ncol + 15) / 16 * 16 * (pair ? 2 : 1) : V;
  if (t.kind == 2)
    t.rt = 2;
  else
    set_cols(t, V <= 16 ? 16 : V <= 32 ? 32 : t.vcols <= 64 ? 64 : 128);
  return t;
}
PairTile pair_synth_tile(int ncol, int pair, int sym, bool f32m, bool uneven, int nr, int norder) {
  PairTile t = pair_tile(ncol, pair, f32m);
  const int rtt = (nr + 15) / 16;
  // Row tiles of the busiest waves of n row blocks of wr row groups: rt each, one
  // more in a block with room for an extra one (of all its waves only those of the
  // last row group have it: lMax=1000, whose 63 tiles fit 7 blocks of 9, 10 real
  // fields of n=2 841 us in 7 blocks, 786 in 8).
  auto row_cost = [rtt](int rt, int wr, int n) { return n * rt + std::max(0, rtt - n * rt * wr); };
  auto full_blocks = [rtt](int rt, int wr) { return (rtt + rt * wr - 1) / (rt * wr); };
  auto row_blocks = [&](int rt, int wr) {
    int n = full_blocks(rt, wr);
    for (int k = n - 1; k > 0 && k * (rt * wr + 1) >= rtt; k--)
      if (row_cost(rt, wr, k) <= row_cost(rt, wr, n)) n = k;
    return n;
  };
  if (t.kind == 2) {
    t.nj = 1;
    t.rt = t.vcols > 4 ? 4 : 2;
    t.wr = t.vcols > 4 ? 2 : 4;
    t.cols = t.vcols > 4 ? 8 : 4;
    t.nblk = row_blocks(t.rt, t.wr);
    return t;
  }
  // Fewer padding columns in groups of 32 are worth more A operands read (64
  // columns in them, lMax=1000: 1356 us, 1174 in one group; 80 columns 1956 and
  // 2265, 96 columns 2047 and 2294; 160 columns 3595 and 3560).
  int cols = t.vcols <= 16 ? 16 : t.vcols <= 32 ? 32 : 64;
  if (!sym && cols == 64 && 5 * padded(t.vcols, 32) <= 4 * padded(t.vcols, 64)) cols = 32;
  if (t.kind == 1 && !uneven && t.vcols > 64 && padded(t.vcols, 128) == padded(t.vcols, 64)) cols = 128;
  auto set = [&](int c) {
    t.cols = c;
    t.nj = c == 128 ? 2 : 1;
    t.rt = c == 16 ? 2 : c == 32 ? 4 : 8;
    t.wr = c == 16 ? 4 : c == 32 ? 2 : 1;
  };
  set(cols);
  auto few = [&](int nblk) { return norder * nblk * (padded(t.vcols, t.cols) / t.cols) < kFewBlocks; };
  t.nblk = row_blocks(t.rt, t.wr);
  if (few(t.nblk)) t.nblk = full_blocks(t.rt, t.wr);
  while (t.cols > 16 && few(t.nblk)) set(t.cols / 2);
  if (t.kind == 0 && t.rt >= 4) {
    const int r6 = t.rt == 8 ? 6 : 3;
    const int n6 = row_blocks(r6, t.wr);
    if (row_cost(r6, t.wr, n6) < row_cost(t.rt, t.wr, t.nblk)) {
      t.rt = r6;
      t.nblk = n6;
    }
  }
  // FP32, at most 16 columns: blocks of 16 row tiles use each coefficient twice as
  // often (lMax=1024, 8 real fields 410 -> 364 us, 1 field 356 -> 352), where enough of
  // them are left (lMax=800, 2403 workgroups: 222 -> 213 and 190 -> 212 us).  FP64, with
  // products twice as long, gains nothing (489 and 500 us).
  if (t.kind == 1 && t.cols == 16) {
    const int n4 = row_blocks(4, 4);
    if (norder * n4 >= 5 * kFewBlocks && row_cost(4, 4, n4) <= row_cost(2, 4, t.nblk)) {
      t.rt = 4;
      t.nblk = n4;
    }
  }
  return t;
}
PairTile pair_anal_tile(int ncol, int pair, bool uneven, int norder) {
  PairTile t = pair_tile(ncol, pair, false);
  t.nblk = 4;  // units of 32 degrees per pass
  if (t.kind == 2) {
    t.nj = t.vcols <= 4 ? 1 : 2;
    t.cols = 4 * t.nj;
    return t;
  }
  if (uneven && t.cols > 32) set_cols(t, 32);
  // 17 .. 24 and 33 .. 40 real fields: tiles of 64 and 128 would multiply a third
  // and more of padding columns, tiles of 16 none (the sums are then as many as the
  // recurrences repeated for them).  n = 1, 24 fields: lMax=256 52 -> 44 us, lMax=512
  // 237 -> 205 us; 40 fields 95 -> 63 and 374 -> 333 us.  96 columns in tiles of 32
  // gain at some degrees and lose at others: lMax=512, n = 2 376 -> 351 us, n = 0
  // 236 -> 257 us.
  if (!uneven && (t.vcols == 48 || t.vcols == 80)) set_cols(t, 16);
  // The same past 128: 144 or 160 columns in groups of 32, 176 or 192 in groups
  // of 64, which take 1.3 and 1.2 times as long a column as groups of 128.  36 .. 48
  // complex fields, n=2: lMax=256 131 -> 101 (40) us, lMax=1000 3917 -> 3247 (40) and
  // 3964 -> 3610 (48) us.
  auto groups = [&](int cols) { return (t.vcols + cols - 1) / cols; };
  if (!uneven && t.cols == 128) {
    const int w[3] = {26 * padded(t.vcols, 32), 24 * padded(t.vcols, 64), 19 * padded(t.vcols, 128)};
    const int k = static_cast<int>(std::min_element(w, w + 3) - w);
    set_cols(t, 32 << k);
  }
  auto few = [&] { return norder * ((norder + 255) / 256) * groups(t.cols) < kFewBlocks; };
  // Fewer padding columns in the half as wide tile (96 columns at lMax=256, which
  // stopped at 64: 94 -> 67 us).
  auto leaner = [&](int cols) { return groups(cols / 2) * (cols / 2) < groups(cols) * cols; };
  bool narrow = few();
  while (narrow && t.cols > 16) {
    set_cols(t, t.cols / 2);
    narrow = few() || (t.cols > 16 && leaner(t.cols));
  }
  return t;
}

hipError_t launch_leg_synth_pair(const LegParams& p0, const PairTile& t, int sym, hipStream_t s) {
  if (!p0.ck || !p0.kf) return hipErrorInvalidValue;  // checkpoint table required
  LegParams p = p0;
  p.n_tsb = t.nblk;
  p.vint = t.vint;
  if (t.kind == 1) {
    if (sym) return hipErrorInvalidValue;
    if (t.rt == 8) return t.nj == 2 ? go_synth<1, 0, 8, 2, 1>(p, s) : go_synth<1, 0, 8, 1, 1>(p, s);
    if (t.rt == 4) return t.wr == 4 ? go_synth<1, 0, 4, 1, 4>(p, s) : go_synth<1, 0, 4, 1, 2>(p, s);
    return go_synth<1, 0, 2, 1, 4>(p, s);
  }
  if (t.kind == 2) {
    if (sym) return t.rt == 2 ? go_synth<2, 1, 2, 1, 4>(p, s) : go_synth<2, 1, 4, 1, 2>(p, s);
    return t.rt == 2 ? go_synth<2, 0, 2, 1, 4>(p, s) : go_synth<2, 0, 4, 1, 2>(p, s);
  }
  if (sym) switch (t.rt) {
      case 8: return go_synth<0, 1, 8, 1, 1>(p, s);
      case 6: return go_synth<0, 1, 6, 1, 1>(p, s);
      case 4: return go_synth<0, 1, 4, 1, 2>(p, s);
      case 3: return go_synth<0, 1, 3, 1, 2>(p, s);
      default: return go_synth<0, 1, 2, 1, 4>(p, s);
    }
  switch (t.rt) {
    case 8: return go_synth<0, 0, 8, 1, 1>(p, s);
    case 6: return go_synth<0, 0, 6, 1, 1>(p, s);
    case 4: return go_synth<0, 0, 4, 1, 2>(p, s);
    case 3: return go_synth<0, 0, 3, 1, 2>(p, s);
    default: return go_synth<0, 0, 2, 1, 4>(p, s);
  }
}

hipError_t launch_leg_anal_pair(const LegParams& p0, const PairTile& t, int sym, hipStream_t s) {
  if (!p0.ck || !p0.kf) return hipErrorInvalidValue;
  LegParams p = p0;
  p.vint = t.vint;
  p.n_cg = (p.ncol + p.cw - 1) / p.cw;
  p.nquad = (p.ntheta + 3) / 4;
  if (t.kind == 2) {
    if (sym) return t.nj == 1 ? go_anal<2, 1, 2, 1>(p, s) : go_anal<2, 1, 2, 2>(p, s);
    return t.nj == 1 ? go_anal<2, 0, 2, 1>(p, s) : go_anal<2, 0, 2, 2>(p, s);
  }
  if (sym) switch (t.rt) {
      case 8: return go_anal<0, 1, 8, 2>(p, s);
      case 4: return go_anal<0, 1, 4, 2>(p, s);
      default: return t.nj == 2 ? go_anal<0, 1, 2, 2>(p, s) : go_anal<0, 1, 2, 1>(p, s);
    }
  switch (t.rt) {
    case 8: return go_anal<0, 0, 8, 2>(p, s);
    case 4: return go_anal<0, 0, 4, 2>(p, s);
    default: return t.nj == 2 ? go_anal<0, 0, 2, 2>(p, s) : go_anal<0, 0, 2, 1>(p, s);
  }
}

}  // namespace gsh
