// Large fp32 matrix products on the bf16 matrix cores (column-major, C = alpha*op(A)*op(B) + beta*C [+ bias] [relu]).
//
// The fp32 matrix instructions run at 1/16 of the bf16 ones (157 against 2500 TFLOP/s nominal), and the vendor library's fp32 products sit at
// their limit: 8192^3 reaches 154 TFLOP/s, 4096x2048x4096 151.  Here every element is cut into three bf16 parts, x = h + m + l, each the
// rounding of what the ones before it leave: 3 x 8 bits and the signs hold all 24 bits of an fp32 number, so h + m + l = x exactly, with
// |m| <= 2^-8 |x| and |l| <= 2^-17 |x|.  Of the nine products of parts all but ll (at most 2^-34 of the whole) are formed, hh in one
// set of fp32 accumulators and the seven small ones in another: the large sums see one rounding per 32 steps of k, and a sum with one term that is not
// zero is rounded as the fp32 instruction rounds it.  (ml and lm reach 2^-24 of the whole together: without them such a sum is off by up to 2^-23.2, and sums
// of equal numbers by as much; they cost a sixth of the speed.)  2-norm of the error against 64 bits, this / vendor fp32: normal data 1000x237x784 8.4e-8/5.0e-7,
// 4096x2048x4096 4.0e-7/1.15e-6, 512x2048x32000 4.0e-7/2.3e-6; all-positive data 4.9e-8/3.8e-7, 3.5e-7/9.9e-7, 1.3e-7/1.4e-6; 2048^3 with one term a sum
// 2.53e-8/2.53e-8 (largest 2^-23.99/2^-24.00), with two 3.14e-8/3.11e-8, with eight 3.8e-8/5.4e-8.
//   * Small numbers: the lower parts of numbers below 2^-109 would leave bf16's range.  Both operands are multiplied by 2^24 on the way in and the
//     sums by 2^-48 on the way out, which keeps every fp32 number, denormals included, whole.
//   * Large numbers, infinities, NaN: a part or a sum that overflows leaves a NaN or an infinity in an accumulator (inf - inf in the split itself
//     if not before).  A wave that finds one in its patch forms these sums again with the fp32 matrix instruction: results beyond
//     2^80, and what is infinite or NaN, come out as that instruction gives them; the others stay.  us, 4096x2048x4096 (vendor 458): 352 on finite data, 324 if all is NaN, 542 with
//     one NaN in A and 731 with one infinity (a row of sums to form again), 1130 if every sum is beyond 2^80.
//
// The cut is made while a tile goes from global memory to LDS (6.5 vector instructions an element, in the shadow of the matrix instructions of the
// SIMD's other wave): no extra pass over the operands, no scratch.  256x128 tile, 8 waves of 64x64, 32 steps of k a stage.  LDS: two stages and the masks
// of sums that are not finite, 153088 bytes (TN), 158464 (NN, TT) or 163840 (NT, all that a compute unit has).  Matrix cores 4096 cycles a stage, LDS about 2070, vector ALU about 2100.  What bounds it is power: 8192^3 runs at 198 TFLOP/s on normal data and at 232 on zeros.
// So the matrix instructions are chosen and ordered by the energy they take on normal data.  From registers alone 32x32x16 reaches 1822 TFLOP/s of bf16 work
// and 16x16x32 2073 (both 2450 to 2480 on zeros): half the traffic to the accumulators.  All eight products of a 16x16 tile follow each other, so that the sums stay
// where they are (3 % over taking the tiles in turn), in an order in which only one operand changes from one to the next (another 2 %; one that changes the first
// operand more often instead is 1 to 2 % slower).  us, before (32x32x16, tiles in turn) / now, the same run: 4096x2048x4096 396/346, TN 410/352, 4096x4096x2048 NT 420/358, 8192^3 6650/5910,
// 32000x2048x512 458/401, 512x2048x32000 TN 414/375, 32000x512x2048 NT 427/374.  TFLOP/s (of fp32 work), this / vendor: 4096x2048x4096 192/150, TN 195/150,
// 4096x4096x2048 NT 194/148, 32000x2048x512 168/137, 512x2048x32000 TN 178/139, 32000x512x2048 NT 188/145, 8192^3 198/154.
#pragma once
#include "knet8_device.h"
#include "knet8_runtime.h"

namespace knet8 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
template <int N> struct __attribute__((packed, aligned(4))) FNu { float v[N]; };   // N elements at any element boundary, one load
using F4u = FNu<4>;

constexpr float kSplitScale = 16777216.0f;              // 2^24
constexpr float kSplitUnscale = 1.0f / (16777216.0f * 16777216.0f);   // 2^-48: both operands are scaled

template <int N> struct SplitParts { unsigned h[N / 2], m[N / 2], l[N / 2]; };

__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));   // v_cvt_pk_bf16_f32, round to nearest even
}
template <int N>
__device__ __forceinline__ SplitParts<N> split_bf16(const float* x) {
  SplitParts<N> r;
#pragma unroll
  for (int i = 0; i < N; i += 2) {
    const float a = x[i] * kSplitScale, b = x[i + 1] * kSplitScale;
    const unsigned h = pack_bf16(a, b);
    const float ra = a - __builtin_bit_cast(float, h << 16), rb = b - __builtin_bit_cast(float, h & 0xffff0000u);
    const unsigned m = pack_bf16(ra, rb);
    const float sa = ra - __builtin_bit_cast(float, m << 16), sb = rb - __builtin_bit_cast(float, m & 0xffff0000u);
    r.h[i / 2] = h; r.m[i / 2] = m; r.l[i / 2] = pack_bf16(sa, sb);
  }
  return r;
}

// One operand's share of a tile: ROWS rows (of op(A), or columns of op(B)) by BK steps of k, fetched as fp32 and kept in LDS as three bf16 parts,
// 16 bytes (8 steps of k) of one row at a time.
// KC: k is the contiguous axis in memory (element (row,k) at p[row*ld + k]): a lane takes 4 steps of k of one row.
// Otherwise the rows are (p[k*ld + row]): a lane takes 4 steps of k of kRows rows next to each other.
template <int ROWS, int BK, int NT, bool KC>
struct SplitLoader {
  static constexpr int kVals = ROWS * BK / NT;
  static constexpr int kRows = KC ? 1 : (kVals >= 16 ? 4 : 2);
  static constexpr int kItems = kVals / (4 * kRows);
  static_assert(kItems >= 1 && kVals % (4 * kRows) == 0 && ROWS % 64 == 0, "tile and workgroup do not match");
  // Where the 16 bytes of a row stand (in units of 16 bytes): in order, or dealt out to four groups, each 64 bytes off the multiples of 256, so that the 16 rows of a
  // fragment lie in all banks once (32 bytes off, which suits reads of 32 rows: 4096x4096x2048 NT 372 us, so 365).  The octets of k of the first form stand
  // 32 bytes off: eight lanes there write the 32 steps of a row.
  static constexpr int kGroup = ROWS / 4 + 4;
  static constexpr int kStride = KC ? ROWS + 2 : 4 * kGroup;      // from one octet of k to the next
  static constexpr int kPart = (BK / 8) * kStride;                // from one part to the next
  static constexpr int kUnits = 3 * kPart;
  static __device__ __forceinline__ int unit(int r) { return KC ? r : (r & 3) * kGroup + (r >> 2); }

  float v[kVals];
  int off[kItems];           // elements from the tile's first row and step (below it for a tile of fewer rows than a lane takes)
  int to[kItems][kRows];     // in units of 8 bytes

  __device__ __forceinline__ void init(int t, int rows, int ld) {   // rows: how many of the matrix are left here (the matrix itself has 4 or more)
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const int e = t + i * NT;
      if (KC) {
        const int r = e / (BK / 4), q = e % (BK / 4), rr = r < rows ? r : rows - 1;   // rows beyond the matrix: any valid row, nothing is made of them
        off[i] = rr * ld + 4 * q;
        to[i][0] = 2 * ((q >> 1) * kStride + r) + (q & 1);
      } else {
        const int g = (e >> 1) % (ROWS / kRows), q = 2 * ((e >> 1) / (ROWS / kRows)) + (e & 1);
        const int r = kRows * g + kRows <= rows ? kRows * g : rows - kRows;           // the matrix's last rows (again) rather than rows beyond it
        off[i] = 4 * q * ld + r;
#pragma unroll
        for (int j = 0; j < kRows; j++) to[i][j] = 2 * ((q >> 1) * kStride + (r + j < 0 ? ROWS / 4 : unit(r + j))) + (q & 1);   // rows before the tile: into the gap after the first group
      }
    }
  }
  // p: the operand at the tile's first row and step
  __device__ __forceinline__ void load(const float* __restrict__ p, int ld) {
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      if constexpr (KC) {
        const F4u q = *reinterpret_cast<const F4u*>(p + off[i]);
#pragma unroll
        for (int j = 0; j < 4; j++) v[4 * i + j] = q.v[j];
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const FNu<kRows> q = *reinterpret_cast<const FNu<kRows>*>(p + (long)j * ld + off[i]);
#pragma unroll
          for (int r = 0; r < kRows; r++) v[4 * (kRows * i + r) + j] = q.v[r];
        }
      }
    }
  }
  __device__ __forceinline__ void load_tail(int t, const float* __restrict__ p, int ld, int kleft) {   // kleft of the BK steps exist
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const int e = t + i * NT;
      const int k = 4 * (KC ? e % (BK / 4) : 2 * ((e >> 1) / (ROWS / kRows)) + (e & 1));
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int r = 0; r < kRows; r++) v[4 * (kRows * i + r) + j] = k + j < kleft ? p[(long)off[i] + (KC ? (long)j : (long)j * ld + r)] : 0.0f;
    }
  }
  __device__ __forceinline__ void store(uint4* __restrict__ s) const {
    uint2* s2 = reinterpret_cast<uint2*>(s);
#pragma unroll
    for (int i = 0; i < kItems; i++)
#pragma unroll
      for (int r = 0; r < kRows; r++) {
        const SplitParts<4> p = split_bf16<4>(v + 4 * (kRows * i + r));
        uint2* d = s2 + to[i][r];
        d[0] = make_uint2(p.h[0], p.h[1]);
        d[2 * kPart] = make_uint2(p.m[0], p.m[1]);
        d[4 * kPart] = make_uint2(p.l[0], p.l[1]);
      }
  }
};

// Workgroup -> (tile of m, tile of n, slice of k).  Workgroups go to the 8 XCDs in turn: give every XCD a run of neighbouring tiles, walked in
// bands of kBand tiles of m, so that the operands' panels are shared in its L2.
__device__ __forceinline__ void split_tile(unsigned b, unsigned total, unsigned tm, unsigned tn, unsigned& im, unsigned& in, unsigned& z) {
  constexpr unsigned kXcd = 8, kBand = 8;
  const unsigned q = total / kXcd, rem = total % kXcd, x = b % kXcd, y = b / kXcd;
  unsigned id = x < rem ? x * (q + 1) + y : rem * (q + 1) + (x - rem) * q + y;
  z = id / (tm * tn);
  id -= z * (tm * tn);
  const unsigned band = id / (kBand * tn), first = band * kBand, h = tm - first < kBand ? tm - first : kBand;
  const unsigned in_band = id - band * (kBand * tn);
  im = first + in_band % h;
  in = in_band / h;
}

template <int BM, int BN, int WM, int WN, int BK, bool TA, bool TB>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN), 2)
void gemm_split_kernel(int m, int n, int k, const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, float* __restrict__ C, int ldc,
                       float alpha, float beta, const float* __restrict__ bias, int act, int kchunk, unsigned splits) {
  constexpr int NT = 64 * (BM / WM) * (BN / WN), FM = WM / 16, FN = WN / 16;
  using LA = SplitLoader<BM, BK, NT, TA>;
  using LB = SplitLoader<BN, BK, NT, !TB>;
  __shared__ uint4 lds[2][LA::kUnits + LB::kUnits];
  __shared__ unsigned long long odd[NT / 64][FN * 4 * FM];   // which sums are not finite (see the end)
  static_assert(sizeof(lds) + sizeof(odd) <= 160 * 1024, "gemm_split_kernel: more LDS than a compute unit has");
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, half = lane >> 5, l32 = lane & 31, quad = lane >> 4, l16 = lane & 15;
  const int wm = (wave % (BM / WM)) * WM, wn = (wave / (BM / WM)) * WN;
  unsigned im, in, z;
  split_tile(blockIdx.x, gridDim.x, (unsigned)((m + BM - 1) / BM), (unsigned)((n + BN - 1) / BN), im, in, z);
  const int i0 = (int)im * BM, j0 = (int)in * BN;
  const int kbeg = (int)z * kchunk, kend = k - kbeg < kchunk ? k : kbeg + kchunk;
  const long sa = TA ? 1 : lda, sb = TB ? ldb : 1;               // elements from one k to the next
  const float* pa = A + (TA ? (long)i0 * lda : i0) + kbeg * sa;
  const float* pb = B + (TB ? (long)j0 : (long)j0 * ldb) + kbeg * sb;
  LA la;
  LB lb;
  la.init(t, m - i0, lda);
  lb.init(t, n - j0, ldb);
  f32x4 acc[FN][FM], low[FN][FM];   // hh, and the seven products of lower weight
#pragma unroll
  for (int a = 0; a < FN; a++)
#pragma unroll
    for (int b = 0; b < FM; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[a][b][r] = low[a][b][r] = 0.0f;
  auto fetch_full = [&]() {
    la.load(pa, lda);
    lb.load(pb, ldb);
    pa += BK * sa;
    pb += BK * sb;
  };
  auto fetch = [&](int k0) {
    if (kend - k0 >= BK) { fetch_full(); return; }
    la.load_tail(t, pa, lda, kend - k0);
    lb.load_tail(t, pb, ldb, kend - k0);
  };
  auto stage = [&](uint4* s) {
    la.store(s);
    lb.store(s + LA::kUnits);
  };
  int ua[FM], ub[FN];   // this lane's rows in the two halves of a buffer, at its octet of k
#pragma unroll
  for (int i = 0; i < FM; i++) ua[i] = quad * LA::kStride + LA::unit(wm + 16 * i + l16);
#pragma unroll
  for (int i = 0; i < FN; i++) ub[i] = LA::kUnits + quad * LB::kStride + LB::unit(wn + 16 * i + l16);
  bf16x8 fa[FM][3];
  auto take_a = [&](const uint4* s) {
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int i = 0; i < FM; i++) fa[i][p] = __builtin_bit_cast(bf16x8, s[ua[i] + p * LA::kPart]);
  };
  auto multiply = [&](const uint4* s, int first, int last) {   // 32 steps of k, column tiles first .. last - 1 of the wave
#pragma unroll
    for (int a = first; a < last; a++) {
      bf16x8 fb[3];
#pragma unroll
      for (int p = 0; p < 3; p++) fb[p] = __builtin_bit_cast(bf16x8, s[ub[a] + p * LB::kPart]);
      // ml, mm ... hh: one operand changes at a time
      constexpr int kA[8] = {2, 2, 1, 1, 1, 0, 0, 0}, kB[8] = {1, 0, 0, 1, 2, 2, 1, 0};
#pragma unroll
      for (int b = 0; b < FM; b++)
#pragma unroll
        for (int o = 0; o < 8; o++) {
          f32x4& c = o < 7 ? low[a][b] : acc[a][b];
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[b][kA[o]], fb[kB[o]], c, 0, 0, 0);
        }
    }
  };
  const int tiles = (kend - kbeg + BK - 1) / BK, full = (kend - kbeg) / BK;
  fetch(kbeg);
  stage(lds[0]);
  if (tiles > 1) fetch(kbeg + BK);
  int cur = 0, i = 0;
  for (; i + 2 < full; i++, cur ^= 1) {
    __syncthreads();
    take_a(lds[cur]);
    multiply(lds[cur], 0, FN / 2);
    la.store(lds[cur ^ 1]);
    la.load(pa, lda);
    pa += BK * sa;
    lb.store(lds[cur ^ 1] + LA::kUnits);
    lb.load(pb, ldb);
    pb += BK * sb;
    multiply(lds[cur], FN / 2, FN);
    __builtin_amdgcn_iglp_opt(0);   // spread the LDS traffic and the cut over the matrix instructions (8192^3 181 -> 184 TFLOP/s, 512x2048x32000 TN 172 -> 174)
  }
  for (; i < tiles; i++, cur ^= 1) {   // the last stages: nothing more to fetch, or less than a stage
    __syncthreads();
    take_a(lds[cur]);
    multiply(lds[cur], 0, FN / 2);
    if (i + 1 < tiles) stage(lds[cur ^ 1]);
    if (i + 2 < tiles) fetch(kbeg + (i + 2) * BK);
    multiply(lds[cur], FN / 2, FN);
  }
#pragma unroll
  for (int a = 0; a < FN; a++)
#pragma unroll
    for (int b = 0; b < FM; b++) acc[a][b] += low[a][b];
  float bad = 0.0f;
#pragma unroll
  for (int a = 0; a < FN; a++)
    if (j0 + wn + 16 * a + l16 < n) {
#pragma unroll
      for (int b = 0; b < FM; b++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (i0 + wm + 16 * b + 4 * quad + r < m) bad += acc[a][b][r] * 0.0f;
    }
  const bool again = __any(bad != 0.0f);   // (NaN: a sum is not finite)
  float* c = C;
  const long ld = ldc;
  if (splits > 1) c += (long)z * m * n;   // this slice's sums; gemm_split_sum_kernel applies the rest
  auto store = [&](float v, int i, int j, float bi) {
    float* d = c + (long)j * ld + i;
    if (splits == 1) {
      v = alpha * v;
      if (beta != 0.0f) v = v + beta * *d;
      if (bias) v = v + bi;
      if (act == 1) v = v > 0.0f ? v : 0.0f;
    }
    *d = v;
  };
#pragma unroll
  for (int b = 0; b < FM; b++) {   // a lane's four sums are neighbours in a column: 16 bytes a store
    const int i = i0 + wm + 16 * b + 4 * quad;
    if (i >= m) continue;
    const bool whole = i + 4 <= m && !again;
    float bi[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (bias && splits == 1) {
#pragma unroll
      for (int r = 0; r < 4; r++) bi[r] = bias[i + r < m ? i + r : i];
    }
#pragma unroll
    for (int a = 0; a < FN; a++) {
      const int j = j0 + wn + 16 * a + l16;
      if (j >= n) continue;
      if (whole) {
        float* d = c + (long)j * ld + i;
        F4u v;
#pragma unroll
        for (int r = 0; r < 4; r++) v.v[r] = acc[a][b][r] * kSplitUnscale;
        if (splits == 1) {
          F4u old = {{0.0f, 0.0f, 0.0f, 0.0f}};
          if (beta != 0.0f) old = *reinterpret_cast<const F4u*>(d);
#pragma unroll
          for (int r = 0; r < 4; r++) {
            v.v[r] = alpha * v.v[r];
            if (beta != 0.0f) v.v[r] = v.v[r] + beta * old.v[r];
            if (bias) v.v[r] = v.v[r] + bi[r];
            if (act == 1) v.v[r] = v.v[r] > 0.0f ? v.v[r] : 0.0f;
          }
        }
        *reinterpret_cast<F4u*>(d) = v;
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (i + r < m && acc[a][b][r] * 0.0f == 0.0f) store(acc[a][b][r] * kSplitUnscale, i + r, j, bi[r]);
      }
    }
  }
  if (!again) return;
  // The sums that are not finite, by the fp32 instruction: 32x32 of the patch at a time, where there are any.  Lanes 0-31 take the first 16 of 32 steps of k and lanes
  // 32-63 the others, so that an operand with k in a row comes in 16-byte loads.  Once all that are wanted are NaN, as in a training run that has diverged, what follows
  // changes nothing.
  constexpr int kStep = 16;
#pragma unroll
  for (int a = 0; a < FN; a++)
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int b = 0; b < FM; b++) {   // bit 16*q + l: column l of the 16x16 tile, row 4*q + r
        const unsigned long long w = __ballot(acc[a][b][r] * 0.0f != 0.0f);
        if (lane == 0) odd[wave][(a * 4 + r) * FM + b] = w;
      }
  __builtin_amdgcn_wave_barrier();   // (a wave reads back what it wrote itself)
#pragma unroll 1
  for (int f = 0; f < FN * FM / 4; f++) {
    const int fi = 32 * (f % (FM / 2)), fj = 32 * (f / (FM / 2));
    const int i = i0 + wm + fi + l32, ja = j0 + wn + fj, jl = ja + l32;
    unsigned want = 0;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int jw = 8 * (r >> 2) + 4 * half + (r & 3);   // the column of the 32x32 patch that the instruction below leaves in register r
      const unsigned long long w = odd[wave][(((fj + jw) / 16) * 4 + (l32 & 3)) * FM + (fi + l32) / 16];
      if (i < m && ja + jw < n) want |= (unsigned)(w >> (16 * (l16 / 4) + jw % 16) & 1u) << r;
    }
    if (!__any(want != 0)) continue;
    const float* p = A + (long)(i < m ? i : m - 1) * (TA ? lda : 1) + (kbeg + kStep * half) * sa;
    const float* q = B + (long)(jl < n ? jl : n - 1) * (TB ? 1 : ldb) + (kbeg + kStep * half) * sb;
    f32x16 sum;
#pragma unroll
    for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll 1
    for (int k0 = kbeg; k0 < kend; k0 += 2 * kStep, p += 2 * kStep * sa, q += 2 * kStep * sb) {
      float va[kStep], vb[kStep];
      if (kend - k0 >= 2 * kStep) {
#pragma unroll
        for (int s = 0; s < kStep; s += 4) {
          const float *ps = p + s * sa, *qs = q + s * sb;
          const F4u x = TA ? *reinterpret_cast<const F4u*>(ps) : F4u{{ps[0], ps[sa], ps[2 * sa], ps[3 * sa]}};
          const F4u y = TB ? F4u{{qs[0], qs[sb], qs[2 * sb], qs[3 * sb]}} : *reinterpret_cast<const F4u*>(qs);
#pragma unroll
          for (int e = 0; e < 4; e++) { va[s + e] = x.v[e]; vb[s + e] = y.v[e]; }
        }
      } else {
        const int left = kend - k0 - kStep * half;
#pragma unroll
        for (int s = 0; s < kStep; s++) { va[s] = s < left ? p[s * sa] : 0.0f; vb[s] = s < left ? q[s * sb] : 0.0f; }
      }
#pragma unroll
      for (int s = 0; s < kStep; s++) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(vb[s], va[s], sum, 0, 0, 0);
      bool done = true;
#pragma unroll
      for (int r = 0; r < 16; r++) done = done && ((want >> r & 1u) == 0 || sum[r] != sum[r]);
      if (__all(done)) break;
    }
    const float bi = (want != 0 && bias && splits == 1) ? bias[i] : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++)
      if (want >> r & 1u) store(sum[r], i, ja + 8 * (r >> 2) + 4 * half + (r & 3), bi);
  }
}

// How many slices of k an m x n x k product is cut into, and its estimated time in us: a stage of 32 steps takes 2.5 with most of the 256 CUs at work, starting
// and storing a tile 7 (fitted to 90 products of 2 to 200 GFLOP); slices, which let few tiles fill the chip, cost a second launch that reads them.
struct SplitPlan { int splits, kchunk; double us; };
inline SplitPlan gemm_split_plan(int m, int n, int k) {
  constexpr size_t kMostPartial = size_t(64) << 20;
  const double ncu = tuning(kTuneNumCUs), tiles = double((m + 255) / 256) * ((n + 127) / 128), stages = (k + 31) / 32;
  SplitPlan best = {1, k, 1e30};
  for (int s = 1; s <= 16; s++) {
    if (s > 1 && (stages / s < 4 || (size_t)s * m * n * sizeof(float) > kMostPartial)) break;
    const double per = (double)(long)((stages + s - 1) / s), turns = (double)(long)((tiles * s + ncu - 1) / ncu);
    double us = turns * (per * 2.5 + 7);
    if (s > 1) us += 4 + (s + 1) * 4.0 * m * n / 5e6;
    if (us < best.us) best = {s, (int)per * 32, us};
  }
  best.splits = (k + best.kchunk - 1) / best.kchunk;
  return best;
}
// True if the product runs here: estimated faster than the vendor's fp32 kernels (140 TFLOP/s and 8 us for the call).  us, this /
// vendor: 1000x2048x4096 101/119, 4096x1792x545 54/80, 255x3000x8005 89/104, 689x8103x920 TN 82/95, 3161x6756x1098 TN 304/410; level: 1880x1085x4387 130/130; not taken:
// 1024x2048x1024 41/35, 3000x3000x400 NT 81/66, 188x6336x1630 44/37, 1785x5130x7191 1094/953 (a last turn that is nearly empty).
// The loaders' offsets within a tile have 32 bits: 255 * ld.
inline bool gemm_split_fits(int m, int n, int k, int lda, int ldb, SplitPlan* plan) {
  const int knob = tuning(kTuneGemmSplit);   // for tests and comparisons: 1 never, 2 wherever the kernel can
  if (m < 4 || n < 4 || k < 1 || lda > (1 << 23) || ldb > (1 << 23) || knob == 1) return false;
  const double flop = 2.0 * m * n * (double)k;
  if (knob != 2 && (m < 64 || n < 64 || k < 64 || flop < 2e9)) return false;
  *plan = gemm_split_plan(m, n, k);
  return knob == 2 || plan->us < flop / 140e6 + 8;
}

// C = act(alpha*sum of the slices [+ beta*C] [+ bias]), slices in order.
__global__ __launch_bounds__(256) void gemm_split_sum_kernel(int m, int n, int splits, const float* __restrict__ partial, float* C, int ldc, float alpha,
                                                             float beta, const float* __restrict__ bias, int act) {
  const long mn = (long)m * n;
  for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < mn; e += (long)gridDim.x * 256) {
    float v = partial[e];
    for (int z = 1; z < splits; z++) v = v + partial[z * mn + e];
    const int i = (int)(e % m), j = (int)(e / m);
    float* d = C + (long)j * ldc + i;
    v = alpha * v;
    if (beta != 0.0f) v = v + beta * *d;
    if (bias) v = v + bias[i];
    if (act == 1) v = v > 0.0f ? v : 0.0f;
    *d = v;
  }
}

inline void launch_gemm_split(hipStream_t stream, bool ta, bool tb, int m, int n, int k, float alpha, const float* A, int lda, const float* B, int ldb,
                             float beta, float* C, int ldc, const float* bias, int act, SplitPlan plan) {
  float* out = C;
  int ldo = ldc;
  Workspace ws;
  if (plan.splits > 1) {
    ws = workspace_for(stream, (size_t)plan.splits * m * n * sizeof(float), 0, true);
    if (ws.partial != nullptr) {
      out = static_cast<float*>(ws.partial);
      ldo = m;
    } else {   // no scratch: k in one piece, which needs none
      plan.splits = 1;
      plan.kchunk = k;
    }
  }
  const long tiles = (long)((m + 255) / 256) * ((n + 127) / 128);
  const dim3 grid((unsigned)(tiles * plan.splits)), block(512);
#define KNET8_SP(TA, TB) hipLaunchKernelGGL((gemm_split_kernel<256, 128, 64, 64, 32, TA, TB>), grid, block, 0, stream, m, n, k, A, lda, B, ldb, out, ldo, alpha, beta, bias, act, plan.kchunk, (unsigned)plan.splits)
  if (!ta && !tb) KNET8_SP(false, false);
  else if (ta && !tb) KNET8_SP(true, false);
  else if (!ta && tb) KNET8_SP(false, true);
  else KNET8_SP(true, true);
#undef KNET8_SP
  if (plan.splits > 1) {
    const long mn = (long)m * n, blocks = (mn + 255) / 256;
    hipLaunchKernelGGL(gemm_split_sum_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream, m, n, plan.splits, out, C, ldc, alpha, beta, bias, act);
  }
  check_launch("gemm (split)");
}

}  // namespace knet8
