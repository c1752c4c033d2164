// Products between the small and the large ones (column-major, C = alpha*op(A)*op(B) + beta*C [+ bias] [relu]) in fp32 and fp64, on the matrix instructions of the type.
//
// A workgroup makes a 32x32 tile of C; its KS waves take a slice of k each, fetch their rows straight into the instruction's registers, two steps of 16 ahead, and their
// tiles meet in LDS: no barrier in the walk, nothing leaves the workgroup but C.  A lane holds two neighbouring rows of either operand, so that one that is contiguous along its rows comes
// in 8-byte (fp64: 16-byte) loads of 128 (256) bytes a row of lanes, and one that is contiguous along k in loads of four steps.  Four 16x16 tiles a wave make half the traffic
// per operation of the 16x16 kernel; 64x64, which would make a quarter, leaves most compute units without a tile at these sizes.
// What bounds it in fp32: 1000x237x1000 is 256 tiles, 3.3 us of matrix instructions on every compute unit, behind 2.5 us of launch and two round trips to memory; in fp64, large, the
// traffic of the tiles (55 TFLOP/s of the 72 that a large product reaches).  us by kernel trace, this / vendor's kernel (whose call costs its caller another 8 us): 1000x237x784 9.6/12.4, 1000x237x1000 10.2/13.9, TN 9.4/12.3,
// 1000x784x237 NT 11.1/12.1, 512^3 7.2/9.1, 712x618x301 8.0/9.6; level: 1000x1000x237 NT 11.6/10.8, 1458x320x509 10.7/11.0; slower: 1719x183x930 TN 15.7/13.6, 512x2048x512 17/15.
// Steps in flight, 2 / 4 / 6: 1000x237x1000 TN 9.4/10.6/10.6, 1458x320x509 10.6/11.2/11.9.
#pragma once
#include "knet8_gemm_small.h"
#include "knet8_gemm_split.h"

namespace knet8 {

// N elements at any element boundary, one load.
template <typename T, int N> struct __attribute__((packed, aligned(sizeof(T)))) Run { T v[N]; };

template <typename T, bool TA, bool TB, int KS>
__global__ __launch_bounds__(KS * kWave) void gemm_mid_kernel(int m, int n, int k, T alpha, const T* __restrict__ A, int lda, const T* __restrict__ B, int ldb, T beta, T* C, int ldc,
                                                              const T* bias, int act, int kslice) {
  constexpr int TS = 32, PITCH = TS + 1, D = 2;
  __shared__ T part[KS][TS * PITCH];
  unsigned im, in, z;
  split_tile(blockIdx.x, gridDim.x, (unsigned)((m + TS - 1) / TS), (unsigned)((n + TS - 1) / TS), im, in, z);
  const int i0 = (int)im * TS, j0 = (int)in * TS;
  const int w = threadIdx.x / kWave, l = threadIdx.x & (kWave - 1), r16 = l & 15, kq = l >> 4;
  const int kbeg = w * kslice, kend = k < kbeg + kslice ? k : kbeg + kslice;
  // rows 2*r16 and 2*r16 + 1 of the tile are this lane's
  struct Operand {
    const T* p[2];
    bool shift;
  };
  Operand oa, ob;
  const int ra = i0 + 2 * r16, rb = j0 + 2 * r16;
  if (TA) { oa.p[0] = A + (long)(ra < m ? ra : m - 1) * lda; oa.p[1] = A + (long)(ra + 1 < m ? ra + 1 : m - 1) * lda; oa.shift = false; }
  else { const int r = ra < m - 2 ? ra : m - 2; oa.p[0] = oa.p[1] = A + r; oa.shift = ra == m - 1; }
  if (!TB) { ob.p[0] = B + (long)(rb < n ? rb : n - 1) * ldb; ob.p[1] = B + (long)(rb + 1 < n ? rb + 1 : n - 1) * ldb; ob.shift = false; }
  else { const int r = rb < n - 2 ? rb : n - 2; ob.p[0] = ob.p[1] = B + r; ob.shift = rb == n - 1; }
  typename Mfma16<T>::Acc acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[a][b][r] = T(0);
  auto load = [&](T (&v)[2][4], const Operand& o, bool kcont, int ld, int kk) {
    if (kcont) {
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const Run<T, 4> q = *reinterpret_cast<const Run<T, 4>*>(o.p[t] + kk);
#pragma unroll
        for (int c = 0; c < 4; c++) v[t][c] = q.v[c];
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const Run<T, 2> q = *reinterpret_cast<const Run<T, 2>*>(o.p[0] + (long)(kk + c) * ld);
        v[0][c] = o.shift ? q.v[1] : q.v[0];
        v[1][c] = q.v[1];
      }
    }
  };
  auto load_tail = [&](T (&v)[2][4], const Operand& o, bool kcont, int ld, int kk) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int e = kcont ? 0 : (t == 0 ? (o.shift ? 1 : 0) : 1);
        v[t][c] = kk + c < kend ? (kcont ? o.p[t][kk + c] : o.p[0][(long)(kk + c) * ld + e]) : T(0);
      }
  };
  T fa[D][2][4], fb[D][2][4];
  auto fetch = [&](int d, int kk) {
    load(fa[d], oa, TA, lda, kk + 4 * kq);
    load(fb[d], ob, !TB, ldb, kk + 4 * kq);
  };
  auto multiply = [&](int d) {
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) acc[a][b] = Mfma16<T>::run(fa[d][a][c], fb[d][b][c], acc[a][b]);
  };
  const int full = kend > kbeg ? (kend - kbeg) / 16 : 0;
#pragma unroll
  for (int d = 0; d < D; d++)
    if (d < full) fetch(d, kbeg + 16 * d);
  int s = 0;
  for (; s + 2 * D <= full; s += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      multiply(d);
      fetch(d, kbeg + 16 * (s + D + d));
    }
  }
  for (; s < full; s += D) {
#pragma unroll
    for (int d = 0; d < D; d++)
      if (s + d < full) {
        multiply(d);
        if (s + D + d < full) fetch(d, kbeg + 16 * (s + D + d));
      }
  }
  if (kbeg + 16 * full < kend) {
    load_tail(fa[0], oa, TA, lda, kbeg + 16 * full + 4 * kq);
    load_tail(fb[0], ob, !TB, ldb, kbeg + 16 * full + 4 * kq);
    multiply(0);
  }
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) part[w][(2 * r16 + b) * PITCH + 2 * Mfma16<T>::row(r, kq) + a] = acc[a][b][r];
  __syncthreads();
  for (int o = threadIdx.x; o < TS * TS; o += KS * kWave) {
    const int i = o % TS, j = o / TS;
    T sum = part[0][j * PITCH + i];
#pragma unroll
    for (int q = 1; q < KS; q++) sum += part[q][j * PITCH + i];
    if (i0 + i < m && j0 + j < n) gemm_store(C + i0 + i + (long)(j0 + j) * ldc, sum, alpha, beta, bias, i0 + i, act);
  }
}
// Waves to a tile: about 1500 in all, two steps of 16 or more each; in fp64, whose long walks are bound by their loads' round trips, four with k >= 500 and two with k >= 250
// whatever the number of tiles (1, 2, 4, 8 waves: 1583x650x1843 131/100/86/86, 3433x719x2289 NT 246/234/219/242, 3117x1375x248 NT 59/58/63/70).
template <typename T>
inline int gemm_mid_waves(long tiles, int k) {
  const int steps = (k + 15) / 16, most = sizeof(T) == 8 ? 8 : 16;
  int ks = 1;
  while (ks < most && tiles * ks < 1500 && steps >= 2 * ks) ks *= 2;
  if (sizeof(T) == 8 && k >= 250 && ks < 2) ks = 2;
  if (sizeof(T) == 8 && k >= 500 && ks < 4) ks = 4;
  return ks;
}

// Where vendor calls cost more than a launch: true if the product is faster here.  small: the rule for small products would have it.  us a call, back to back from a Python process:
// fp32 against the 16x16 kernel: faster with 160 tiles and more (1000x237x100 TN 3.7/4.2, 512^3 6.8/8.6), sooner where that kernel's loads along k start off the 16-byte
//   boundaries (277x454x558 6.5/7.9); with fewer its waves are too few (100x237x1000 9.8/4.9, 399x651x243 6.6/5.5).  Against hipBLASLt: 291x460x433 TN 6.0/10.4, 307x706x605 TN 7.4/10.6, 1000x237x1000 TN 9.0/11.0; beyond 5.3e8 flop or long k
//   its larger tiles are ahead (1719x183x930 TN 14.4/12.3, 512x512x2048 NT 16.4/14.9, 152x1600x1600 13.3/11.0).  Short k over many tiles is nearly all stores of C.  Where m comes in whole
//   128s and n in whole 16s, as its tiles do, hipBLASLt's are ahead from about 6500 tiles on, fewer with more steps of k to each: 8192x8192x1 59/51, 4096x4096x4 20.7/17.9, 8704x1536x8 TN
//   21.7/15.9, 14592x640x20 TN 18.7/14.2, 10496x448x48 NT 14.4/11.5; at other sizes they do work for padding: 3000x3000x4 14.1/19.0, 7256x12328x2 NT 96/104, 108054x84x14 17.5/30.8.  (764 products
//   with k up to 260: the sum of log(time / the better time) is 25.7 without this line, 11.0 with it.)
// fp64, where hipBLASLt's kernels (the copy that PyTorch brings) reach 25 TFLOP/s: 979x200x870 TN 12.8/39.7, 1392x1234x1194 79/185, 2549x2683x1193 TN 330/847, 906x1912x63 11.8/13.0;
//   not short k over many tiles: 2973x1218x64 TN 24.9/21.2.  Against the 16x16 kernel 120x1026x946 TN 14.6/31.3, 531x295x494 8.6/12.9, 204x859x279 TN 7.5/10.9; level: 968x122x376 7.0/6.9;
//   few tiles: 212x155x1981 NT 21.9/13.4.
template <typename T>
inline bool gemm_mid_fits(bool ta, bool tb, int m, int n, int k, int lda, int ldb, bool small) {
  const double tiles = (m + 31) / 32 * 1.0 * ((n + 31) / 32), flop = 2048 * tiles * k;
  if (sizeof(T) == 8) {
    if (m < 2 || n < 2 || k < 16 || k > 8192) return false;
    if (tiles * gemm_mid_waves<T>((long)tiles, k) * kWave >= 4294967296.0) return false;   // a grid has fewer than 2^32 threads (131072^2 outputs, k >= 500); in fp32 the flop are far below that
    return small ? tiles >= 128 && k >= 150 : tiles >= 32 && !(k < 100 && tiles > 3500);
  }
  if (m < 32 || n < 32 || k > 1500 || flop > (k <= 1000 ? 5.3e8 : 3.5e8)) return false;
  if (!small) return tiles >= 64 && !(k <= 64 && m % 128 == 0 && n % 16 == 0 && tiles + 80.0 * k > 6500);
  const double padded = 512.0 * ((m + 15) / 16) * ((n + 15) / 16) * k;
  const bool narrow = (ta && lda % 4 != 0) || (!tb && ldb % 4 != 0);
  return tiles >= 160 && padded >= (narrow ? 6e7 : 1.3e8);
}

template <typename T>
inline void launch_gemm_mid(hipStream_t stream, bool ta, bool tb, int m, int n, int k, T alpha, const T* A, int lda, const T* B, int ldb, T beta, T* C, int ldc, const T* bias, int act) {
  const long tiles = (long)((m + 31) / 32) * ((n + 31) / 32);
  const int ks = gemm_mid_waves<T>(tiles, k), kslice = ((k + 15) / 16 + ks - 1) / ks * 16;
#define KNET8_MIDK(TA, TB, KS) hipLaunchKernelGGL((gemm_mid_kernel<T, TA, TB, KS>), dim3((unsigned)tiles), dim3(KS * kWave), 0, stream, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, bias, act, kslice)
#define KNET8_MID(TA, TB) do { if (ks == 1) KNET8_MIDK(TA, TB, 1); else if (ks == 2) KNET8_MIDK(TA, TB, 2); else if (ks == 4) KNET8_MIDK(TA, TB, 4); else if (ks == 8) KNET8_MIDK(TA, TB, 8); \
                               else if constexpr (sizeof(T) == 4) KNET8_MIDK(TA, TB, 16); } while (0)
  if (!ta && !tb) KNET8_MID(false, false);
  else if (ta && !tb) KNET8_MID(true, false);
  else if (!ta && tb) KNET8_MID(false, true);
  else KNET8_MID(true, true);
#undef KNET8_MID
#undef KNET8_MIDK
}

}  // namespace knet8
