// Schur-update GEMM of the multifrontal factorization on MFMA (gfx950).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mf.hpp"
#include "mfma.hpp"

namespace rf {

// 16 bytes of consecutive entries at an entry-aligned address: one access
// (gfx950 runs in unaligned access mode; the front leading dimension m is
// arbitrary).
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// The MFMA block of the Schur update: BS x BS outputs, KS k per instruction;
// lane l supplies the first operand's entry [l % BS][l / BS] and the second's
// [l / BS][l % BS], and its output register e is column ocol(l, e) of the
// first operand's index, l % BS of the second's.  FP32 takes the 32 x 32
// block: per k it needs half the LDS operand reads of the 16 x 16 one.
template <typename T>
struct GemmMfma;
template <>
struct GemmMfma<float> {
  static constexpr int BS = 32, KS = 2, E = 4, NACC = 16;
  using acc_t = v16f;
  using unaligned_t = f4u;
  using lds_t = v4f;
  __device__ static acc_t op(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
  __device__ static int ocol(int lane, int e) { return 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); }
};
template <>
struct GemmMfma<double> {
  static constexpr int BS = 16, KS = 4, E = 2, NACC = 4;
  using acc_t = v4d;
  using unaligned_t = d2u;
  using lds_t = v2d;
  __device__ static acc_t op(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ static int ocol(int lane, int e) { return (lane >> 4) + 4 * e; }
};

// Workgroup bid of a launch runs on XCD bid % 8 (round-robin dispatch).  Every
// group of 512 tiles, what the chip holds at once, is dealt to the XCDs in
// runs of 64: the list goes through a front in blocks of GT_SUPER x GT_SUPER
// tiles, so a run shares 16 panels, which stay in that XCD's L2, instead of
// the 64 and more of tiles taken in turn.  The rest of the list stays in turn,
// so that its fronts of long K spread over the chip.  A bijection on [0, nb).
template <int NS>
__device__ __forceinline__ int gemm_order(int bid, int nb) {
  constexpr int RUN = GT_SUPER * GT_SUPER * NS;
  const int g = bid / (8 * RUN);
  if ((g + 1) * 8 * RUN > nb) return bid;
  const int x = bid & 7, s = (bid % (8 * RUN)) >> 3;
  return g * 8 * RUN + x * RUN + s;
}

// C[r0:r0+TM, c0:min(c0+TN, cend)) -= (L[r0:, k0:k1] D[k0:k1]) L[c0:, k0:k1]^T
// on one TM x TN tile of a column-major front.  The launch covers a list of
// 128 x 128 tiles with NS = (128 / TM)(128 / TN) workgroups each; one whose
// part starts outside the tile's valid rows and columns or lies above the
// diagonal returns at once (NS = 1 with a smaller tile is for lists of tiles
// that need no more than their first part).
//
// Four waves, 2 x 2, each own a TM/2 x TN/2 block.  The MFMA's first operand
// runs over C's columns, so that the lanes of an output register hold BS
// consecutive rows of the front (coalesced C access).
//  - Global loads: 16 bytes down a column of each panel per thread.  A group
//    of rows that starts at or beyond the last valid row starts at that row
//    instead; it then reads up to E - 1 entries past the column (the next
//    column's unused upper part, or the arena's padding), which reach only C
//    entries that are not stored.  Columns beyond k1 are clamped to k1 - 1 and
//    their D is 0; no load carries a mask.
//  - LDS holds KT columns as they lie in the front, [k][row], so a thread's
//    loads are stored as they are and an MFMA operand read is one entry per
//    lane along the rows (consecutive banks).  D multiplies the B panel at the
//    store.  Two buffers, one barrier per KT columns.
//  - PD tiles of KT columns are in flight in registers, in straight-line code:
//    each step issues the loads PD tiles ahead, the products of the current
//    tile, then stores the next tile.
// An accumulator receives its products in the order of k whatever the tile, so
// every shape gives identical results.
//
// Bound by the MFMA rate where K and the tile count are large, by C traffic
// and the fill of the chip where K is small.  Measured TFLOP/s of a front of m
// rows, K pivots, FP32 128 x 128 / 128 x 64 / 64 x 64 (FP64 128 x 64 / 64 x 64):
//   m = 18000, K = 3000 (7021 tiles): 127 / 122 / 109   (65 / 56)
//   m = 16383, K =  256 (8001 tiles): 102 / 102 / 102   (55 / 54)
//   m =  3001, K =  256  (253 tiles):  61 /  62 /  64   (36 / 39)
//   m =  2500, K = 1000   (78 tiles):  28 /  45 /  47   (24 / 26)
// against 118, 91, 55 and 21 (64, 52, 32 and 14) of the best of five kernels
// with 128 x 128 tiles, k-contiguous LDS rows, 16 x 16 blocks and one tile of
// up to 64 (32) columns in flight; without the list's order by blocks the FP64
// 128 x 64 shape reached 59 at the first size.
template <typename T, int TM, int TN, int KT, int PD, int NS>
__device__ __forceinline__ void gemm_tile(const FrontDesc* __restrict__ fd, const GemmTile* __restrict__ tiles,
                                          T* __restrict__ arena, const double* __restrict__ dpiv) {
  using M = GemmMfma<T>;
  using U = typename M::unaligned_t;
  using V = typename M::lds_t;
  constexpr int WM = TM / 2, WN = TN / 2, BM = WM / M::BS, BN = WN / M::BS, E = M::E;
  constexpr int QA = TM / E, QB = TN / E;        // 16-byte groups per column
  constexpr int CA = 256 / QA, CB = 256 / QB;    // columns per load of the workgroup
  constexpr int LA = KT / CA, LB = KT / CB;      // loads per thread and tile of KT columns
  static_assert(LA * CA == KT && LB * CB == KT && PD % 2 == 0, "KT columns are whole loads, PD keeps buffer parity");
  __shared__ __attribute__((aligned(16))) T As[2][KT][TM];
  __shared__ __attribute__((aligned(16))) T Bs[2][KT][TN];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int wg = gemm_order<NS>(blockIdx.x, gridDim.x);
  const GemmTile t = tiles[wg / NS];
  const int part = wg % NS;
  constexpr int NR = NS == 1 ? 1 : GT_M / TM;
  const int r0 = t.r0 + (part % NR) * TM, c0 = t.c0 + (part / NR) * TN;
  const FrontDesc d = fd[t.front];
  if (r0 >= d.m || c0 >= t.cend || c0 > r0 + TM - 1) return;
  T* F = arena + d.off;
  const int64_t m = d.m;
  const int qa = tid % QA, ca = tid / QA, qb = tid % QB, cb = tid / QB;
  const T* pa = F + min(r0 + E * qa, d.m - 1);
  const T* pb = F + min(c0 + E * qb, t.cend - 1);
  struct Stage {
    U ra[LA], rb[LB];
    double rd[LB];
    int kl;
  };
  auto gload = [&](Stage& s, int kb) {
    s.kl = kb;
#pragma unroll
    for (int i = 0; i < LA; ++i)
      s.ra[i] = *reinterpret_cast<const U*>(pa + static_cast<int64_t>(min(kb + ca + CA * i, t.k1 - 1)) * m);
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int c = min(kb + cb + CB * i, t.k1 - 1);
      s.rb[i] = *reinterpret_cast<const U*>(pb + static_cast<int64_t>(c) * m);
      s.rd[i] = dpiv[d.start + c];
    }
  };
  auto store = [&](const Stage& s, int buf) {
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      V v;
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = s.ra[i][e];
      *reinterpret_cast<V*>(&As[buf][ca + CA * i][E * qa]) = v;
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const T dk = s.kl + cb + CB * i < t.k1 ? static_cast<T>(s.rd[i]) : T(0);
      V v;
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = s.rb[i][e] * dk;
      *reinterpret_cast<V*>(&Bs[buf][cb + CB * i][E * qb]) = v;
    }
  };
  typename M::acc_t acc[BN][BM];
#pragma unroll
  for (int j = 0; j < BN; ++j)
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
      for (int e = 0; e < M::NACC; ++e) acc[j][i][e] = 0;
  const int lr = lane & (M::BS - 1), lk = lane / M::BS;
  auto products = [&](int buf) {
    const T* ap = &As[buf][lk][wm * WM + lr];
    const T* bp = &Bs[buf][lk][wn * WN + lr];
#pragma unroll
    for (int k = 0; k < KT; k += M::KS) {
      T a[BM], b[BN];
#pragma unroll
      for (int i = 0; i < BM; ++i) a[i] = ap[k * TM + M::BS * i];
#pragma unroll
      for (int j = 0; j < BN; ++j) b[j] = bp[k * TN + M::BS * j];
#pragma unroll
      for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j) acc[j][i] = M::op(b[j], a[i], acc[j][i]);
    }
  };
  const int nt = (t.k1 - t.k0 + KT - 1) / KT;
  Stage s[PD];
#pragma unroll
  for (int p = 0; p < PD; ++p) gload(s[p], t.k0 + p * KT);
  store(s[0], 0);
  __syncthreads();
  int q = 0;
  for (; q + PD < nt; q += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      gload(s[u], t.k0 + (q + u + PD) * KT);
      products(u & 1);
      store(s[(u + 1) % PD], (u + 1) & 1);
      __syncthreads();
    }
  }
#pragma unroll
  for (int u = 0; u < PD; ++u) {
    products(u & 1);
    if (q + u + 1 >= nt) break;
    if (u + 1 < PD) store(s[(u + 1) % PD], (u + 1) & 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < BM; ++i) {
    const int row = r0 + wm * WM + M::BS * i + lr;
    const int rowc = min(row, d.m - 1);
    // all reads of a block row before its writes, so that they overlap
    T cv[BN][M::NACC];
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int e = 0; e < M::NACC; ++e)
        cv[j][e] = F[rowc + static_cast<int64_t>(min(c0 + wn * WN + M::BS * j + M::ocol(lane, e), t.cend - 1)) * m];
    if (row >= d.m) continue;
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
      for (int e = 0; e < M::NACC; ++e) {
        const int c = c0 + wn * WN + M::BS * j + M::ocol(lane, e);
        if (c < t.cend) F[row + static_cast<int64_t>(c) * m] = cv[j][e] - acc[j][i][e];
      }
  }
}

template <typename T, int TM, int TN, int KT, int PD, int NS, int W>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(W))) void k_gemm(
    const FrontDesc* __restrict__ fd, const GemmTile* __restrict__ tiles, T* __restrict__ arena,
    const double* __restrict__ dpiv) {
  gemm_tile<T, TM, TN, KT, PD, NS>(fd, tiles, arena, dpiv);
}

enum GemmShape { GEMM_64x64 = 0, GEMM_128x64 = 1, GEMM_128x128 = 2 };
// FP64 128 x 128 needs 64 accumulator registers more, spills, and is slower
// than 128 x 64 at every size measured (m = 16383, K = 2048: 61 against 62
// TFLOP/s, m = 12000, K = 256: 46 against 53): FP64 factors have two shapes.
template <typename T>
constexpr int kGemmShapes = std::is_same<T, float>::value ? 3 : 2;

}  // namespace rf
