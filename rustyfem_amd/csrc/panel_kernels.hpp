// Inner pivot step of the multifrontal LDL^T on gfx950: one 64-column pivot
// block B = [j0, j0 + jb) of each front, inside an outer block [J0, J0 + 256).
#pragma once
#include <hip/hip_runtime.h>

#include "lane_ops.hpp"
#include "mf.hpp"
#include "mfma.hpp"

namespace rf {

// orders the LDS accesses of one wave
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDL^T of the jb x jb pivot block (jb <= 64) and the inverse of its unit
// lower factor, blocked by 16 columns, by all four waves of the workgroup.
//   in:  A[q][i] = A_BB[i][q] (column q, row i), zero outside jb x jb; the
//        16 x 16 tiles above the diagonal ones are not read
//   out: A's lower triangle holds L below the diagonal and D on it (the
//        identity beyond jb); dout[i] = D_i (0 beyond jb); V[q][i] =
//        L^-1[i][q] for q <= i < jb, anything elsewhere; the pivot
//        test (src/sparse.rs:528-531) against orig = the original diagonal of
//        lane i of wave 0, the first failing equation eq0 + i wins in *err (no
//        test when err is null)
//   T:   scratch of kLdltScratch doubles
// Block column b: wave 0 eliminates its 16 columns for every row (lane i
// owns row i, columns 16b..16b+15 in registers; step j reads the pivot row
// from the lanes' registers); then the waves apply the block's update
// -L[:, blk] D[blk] L[:, blk]^T to the trailing lower 16 x 16 tiles with FP64
// MFMA (K = 16).  While wave 0 eliminates block column b the other waves
// complete row b - 1 of the inverse and sum for row b.
//
// Bound by the chain of 64 pivots (divide, lane read, fused multiply-add) in
// one wave, 284 cycles a pivot of about 35 instructions (a division without its
// scaling steps left it the same), 65% of a 64-column block's 28,000 cycles.
// What went: the inverse after the elimination instead of beside it, passes
// that only wrote zeros (33,000 cycles with them).
constexpr int kLdltScratch = 6 * 16 * 17;

__device__ __forceinline__ void block_ldlt_blk(double (*A)[NB + 1], double (*V)[NB + 2], double* T, double* dout,
                                               int jb, double orig, int64_t eq0,
                                               unsigned long long* err) {
  using M = Mfma<double>;
  constexpr int BS = 16, BP = BS + 1;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // identity beyond jb, so that every step below is uniform; the 16-column
  // blocks past jb (nbe on) stay identity and are skipped
  const int nbe = __builtin_amdgcn_readfirstlane((jb + BS - 1) / BS);
  if (tid < NB && tid >= jb) A[tid][tid] = 1.0;
  __syncthreads();
  // The inverse's column of blocks be = w - 1 belongs to wave w = 1, 2, 3:
  // V_ab = -V_aa sum_{c=b}^{a-1} L_ac V_cb.  row_sum(a) leaves the sum in the
  // wave's Tw; row_end(a) inverts L_aa (every wave for itself) and completes
  // the block.  V_aa is stored by the wave of column a, V_33 by wave 1.
  const int be = wave - 1;
  double* Tw = T + be * 2 * BS * BP;  // Tw[j * BP + i] = sum[i][j]
  double* Uw = Tw + BS * BP;          // Uw[q * BP + i] = V_aa[i][q]
  auto row_sum = [&](int a) {
    M::acc_t t = M::acc_t{0, 0, 0, 0};
#pragma unroll 1
    for (int c = be; c < a; ++c)
#pragma unroll
      for (int s4 = 0; s4 < BS / 4; ++s4) {
        const int k = BS * c + 4 * s4 + g;
        t = M::op(A[k][BS * a + l16], V[BS * be + l16][k], t);
      }
    // register r holds row g + 4 r, column l16
#pragma unroll
    for (int r = 0; r < 4; ++r) Tw[l16 * BP + g + 4 * r] = t[r];
  };
  auto row_end = [&](int a) {
    const int r0 = BS * a;
    // column l16 of L_aa^-1 (unit lower), the same in every lane group
    double x[BS];
#pragma unroll
    for (int i = 0; i < BS; ++i) x[i] = i == l16 ? 1.0 : 0.0;
#pragma unroll
    for (int p = 0; p < BS - 1; ++p)
#pragma unroll
      for (int i = p + 1; i < BS; ++i) x[i] = fma(-A[r0 + p][r0 + i], x[p], x[i]);
    if (g == 0) {
      if (be == a || (a == 3 && be == 0)) {
#pragma unroll
        for (int i = 0; i < BS; ++i) V[r0 + l16][r0 + i] = x[i];
      }
      if (be < a) {
#pragma unroll
        for (int i = 0; i < BS; ++i) Uw[l16 * BP + i] = x[i];
      }
    }
    wave_lds_sync();
    if (be < a) {
      M::acc_t o = M::acc_t{0, 0, 0, 0};
#pragma unroll
      for (int s4 = 0; s4 < BS / 4; ++s4) {
        const int k = 4 * s4 + g;
        o = M::op(Uw[k * BP + l16], Tw[l16 * BP + k], o);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) V[BS * be + l16][r0 + g + 4 * r] = -o[r];
    }
    wave_lds_sync();
  };
  // (not unrolled: the kernel's code is read once per launch, and its length
  // costs more than the loop)
#pragma unroll 1
  for (int b = 0; b <= nbe; ++b) {
    const int c0 = BS * b;
    if (wave != 0) {
      if (b > 0) row_end(b - 1);
      if (be < b && b < nbe) row_sum(b);
    } else if (b < nbe) {
      double r[BS];
#pragma unroll
      for (int q = 0; q < BS; ++q) r[q] = A[c0 + q][lane];
#pragma unroll
      for (int jj = 0; jj < BS; ++jj) {
        const double l = r[jj] / readlane_d(r[jj], c0 + jj);
#pragma unroll
        for (int q = jj + 1; q < BS; ++q) r[q] = fma(-l, readlane_d(r[jj], c0 + q), r[q]);
        if (lane > c0 + jj) r[jj] = l;
      }
      if (lane >= c0) {
#pragma unroll
        for (int q = 0; q < BS; ++q) A[c0 + q][lane] = r[q];
      }
    } else {
      // D and the pivot test beside the inverse's last row
      const double dl = A[lane][lane];
      if (err != nullptr && lane < jb && (!(orig > 0.0) || !(dl > 1e-12 * orig)))
        atomicMin(err, static_cast<unsigned long long>(eq0 + lane));
      dout[lane] = lane < jb ? dl : 0.0;
    }
    __syncthreads();
    // trailing lower tiles (ti, tc), b < tc <= ti < nbe, one per wave
    const int nt = nbe - 1 - b;
    for (int tt = wave; tt < nt * (nt + 1) / 2; tt += 4) {
      int ti = b + 1, rem = tt;
      while (rem >= ti - b) {
        rem -= ti - b;
        ++ti;
      }
      const int tc = b + 1 + rem;
      // output (row 16 ti + g + 4 r, column 16 tc + l16) in register r
      M::acc_t acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = A[BS * tc + l16][BS * ti + g + 4 * r];
#pragma unroll
      for (int s4 = 0; s4 < BS / 4; ++s4) {
        const int k = c0 + 4 * s4 + g;
        acc = M::op(-A[k][BS * ti + l16] * A[k][k], A[k][BS * tc + l16], acc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) A[BS * tc + l16][BS * ti + g + 4 * r] = acc[r];
    }
    if (nt > 0) __syncthreads();
  }
}

// The left-looking update of a pivot block reads the 0 to 3 earlier blocks of
// its outer block, one block of 64 columns at a time: a block's loads are
// issued before the products of the block before it, and what every wave would
// convert and scale for itself (L to FP64, times D) is done once, when it is
// stored to LDS.  Rows beyond jb (or beyond the front) are clamped to a valid
// row: they only reach update entries that are discarded.  The MFMA order over
// k is that of one k-step of 4 at a time (lane group g = lane / 16 takes
// k = 4 t + g at step t), the order of the fused panel kernel, so both give
// identical factors.
//
// Measured per launch, against staging all earlier columns as they are and
// converting in the product loop, whole pivot blocks instead of their lower
// tiles and W's zero blocks included: k_pdiag 21.7 -> 17.2 us, k_prow 13.1 ->
// 10.9 us (31x19x23 block, FP32 factor), 22.9 -> 19.7 and 15.3 -> 12.8 us
// (100k-DOF plate, FP64), 180 -> 161 and 137 -> 114 us (512 plates at once).
//
// k_pdiag (one workgroup per front): C_BB = Y D Y^T with Y = L[B, J0:j0],
// A_BB = F_BB - C_BB, then block_ldlt_blk; writes D and V = L_BB^-1 (the
// arena's pivot block stays as assembled).
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_pdiag(
    const FrontDesc* __restrict__ fd, const PanelTile* __restrict__ tiles,
                                               const T* __restrict__ arena, double* __restrict__ dpiv,
                                               const double* __restrict__ adiag, double* __restrict__ vbuf,
                                               unsigned long long* __restrict__ err) {
  using M = Mfma<double>;
  constexpr int PY = NB + 2;
  constexpr int YBYTES = 2 * NB * PY * 8;
  constexpr int ABYTES = NB * (NB + 1) * 8;  // Ad, factored in place
  constexpr int TOFF = (ABYTES + 15) / 16 * 16;  // the inverse's scratch after Ad
  constexpr int VOFF = TOFF + kLdltScratch * 8;  // then Vs
  constexpr int LBYTES = VOFF + NB * (NB + 2) * 8;
  // the update's staging and the factorization's buffers share one region
  // (79 KB in all), so that two workgroups fit in a CU's LDS
  __shared__ __attribute__((aligned(16))) unsigned char smem[YBYTES > LBYTES ? YBYTES : LBYTES];
  __shared__ double dd[NB];
  double(*Vs)[NB + 2] = reinterpret_cast<double(*)[NB + 2]>(smem + VOFF);  // Vs[q][i] = L^-1[i][q]
  double(*Yd)[PY] = reinterpret_cast<double(*)[PY]>(smem);                    // Yd[k][i] = L[j0 + i, p0 + k]
  double(*Zd)[PY] = reinterpret_cast<double(*)[PY]>(smem + NB * PY * 8);      // Yd[k][i] D[p0 + k]
  double(*Ad)[NB + 1] = reinterpret_cast<double(*)[NB + 1]>(smem);                  // after the update
  const PanelTile t = tiles[blockIdx.x];
  const FrontDesc d = fd[t.front];
  const int jb = t.jb, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const T* F = arena + d.off;
  const int64_t m = d.m;
  // the block's ten lower 16 x 16 tiles (row, column), three per wave at most:
  // (0,0) (3,0) | (1,0) (1,1) | (2,0) (2,1) (2,2) | (3,1) (3,2) (3,3); the
  // first two waves repeat their last one
  constexpr int NT = 3;
  const int l16 = lane & 15;
  int tr[NT], tc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    tr[n] = 16 * (wave == 0 ? (n == 0 ? 0 : 3) : wave);
    tc[n] = 16 * (wave == 0 ? 0 : wave == 1 ? min(n, 1) : wave == 2 ? n : n + 1);
  }
  // the original diagonal of lane i's pivot (for the test after the
  // elimination) and the block's own entries (lower triangle, mirrored)
  const double orig = lane < jb ? adiag[static_cast<int64_t>(d.start) + t.j0 + lane] : 1.0;
  // (read before the update in FP32; in FP64 after it, where the 32 registers
  // they take would push the update past two waves per SIMD)
  constexpr bool kEarly = sizeof(T) == 4;
  T fb[NT][4];
  auto load_fb = [&]() {
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = tr[n] + l16, q = tc[n] + M::orow(lane, r);
        const int hi = min(max(i, q), jb - 1), lo = min(min(i, q), jb - 1);
        fb[n][r] = F[t.j0 + hi + static_cast<int64_t>(t.j0 + lo) * m];
      }
  };
  if constexpr (kEarly) load_fb();
  M::acc_t cb[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) cb[n] = M::acc_t{0, 0, 0, 0};
  const int nblk = (t.j0 - t.J0) / NB, g = lane >> 4;
  const T* Fy = F + t.j0 + min(lane, jb - 1);
  // thread (lane, wave) loads row `lane` of the columns wave + 4 s
  T ry[NB / 4];
  double rd = 0.0;
  auto yload = [&](int p0) {
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) ry[s] = Fy[static_cast<int64_t>(p0 + wave + 4 * s) * m];
    rd = dpiv[d.start + p0 + lane];
  };
  if (nblk > 0) yload(t.J0);
#pragma unroll 1
  for (int c = 0; c < nblk; ++c) {
    lds_barrier();
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
      const double y = static_cast<double>(ry[s]);
      Yd[wave + 4 * s][lane] = y;
      Zd[wave + 4 * s][lane] = y * readlane_d(rd, wave + 4 * s);
    }
    lds_barrier();
    if (c + 1 < nblk) yload(t.J0 + (c + 1) * NB);
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
      const double* z = Zd[4 * s + g] + l16;
      const double* y = Yd[4 * s + g] + l16;
      const double y0 = y[tr[0]], y1 = y[tr[1]];
#pragma unroll
      for (int n = 0; n < NT; ++n) cb[n] = M::op(z[tc[n]], n == 0 ? y0 : y1, cb[n]);
    }
  }
  if constexpr (!kEarly) load_fb();
  __syncthreads();
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = tr[n] + l16, q = tc[n] + M::orow(lane, r);
      Ad[q][i] = (i < jb && q < jb) ? static_cast<double>(fb[n][r]) - cb[n][r] : 0.0;
    }
  __syncthreads();
  block_ldlt_blk(Ad, Vs, reinterpret_cast<double*>(smem + TOFF), dd, jb, orig,
                 static_cast<int64_t>(d.start) + t.j0, err);
  __syncthreads();
  // only the jb x jb block: the buffer is zero outside it from its
  // allocation on (and every pivot step of the plan writes the same jb)
  double* vb = vbuf + static_cast<int64_t>(t.task) * NB * NB + wave * 16 * NB + lane;
  double vo[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) vo[u] = lane >= wave * 16 + u ? Vs[wave * 16 + u][lane] : 0.0;
#pragma unroll
  for (int u = 0; u < 16; ++u)
    if (wave * 16 + u < jb && lane < jb) vb[u * NB] = vo[u];
  if (tid < jb) dpiv[d.start + t.j0 + tid] = dd[tid];
}

// k_prow (one workgroup per 64-row tile below the block): C_R = X D Y^T with
// X = L[r0:r0+64, J0:j0] (in registers, in the MFMA operand layout), then
// L_R = (F_R - C_R) L_BB^-T D^-1 on MFMA with W built from V and D.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_prow(
    const FrontDesc* __restrict__ fd, const PanelTile* __restrict__ tiles, T* __restrict__ arena,
    const double* __restrict__ dpiv, const double* __restrict__ vbuf) {
  using M = Mfma<double>;
  constexpr int PY = NB + 2;
  constexpr int YBYTES = NB * PY * 8;
  constexpr int WBYTES = NB * (NB + 1) * 8;
  __shared__ __attribute__((aligned(16))) unsigned char smem[YBYTES > WBYTES ? YBYTES : WBYTES];
  __shared__ double dinv[NB];
  double(*Zd)[PY] = reinterpret_cast<double(*)[PY]>(smem);  // Zd[k][i] = L[j0 + i, p0 + k] D[p0 + k]
  double(*Wd)[NB + 1] = reinterpret_cast<double(*)[NB + 1]>(smem);  // W[p][q] = L_BB^-1[q][p], after the update
  const PanelTile t = tiles[blockIdx.x];
  const FrontDesc d = fd[t.front];
  const int jb = t.jb, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  T* F = arena + d.off;
  const int64_t m = d.m;
  // the pivot block's inverse and D (written by the previous launch) first
  const double* vb = vbuf + static_cast<int64_t>(t.task) * NB * NB;
  double wv[NB * NB / 256];
#pragma unroll
  for (int s = 0; s < NB * NB / 256; ++s) {
    const int idx = tid + 256 * s;  // zero outside the jb x jb block
    wv[s] = (idx / NB < jb && idx % NB < jb) ? vb[idx] : 0.0;
  }
  const double dv = tid < jb ? dpiv[d.start + t.j0 + tid] : 1.0;
  const int i = wave * 16 + (lane & 15);
  const int row = t.r0 + i;
  const int rowc = min(row, d.m - 1);
  // A_R entries of this lane
  T fa[4][4];
#pragma unroll
  for (int bj = 0; bj < 4; ++bj)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int q = min(bj * 16 + M::orow(lane, r), jb - 1);
      fa[bj][r] = F[rowc + static_cast<int64_t>(t.j0 + q) * m];
    }
  M::acc_t cr[4];
#pragma unroll
  for (int bj = 0; bj < 4; ++bj) cr[bj] = M::acc_t{0, 0, 0, 0};
  const int nblk = (t.j0 - t.J0) / NB, g = lane / 16;
  const T* Fy = F + t.j0 + min(lane, jb - 1);
  const T* Fx = F + rowc;
  T ry[NB / 4], rx[NB / 4];
  double rd = 0.0;
  auto yload = [&](int p0) {
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
      ry[s] = Fy[static_cast<int64_t>(p0 + wave + 4 * s) * m];
      rx[s] = Fx[static_cast<int64_t>(p0 + 4 * s + g) * m];
    }
    rd = dpiv[d.start + p0 + lane];
  };
  if (nblk > 0) yload(t.J0);
#pragma unroll 1
  for (int c = 0; c < nblk; ++c) {
    lds_barrier();
    T xc[NB / 4];
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
      Zd[wave + 4 * s][lane] = static_cast<double>(ry[s]) * readlane_d(rd, wave + 4 * s);
      xc[s] = rx[s];
    }
    lds_barrier();
    if (c + 1 < nblk) yload(t.J0 + (c + 1) * NB);
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
      const double bx = static_cast<double>(xc[s]);
#pragma unroll
      for (int bj = 0; bj < 4; ++bj) cr[bj] = M::op(Zd[4 * s + g][bj * 16 + (lane & 15)], bx, cr[bj]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < NB * NB / 256; ++s) {
    const int idx = tid + 256 * s, q = idx % NB, p = idx / NB;
    Wd[p][q] = q < jb ? wv[s] : 0.0;
  }
  if (tid < NB) dinv[tid] = tid < jb ? 1.0 / dv : 0.0;
  // A_R = F_R - C_R stays in the registers that hold C_R: at TRSM step s the
  // lane's B operand is column 4s + lane/16 of its row, which is register
  // (s / 4, s % 4) of cr
  double ar[16];
#pragma unroll
  for (int bj = 0; bj < 4; ++bj)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int q = bj * 16 + M::orow(lane, r);
      ar[bj * 4 + r] = (row < d.m && q < jb) ? static_cast<double>(fa[bj][r]) - cr[bj][r] : 0.0;
    }
  __syncthreads();
  M::acc_t o[4];
#pragma unroll
  for (int bj = 0; bj < 4; ++bj) o[bj] = M::acc_t{0, 0, 0, 0};
  // (W is triangular: column block bj takes the first 4 bj + 4 steps)
#pragma unroll
  for (int s4 = 0; s4 < 16; ++s4) {
    const int kr = 4 * s4 + lane / 16;
#pragma unroll
    for (int bj = s4 / 4; bj < 4; ++bj) o[bj] = M::op(Wd[kr][bj * 16 + (lane & 15)], ar[s4], o[bj]);
  }
  if (row < d.m) {
#pragma unroll
    for (int bj = 0; bj < 4; ++bj)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int q = bj * 16 + M::orow(lane, r);
        if (q < jb) F[row + static_cast<int64_t>(t.j0 + q) * m] = T(o[bj][r] * dinv[q]);
      }
  }
}

}  // namespace rf
