// HIP kernels (gfx950) of the learned smoother's network: forward (the
// smoother's blocks from the matrix) and backward (parameter gradients from
// dL/dM), and a training handle that evaluates the smoothing loss
//   L = mean_v  e_nu^T A e_nu / e_0^T A e_0,   e_{k+1} = (I - M A) e_k,
// and its gradient by the adjoint recursion
//   g_nu = 2 A e_nu / (nvec e_0^T A e_0),
//   dL/dM += -g_{k+1} (A e_k)^T   (on M's block pattern),
//   g_k = g_{k+1} - A M g_{k+1}   (A and M symmetric).
// All reductions run in a fixed order (no atomics), so results are
// reproducible bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "amg.hpp"
#include "mfma.hpp"
#include "mpnn.hpp"
#include "mpnn_train.hpp"

namespace rf {

#define MCHK(expr)                                                                                   \
  do {                                                                                               \
    hipError_t e_ = (expr);                                                                          \
    if (e_ != hipSuccess) {                                                                          \
      char b_[512];                                                                                  \
      snprintf(b_, sizeof b_, "HIP error %s at %s:%d: %s", hipGetErrorString(e_), __FILE__, __LINE__, #expr); \
      throw std::runtime_error(b_);                                                                  \
    }                                                                                                \
  } while (0)

namespace {

constexpr int F = MPNN_F, H = MPNN_H;
constexpr int OW1 = 0, OB1 = H * F, OW2 = OB1 + H, OB2 = OW2 + H * 3 * H, OW3 = OB2 + H, OB3 = OW3 + 9 * H;
static_assert(OB3 + 9 == MPNN_NPARAMS, "parameter layout");
constexpr int TB = 256;

unsigned blocks_for(int64_t n) { return static_cast<unsigned>(std::max<int64_t>(1, (n + TB - 1) / TB)); }

template <typename T>
T* dnew(int64_t count) {
  T* p = nullptr;
  MCHK(hipMalloc(&p, static_cast<size_t>(std::max<int64_t>(count, 1)) * sizeof(T)));
  return p;
}

__device__ inline double relu(double v) { return v > 0.0 ? v : 0.0; }

// row of every block, node scales s_i = sqrt(3 / trace(A_ii))
__global__ void k_mg_rows(int64_t nb, const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                          const double* __restrict__ val, int32_t* __restrict__ row, double* __restrict__ scale) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (i >= nb) return;
  double tr = 0.0;
  for (int64_t e = ptr[i]; e < ptr[i + 1]; ++e) {
    row[e] = static_cast<int32_t>(i);
    if (idx[e] == i) tr = val[9 * e] + val[9 * e + 4] + val[9 * e + 8];
  }
  scale[i] = tr > 0.0 ? sqrt(3.0 / tr) : 1.0;
}

// rev(e): the position of block (j, i) for block e = (i, j); -1 if absent
__global__ void k_mg_rev(int64_t nnzb, const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                         const int32_t* __restrict__ row, int32_t* __restrict__ rev) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (e >= nnzb) return;
  const int32_t i = row[e], j = idx[e];
  int64_t lo = ptr[j], hi = ptr[j + 1] - 1, found = -1;
  while (lo <= hi) {
    const int64_t mid = (lo + hi) / 2;
    if (idx[mid] == i) {
      found = mid;
      break;
    }
    if (idx[mid] < i) lo = mid + 1;
    else hi = mid - 1;
  }
  rev[e] = static_cast<int32_t>(found);
}

__global__ void k_mg_feat(int64_t nnzb, const int32_t* __restrict__ row, const int32_t* __restrict__ idx,
                          const double* __restrict__ val, const double* __restrict__ scale, double* __restrict__ feat) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (e >= nnzb) return;
  const int32_t i = row[e], j = idx[e];
  const double s = scale[i] * scale[j];
  for (int q = 0; q < 9; ++q) feat[F * e + q] = s * val[9 * e + q];
  feat[F * e + 9] = i == j ? 1.0 : 0.0;
}

// The 64 columns [W2b^T | W2c^T] of the second layer's node parts: entry
// (b, c) is W2[c][H + b] for c < H and W2[c - H][2H + b] above.
__device__ __forceinline__ double w2_node(const double* __restrict__ prm, int b, int c) {
  return prm[OW2 + (c & (H - 1)) * 3 * H + (c < H ? H : 2 * H) + b];
}

constexpr int NPW = 4;  // nodes per wave of the per-node kernels

// Per node i: the edge messages' first layer pre1_e = W1 x_e + b1 of its
// blocks, n_i = mean relu(pre1_e), and the node's share of the second layer,
// P_i = W2b n_i + b2 and Q_i = W2c n_i (W2 [m_e; n_i; n_j] = W2a m_e + W2b n_i
// + W2c n_j, so that the 64 node columns are multiplied once per node and not
// once per block).
// One wave per node at a time: lane = (half, hidden unit), each half takes
// every other block of the row, a block's 32 outputs are one 256-byte store.
// Bound by those stores: 53 us for 24^3 cubes (210,694 blocks, 54 MB of pre1).
__global__ __launch_bounds__(TB) void k_mg_l1(int64_t nb, const double* __restrict__ prm,
                                              const int64_t* __restrict__ ptr, const double* __restrict__ feat,
                                              double* __restrict__ pre1, double* __restrict__ node,
                                              double* __restrict__ pq) {
  static_assert(H == 32 && F == 10, "lane = (half, hidden unit)");
  __shared__ double wn[H][2 * H];
  __shared__ double ns[TB / 64][H];
  for (int t = threadIdx.x; t < H * 2 * H; t += TB) wn[t / (2 * H)][t % (2 * H)] = w2_node(prm, t / (2 * H), t % (2 * H));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, a = lane & 31, half = lane >> 5;
  double w1[F];
#pragma unroll
  for (int q = 0; q < F; ++q) w1[q] = prm[OW1 + a * F + q];
  const double b1 = prm[OB1 + a], b2 = half == 0 ? prm[OB2 + a] : 0.0;
  __syncthreads();
  for (int w = 0; w < NPW; ++w) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * (TB / 64) + wave) * NPW + w;
    const bool in = i < nb;
    const int64_t e0 = in ? ptr[i] : 0, e1 = in ? ptr[i + 1] : 0;
    double acc = 0.0;
    for (int64_t e = e0 + half; e < e1; e += 2) {
      double v = b1;
#pragma unroll
      for (int q = 0; q < F; ++q) v += w1[q] * feat[F * e + q];
      pre1[H * e + a] = v;
      acc += relu(v);
    }
    acc += __shfl_xor(acc, 32, 64);
    const double n = acc * (1.0 / static_cast<double>(max<int64_t>(1, e1 - e0)));
    if (half == 0) ns[wave][a] = n;
    __syncthreads();
    double v = b2;
#pragma unroll
    for (int b = 0; b < H; ++b) v += wn[b][lane] * ns[wave][b];
    if (in) {
      if (half == 0) node[H * i + a] = n;
      pq[2 * H * i + lane] = v;
    }
    __syncthreads();
  }
}

// Rows of a 32-unit layer as MFMA rows: row rho of tile t is unit
// 8 (rho % 4) + 4 t + rho / 4, so that lane group g holds units 8 g .. 8 g + 7
// of its column in the two tiles' output registers: 64 consecutive bytes in
// memory, and, in that order, the lane's operands of the next layer's steps.
__device__ __forceinline__ int unit_of(int t, int rho) { return 8 * (rho & 3) + 4 * t + (rho >> 2); }

// eight consecutive doubles at a 64-byte aligned address
__device__ __forceinline__ void load8(const double* __restrict__ p, double (&v)[8]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const v2d w = reinterpret_cast<const v2d*>(p)[q];
    v[2 * q] = w[0];
    v[2 * q + 1] = w[1];
  }
}
__device__ __forceinline__ void store8(double* __restrict__ p, const double (&v)[8]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) reinterpret_cast<v2d*>(p)[q] = v2d{v[2 * q], v[2 * q + 1]};
}

// Second layer and output of 16 blocks per wave pass on FP64 MFMA:
// h = W2a relu(pre1_e) + P_i + Q_j (16 MFMAs), o = W3 relu(h) + b3 (8 more,
// the output registers of the first product are the operands of the second).
// Column of the MFMA = block, step s of lane group g = unit 8 g + s.  Bound by
// the reads of pre1, P, Q and the writes of pre2.  210,694 blocks: one thread
// per block, W2 over 96 inputs in VALU FMAs with 256-byte lane strides, 99 us;
// this, 49 us.
__global__ __launch_bounds__(TB) void k_mg_l2(int64_t nnzb, const double* __restrict__ prm,
                                              const int32_t* __restrict__ row, const int32_t* __restrict__ idx,
                                              const double* __restrict__ pre1, const double* __restrict__ pq,
                                              double* __restrict__ pre2, double* __restrict__ out) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  double wa[2][8], w3[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
#pragma unroll
    for (int t = 0; t < 2; ++t) wa[t][s] = prm[OW2 + unit_of(t, c) * 3 * H + 8 * g + s];
    w3[s] = c < 9 ? prm[OW3 + c * H + 8 * g + s] : 0.0;
  }
  double b3[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) b3[r] = g + 4 * r < 9 ? prm[OB3 + g + 4 * r] : 0.0;
  const int64_t nw = static_cast<int64_t>(gridDim.x) * (TB / 64);
  for (int64_t w = static_cast<int64_t>(blockIdx.x) * (TB / 64) + (threadIdx.x >> 6); w * 16 < nnzb; w += nw) {
    const int64_t e = min(w * 16 + c, nnzb - 1);  // the last pass repeats the last block
    const bool in = w * 16 + c < nnzb;
    double m[8], p[8], q[8];
    load8(pre1 + H * e + 8 * g, m);
    load8(pq + 2 * H * static_cast<int64_t>(row[e]) + 8 * g, p);
    load8(pq + 2 * H * static_cast<int64_t>(idx[e]) + H + 8 * g, q);
    v4d acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] = p[4 * t + r] + q[4 * t + r];
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = Mfma<double>::op(wa[t][s], relu(m[s]), acc[t]);
    double h[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) h[s] = acc[s >> 2][s & 3];
    if (in) store8(pre2 + H * e + 8 * g, h);
    v4d o = v4d{b3[0], b3[1], b3[2], 0.0};
#pragma unroll
    for (int s = 0; s < 8; ++s) o = Mfma<double>::op(w3[s], relu(h[s]), o);
    if (in) {
#pragma unroll
      for (int r = 0; r < 3; ++r)
        if (g + 4 * r < 9) out[9 * e + g + 4 * r] = o[r];
    }
  }
}

__global__ void k_mg_out(int64_t nnzb, const int32_t* __restrict__ row, const int32_t* __restrict__ idx,
                         const int32_t* __restrict__ rev, const double* __restrict__ scale,
                         const double* __restrict__ out, double* __restrict__ m) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (e >= nnzb) return;
  const int32_t i = row[e], j = idx[e];
  const int64_t t = rev[e];
  const double s = scale[i] * scale[j];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double g = 0.5 * (out[9 * e + 3 * r + c] + out[9 * t + 3 * c + r]);
      m[9 * e + 3 * r + c] = s * (g + ((i == j && r == c) ? MPNN_OMEGA : 0.0));
    }
}

// Backward of the output and second layers, 16 blocks per wave pass on FP64
// MFMA with the layout of k_mg_l2:
//   go_e = dL/dO_e = (s_i s_j) (dL/dM_e + dL/dM_rev(e)^T) / 2
//   d2_e = (W3^T go_e) where pre2_e > 0         (dL/dpre2)
//   dm_e = W2a^T d2_e                           (dL/dm_e through this layer)
// Lane group g < 3 supplies row g of the 3 x 3 block as steps 0..2 of the
// first product; the node parts of the layer follow in k_mg_bnode from sums
// of d2 alone.  210,694 blocks: with the 96-wide W2^T d2 per block and one
// thread per block 136 us (dL/dO in a pass before it); this, 56 us (bound by pre2, d2 and dm: 3 x 54 MB).
__global__ __launch_bounds__(TB) void k_mg_b2(int64_t nnzb, const double* __restrict__ prm,
                                              const int32_t* __restrict__ row, const int32_t* __restrict__ idx,
                                              const int32_t* __restrict__ rev, const double* __restrict__ scale,
                                              const double* __restrict__ gm, const double* __restrict__ pre2,
                                              double* __restrict__ go, double* __restrict__ d2,
                                              double* __restrict__ dm) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  double w3t[2][3], wat[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int u = unit_of(t, c);
#pragma unroll
    for (int s = 0; s < 3; ++s) w3t[t][s] = g < 3 ? prm[OW3 + (3 * g + s) * H + u] : 0.0;
#pragma unroll
    for (int s = 0; s < 8; ++s) wat[t][s] = prm[OW2 + (8 * g + s) * 3 * H + u];
  }
  const int64_t nw = static_cast<int64_t>(gridDim.x) * (TB / 64);
  for (int64_t w = static_cast<int64_t>(blockIdx.x) * (TB / 64) + (threadIdx.x >> 6); w * 16 < nnzb; w += nw) {
    const int64_t e = min(w * 16 + c, nnzb - 1);
    const bool in = w * 16 + c < nnzb;
    const double sc = 0.5 * (scale[row[e]] * scale[idx[e]]);
    const int64_t t9 = 9 * static_cast<int64_t>(rev[e]);
    double gv[3] = {0.0, 0.0, 0.0};
    if (g < 3) {
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        gv[s] = sc * (gm[9 * e + 3 * g + s] + gm[t9 + 3 * s + g]);
        if (in) go[9 * e + 3 * g + s] = gv[s];
      }
    }
    double pre[8], d[8];
    load8(pre2 + H * e + 8 * g, pre);
    v4d acc[2] = {v4d{0, 0, 0, 0}, v4d{0, 0, 0, 0}};
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = Mfma<double>::op(w3t[t][s], gv[s], acc[t]);
#pragma unroll
    for (int s = 0; s < 8; ++s) d[s] = pre[s] > 0.0 ? acc[s >> 2][s & 3] : 0.0;
    if (in) store8(d2 + H * e + 8 * g, d);
    acc[0] = v4d{0, 0, 0, 0};
    acc[1] = v4d{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t] = Mfma<double>::op(wat[t][s], d[s], acc[t]);
#pragma unroll
    for (int s = 0; s < 8; ++s) d[s] = acc[s >> 2][s & 3];
    if (in) store8(dm + H * e + 8 * g, d);
  }
}

// Per node i: S_i = sum of d2 over the blocks of row i (where n_i is the row's
// node), R_i = the same over their reverses (where it is the column's), and
// dL/dn_i = W2b^T S_i + W2c^T R_i, times 1 / deg for the mean.  Half 0 of the
// wave sums S, half 1 R.  210,694 blocks: from the 96-wide dz of every block
// and its reverse 92 us (and 81 us for dpre1 as a pass of its own); this, 44 us.
__global__ __launch_bounds__(TB) void k_mg_bnode(int64_t nb, const double* __restrict__ prm,
                                                 const int64_t* __restrict__ ptr, const int32_t* __restrict__ rev,
                                                 const double* __restrict__ d2, double* __restrict__ sr,
                                                 double* __restrict__ dnode) {
  __shared__ double wt[2 * H][H + 1];  // wt[c][b]: w2_node(b, c)
  __shared__ double ss[TB / 64][2 * H];
  for (int t = threadIdx.x; t < H * 2 * H; t += TB) wt[t % (2 * H)][t / (2 * H)] = w2_node(prm, t / (2 * H), t % (2 * H));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, a = lane & 31, half = lane >> 5;
  __syncthreads();
  for (int w = 0; w < NPW; ++w) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * (TB / 64) + wave) * NPW + w;
    const bool in = i < nb;
    const int64_t e0 = in ? ptr[i] : 0, e1 = in ? ptr[i + 1] : 0;
    double acc = 0.0;
#pragma unroll 4
    for (int64_t e = e0; e < e1; ++e) acc += d2[H * (half == 0 ? e : static_cast<int64_t>(rev[e])) + a];
    ss[wave][lane] = acc;
    __syncthreads();
    // output b = a; half 0 adds S's terms, half 1 R's
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < H; ++q) v += wt[H * half + q][a] * ss[wave][H * half + q];
    v += __shfl_xor(v, 32, 64);
    if (in) {
      sr[2 * H * i + lane] = acc;
      if (half == 0) dnode[H * i + a] = v * (1.0 / static_cast<double>(max<int64_t>(1, e1 - e0)));
    }
    __syncthreads();
  }
}

// Parameter gradients as FP64-MFMA products over the blocks and the nodes
// (K = 210,694 blocks for 3,753 parameters): every wave sums its share of the
// blocks, the four waves of a workgroup are added through LDS and the
// workgroups' partial sums by k_mg_wsum, all in a fixed order.
// Workgroups < neb take blocks:
//   W2a (a, b) += d2 relu(pre1)^T, W1 (a, f) += dpre1 feat^T with dpre1 =
//   dm + dnode where pre1 > 0, W3 (q, a) += go relu(pre2)^T, and the biases
//   as the sums of d2, dpre1 and go;
// the others take nodes: W2b += S n^T, W2c += R n^T (the sums over the blocks
// of a row share n).  Step k of lane group g is block (node) 4 k + g; lane
// l % 16 is the row of A and the column of B, so that a group's operand load is
// 128 consecutive bytes.  One workgroup per parameter, each reading every
// block, took 17.3 ms on 210,694 blocks; this 91 us and k_mg_wsum 7 us.
constexpr int WG_OUT = static_cast<int>(MPNN_NPARAMS);
__device__ __forceinline__ void wg_tile(double* __restrict__ red, int row0, int nrow, int ncol, int ld, const v4d& acc,
                                        int g, int c) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (g + 4 * r < nrow && c < ncol) red[row0 + (g + 4 * r) * ld + c] += acc[r];
}
__device__ __forceinline__ double group4_sum(double v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

__global__ __launch_bounds__(TB) void k_mg_wgrad(int64_t nnzb, int64_t nb, int neb, const int32_t* __restrict__ row,
                                                 const double* __restrict__ feat, const double* __restrict__ pre1,
                                                 const double* __restrict__ node, const double* __restrict__ pre2,
                                                 const double* __restrict__ go, const double* __restrict__ d2,
                                                 const double* __restrict__ dm, const double* __restrict__ dnode,
                                                 const double* __restrict__ sr, double* __restrict__ part) {
  using M = Mfma<double>;
  __shared__ double red[WG_OUT];
  for (int t = threadIdx.x; t < WG_OUT; t += TB) red[t] = 0.0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const v4d z4 = v4d{0, 0, 0, 0};
  if (static_cast<int>(blockIdx.x) < neb) {
    v4d w2[2][2], w1[2], w3[2];
    double s2[2] = {0.0, 0.0}, s1[2] = {0.0, 0.0}, s3 = 0.0;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      w2[t][0] = w2[t][1] = w1[t] = w3[t] = z4;
    }
    const int64_t nw = static_cast<int64_t>(neb) * (TB / 64);
#pragma unroll 2
    for (int64_t k = static_cast<int64_t>(blockIdx.x) * (TB / 64) + wave; k * 4 < nnzb; k += nw) {
      const int64_t e = min(k * 4 + g, nnzb - 1);
      const double live = k * 4 + g < nnzb ? 1.0 : 0.0;  // the A operands of blocks past the last are 0
      const int64_t i = row[e];
      double dv[2], pv[2], hv[2], uv[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        dv[t] = live * d2[H * e + 16 * t + c];
        pv[t] = pre1[H * e + 16 * t + c];
        hv[t] = relu(pre2[H * e + 16 * t + c]);
        uv[t] = live * (dm[H * e + 16 * t + c] + dnode[H * i + 16 * t + c]);
      }
      const double fv = c < F ? feat[F * e + c] : 0.0;
      const double gv = c < 9 ? live * go[9 * e + c] : 0.0;
      s3 += gv;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        uv[t] = pv[t] > 0.0 ? uv[t] : 0.0;
        s2[t] += dv[t];
        s1[t] += uv[t];
        w1[t] = M::op(uv[t], fv, w1[t]);
        w3[t] = M::op(gv, hv[t], w3[t]);
#pragma unroll
        for (int u = 0; u < 2; ++u) w2[t][u] = M::op(dv[t], relu(pv[u]), w2[t][u]);
      }
    }
    for (int w = 0; w < TB / 64; ++w) {
      __syncthreads();
      if (wave != w) continue;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int u = 0; u < 2; ++u) wg_tile(red, OW2 + 16 * t * 3 * H + 16 * u, 16, 16, 3 * H, w2[t][u], g, c);
        wg_tile(red, OW1 + 16 * t * F, 16, F, F, w1[t], g, c);
        wg_tile(red, OW3 + 16 * t, 9, 16, H, w3[t], g, c);
        const double b2 = group4_sum(s2[t]), b1 = group4_sum(s1[t]);
        if (g == 0) {
          red[OB2 + 16 * t + c] += b2;
          red[OB1 + 16 * t + c] += b1;
        }
      }
      const double b3 = group4_sum(s3);
      if (g == 0 && c < 9) red[OB3 + c] += b3;
    }
  } else {
    v4d w2[2][2][2];  // [b or c part][a tile][b tile]
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int t = 0; t < 2; ++t) w2[p][t][0] = w2[p][t][1] = z4;
    const int64_t nw = static_cast<int64_t>(gridDim.x - neb) * (TB / 64);
#pragma unroll 2
    for (int64_t k = static_cast<int64_t>(blockIdx.x - neb) * (TB / 64) + wave; k * 4 < nb; k += nw) {
      const int64_t i = min(k * 4 + g, nb - 1);
      const double live = k * 4 + g < nb ? 1.0 : 0.0;
      double nv[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) nv[u] = node[H * i + 16 * u + c];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const double sv = live * sr[2 * H * i + H * p + 16 * t + c];
#pragma unroll
          for (int u = 0; u < 2; ++u) w2[p][t][u] = M::op(sv, nv[u], w2[p][t][u]);
        }
    }
    for (int w = 0; w < TB / 64; ++w) {
      __syncthreads();
      if (wave != w) continue;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int u = 0; u < 2; ++u)
            wg_tile(red, OW2 + 16 * t * 3 * H + H * (p + 1) + 16 * u, 16, 16, 3 * H, w2[p][t][u], g, c);
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < WG_OUT; t += TB) part[static_cast<int64_t>(blockIdx.x) * WG_OUT + t] = red[t];
}

// grad[p] = sum of the workgroups' partial sums: 64 parameters per workgroup,
// its four waves take every fourth partial sum
__global__ __launch_bounds__(TB) void k_mg_wsum(int np, const double* __restrict__ part, double* __restrict__ grad) {
  __shared__ double red[TB / 64][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int p = blockIdx.x * 64 + lane;
  double s = 0.0;
  if (p < WG_OUT)
#pragma unroll 8
    for (int q = wave; q < np; q += TB / 64) s += part[static_cast<int64_t>(q) * WG_OUT + p];
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && p < WG_OUT) grad[p] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// ------------------------------------------------------------ training loss

// The nvec vectors of the loss are interleaved (entry t of vector v at
// [t nvec + v]): the vectors of one node share its blocks, and a block's
// products read consecutive entries.

// x (n x nvec column-major) -> interleaved
__global__ __launch_bounds__(TB) void k_interleave(int64_t n, int nvec, const double* __restrict__ x,
                                                   double* __restrict__ y) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (t < n * nvec) y[t] = x[(t % nvec) * n + t / nvec];
}

// Y = A X, or with `from`, Y = from - A X (A: 3x3 blocks).  Four lanes per
// (node, vector) take every fourth block of the row; the vectors of a node
// are adjacent lanes.  210,694 blocks, 8 vectors: one thread per (node,
// vector), vectors column by column, 34 us; this, 13 us.
__global__ __launch_bounds__(TB) void k_bsr3_mv(int64_t nb, int nvec, const int64_t* __restrict__ ptr,
                                                const int32_t* __restrict__ idx, const double* __restrict__ val,
                                                const double* __restrict__ x, const double* from,
                                                double* y) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  const int64_t w = t >> 6;
  // a wave: 16 (node, vector) pairs, sub-lane = which quarter of the row's blocks
  const int64_t p = w * 16 + (t & 15);
  const int sub = static_cast<int>((t >> 4) & 3);
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  const bool in = p < nb * nvec;
  const int64_t i = in ? p / nvec : 0;
  const int v = static_cast<int>(in ? p % nvec : 0);
  if (in) {
    const int64_t e1 = ptr[i + 1];
#pragma unroll 2
    for (int64_t e = ptr[i] + sub; e < e1; e += 4) {
      const double* b = val + 9 * e;
      const double* xj = x + 3 * static_cast<int64_t>(idx[e]) * nvec + v;
      const double x0 = xj[0], x1 = xj[nvec], x2 = xj[2 * nvec];
      a0 += b[0] * x0 + b[1] * x1 + b[2] * x2;
      a1 += b[3] * x0 + b[4] * x1 + b[5] * x2;
      a2 += b[6] * x0 + b[7] * x1 + b[8] * x2;
    }
  }
  a0 = group4_sum(a0);
  a1 = group4_sum(a1);
  a2 = group4_sum(a2);
  if (in && sub < 3) {
    const double s = sub == 0 ? a0 : sub == 1 ? a1 : a2;
    const int64_t o = (3 * i + sub) * nvec + v;
    y[o] = from ? from[o] - s : s;
  }
}

// partial sums of x_v . y_v (part 0) and z_v . w_v (part 1) over NDB chunks
// of the rows: out[part][chunk][v]; a workgroup's 256 threads take (row,
// vector) pairs, the rows of one vector added in a fixed order
constexpr int NDB = 128;
__global__ __launch_bounds__(TB) void k_dots(int64_t n, int nvec, const double* __restrict__ x,
                                             const double* __restrict__ y, const double* __restrict__ z,
                                             const double* __restrict__ w, double* __restrict__ out) {
  __shared__ double red[TB];
  const double* a = blockIdx.y == 0 ? x : z;
  const double* b = blockIdx.y == 0 ? y : w;
  const int64_t r0 = n * blockIdx.x / NDB, r1 = n * (blockIdx.x + 1) / NDB;
  // vectors in passes of at most TB
  for (int v0 = 0; v0 < nvec; v0 += TB) {
    const int nv = min(TB, nvec - v0), rows = TB / nv;
    const int v = static_cast<int>(threadIdx.x) % nv, rr = static_cast<int>(threadIdx.x) / nv;
    double s = 0.0;
    if (rr < rows)
      for (int64_t r = r0 + rr; r < r1; r += rows) s += a[r * nvec + v0 + v] * b[r * nvec + v0 + v];
    __syncthreads();
    red[threadIdx.x] = s;
    __syncthreads();
    if (rr == 0) {
      for (int q = 1; q < rows; ++q) s += red[q * nv + v];
      out[(static_cast<int64_t>(blockIdx.y) * NDB + blockIdx.x) * nvec + v0 + v] = s;
    }
  }
}

// out[part][v] = the NDB partial sums in order, one thread each
__global__ __launch_bounds__(TB) void k_dots_sum(int nvec, const double* __restrict__ part, double* __restrict__ out) {
  const int t = blockIdx.x * TB + threadIdx.x;
  if (t >= 2 * nvec) return;
  const double* p = part + static_cast<int64_t>(t / nvec) * NDB * nvec + t % nvec;
  double s = 0.0;
#pragma unroll 16
  for (int q = 0; q < NDB; ++q) s += p[static_cast<int64_t>(q) * nvec];
  out[t] = s;
}

// g_v = 2 (A e)_v / (nvec den_v)
__global__ __launch_bounds__(TB) void k_gscale(int64_t n, int nvec, const double* __restrict__ ae,
                                               const double* __restrict__ den, double* __restrict__ g) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (t >= n * nvec) return;
  g[t] = 2.0 * ae[t] / (static_cast<double>(nvec) * den[t % nvec]);
}

// gm_e = (first ? 0 : gm_e) - sum_v g[i] y[j]^T on the block pattern
__global__ __launch_bounds__(TB) void k_outer(int64_t nnzb, int nvec, int first, const int32_t* __restrict__ row,
                                              const int32_t* __restrict__ idx, const double* __restrict__ g,
                                              const double* __restrict__ y, double* __restrict__ gm) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (e >= nnzb) return;
  const double* gi = g + 3 * static_cast<int64_t>(row[e]) * nvec;
  const double* yj = y + 3 * static_cast<int64_t>(idx[e]) * nvec;
  double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int v = 0; v < nvec; ++v)
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[3 * r + c] += gi[r * nvec + v] * yj[c * nvec + v];
#pragma unroll
  for (int q = 0; q < 9; ++q) gm[9 * e + q] = (first ? 0.0 : gm[9 * e + q]) - acc[q];
}

}  // namespace

MpnnGraph::MpnnGraph(int64_t nb, int64_t nnzb, const int64_t* d_ptr, const int32_t* d_idx, const double* d_val,
                     hipStream_t s)
    : nb_(nb), nnzb_(nnzb), ptr_(d_ptr), idx_(d_idx), s_(s) {
  row_ = dnew<int32_t>(nnzb);
  rev_ = dnew<int32_t>(nnzb);
  scale_ = dnew<double>(nb);
  feat_ = dnew<double>(nnzb * F);
  pre1_ = dnew<double>(nnzb * H);
  node_ = dnew<double>(nb * H);
  pq_ = dnew<double>(nb * 2 * H);
  pre2_ = dnew<double>(nnzb * H);
  out_ = dnew<double>(nnzb * 9);
  k_mg_rows<<<blocks_for(nb), TB, 0, s_>>>(nb, d_ptr, d_idx, d_val, row_, scale_);
  k_mg_rev<<<blocks_for(nnzb), TB, 0, s_>>>(nnzb, d_ptr, d_idx, row_, rev_);
  k_mg_feat<<<blocks_for(nnzb), TB, 0, s_>>>(nnzb, row_, d_idx, d_val, scale_, feat_);
  MCHK(hipGetLastError());
  std::vector<int32_t> rv(static_cast<size_t>(nnzb));
  MCHK(hipMemcpyAsync(rv.data(), rev_, nnzb * sizeof(int32_t), hipMemcpyDeviceToHost, s_));
  MCHK(hipStreamSynchronize(s_));
  for (int32_t v : rv)
    if (v < 0) throw std::runtime_error("learned smoother: the block pattern is not structurally symmetric");
}

MpnnGraph::~MpnnGraph() {
  for (void* p : {static_cast<void*>(row_), static_cast<void*>(rev_), static_cast<void*>(scale_),
                  static_cast<void*>(feat_), static_cast<void*>(pre1_), static_cast<void*>(node_),
                  static_cast<void*>(pq_), static_cast<void*>(pre2_), static_cast<void*>(out_),
                  static_cast<void*>(go_), static_cast<void*>(d2_), static_cast<void*>(dm_), static_cast<void*>(sr_),
                  static_cast<void*>(dnode_), static_cast<void*>(part_)})
    if (p) (void)hipFree(p);
}

namespace {
// workgroups of the kernels that walk 16 blocks per wave pass
unsigned walk_blocks(int64_t nnzb) {
  return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(1024, (nnzb + 16 * (TB / 64) - 1) / (16 * (TB / 64)))));
}
unsigned node_blocks(int64_t nb) {
  constexpr int64_t per = NPW * (TB / 64);
  return static_cast<unsigned>(std::max<int64_t>(1, (nb + per - 1) / per));
}
// workgroups of the gradient products over blocks and over nodes: about 32
// steps of four per wave, at most one workgroup per CU (small systems take
// fewer, so that the partial sums stay small)
int wgrad_blocks(int64_t count) {
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(256, (count + 4 * 32 * (TB / 64) - 1) / (4 * 32 * (TB / 64)))));
}
}  // namespace

void MpnnGraph::forward(const double* d_params, double* d_m) {
  k_mg_l1<<<node_blocks(nb_), TB, 0, s_>>>(nb_, d_params, ptr_, feat_, pre1_, node_, pq_);
  k_mg_l2<<<walk_blocks(nnzb_), TB, 0, s_>>>(nnzb_, d_params, row_, idx_, pre1_, pq_, pre2_, out_);
  k_mg_out<<<blocks_for(nnzb_), TB, 0, s_>>>(nnzb_, row_, idx_, rev_, scale_, out_, d_m);
  MCHK(hipGetLastError());
}

void MpnnGraph::backward(const double* d_params, const double* d_gm, double* d_grad) {
  const int neb = wgrad_blocks(nnzb_), nnb = wgrad_blocks(nb_);
  if (!go_) {
    go_ = dnew<double>(nnzb_ * 9);
    d2_ = dnew<double>(nnzb_ * H);
    dm_ = dnew<double>(nnzb_ * H);
    sr_ = dnew<double>(nb_ * 2 * H);
    dnode_ = dnew<double>(nb_ * H);
    part_ = dnew<double>(static_cast<int64_t>(neb + nnb) * WG_OUT);
  }
  k_mg_b2<<<walk_blocks(nnzb_), TB, 0, s_>>>(nnzb_, d_params, row_, idx_, rev_, scale_, d_gm, pre2_, go_, d2_, dm_);
  k_mg_bnode<<<node_blocks(nb_), TB, 0, s_>>>(nb_, d_params, ptr_, rev_, d2_, sr_, dnode_);
  k_mg_wgrad<<<static_cast<unsigned>(neb + nnb), TB, 0, s_>>>(nnzb_, nb_, neb, row_, feat_, pre1_, node_, pre2_, go_,
                                                            d2_, dm_, dnode_, sr_, part_);
  k_mg_wsum<<<(WG_OUT + 63) / 64, TB, 0, s_>>>(neb + nnb, part_, d_grad);
  MCHK(hipGetLastError());
}

// ------------------------------------------------------------ training handle

namespace {

class TrainerImpl final : public MpnnTrainer {
 public:
  TrainerImpl(int64_t n, const int64_t* colptr, const int64_t* rowidx, const double* val) : n_(n) {
    if (n % 3 != 0) throw std::runtime_error("learned smoother: 3 DOFs per node expected");
    MCHK(hipStreamCreate(&s_));
    nb_ = n / 3;
    const Csr a = csr_from_lower(n, colptr, rowidx, val);
    // 3x3 blocks of nodes i = row / 3 (natural node-major numbering)
    std::vector<int64_t> bptr(nb_ + 1, 0);
    std::vector<int32_t> bidx;
    std::vector<double> bval;
    std::vector<int64_t> pos(nb_, -1);
    for (int64_t bi = 0; bi < nb_; ++bi) {
      std::vector<int32_t> cols;
      for (int r = 0; r < 3; ++r)
        for (int64_t p = a.ptr[3 * bi + r]; p < a.ptr[3 * bi + r + 1]; ++p) cols.push_back(a.idx[p] / 3);
      std::sort(cols.begin(), cols.end());
      cols.erase(std::unique(cols.begin(), cols.end()), cols.end());
      for (int32_t c : cols) {
        pos[c] = static_cast<int64_t>(bidx.size());
        bidx.push_back(c);
      }
      bval.resize(bidx.size() * 9, 0.0);
      for (int r = 0; r < 3; ++r)
        for (int64_t p = a.ptr[3 * bi + r]; p < a.ptr[3 * bi + r + 1]; ++p)
          bval[9 * pos[a.idx[p] / 3] + 3 * r + a.idx[p] % 3] = a.val[p];
      for (int32_t c : cols) pos[c] = -1;
      bptr[bi + 1] = static_cast<int64_t>(bidx.size());
    }
    nnzb_ = bptr[nb_];
    ptr_ = upload(bptr);
    idx_ = upload(bidx);
    val_ = upload(bval);
    hptr_ = bptr;
    hidx_ = bidx;
    graph_ = std::make_unique<MpnnGraph>(nb_, nnzb_, ptr_, idx_, val_, s_);
    prm_ = dnew<double>(MPNN_NPARAMS);
    grad_ = dnew<double>(MPNN_NPARAMS);
    m_ = dnew<double>(nnzb_ * 9);
    gm_ = dnew<double>(nnzb_ * 9);
    MCHK(hipStreamSynchronize(s_));
  }
  ~TrainerImpl() override {
    graph_.reset();
    for (void* p : {static_cast<void*>(ptr_), static_cast<void*>(idx_), static_cast<void*>(val_),
                    static_cast<void*>(prm_), static_cast<void*>(grad_), static_cast<void*>(m_),
                    static_cast<void*>(gm_), static_cast<void*>(vec_), static_cast<void*>(dot_)})
      if (p) (void)hipFree(p);
    if (s_) (void)hipStreamDestroy(s_);
  }

  int64_t nnzb() const override { return nnzb_; }

  void smoother(const double* params, double* blocks, int64_t* ptr, int32_t* idx) override {
    MCHK(hipMemcpyAsync(prm_, params, MPNN_NPARAMS * sizeof(double), hipMemcpyHostToDevice, s_));
    graph_->forward(prm_, m_);
    if (blocks) MCHK(hipMemcpyAsync(blocks, m_, nnzb_ * 9 * sizeof(double), hipMemcpyDeviceToHost, s_));
    MCHK(hipStreamSynchronize(s_));
    if (ptr) std::copy(hptr_.begin(), hptr_.end(), ptr);
    if (idx) std::copy(hidx_.begin(), hidx_.end(), idx);
  }

  double loss(const double* params, const double* e0, int nvec, int nu, double* grad) override {
    if (nvec < 1 || nu < 1) throw std::runtime_error("learned smoother loss: nvec and nu must be positive");
    const int64_t len = n_ * nvec;
    // vectors (interleaved): E_0..E_nu, Y_0..Y_{nu-1}, T, G, AE
    const int64_t need = len * (2 * static_cast<int64_t>(nu) + 4);
    if (need > cap_) {
      if (vec_) MCHK(hipFree(vec_));
      vec_ = nullptr;
      cap_ = 0;
      vec_ = dnew<double>(need);
      cap_ = need;
    }
    if (nvec > dcap_) {
      if (dot_) MCHK(hipFree(dot_));
      dot_ = nullptr;
      dcap_ = 0;
      dot_ = dnew<double>(2 * static_cast<int64_t>(nvec) * (NDB + 1));
      dcap_ = nvec;
    }
    double* E = vec_;
    double* Y = E + len * (nu + 1);
    double* T = Y + len * nu;
    double* G = T + len;
    double* AE = G + len;
    MCHK(hipMemcpyAsync(prm_, params, MPNN_NPARAMS * sizeof(double), hipMemcpyHostToDevice, s_));
    graph_->forward(prm_, m_);
    MCHK(hipMemcpyAsync(nvec > 1 ? T : E, e0, len * sizeof(double), hipMemcpyHostToDevice, s_));
    const unsigned gv = static_cast<unsigned>((nb_ * nvec * 4 + TB - 1) / TB), gl = blocks_for(len);
    if (nvec > 1) k_interleave<<<gl, TB, 0, s_>>>(n_, nvec, T, E);
    for (int k = 0; k < nu; ++k) {
      k_bsr3_mv<<<gv, TB, 0, s_>>>(nb_, nvec, ptr_, idx_, val_, E + k * len, nullptr, Y + k * len);
      k_bsr3_mv<<<gv, TB, 0, s_>>>(nb_, nvec, ptr_, idx_, m_, Y + k * len, E + k * len, E + (k + 1) * len);
    }
    k_bsr3_mv<<<gv, TB, 0, s_>>>(nb_, nvec, ptr_, idx_, val_, E + nu * len, nullptr, AE);
    double* dpart = dot_ + 2 * nvec;
    k_dots<<<dim3(NDB, 2), TB, 0, s_>>>(n_, nvec, E + nu * len, AE, E, Y, dpart);
    k_dots_sum<<<blocks_for(2 * nvec), TB, 0, s_>>>(nvec, dpart, dot_);
    MCHK(hipGetLastError());
    std::vector<double> dh(2 * nvec);
    if (grad) {
      k_gscale<<<gl, TB, 0, s_>>>(n_, nvec, AE, dot_ + nvec, G);
      for (int k = nu - 1; k >= 0; --k) {
        k_outer<<<blocks_for(nnzb_), TB, 0, s_>>>(nnzb_, nvec, k == nu - 1 ? 1 : 0, graph_->rows(), idx_, G,
                                                  Y + k * len, gm_);
        if (k > 0) {
          k_bsr3_mv<<<gv, TB, 0, s_>>>(nb_, nvec, ptr_, idx_, m_, G, nullptr, T);
          k_bsr3_mv<<<gv, TB, 0, s_>>>(nb_, nvec, ptr_, idx_, val_, T, G, G);
        }
      }
      graph_->backward(prm_, gm_, grad_);
      MCHK(hipMemcpyAsync(grad, grad_, MPNN_NPARAMS * sizeof(double), hipMemcpyDeviceToHost, s_));
    }
    MCHK(hipMemcpyAsync(dh.data(), dot_, 2 * nvec * sizeof(double), hipMemcpyDeviceToHost, s_));
    MCHK(hipStreamSynchronize(s_));
    double l = 0.0;
    for (int v = 0; v < nvec; ++v) l += dh[v] / dh[nvec + v];
    return l / nvec;
  }

 private:
  template <typename T>
  T* upload(const std::vector<T>& h) {
    T* p = dnew<T>(static_cast<int64_t>(h.size()));
    if (!h.empty()) MCHK(hipMemcpyAsync(p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, s_));
    return p;
  }

  int64_t n_ = 0, nb_ = 0, nnzb_ = 0, cap_ = 0, dcap_ = 0;
  hipStream_t s_ = nullptr;
  int64_t* ptr_ = nullptr;
  int32_t* idx_ = nullptr;
  double *val_ = nullptr, *prm_ = nullptr, *grad_ = nullptr, *m_ = nullptr, *gm_ = nullptr, *vec_ = nullptr,
         *dot_ = nullptr;
  std::vector<int64_t> hptr_;
  std::vector<int32_t> hidx_;
  std::unique_ptr<MpnnGraph> graph_;
};

}  // namespace

int64_t mpnn_nparams() { return MPNN_NPARAMS; }

std::unique_ptr<MpnnTrainer> make_mpnn_trainer(int64_t n, const int64_t* colptr, const int64_t* rowidx,
                                               const double* val) {
  return std::make_unique<TrainerImpl>(n, colptr, rowidx, val);
}

}  // namespace rf
