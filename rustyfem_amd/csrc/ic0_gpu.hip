// IC(0) on the GPU (gfx950): factorization and application of
// A ~ L D L^T with L unit lower triangular on the strictly lower pattern of A
// (src/solver/iterative/csr.rs:219-324).
//
// Both run level by level over the dependency graph of L: row i of L (and of
// the forward solve) needs the rows j < i of its pattern, so a row's level is
// one more than the highest level among them; the backward solve runs on the
// transpose U = L^T with the levels of the reversed graph.  Rows of one level
// are independent and go to one launch.
//
// Factorization (csr.rs:259-293): one wave per row.  The wave holds its row
// (columns and values) in LDS; for every entry j of the row, in increasing
// order, the lanes stride over row j of L, find each column k in the row's
// own columns by binary search, and sum L_ik d_k L_jk; L_ij = (A_ij - sum) /
// d_j.  Then d_i = A_ii (1 + shift) - sum_j L_ij^2 d_j, and a pivot that is
// not above 1e-12 |A_ii| marks the attempt failed; the host retries with the
// shift sequence of csr.rs:250-256 (1e-3, then 4x).
//
// Application (csr.rs:296-316): y = L^-1 r, then z = L^-T D^-1 y.  Rows of one
// node depend on each other but share their other columns, so they are taken
// as one group (up to three rows), which divides the levels by the node's DOF
// count.  One workgroup walks all levels with the recent values of the
// solution in LDS (k_ic0_sweep); where the levels are wide enough to feed the
// whole GPU, a dependency reaches further back than the LDS ring, or the levels
// are so many and narrow that their padded records outgrow the factor
// (ic0_plan.cpp), every level of rows is a launch (k_ic0_fwd / k_ic0_bwd, 16
// lanes per row).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <vector>

#include "ic0.hpp"
#include "ic0_plan.hpp"
#include "lane_ops.hpp"

namespace rf {

#define ICHK(expr)                                                                                   \
  do {                                                                                               \
    hipError_t e_ = (expr);                                                                          \
    if (e_ != hipSuccess) {                                                                          \
      char b_[512];                                                                                  \
      snprintf(b_, sizeof b_, "HIP error %s at %s:%d: %s", hipGetErrorString(e_), __FILE__, __LINE__, #expr); \
      throw std::runtime_error(b_);                                                                  \
    }                                                                                                \
  } while (0)

namespace {

constexpr int TB = 256;  // threads per block of the solve kernels
constexpr int G = 16;    // lanes per row in the solves

template <typename T>
struct Dev {
  T* p = nullptr;
  size_t n = 0;
  Dev() = default;
  Dev(const Dev&) = delete;
  Dev& operator=(const Dev&) = delete;
  ~Dev() {
    if (p) (void)hipFree(p);
  }
  void alloc(size_t count) {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = count;
    ICHK(hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)));
  }
  void free() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void put(const std::vector<T>& v) {
    alloc(v.size());
    if (!v.empty()) ICHK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  }
};

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// One wave per row of the level list[lb, lb + gridDim.x).
__global__ __launch_bounds__(64) void k_ic0_factor(int64_t lb, const int32_t* __restrict__ list,
                                                   const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                                   const double* __restrict__ aval, double* lval,
                                                   const double* __restrict__ diag, double* d, double shift,
                                                   int32_t* fail) {
  __shared__ int32_t ci[IC0_MAX_ROW];
  __shared__ double cv[IC0_MAX_ROW];
  const int lane = threadIdx.x;
  const int i = list[lb + blockIdx.x];
  const int64_t lo = ptr[i];
  const int len = static_cast<int>(ptr[i + 1] - lo);
  for (int q = lane; q < len; q += 64) {
    ci[q] = idx[lo + q];
    cv[q] = aval[lo + q];
  }
  __syncthreads();
  for (int p = 0; p < len; ++p) {
    const int j = ci[p];
    const int64_t jhi = ptr[j + 1];
    double s = 0.0;
    for (int64_t q = ptr[j] + lane; q < jhi; q += 64) {
      const int k = idx[q];
      // k < j for every entry of row j, so its partner in row i lies in ci[0, p)
      int a = 0, b = p;
      while (a < b) {
        const int m = (a + b) >> 1;
        if (ci[m] < k) a = m + 1;
        else b = m;
      }
      if (a < p && ci[a] == k) s += cv[a] * d[k] * lval[q];
    }
    s = wave_sum(s);
    if (lane == 0) cv[p] = (cv[p] - s) / d[j];
    __syncthreads();
  }
  double t = 0.0;
  for (int q = lane; q < len; q += 64) {
    const double v = cv[q];
    t += v * v * d[ci[q]];
    lval[lo + q] = v;
  }
  t = wave_sum(t);
  if (lane == 0) {
    const double di = diag[i] * (1.0 + shift) - t;
    d[i] = di;
    if (!(di > 1e-12 * fabs(diag[i]))) *fail = 1;
  }
}

// dst[q] = src[tmap[q]]: the factor's values in the order of U's rows
__global__ __launch_bounds__(TB) void k_gather(int64_t n, const int64_t* __restrict__ tmap,
                                               const double* __restrict__ src, double* __restrict__ dst) {
  for (int64_t q = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x; q < n; q += static_cast<int64_t>(gridDim.x) * TB)
    dst[q] = src[tmap[q]];
}

// y_i = r_i - sum_j L_ij y_j for the rows list[lb, le)
__global__ __launch_bounds__(TB) void k_ic0_fwd(int64_t lb, int64_t le, const int32_t* __restrict__ list,
                                                const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                                const double* __restrict__ val, const double* __restrict__ r, double* y,
                                                const int32_t* done) {
  if (done && *done) return;
  const int64_t t = lb + (static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x) / G;
  const int g = threadIdx.x & (G - 1);
  if (t >= le) return;  // whole groups leave together
  const int i = list[t];
  const int64_t hi = ptr[i + 1];
  double s = 0.0;
  for (int64_t p = ptr[i] + g; p < hi; p += G) s += val[p] * y[idx[p]];
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (g == 0) y[i] = r[i] - s;
}

// z_j = y_j / d_j - sum_i U_ji z_i for the rows list[lb, le) of U = L^T
__global__ __launch_bounds__(TB) void k_ic0_bwd(int64_t lb, int64_t le, const int32_t* __restrict__ list,
                                                const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                                const double* __restrict__ val, const double* __restrict__ y,
                                                const double* __restrict__ d, double* z, const int32_t* done) {
  if (done && *done) return;
  const int64_t t = lb + (static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x) / G;
  const int g = threadIdx.x & (G - 1);
  if (t >= le) return;
  const int j = list[t];
  const int64_t hi = ptr[j + 1];
  double s = 0.0;
  for (int64_t p = ptr[j] + g; p < hi; p += G) s += val[p] * z[idx[p]];
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (g == 0) z[j] = y[j] / d[j] - s;
}

// y_i /= d_i
__global__ __launch_bounds__(TB) void k_ic0_div(int64_t n, const double* __restrict__ d, double* __restrict__ y,
                                                const int32_t* done) {
  if (done && *done) return;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (i < n) y[i] /= d[i];
}

// ------------------------------------------------------- one-workgroup sweep

typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef int32_t v2i __attribute__((ext_vector_type(2)));
typedef double d2 __attribute__((ext_vector_type(2)));

// Substitution with one strictly triangular factor by one workgroup: forward
// (DIR = 1) out = L^-1 rin, backward (DIR = -1) out = U^-1 rin.
//
// A level is one or more rounds of SWS groups, SWG lanes each; the lanes take
// the group's columns SWG apart, read the earlier solution values from the LDS
// ring, sum across the lanes by DPP, and lane r finishes row r.  Between levels
// the waves meet at a barrier that waits for LDS alone, so the records of the
// next SWD rounds stay in flight: a level costs an LDS round trip instead of a
// launch.  The host checks that no dependency is older than the ring.
//
// Bound by the instructions and memory accesses that one compute unit issues:
// hence records that need no address, index or bounds arithmetic (columns are
// ring offsets, what a record does not fill points at the ring's 0), 16-byte
// loads of consecutive lanes only, and the group's triangle inverted once.
// 20^3 block (26,460 rows, 420 row levels, 140 of groups), per sweep: one
// launch per row level 1,430 us; columns and values row by row in the
// factor's order 294-355 us (more loads, selects and address arithmetic); this
// 209 us (1.0 us per round of 88 KB, 93 GB/s: the rate of one unit's L1).
template <int R, int NC, int DIR>
__global__ __launch_bounds__(SWT) void k_ic0_sweep(int rounds, const uint32_t* __restrict__ word0,
                                                   const v4i* __restrict__ rec, const int32_t* __restrict__ tptr,
                                                   const int32_t* __restrict__ tcol, const double* __restrict__ tval,
                                                   const double* __restrict__ rin, double* __restrict__ out,
                                                   const int32_t* done) {
  if (done && *done) return;
  using Rec = SweepRecord<R, NC>;
  constexpr int RB = SWS * R * 8;                 // ring bytes of a round
  constexpr int RW = ring_rounds(R) * RB;         // of the ring
  __shared__ double ring[RING + 1];
  char* rb = reinterpret_cast<char*>(ring);
  const int lane = threadIdx.x & (SWG - 1), slot = threadIdx.x / SWG;
  if (threadIdx.x == 0) ring[ring_rounds(R) * SWS * R] = 0.0;
  lds_barrier();
  struct Stage {
    // exactly what is used: a register that a load fills and nothing reads is
    // reused at once, and its next writer then waits for the load
    int32_t w[Rec::NI];
    double d[Rec::ND];
    uint32_t word;
    double rv;
  };
  // round t's record for this thread
  const char* mine = reinterpret_cast<const char*>(rec + (threadIdx.x >> 6) * (Rec::GRANULES * 64) + (threadIdx.x & 63));
  auto fetch = [&](Stage& s, int t) {
    const char* p = mine + static_cast<int64_t>(t) * ((SWT / 64) * Rec::GRANULES * 64 * 16);
#pragma unroll
    for (int w = 0; w + 4 <= Rec::NI; w += 4) {
      const v4i g = *reinterpret_cast<const v4i*>(p + 256 * w);
#pragma unroll
      for (int e = 0; e < 4; ++e) s.w[w + e] = g[e];
    }
    constexpr int W0 = Rec::NI / 4 * 4;
    if constexpr (Rec::NI % 4 == 2) {
      const v2i g = *reinterpret_cast<const v2i*>(p + 256 * W0);
      s.w[W0] = g[0];
      s.w[W0 + 1] = g[1];
    } else if constexpr (Rec::NI % 4 == 3) {
      const v2i g = *reinterpret_cast<const v2i*>(p + 256 * W0);
      s.w[W0] = g[0];
      s.w[W0 + 1] = g[1];
      s.w[W0 + 2] = *reinterpret_cast<const int32_t*>(p + 256 * W0 + 8);
    }
    static_assert(Rec::NI % 4 != 1, "2, 3 or 5 columns and a word");
    const char* pd = p + Rec::GI * 1024;
#pragma unroll
    for (int q = 0; q + 2 <= Rec::ND; q += 2) {
      const d2 g = *reinterpret_cast<const d2*>(pd + 512 * q);
      s.d[q] = g[0];
      s.d[q + 1] = g[1];
    }
    if constexpr (Rec::ND % 2 == 1) s.d[Rec::ND - 1] = *reinterpret_cast<const double*>(pd + 512 * (Rec::ND - 1));
    // lanes past the group's rows read its first row (an empty slot: row 0)
    const int row = static_cast<int>(s.word >> 4), cnt = (s.word >> 2) & 3;
    s.rv = rin[row + (lane < cnt ? DIR * lane : 0)];
  };
  int base = 0;  // ring offset of the round
  auto step = [&](Stage& s, int t) {
    double a[R];
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = lane == r ? -s.rv : 0.0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const double y = *reinterpret_cast<const double*>(rb + s.w[c]);
#pragma unroll
      for (int r = 0; r < R; ++r) a[r] = fma(s.d[c * R + r], y, a[r]);
    }
    if (s.word & SW_TAIL) {
      const int32_t* tp = tptr + t * SWS + slot;
      for (int q = tp[0] + lane; q < tp[1]; q += SWG) {
        const double y = *reinterpret_cast<const double*>(rb + tcol[q]);
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = fma(tval[static_cast<int64_t>(q) * R + r], y, a[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = half_row_sum(a[r]);
    // a = -t; x_r = t_r + sum_{q < r} coef_q t_q (not with zeros for the other
    // q: a row must not receive what is not finite in a later one)
    double x = a[0];
#pragma unroll
    for (int r = 1; r < R; ++r) {
      double t = a[r];
#pragma unroll
      for (int q = 0; q < r; ++q) t = fma(s.d[NC * R + q], a[q], t);
      if (lane == r) x = t;
    }
    x = -x;
    const int cnt = (s.word >> 2) & 3;
    if (lane < cnt) {
      *reinterpret_cast<double*>(rb + base + slot * (R * 8) + lane * 8) = x;
      out[static_cast<int>(s.word >> 4) + DIR * lane] = x;
    }
    if (__builtin_amdgcn_readfirstlane(s.word) & SW_LAST) lds_barrier();
    base = base + RB == RW ? 0 : base + RB;
    s.word = static_cast<uint32_t>(s.w[NC]);
    __builtin_amdgcn_sched_barrier(0);
    fetch(s, t + SWD);
    __builtin_amdgcn_sched_barrier(0);
  };
  Stage s[SWD];
#pragma unroll
  for (int q = 0; q < SWD; ++q) s[q].word = word0[q * SWS + slot];
  // in this order, as in the loop: the waits inside the loop are set for the
  // fewest loads that any path to it leaves behind
#pragma unroll
  for (int q = 0; q < SWD; ++q) {
    __builtin_amdgcn_sched_barrier(0);
    fetch(s[q], q);
  }
  __builtin_amdgcn_sched_barrier(0);
  // rounds is a multiple of SWD, followed by SWD empty ones
  for (int t = 0; t < rounds; t += SWD) {
#pragma unroll
    for (int q = 0; q < SWD; ++q) step(s[q], t + q);
  }
}

// The records (and tails) of a sweep from its schedule: lane by lane of every
// slot, the ring places of its columns and the factor's values.  map: the place
// of entry p of (ptr, idx) in lval (null: p).  The host only lays out the
// schedule, in two threads beside the factorization: setup of the 20^3 block
// 92 ms with the records built entry by entry on the host, 67 ms so (66 without
// sweeps); plate of 500 x 200 quadrilaterals 160, 96 and 95 ms.
template <int R, int NC, int DIR>
__global__ __launch_bounds__(TB) void k_ic0_records(int64_t slots, const uint32_t* __restrict__ words,
                                                    const int32_t* __restrict__ ring, const int32_t* __restrict__ tptr,
                                                    const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                                    const int64_t* __restrict__ map, const double* __restrict__ lval,
                                                    v4i* __restrict__ rec, int32_t* __restrict__ tcol,
                                                    double* __restrict__ tval) {
  using Rec = SweepRecord<R, NC>;
  const int64_t th = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  const int64_t q = th / SWG;
  const int lane = static_cast<int>(th % SWG);
  if (q >= slots) return;
  const uint32_t word = words[q];
  const int64_t f = slot_row(word);
  const int cnt = slot_rows(word);
  const int64_t p0 = ptr[f], k = cnt ? ptr[f + 1] - p0 : 0;
  auto value = [&](int64_t p) { return lval[map ? map[p] : p]; };
  int64_t rowp[R];  // row r's entries of the shared columns
#pragma unroll
  for (int r = 0; r < R; ++r) rowp[r] = ptr[r < cnt ? f + DIR * r : f] + (DIR > 0 ? 0 : r);
  int32_t w[4 * Rec::GI] = {};
  double d[2 * Rec::GD] = {};
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int64_t j = c * SWG + lane;
    w[c] = j < k ? ring[idx[p0 + j]] : ring_rounds(R) * SWS * R * 8;
#pragma unroll
    for (int r = 0; r < R; ++r) d[c * R + r] = (j < k && r < cnt) ? value(rowp[r] + j) : 0.0;
  }
  w[NC] = static_cast<int32_t>(words[q + SWD * SWS]);
  // the coefficients of the group's rows: x_1 = t_1 - l_10 t_0,
  // x_2 = t_2 + (l_21 l_10 - l_20) t_0 - l_21 t_1
  if constexpr (R > 1) {
    // row r's entry in the group's row m (m < r)
    auto own = [&](int r, int m) { return value(ptr[f + DIR * r] + (DIR > 0 ? k + m : r - 1 - m)); };
    if (lane == 1 && cnt > 1) d[NC * R] = -own(1, 0);
    if constexpr (R > 2) {
      if (lane == 2 && cnt > 2) {
        const double l21 = own(2, 1);
        d[NC * R] = l21 * own(1, 0) - own(2, 0);
        d[NC * R + 1] = -l21;
      }
    }
  }
  const int64_t in = th % SWT;
  v4i* o = rec + ((q / SWS) * (SWT / 64) + in / 64) * (Rec::GRANULES * 64) + in % 64;
#pragma unroll
  for (int g = 0; g < Rec::GI; ++g) o[64 * g] = v4i{w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]};
#pragma unroll
  for (int g = 0; g < Rec::GD; ++g)
    o[64 * (Rec::GI + g)] = __builtin_bit_cast(v4i, d2{d[2 * g], d[2 * g + 1]});
  if (word & SW_TAIL) {
    const int64_t t0 = static_cast<int64_t>(tptr[q]) - SWG * NC;
    for (int64_t j = SWG * NC + lane; j < k; j += SWG) {
      tcol[t0 + j] = ring[idx[p0 + j]];
#pragma unroll
      for (int r = 0; r < R; ++r) tval[(t0 + j) * R + r] = r < cnt ? value(rowp[r] + j) : 0.0;
    }
  }
}

// f(R, NC) for a plan's constants
template <typename F>
void with_constants(int R, int NC, F f) {
  auto nc = [&](auto r) {
    if (NC == 2) f(r, std::integral_constant<int, 2>());
    else if (NC == 3) f(r, std::integral_constant<int, 3>());
    else f(r, std::integral_constant<int, 5>());
  };
  if (R == 1) nc(std::integral_constant<int, 1>());
  else if (R == 2) nc(std::integral_constant<int, 2>());
  else nc(std::integral_constant<int, 3>());
}

class Ic0Impl final : public Ic0Gpu {
 public:
  Ic0Impl(const Csr& a, hipStream_t s);
  void apply(const double* r, double* z, const int32_t* done) override;
  double shift() const override { return shift_; }
  int64_t forward_levels() const override { return static_cast<int64_t>(foff_.size()) - 1; }
  int64_t backward_levels() const override { return static_cast<int64_t>(boff_.size()) - 1; }
  double factor_ms() const override { return factor_ms_; }
  int attempts() const override { return attempts_; }
  bool sweeps() const override { return bw_.R > 0; }
  int64_t sweep_levels(int dir) const override { return dir > 0 ? fw_.levels : bw_.levels; }
  int64_t sweep_bytes() const override { return fw_.bytes + bw_.bytes; }

 private:
  struct Sweep {
    int R = 0, NC = 0, rounds = 0;
    int64_t levels = 0, bytes = 0;
    Dev<uint32_t> words;
    Dev<int32_t> tptr, tcol;
    Dev<v4i> rec;
    Dev<double> tval;
  };
  template <int DIR>
  void make_sweep(Sweep& w, const SweepPlan& S, const int64_t* ptr, const int32_t* idx, const int64_t* map);
  template <int DIR>
  void launch_sweep(const Sweep& w, const double* rin, double* out, const int32_t* done);

  int64_t n_ = 0;
  hipStream_t s_;
  Sweep fw_, bw_;
  std::vector<int64_t> foff_, boff_;
  Dev<int64_t> lptr_, uptr_, tmap_;
  Dev<int32_t> lidx_, uidx_, flist_, blist_, fail_;
  Dev<double> aval_, lval_, uval_, diag_, d_, y_;
  double shift_ = 0.0, factor_ms_ = 0.0;
  int attempts_ = 0;
};

Ic0Impl::Ic0Impl(const Csr& a, hipStream_t s) : n_(a.nrows), s_(s) {
  const auto t0 = std::chrono::steady_clock::now();
  const int64_t n = n_;
  if (a.ncols != n) throw std::runtime_error("IC(0): square matrix required");
  if (n >= (int64_t(1) << 31)) throw std::runtime_error("IC(0): too many rows");
  // strictly lower L row-wise and the diagonal (csr.rs:231-247)
  std::vector<int64_t> lptr(n + 1, 0);
  std::vector<int32_t> lidx;
  std::vector<double> aval, diag(n, 0.0);
  lidx.reserve(static_cast<size_t>(a.nnz() / 2 + 1));
  aval.reserve(static_cast<size_t>(a.nnz() / 2 + 1));
  for (int64_t i = 0; i < n; ++i) {
    int32_t prev = -1;
    for (int64_t p = a.ptr[i]; p < a.ptr[i + 1]; ++p) {
      const int32_t j = a.idx[p];
      if (j < i) {
        if (j <= prev) throw std::runtime_error("IC(0): rows must be sorted without duplicates");
        prev = j;
        lidx.push_back(j);
        aval.push_back(a.val[p]);
      } else if (j == i) {
        diag[i] += a.val[p];
      }
    }
    lptr[i + 1] = static_cast<int64_t>(lidx.size());
    if (lptr[i + 1] - lptr[i] > IC0_MAX_ROW)
      throw std::runtime_error("IC(0): a row of L holds more than " + std::to_string(IC0_MAX_ROW) + " entries");
  }
  const int64_t nnz = lptr[n];
  // the rows' levels, U = L^T row-wise and the map into L's values; the
  // one-workgroup sweeps where they pay are planned beside the factorization
  const char* env = std::getenv("RUSTYFEM_IC0_LEVELS");
  const bool plan = n && !(env && *env && *env != '0');
  std::vector<int32_t> flist, blist, uidx;
  std::vector<int64_t> uptr, tmap;
  std::future<SweepPlan> fplan, bplan;  // (after what they read: destroyed before it)
  int32_t count = 0;
  std::vector<int32_t> lev = row_levels(n, lptr, lidx, 1, count);
  if (plan) fplan = std::async([&, count] { return plan_sweep(n, lptr, lidx, count, 1); });
  by_level(lev, count, flist, foff_);
  transpose_pattern(n, lptr, lidx, uptr, uidx, tmap);
  lev = row_levels(n, uptr, uidx, -1, count);
  if (plan) bplan = std::async([&, count] { return plan_sweep(n, uptr, uidx, count, -1); });
  by_level(lev, count, blist, boff_);

  lptr_.put(lptr);
  lidx_.put(lidx);
  aval_.put(aval);
  diag_.put(diag);
  flist_.put(flist);
  lval_.alloc(nnz);
  d_.alloc(n);
  y_.alloc(n);
  fail_.alloc(1);

  // factor, with the diagonal shift of csr.rs:250-256 on breakdown
  double shift = 0.0;
  for (;;) {
    ++attempts_;
    ICHK(hipMemsetAsync(fail_.p, 0, sizeof(int32_t), s_));
    for (size_t l = 0; l + 1 < foff_.size(); ++l) {
      const int64_t rows = foff_[l + 1] - foff_[l];
      k_ic0_factor<<<static_cast<unsigned>(rows), 64, 0, s_>>>(foff_[l], flist_.p, lptr_.p, lidx_.p, aval_.p, lval_.p,
                                                              diag_.p, d_.p, shift, fail_.p);
    }
    ICHK(hipGetLastError());
    int32_t fail = 0;
    ICHK(hipMemcpyAsync(&fail, fail_.p, sizeof fail, hipMemcpyDeviceToHost, s_));
    ICHK(hipStreamSynchronize(s_));
    if (!fail) break;
    if (attempts_ >= 40) throw std::runtime_error("IC(0): no positive factorization up to shift " + std::to_string(shift));
    shift = shift == 0.0 ? 1e-3 : shift * 4.0;
  }
  shift_ = shift;
  uptr_.put(uptr);
  uidx_.put(uidx);
  tmap_.put(tmap);
  SweepPlan fw, bw;
  if (plan) {
    fw = fplan.get();
    bw = bplan.get();
  }
  if (fw.R && bw.R) {
    make_sweep<1>(fw_, fw, lptr_.p, lidx_.p, nullptr);
    make_sweep<-1>(bw_, bw, uptr_.p, uidx_.p, tmap_.p);
    // only the launches per level read these
    uptr_.free();
    uidx_.free();
    tmap_.free();
  } else {
    blist_.put(blist);
    uval_.alloc(nnz);
    if (nnz) {
      const unsigned g = static_cast<unsigned>(std::min<int64_t>(1024, (nnz + TB - 1) / TB));
      k_gather<<<g, TB, 0, s_>>>(nnz, tmap_.p, lval_.p, uval_.p);
      ICHK(hipGetLastError());
    }
  }
  ICHK(hipStreamSynchronize(s_));
  factor_ms_ = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

template <int DIR>
void Ic0Impl::make_sweep(Sweep& w, const SweepPlan& S, const int64_t* ptr, const int32_t* idx, const int64_t* map) {
  const int64_t slots = (S.rounds + SWD) * SWS;
  Dev<int32_t> ring;
  ring.put(S.ring);
  w.words.put(S.words);
  w.tptr.put(S.tptr);
  w.tcol.alloc(S.tptr.back());
  w.tval.alloc(static_cast<size_t>(S.tptr.back()) * S.R);
  w.rec.alloc(static_cast<size_t>(slots * SWG * record_granules(S.R, S.NC)));
  with_constants(S.R, S.NC, [&](auto r, auto nc) {
    k_ic0_records<r(), nc(), DIR><<<static_cast<unsigned>((slots * SWG + TB - 1) / TB), TB, 0, s_>>>(
        slots, w.words.p, ring.p, w.tptr.p, ptr, idx, map, lval_.p, w.rec.p, w.tcol.p, w.tval.p);
  });
  ICHK(hipGetLastError());
  ICHK(hipStreamSynchronize(s_));  // the ring places live until here
  w.rounds = static_cast<int>(S.rounds);
  w.R = S.R;
  w.NC = S.NC;
  w.levels = S.levels;
  w.bytes = S.bytes;
}

template <int DIR>
void Ic0Impl::launch_sweep(const Sweep& w, const double* rin, double* out, const int32_t* done) {
  with_constants(w.R, w.NC, [&](auto r, auto nc) {
    k_ic0_sweep<r(), nc(), DIR><<<1, SWT, 0, s_>>>(w.rounds, w.words.p, w.rec.p, w.tptr.p, w.tcol.p, w.tval.p, rin, out,
                                                   done);
  });
}

void Ic0Impl::apply(const double* r, double* z, const int32_t* done) {
  if (sweeps()) {
    launch_sweep<1>(fw_, r, y_.p, done);
    k_ic0_div<<<static_cast<unsigned>((n_ + TB - 1) / TB), TB, 0, s_>>>(n_, d_.p, y_.p, done);
    launch_sweep<-1>(bw_, y_.p, z, done);
    ICHK(hipGetLastError());
    return;
  }
  for (size_t l = 0; l + 1 < foff_.size(); ++l) {
    const int64_t rows = foff_[l + 1] - foff_[l];
    const unsigned g = static_cast<unsigned>((rows * G + TB - 1) / TB);
    k_ic0_fwd<<<g, TB, 0, s_>>>(foff_[l], foff_[l + 1], flist_.p, lptr_.p, lidx_.p, lval_.p, r, y_.p, done);
  }
  for (size_t l = 0; l + 1 < boff_.size(); ++l) {
    const int64_t rows = boff_[l + 1] - boff_[l];
    const unsigned g = static_cast<unsigned>((rows * G + TB - 1) / TB);
    k_ic0_bwd<<<g, TB, 0, s_>>>(boff_[l], boff_[l + 1], blist_.p, uptr_.p, uidx_.p, uval_.p, y_.p, d_.p, z, done);
  }
  ICHK(hipGetLastError());
}

}  // namespace

std::unique_ptr<Ic0Gpu> make_ic0_gpu(const Csr& a, hipStream_t s) { return std::make_unique<Ic0Impl>(a, s); }

}  // namespace rf
