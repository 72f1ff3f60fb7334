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
// whole GPU, or a dependency reaches further back than the LDS ring, every
// level of rows is a launch (k_ic0_fwd / k_ic0_bwd, 16 lanes per row).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include <string>
#include <vector>

#include "ic0.hpp"
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

// dst[q] = src[tmap[q]] (0 where the map is negative): the factor's values in
// the order of U's rows, or of a sweep's stream
__global__ __launch_bounds__(TB) void k_gather(int64_t n, const int64_t* __restrict__ tmap,
                                               const double* __restrict__ src, double* __restrict__ dst) {
  for (int64_t q = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x; q < n; q += static_cast<int64_t>(gridDim.x) * TB) {
    const int64_t t = tmap[q];
    dst[q] = t >= 0 ? src[t] : 0.0;
  }
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

constexpr int SWT = 512;           // threads of the sweep's workgroup
constexpr int SWG = 8;             // lanes per group
constexpr int SWS = SWT / SWG;     // groups per round
constexpr int SWD = 3;             // rounds whose records are in flight
constexpr int RING = 20000;        // solution values kept in LDS (160 KB with the entry that stays 0)
// rounds of R values per slot that the ring holds
constexpr int ring_rounds(int R) { return RING / (SWS * R); }

// A round's slot holds one group of up to R rows: a word per slot with the
// group's first row (its others follow in the sweep's direction), the number
// of its rows, and two flags.
constexpr uint32_t SW_LAST = 1;    // the last round of its level (in every slot of the round)
constexpr uint32_t SW_TAIL = 2;    // columns beyond the record
__host__ __device__ constexpr uint32_t slot_word(int64_t row, int cnt, uint32_t flags) {
  return static_cast<uint32_t>(row) << 4 | static_cast<uint32_t>(cnt) << 2 | flags;
}

// A thread's record of one round: NC columns (LDS byte offsets of their values
// in the ring), the slot's word SWD rounds later, the columns' R factor
// values each, and, for row r < R of the group in lane r, the coefficients of
// t_0 .. t_{R-2} in x_r (the inverse of the group's unit triangle).  Stored in
// 16-byte granules interleaved over the wave's lanes.
template <int R, int NC>
struct SweepRecord {
  static constexpr int NI = NC + 1, ND = NC * R + R - 1;
  static constexpr int GI = (NI + 3) / 4, GD = (ND + 1) / 2;  // granules of words, of doubles
  static constexpr int GRANULES = GI + GD;
};

// sum over 8 consecutive lanes, in every lane: quad_perm [1,0,3,2], quad_perm
// [2,3,0,1], row_half_mirror
__device__ __forceinline__ double half_row_sum(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x141>(v);
  return v;
}

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
// 194 us (0.9 us per round of 88 KB, 98 GB/s: the rate of one unit's L1).
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
    // a = -t; x_r = t_r + sum_q coef_q t_q
    double x = a[0];
#pragma unroll
    for (int r = 1; r < R; ++r)
      if (lane == r) x = a[r];
#pragma unroll
    for (int q = 0; q + 1 < R; ++q) x = fma(s.d[NC * R + q], a[q], x);
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

// the factor values of the records: double q of the stream is lval[map[q]], 0
// where the map is negative (map given for the doubles in stream order)
__global__ __launch_bounds__(TB) void k_ic0_records(int64_t n, const int32_t* __restrict__ map,
                                                    const int64_t* __restrict__ place,
                                                    const double* __restrict__ lval, double* __restrict__ rec) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (q < n) rec[place[q]] = lval[map[q]];
}

// coefficients of a group's rows: x_1 = t_1 - l_10 t_0, x_2 = t_2 + (l_21 l_10
// - l_20) t_0 - l_21 t_1; `at` holds their places in the stream
struct SweepCoef { int32_t l10, l20, l21, pad; int64_t at[3]; };
__global__ __launch_bounds__(TB) void k_ic0_coefs(int64_t n, const SweepCoef* __restrict__ c,
                                                  const double* __restrict__ lval, double* __restrict__ rec) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * TB + threadIdx.x;
  if (q >= n) return;
  const SweepCoef s = c[q];
  const double l10 = lval[s.l10];
  rec[s.at[0]] = -l10;
  if (s.l20 >= 0) {
    const double l20 = lval[s.l20], l21 = lval[s.l21];
    rec[s.at[1]] = l21 * l10 - l20;
    rec[s.at[2]] = -l21;
  }
}

// rows grouped by level: list (rows in increasing order within a level) and
// the level offsets
void by_level(const std::vector<int32_t>& lev, int32_t nlev, std::vector<int32_t>& list, std::vector<int64_t>& off) {
  off.assign(static_cast<size_t>(nlev) + 1, 0);
  for (int32_t l : lev) ++off[l + 1];
  for (int32_t l = 0; l < nlev; ++l) off[l + 1] += off[l];
  list.resize(lev.size());
  std::vector<int64_t> pos(off.begin(), off.end() - 1);
  for (size_t i = 0; i < lev.size(); ++i) list[pos[lev[i]]++] = static_cast<int32_t>(i);
}

// The schedule and stream of one sweep over the strictly triangular rows
// (ptr, idx: columns sorted; forward: columns below the row, dir = 1;
// backward: above it, dir = -1).  src[p] is the factor value of entry p.
struct SweepPlan {
  int R = 0;                    // rows per group (1, 2 or 3); 0: not possible
  int NC = 0;                   // columns per lane in a record (2, 3 or 5)
  int64_t levels = 0, rounds = 0;
  std::vector<uint32_t> word0;  // the slots' words of the first SWD rounds
  std::vector<int32_t> rec;     // the records' words (the doubles' places 0)
  std::vector<int32_t> vmap;    // factor values and their places among the records' doubles
  std::vector<int64_t> place;
  std::vector<SweepCoef> coef;
  std::vector<int32_t> tptr, tcol, tmap;  // the tails: slots' offsets, ring offsets, R factor values (-1: 0) each
};

template <int R, int NC>
void fill_records(SweepPlan& S, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx,
                  const std::vector<int64_t>* src, int dir, const std::vector<int32_t>& first,
                  const std::vector<int32_t>& cnt, const std::vector<int32_t>& slot_group,
                  const std::vector<int32_t>& slot_of, const std::vector<int32_t>& group_of,
                  const std::vector<uint32_t>& words) {
  using Rec = SweepRecord<R, NC>;
  auto entry = [&](int64_t p) { return static_cast<int32_t>(src ? (*src)[p] : p); };
  const int64_t waves = S.rounds + SWD, per = static_cast<int64_t>(SWT / 64) * Rec::GRANULES * 64 * 4;
  S.rec.assign(static_cast<size_t>(waves * per), 0);
  // word w of the lane of (round, slot): granule w / 4
  auto word_at = [&](int64_t q, int lane, int w) {
    const int64_t t = q / SWS, th = (q % SWS) * SWG + lane;
    return ((t * (SWT / 64) + th / 64) * Rec::GRANULES + w / 4) * 256 + (th % 64) * 4 + w % 4;
  };
  auto double_at = [&](int64_t q, int lane, int d) { return word_at(q, lane, 4 * Rec::GI + 2 * d) / 2; };
  constexpr int32_t zero = ring_rounds(R) * SWS * R * 8;
  S.tptr.assign(static_cast<size_t>(waves * SWS) + 1, 0);
  S.vmap.reserve(idx.size());
  S.place.reserve(idx.size());
  for (int64_t q = 0; q < waves * SWS; ++q) {
    S.tptr[q] = static_cast<int32_t>(S.tcol.size());
    const int64_t next = q + static_cast<int64_t>(SWD) * SWS;
    const uint32_t nw = next < static_cast<int64_t>(words.size()) ? words[next] : 0;
    for (int lane = 0; lane < SWG; ++lane) {
      for (int c = 0; c < NC; ++c) S.rec[word_at(q, lane, c)] = zero;
      S.rec[word_at(q, lane, NC)] = static_cast<int32_t>(nw);
    }
    const int32_t g = q < static_cast<int64_t>(slot_group.size()) ? slot_group[q] : -1;
    if (g < 0) continue;
    const int64_t f = first[g];
    const int c = cnt[g];
    const int64_t k = ptr[f + 1] - ptr[f];
    int64_t rowp[R];  // row r's entries of the shared columns
    for (int r = 0; r < R; ++r) rowp[r] = ptr[f + dir * std::min(r, c - 1)] + (dir > 0 ? 0 : std::min(r, c - 1));
    for (int64_t j = 0; j < k; ++j) {
      const int32_t col = idx[ptr[f] + j], cg = group_of[col];
      const int64_t cq = slot_of[cg];
      const int32_t at = static_cast<int32_t>(
          ((cq / SWS % ring_rounds(R)) * SWS * R + (cq % SWS) * R + dir * (col - first[cg])) * 8);
      if (j < SWG * NC) {
        const int lane = static_cast<int>(j % SWG), cc = static_cast<int>(j / SWG);
        S.rec[word_at(q, lane, cc)] = at;
        for (int r = 0; r < c; ++r) {
          S.vmap.push_back(entry(rowp[r] + j));
          S.place.push_back(double_at(q, lane, cc * R + r));
        }
      } else {
        S.tcol.push_back(at);
        for (int r = 0; r < R; ++r) S.tmap.push_back(r < c ? entry(rowp[r] + j) : -1);
      }
    }
    if (c > 1) {
      // row r's entry in the group's row m (m < r)
      auto own = [&](int r, int m) {
        const int64_t row = f + dir * r;
        return entry(dir > 0 ? ptr[row] + k + m : ptr[row] + (r - 1 - m));
      };
      SweepCoef co{own(1, 0), -1, -1, 0, {double_at(q, 1, NC * R), 0, 0}};
      if (c > 2) {
        co.l20 = own(2, 0);
        co.l21 = own(2, 1);
        co.at[1] = double_at(q, 2, NC * R);
        co.at[2] = double_at(q, 2, NC * R + 1);
      }
      S.coef.push_back(co);
    }
  }
  S.tptr.back() = static_cast<int32_t>(S.tcol.size());
}

// One workgroup's sweep against a launch per row level, measured per
// application on C3D8 blocks (both sweeps, row levels in brackets):
//   8^3 (168) 138 against 896 us, 16^3 (336) 319 / 2,205, 24^3 (504) 702 / 4,386,
//   32^3 (672) 1,383 / 5,258, 40^3 (840) 2,551 / 7,099, 56^3 (1,176) 10,932 / 11,095.
// That is about 0.2 us per level and 0.9 us per round of 64 groups, 1.7 us per
// round where the records exceed the Infinity Cache and come from HBM,
// against 3.4 us per launch (more where a level has thousands of rows).
bool sweep_pays(int64_t levels, int64_t rounds, int R, int NC) {
  const double bytes = static_cast<double>(rounds) * SWT * 8 * (NC * R + R + (NC + 1) / 2 + 1);
  return 0.2 * static_cast<double>(levels) + (bytes < 128e6 ? 0.9 : 1.7) * static_cast<double>(rounds) <
         3.4 * R * static_cast<double>(levels);
}

SweepPlan plan_sweep(int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx,
                     const std::vector<int64_t>* src, int dir) {
  SweepPlan S;
  if (n >= (int64_t(1) << 28) || idx.size() >= (size_t(1) << 30)) return S;
  // groups: consecutive rows (in elimination order) whose columns are the
  // first row's columns and the rows of the group before them
  std::vector<int32_t> first, cnt;  // first row and rows of every group, in elimination order
  auto build = [&](int R) {
    first.clear();
    cnt.clear();
    for (int64_t e = 0; e < n; ++e) {
      const int64_t row = dir > 0 ? e : n - 1 - e;
      bool join = false;
      if (!first.empty() && cnt.back() < R) {
        const int64_t f = first.back();
        const int c = cnt.back();
        const int64_t k = ptr[f + 1] - ptr[f];
        if (ptr[row + 1] - ptr[row] == k + c) {
          // the group's rows come last (forward) or first (backward)
          const int32_t* own = idx.data() + ptr[row] + (dir > 0 ? k : 0);
          const int32_t* ext = idx.data() + ptr[row] + (dir > 0 ? 0 : c);
          const int32_t lo = static_cast<int32_t>(dir > 0 ? f : row + 1);
          join = std::equal(ext, ext + k, idx.data() + ptr[f]);
          for (int q = 0; join && q < c; ++q) join = own[q] == lo + q;
        }
      }
      if (join) {
        ++cnt.back();
      } else {
        first.push_back(static_cast<int32_t>(row));
        cnt.push_back(1);
      }
    }
  };
  // the largest group size that wastes at most a quarter of its rows
  int R = 3;
  for (; R > 1; --R) {
    build(R);
    if (static_cast<double>(n) >= 0.75 * R * static_cast<double>(first.size())) break;
  }
  if (R == 1) build(1);
  const int64_t ng = static_cast<int64_t>(first.size());
  std::vector<int32_t> group_of(n), lev(ng, 0);
  for (int64_t g = 0; g < ng; ++g)
    for (int c = 0; c < cnt[g]; ++c) group_of[first[g] + dir * c] = static_cast<int32_t>(g);
  int32_t nlev = ng ? 1 : 0;
  for (int64_t g = 0; g < ng; ++g) {
    int32_t l = 0;
    for (int64_t p = ptr[first[g]]; p < ptr[first[g] + 1]; ++p) l = std::max(l, lev[group_of[idx[p]]] + 1);
    lev[g] = l;
    nlev = std::max(nlev, l + 1);
  }
  std::vector<int32_t> list;
  std::vector<int64_t> off;
  by_level(lev, nlev, list, off);
  // columns per lane for nearly every group (19 of 20), at most 5
  int64_t over[2] = {0, 0};
  for (int64_t g = 0; g < ng; ++g)
    for (int q = 0; q < 2; ++q) over[q] += ptr[first[g] + 1] - ptr[first[g]] > SWG * (2 + q);
  const int NC = 20 * over[0] <= ng ? 2 : 20 * over[1] <= ng ? 3 : 5;
  // a level's groups in order over the slots of its rounds
  std::vector<int32_t> slot_group, slot_of(ng);
  std::vector<uint32_t> words;
  for (int32_t l = 0; l < nlev; ++l) {
    int64_t oldest = INT64_MAX;  // round of the oldest value the level reads
    for (int64_t q = off[l]; q < off[l + 1]; ++q) {
      const int32_t g = list[q];
      slot_of[g] = static_cast<int32_t>(slot_group.size());
      slot_group.push_back(g);
      const int64_t f = first[g], k = ptr[f + 1] - ptr[f];
      words.push_back(slot_word(f, cnt[g], k > SWG * NC ? SW_TAIL : 0));
      for (int64_t p = ptr[f]; p < ptr[f + 1]; ++p) oldest = std::min<int64_t>(oldest, slot_of[group_of[idx[p]]] / SWS);
    }
    while (slot_group.size() % SWS) {
      slot_group.push_back(-1);
      words.push_back(0);
    }
    // the level's own values must not reach the ring place of one it reads
    const int64_t end = static_cast<int64_t>(slot_group.size()) / SWS;
    if (oldest != INT64_MAX && end - 1 - oldest > ring_rounds(R) - 1) return S;
    for (size_t q = slot_group.size() - SWS; q < slot_group.size(); ++q) words[q] |= SW_LAST;
  }
  S.rounds = (static_cast<int64_t>(slot_group.size()) / SWS + SWD - 1) / SWD * SWD;
  // the tail loops of the sweep index rounds in 32 bits
  if ((S.rounds + SWD) * SWS >= (int64_t(1) << 31) || !sweep_pays(nlev, S.rounds, R, NC)) return S;
  S.word0.assign(static_cast<size_t>(SWD) * SWS, 0);
  for (size_t q = 0; q < S.word0.size() && q < words.size(); ++q) S.word0[q] = words[q];
  S.R = R;
  S.NC = NC;
  S.levels = nlev;
  auto fill = [&](auto f) { f(S, ptr, idx, src, dir, first, cnt, slot_group, slot_of, group_of, words); };
  switch (10 * R + NC) {
    case 12: fill(fill_records<1, 2>); break;
    case 13: fill(fill_records<1, 3>); break;
    case 15: fill(fill_records<1, 5>); break;
    case 22: fill(fill_records<2, 2>); break;
    case 23: fill(fill_records<2, 3>); break;
    case 25: fill(fill_records<2, 5>); break;
    case 32: fill(fill_records<3, 2>); break;
    case 33: fill(fill_records<3, 3>); break;
    default: fill(fill_records<3, 5>); break;
  }
  return S;
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

 private:
  struct Sweep {
    int R = 0, NC = 0, rounds = 0;
    Dev<uint32_t> word0;
    Dev<int32_t> rec, tptr, tcol;
    Dev<double> tval;
  };
  void make_sweep(Sweep& w, const SweepPlan& S);
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
  // forward levels: 1 + the highest level of the row's columns
  std::vector<int32_t> lev(n, 0);
  int32_t nf = n ? 1 : 0;
  for (int64_t i = 0; i < n; ++i) {
    int32_t l = 0;
    for (int64_t p = lptr[i]; p < lptr[i + 1]; ++p) l = std::max(l, lev[lidx[p]] + 1);
    lev[i] = l;
    nf = std::max(nf, l + 1);
  }
  std::vector<int32_t> flist, blist;
  by_level(lev, nf, flist, foff_);
  // U = L^T row-wise (columns increasing) and the map into L's values
  std::vector<int64_t> uptr(n + 1, 0), tmap(nnz);
  std::vector<int32_t> uidx(nnz);
  for (int64_t p = 0; p < nnz; ++p) ++uptr[lidx[p] + 1];
  for (int64_t j = 0; j < n; ++j) uptr[j + 1] += uptr[j];
  {
    std::vector<int64_t> pos(uptr.begin(), uptr.end() - 1);
    for (int64_t i = 0; i < n; ++i)
      for (int64_t p = lptr[i]; p < lptr[i + 1]; ++p) {
        const int64_t q = pos[lidx[p]]++;
        uidx[q] = static_cast<int32_t>(i);
        tmap[q] = p;
      }
  }
  // backward levels on U: row j needs the rows i > j of its pattern
  std::vector<int32_t> blev(n, 0);
  int32_t nbk = n ? 1 : 0;
  for (int64_t j = n - 1; j >= 0; --j) {
    int32_t l = 0;
    for (int64_t q = uptr[j]; q < uptr[j + 1]; ++q) l = std::max(l, blev[uidx[q]] + 1);
    blev[j] = l;
    nbk = std::max(nbk, l + 1);
  }
  by_level(blev, nbk, blist, boff_);

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
  const char* env = std::getenv("RUSTYFEM_IC0_LEVELS");
  if (n && !(env && *env && *env != '0')) {
    // the one-workgroup sweeps where they pay (sweep_pays)
    const SweepPlan f = plan_sweep(n, lptr, lidx, nullptr, 1);
    if (f.R) {
      const SweepPlan b = plan_sweep(n, uptr, uidx, &tmap, -1);
      if (b.R) {
        make_sweep(fw_, f);
        make_sweep(bw_, b);
      }
    }
  }
  if (!bw_.R) {
    uptr_.put(uptr);
    uidx_.put(uidx);
    tmap_.put(tmap);
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

void Ic0Impl::make_sweep(Sweep& w, const SweepPlan& S) {
  w.word0.put(S.word0);
  w.rec.put(S.rec);
  w.tptr.put(S.tptr);
  w.tcol.put(S.tcol);
  Dev<int32_t> vmap;
  Dev<int64_t> place, tmap;
  Dev<SweepCoef> coef;
  vmap.put(S.vmap);
  place.put(S.place);
  coef.put(S.coef);
  tmap.put(std::vector<int64_t>(S.tmap.begin(), S.tmap.end()));
  w.tval.alloc(S.tmap.size());
  double* rec = reinterpret_cast<double*>(w.rec.p);
  auto blocks = [](size_t c) { return static_cast<unsigned>((c + TB - 1) / TB); };
  if (!S.vmap.empty())
    k_ic0_records<<<blocks(S.vmap.size()), TB, 0, s_>>>(static_cast<int64_t>(S.vmap.size()), vmap.p, place.p, lval_.p, rec);
  if (!S.coef.empty())
    k_ic0_coefs<<<blocks(S.coef.size()), TB, 0, s_>>>(static_cast<int64_t>(S.coef.size()), coef.p, lval_.p, rec);
  if (!S.tmap.empty())
    k_gather<<<std::min(1024u, blocks(S.tmap.size())), TB, 0, s_>>>(static_cast<int64_t>(S.tmap.size()), tmap.p, lval_.p,
                                                                   w.tval.p);
  ICHK(hipGetLastError());
  ICHK(hipStreamSynchronize(s_));  // the maps live until here
  w.rounds = static_cast<int>(S.rounds);
  w.R = S.R;
  w.NC = S.NC;
}

template <int DIR>
void Ic0Impl::launch_sweep(const Sweep& w, const double* rin, double* out, const int32_t* done) {
  auto go = [&](auto kernel) {
    kernel<<<1, SWT, 0, s_>>>(w.rounds, w.word0.p, reinterpret_cast<const v4i*>(w.rec.p), w.tptr.p, w.tcol.p, w.tval.p,
                              rin, out, done);
  };
  switch (10 * w.R + w.NC) {
    case 12: go(k_ic0_sweep<1, 2, DIR>); break;
    case 13: go(k_ic0_sweep<1, 3, DIR>); break;
    case 15: go(k_ic0_sweep<1, 5, DIR>); break;
    case 22: go(k_ic0_sweep<2, 2, DIR>); break;
    case 23: go(k_ic0_sweep<2, 3, DIR>); break;
    case 25: go(k_ic0_sweep<2, 5, DIR>); break;
    case 32: go(k_ic0_sweep<3, 2, DIR>); break;
    case 33: go(k_ic0_sweep<3, 3, DIR>); break;
    default: go(k_ic0_sweep<3, 5, DIR>); break;
  }
}

void Ic0Impl::apply(const double* r, double* z, const int32_t* done) {
  if (bw_.R) {
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
