// Schedule of the IC(0) sweeps: groups of rows, their levels, and the round
// and slot of every group in the one-workgroup sweep (ic0_gpu.hip).
#include "ic0_plan.hpp"

#include <algorithm>

namespace rf {

void by_level(const std::vector<int32_t>& lev, int32_t nlev, std::vector<int32_t>& list, std::vector<int64_t>& off) {
  off.assign(nlev + 1, 0);
  for (int32_t l : lev) ++off[l + 1];
  for (int32_t l = 0; l < nlev; ++l) off[l + 1] += off[l];
  list.resize(lev.size());
  std::vector<int64_t> pos(off.begin(), off.end() - 1);
  for (size_t i = 0; i < lev.size(); ++i) list[pos[lev[i]]++] = static_cast<int32_t>(i);
}

std::vector<int32_t> row_levels(int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx, int dir,
                                int32_t& count) {
  std::vector<int32_t> lev(n, 0);
  count = n ? 1 : 0;
  for (int64_t e = 0; e < n; ++e) {
    const int64_t i = dir > 0 ? e : n - 1 - e;
    int32_t l = 0;
    for (int64_t p = ptr[i]; p < ptr[i + 1]; ++p) l = std::max(l, lev[idx[p]] + 1);
    lev[i] = l;
    count = std::max(count, l + 1);
  }
  return lev;
}

void transpose_pattern(int64_t n, const std::vector<int64_t>& lptr, const std::vector<int32_t>& lidx,
                       std::vector<int64_t>& uptr, std::vector<int32_t>& uidx, std::vector<int64_t>& tmap) {
  const int64_t nnz = lptr[n];
  uptr.assign(n + 1, 0);
  uidx.resize(nnz);
  tmap.resize(nnz);
  for (int64_t p = 0; p < nnz; ++p) ++uptr[lidx[p] + 1];
  for (int64_t j = 0; j < n; ++j) uptr[j + 1] += uptr[j];
  std::vector<int64_t> pos(uptr.begin(), uptr.end() - 1);
  for (int64_t i = 0; i < n; ++i)
    for (int64_t p = lptr[i]; p < lptr[i + 1]; ++p) {
      const int64_t q = pos[lidx[p]]++;
      uidx[q] = static_cast<int32_t>(i);
      tmap[q] = p;
    }
}

namespace {

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

// groups: consecutive rows (in elimination order) whose columns are the first
// row's columns and the rows of the group before them; first row and rows of
// every group
void groups(int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx, int dir, int R,
            std::vector<int32_t>& first, std::vector<int32_t>& cnt) {
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
}

}  // namespace

SweepPlan plan_sweep(int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx, int64_t levels,
                     int dir) {
  SweepPlan S;
  if (n >= (int64_t(1) << 28) || idx.size() >= (size_t(1) << 30)) return S;
  std::vector<int32_t> first, cnt;
  // the largest group size that wastes at most a quarter of its rows
  int R = 3;
  for (; R > 1; --R) {
    groups(n, ptr, idx, dir, R, first, cnt);
    if (static_cast<double>(n) >= 0.75 * R * static_cast<double>(first.size())) break;
    if (static_cast<int64_t>(first.size()) == n) R = 2;  // single rows
  }
  if (R == 1 && static_cast<int64_t>(first.size()) != n) groups(n, ptr, idx, dir, 1, first, cnt);
  const int64_t ng = static_cast<int64_t>(first.size());
  // no more levels than of rows, and full rounds: most of what will not pay
  // ends here
  if (!sweep_pays(levels, ng / SWS, R, 2)) return S;
  std::vector<int32_t> group_of(n), lev(ng, 0);
  for (int64_t g = 0; g < ng; ++g)
    for (int c = 0; c < cnt[g]; ++c) group_of[first[g] + dir * c] = static_cast<int32_t>(g);
  int32_t nlev = ng ? 1 : 0;
  int64_t over[2] = {0, 0};
  for (int64_t g = 0; g < ng; ++g) {
    int32_t l = 0;
    const int64_t k = ptr[first[g] + 1] - ptr[first[g]];
    for (int64_t p = ptr[first[g]]; p < ptr[first[g]] + k; ++p) l = std::max(l, lev[group_of[idx[p]]] + 1);
    lev[g] = l;
    nlev = std::max(nlev, l + 1);
    for (int q = 0; q < 2; ++q) over[q] += k > SWG * (2 + q);
  }
  std::vector<int32_t> list;
  std::vector<int64_t> off;
  by_level(lev, nlev, list, off);
  // columns per lane for nearly every group (19 of 20), at most 5
  const int NC = 20 * over[0] <= ng ? 2 : 20 * over[1] <= ng ? 3 : 5;
  int64_t rounds = 0;
  for (int32_t l = 0; l < nlev; ++l) rounds += (off[l + 1] - off[l] + SWS - 1) / SWS;
  rounds = (rounds + SWD - 1) / SWD * SWD;
  // the tail loops of the sweep index rounds in 32 bits
  if ((rounds + SWD) * SWS >= (int64_t(1) << 31) || !sweep_pays(nlev, rounds, R, NC)) return S;
  // a level's groups in order over the slots of its rounds
  std::vector<uint32_t> words(static_cast<size_t>((rounds + 2 * SWD) * SWS), 0);
  std::vector<int32_t> ring(n), round_of(ng);
  int64_t round = 0, tails = 0;
  for (int32_t l = 0; l < nlev; ++l) {
    const int64_t count = off[l + 1] - off[l], end = round + (count + SWS - 1) / SWS;
    int64_t oldest = INT64_MAX;  // round of the oldest value the level reads
    for (int64_t q = 0; q < count; ++q) {
      const int32_t g = list[off[l] + q];
      const int64_t f = first[g], k = ptr[f + 1] - ptr[f], slot = round * SWS + q;
      round_of[g] = static_cast<int32_t>(slot / SWS);
      words[slot] = slot_word(f, cnt[g], k > SWG * NC ? SW_TAIL : 0);
      const int64_t at = (slot / SWS % ring_rounds(R)) * (SWS * R) + (slot % SWS) * R;
      for (int c = 0; c < cnt[g]; ++c) ring[f + dir * c] = static_cast<int32_t>(at + c) * 8;
      for (int64_t p = ptr[f]; p < ptr[f + 1]; ++p) oldest = std::min<int64_t>(oldest, round_of[group_of[idx[p]]]);
      tails += std::max<int64_t>(0, k - SWG * NC);
    }
    // the level's own values must not reach the ring place of one it reads
    if (oldest != INT64_MAX) S.reach = std::max(S.reach, end - 1 - oldest);
    if (S.reach > ring_rounds(R) - 1) return S;
    for (int64_t q = (end - 1) * SWS; q < end * SWS; ++q) words[q] |= SW_LAST;
    round = end;
  }
  S.tptr.assign(static_cast<size_t>((rounds + SWD) * SWS) + 1, 0);
  if (tails > 0)
    for (size_t q = 0; q + 1 < S.tptr.size(); ++q) {
      const int64_t f = slot_row(words[q]);
      S.tptr[q + 1] = S.tptr[q];
      if (words[q] & SW_TAIL) S.tptr[q + 1] += static_cast<int32_t>(ptr[f + 1] - ptr[f] - SWG * NC);
    }
  S.R = R;
  S.NC = NC;
  S.levels = nlev;
  S.rounds = rounds;
  S.bytes = (rounds + SWD) * SWT * record_granules(R, NC) * 16 + tails * (4 + 8 * R);
  S.words = std::move(words);
  S.ring = std::move(ring);
  return S;
}

}  // namespace rf
