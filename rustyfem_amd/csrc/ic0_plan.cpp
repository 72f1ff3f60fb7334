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

// One workgroup's sweep against a launch per level of rows: 0.1 us per level,
// and per round 0.25 us and the load rate of one compute unit for its records
// (0.065 us per 8 KB granule row; 0.13 from HBM, where the records of a
// direction and what else the iteration reads exceed the Infinity Cache),
// against at least 3.4 us per launch.  Measured, both directions together, us:
//                              rows of a group, columns a lane, row levels, rounds: sweeps / launches
//   hexahedra 8^3 / 40^3                 3, 5,  168 /  840,   57 / 1209:    142 /  2,450    1,260 /  7,010
//   hexahedra 48^3 / 56^3                3, 5, 1008 / 1176, 1992 / 3054:  7,090 / 10,930    9,540 / 11,100
//   tetrahedra 20^3 / 40^3               3, 3,  180 /  360,  168 / 1116:    276 /  1,630    1,380 /  3,040
//   quadrilaterals 500 x 200 / 800 x 700 2, 2, 1800 / 4400, 2064 / 10026: 2,080 / 16,500   13,200 / 28,300
//   2D Laplacian 300^2 / 500^2 / 800^2   1, 2,  599 /  999 / 1599, 1716 / 4410 / 10803:
//                                           1,220 / 3,130 / 11,800         4,300 / 7,790 / 11,200
//   3D Laplacian 24^3 / 48^3             1, 2,   70 /  142,  255 / 1800:    203 /  1,225      510 /  1,130
//   chain 1,000 / band of 5,000 rows     1, 2 / 5, 1000 / 5000, 1002 / 5001: 669 / 8,365     7,400 / 37,000
bool sweep_pays(int64_t row_levels, int64_t levels, int64_t rounds, int R, int NC) {
  const double granules = static_cast<double>(record_granules(R, NC)), n = static_cast<double>(rounds);
  const bool cached = n * SWT * 16 * granules < 128e6;
  return 0.1 * static_cast<double>(levels) + (0.25 + granules * (cached ? 0.065 : 0.13)) * n <
         3.4 * static_cast<double>(row_levels);
}

// Every round streams full records for its 64 slots (16 to 90 KB), also where
// its level holds one group: a chain of 10^6 rows would take 16 GB for 12 MB of
// factor.  A sweep may take 16 times the factor instead (a level of five groups
// on average, whatever the size), or 256 MB, one thousandth of the memory: a
// chain of up to 15,000 rows (10,000: 9.4 ms an application, 74.6 with a launch
// per level).
double stream_limit(int64_t n, int64_t nnz) {
  return 256e6 + 16.0 * (12.0 * static_cast<double>(nnz) + 16.0 * static_cast<double>(n));
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
  // full rounds alone: most of what will not pay ends here
  if (!sweep_pays(levels, 0, ng / SWS, R, 2)) return S;
  std::vector<int32_t> at(n), lev(ng), low(ng);  // per row: its group's level; per group: level, lowest one read
  int32_t nlev = ng ? 1 : 0;
  int64_t over[2] = {0, 0}, beyond[3] = {0, 0, 0};  // groups of more columns than 2, 3; columns beyond 2, 3, 5
  for (int64_t g = 0; g < ng; ++g) {
    int32_t l = 0, lo = INT32_MAX;
    const int64_t k = ptr[first[g] + 1] - ptr[first[g]];
    for (int64_t p = ptr[first[g]]; p < ptr[first[g]] + k; ++p) {
      const int32_t c = at[idx[p]];
      l = std::max(l, c + 1);
      lo = std::min(lo, c);
    }
    lev[g] = l;
    low[g] = lo;
    for (int c = 0; c < cnt[g]; ++c) at[first[g] + dir * c] = l;
    nlev = std::max(nlev, l + 1);
    for (int q = 0; q < 2; ++q) over[q] += k > SWG * (2 + q);
    for (int q = 0; q < 3; ++q) beyond[q] += std::max<int64_t>(0, k - SWG * (q == 2 ? 5 : 2 + q));
  }
  std::vector<int32_t> list;
  std::vector<int64_t> off;
  by_level(lev, nlev, list, off);
  // columns per lane for nearly every group (19 of 20), at most 5
  const int NC = 20 * over[0] <= ng ? 2 : 20 * over[1] <= ng ? 3 : 5;
  int64_t rounds = 0;
  for (int32_t l = 0; l < nlev; ++l) rounds += (off[l + 1] - off[l] + SWS - 1) / SWS;
  rounds = (rounds + SWD - 1) / SWD * SWD;
  const int64_t tails = beyond[NC == 5 ? 2 : NC - 2];
  S.bytes = (rounds + SWD) * SWT * record_granules(R, NC) * 16 + tails * (4 + 8 * R);
  if (static_cast<double>(S.bytes) > stream_limit(n, static_cast<int64_t>(idx.size()))) return S;
  // the tail loops of the sweep index rounds in 32 bits
  if ((rounds + SWD) * SWS >= (int64_t(1) << 31) || !sweep_pays(levels, nlev, rounds, R, NC)) return S;
  // a level's groups in order over the slots of its rounds
  std::vector<uint32_t> words(static_cast<size_t>((rounds + 2 * SWD) * SWS), 0);
  std::vector<int32_t> ring(n);
  std::vector<int64_t> start(nlev);  // the levels' first rounds
  int64_t round = 0;
  for (int32_t l = 0; l < nlev; ++l) {
    const int64_t count = off[l + 1] - off[l], end = round + (count + SWS - 1) / SWS;
    start[l] = round;
    int32_t lo = INT32_MAX;
    for (int64_t q = 0; q < count; ++q) {
      const int32_t g = list[off[l] + q];
      const int64_t f = first[g], slot = round * SWS + q;
      words[slot] = slot_word(f, cnt[g], ptr[f + 1] - ptr[f] > SWG * NC ? SW_TAIL : 0);
      const int64_t o = (slot / SWS % ring_rounds(R)) * (SWS * R) + (slot % SWS) * R;
      for (int c = 0; c < cnt[g]; ++c) ring[f + dir * c] = static_cast<int32_t>(o + c) * 8;
      lo = std::min(lo, low[g]);
    }
    // the level's own values must not reach the ring place of one it reads
    // (taken as the first of that value's level)
    if (lo != INT32_MAX) S.reach = std::max(S.reach, end - 1 - start[lo]);
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
  S.words = std::move(words);
  S.ring = std::move(ring);
  return S;
}

std::string check_sweep(const SweepPlan& S, int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx,
                        int dir) {
  const int per = SWS * S.R, places = ring_rounds(S.R) * per;
  std::vector<int32_t> owner(places, -1);
  std::vector<uint8_t> seen(n, 0);
  int64_t rows = 0, levels = 0, tails = 0;
  if (S.words.size() != static_cast<size_t>((S.rounds + 2 * SWD) * SWS) || S.rounds % SWD) return "rounds";
  for (int64_t r0 = 0; r0 < S.rounds;) {
    int64_t r1 = r0;
    while (r1 < S.rounds && !(S.words[r1 * SWS] & SW_LAST)) ++r1;
    if (r1 == S.rounds) break;  // the empty rounds at the end
    ++r1;
    ++levels;
    for (int64_t q = r0 * SWS; q < r1 * SWS; ++q) {
      const uint32_t w = S.words[q];
      if (((w & SW_LAST) != 0) != (q >= (r1 - 1) * SWS)) return "a round's slots disagree on the level's end";
      for (int c = 0; c < slot_rows(w); ++c) {
        const int64_t row = slot_row(w) + dir * c;
        const int64_t at = (q / SWS % ring_rounds(S.R)) * per + (q % SWS) * S.R + c;
        if (c >= S.R || row < 0 || row >= n || seen[row]) return "a row is out of range or taken twice";
        if (S.ring[row] != at * 8) return "a row's ring place is not its slot's";
        seen[row] = 1;
        owner[at] = static_cast<int32_t>(row);
        ++rows;
      }
    }
    for (int64_t q = r0 * SWS; q < r1 * SWS; ++q) {
      const uint32_t w = S.words[q];
      if (!slot_rows(w)) continue;
      const int64_t f = slot_row(w), k = ptr[f + 1] - ptr[f];
      if (((w & SW_TAIL) != 0) != (k > SWG * S.NC)) return "the tail flag does not fit the row";
      if (S.tptr[q] != tails) return "the tails overlap";
      if (w & SW_TAIL) tails += k - SWG * S.NC;
      for (int c = 0; c < slot_rows(w); ++c) {
        const int64_t p = ptr[f + dir * c] + (dir > 0 ? 0 : c), o = ptr[f + dir * c] + (dir > 0 ? k : 0);
        if (ptr[f + dir * c + 1] - ptr[f + dir * c] != k + c || !std::equal(idx.data() + p, idx.data() + p + k, idx.data() + ptr[f]))
          return "a group's rows differ in their columns";
        for (int u = 0; u < c; ++u)
          if (idx[o + u] != (dir > 0 ? f + u : f - c + 1 + u)) return "a group's triangle is not full";
      }
      for (int64_t p = ptr[f]; p < ptr[f] + k; ++p) {
        if (owner[S.ring[idx[p]] / 8] != idx[p]) return "a value is read before it is written or after its place was reused";
        if (seen[idx[p]] == 1) return "a level reads its own value";
      }
    }
    // 2: of an earlier level
    for (int64_t q = r0 * SWS; q < r1 * SWS; ++q)
      for (int c = 0; c < slot_rows(S.words[q]); ++c) seen[slot_row(S.words[q]) + dir * c] = 2;
    r0 = r1;
  }
  return rows == n && levels == S.levels ? "" : "rows or levels are missing";
}

}  // namespace rf
