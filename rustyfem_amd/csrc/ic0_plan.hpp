// Schedule of the IC(0) sweeps (host only): which rows form a group, and in
// which round and slot of the one-workgroup sweep every group is taken.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

namespace rf {

#ifdef __HIP__
#define RF_HOST_DEVICE __host__ __device__
#else
#define RF_HOST_DEVICE
#endif

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
RF_HOST_DEVICE constexpr uint32_t slot_word(int64_t row, int cnt, uint32_t flags) {
  return static_cast<uint32_t>(row) << 4 | static_cast<uint32_t>(cnt) << 2 | flags;
}
RF_HOST_DEVICE constexpr int32_t slot_row(uint32_t w) { return static_cast<int32_t>(w >> 4); }
RF_HOST_DEVICE constexpr int slot_rows(uint32_t w) { return static_cast<int>(w >> 2) & 3; }

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
constexpr int64_t record_granules(int R, int NC) { return (NC + 4) / 4 + (NC * R + R) / 2; }
static_assert(record_granules(3, 5) == SweepRecord<3, 5>::GRANULES && record_granules(1, 2) == SweepRecord<1, 2>::GRANULES &&
                  record_granules(2, 3) == SweepRecord<2, 3>::GRANULES,
              "the same count");

// One sweep over the strictly triangular rows (ptr, idx: columns sorted;
// forward: columns below the row, dir = 1; backward: above it, dir = -1).
struct SweepPlan {
  int R = 0;                    // rows per group (1, 2 or 3); 0: no sweep
  int NC = 0;                   // columns per lane in a record (2, 3 or 5)
  int64_t levels = 0;           // of groups
  int64_t rounds = 0;           // a multiple of SWD
  int64_t reach = 0;            // most rounds between a level's last one and the first of a level it reads
  int64_t bytes = 0;            // streamed by a sweep: records, tails
  std::vector<uint32_t> words;  // the slots' words, of rounds + 2 SWD rounds
  std::vector<int32_t> ring;    // per row: the byte offset of its value in the ring
  std::vector<int32_t> tptr;    // per slot of rounds + SWD rounds: its first tail column
};

// levels: those of the single rows (a launch each without the sweep).  The
// plan's R is 0 where a sweep is not possible, would not pay or would stream
// more than a small multiple of the factor.
SweepPlan plan_sweep(int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx, int64_t levels,
                     int dir);

// the rows' levels of a triangle: one more than the highest among the row's columns
std::vector<int32_t> row_levels(int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx, int dir,
                                int32_t& count);

// U = L^T row-wise (columns increasing) and the map into L's values
void transpose_pattern(int64_t n, const std::vector<int64_t>& lptr, const std::vector<int32_t>& lidx,
                       std::vector<int64_t>& uptr, std::vector<int32_t>& uidx, std::vector<int64_t>& tmap);

// rows grouped by level: list (rows in increasing order within a level) and
// the level offsets
void by_level(const std::vector<int32_t>& lev, int32_t nlev, std::vector<int32_t>& list, std::vector<int64_t>& off);

// Static check of a plan with R > 0 against its triangle: every row is taken
// once, by a group whose columns it shares; what a level reads was written by
// an earlier level and is still in the ring once everything that the level
// writes has been written (its waves are not held together).  Empty when
// sound.
std::string check_sweep(const SweepPlan& S, int64_t n, const std::vector<int64_t>& ptr, const std::vector<int32_t>& idx,
                        int dir);

}  // namespace rf
