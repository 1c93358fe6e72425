// Balanced decode: a fixed number of workgroups shares the keys of all sequences evenly, from the
// lengths as they are on the device (the host never reads them). Every wave of both split kernels
// derives the same schedule; the workgroup that starts a row leaves the row's slots for the merge pass
// (DecodeArgs::row_slots).
//
// A sequence's keys are cut into units of 2^unit_shift keys. A row is one work head (the KV heads and
// query heads that one workgroup serves together) of one sequence: its units and then
// DecodeArgs::ramp_units without keys, about what starting a row costs a workgroup. Sequence 0's rows,
// then sequence 1's, and so on, form one line, and workgroup w takes positions [w chunk, (w + 1) chunk)
// of it, one segment per row that it crosses. chunk is the line's length over the workgroups, rounded
// up. If every row can have workgroups of its own with a chunk no larger than that, rows are padded to
// whole chunks instead and no workgroup runs more than one segment.
//
// A row's first kRowSlots partials have places of their own; the partial of workgroup w for row r
// beyond them goes to overflow slot w + r: along the line each step to the next segment raises exactly
// one of the two, so overflow slots are distinct.
//
// Everything is wave-uniform or per lane: lane l holds the unit counts of sequences l per .. l per +
// per - 1 (per = ceil(B / 64) <= 4), prefix sums run across the lanes, and no LDS or barrier is used.
#pragma once

#include "gfx950.hpp"
#include "launch.hpp"

namespace fl {
namespace decode {

struct Schedule {
  static constexpr int kPer = kMaxBalancedBatch / 64;
  int keys[kPer];  // of the lane's sequences
  int size[kPer];  // positions of one row of each
  int before;      // positions of one row each of the sequences of lower lanes
  int through;     // ... and of the lane's own
  int per;         // sequences per lane
  int rows;        // rows per sequence
  int chunk;       // positions per workgroup
  float inv_chunk;
  int total;       // positions of the line
};

// Inclusive prefix sum over the wave's lanes, on DPP moves (no LDS): within rows of 16 lanes, then row
// 0's sum into row 1 and row 2's into row 3, then the lower half's into the upper.
__device__ __forceinline__ int wave_inclusive_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return x;
}

// floor and ceil of n / c for n in [0, 2^22] (the host keeps the line within that) and c >= 1, with r =
// 1 / c to within an ulp: n r is off from n / c by less than 2 / c, so its integer part is the floor or
// one off it, which the remainder tells. A reciprocal and a few instructions where the integer
// division is some forty, on the path to a workgroup's first load.
__device__ __forceinline__ int floor_div(int n, int c, float r) {
  int q = static_cast<int>(static_cast<float>(n) * r);
  const int rem = n - q * c;
  q += rem >= c ? 1 : 0;
  q -= rem < 0 ? 1 : 0;
  return q;
}
__device__ __forceinline__ int ceil_div(int n, int c, float r) { return floor_div(n + c - 1, c, r); }
__device__ __forceinline__ float reciprocal(int c) { return __builtin_amdgcn_rcpf(static_cast<float>(c)); }

__device__ __forceinline__ int sequence_keys(const DecodeArgs& a, int b) {
  // Lengths are not checked on the host (that would need a sync); clamped to the cache so an
  // out-of-range value cannot read outside it.
  return min(max(a.seq_lens[b], 0), a.max_seqlen);
}

__device__ __forceinline__ int units_of(const DecodeArgs& a, int keys) {
  return (keys + (1 << a.unit_shift) - 1) >> a.unit_shift;
}

__device__ __forceinline__ Schedule make_schedule(const DecodeArgs& a, int rows) {
  Schedule s;
  const int lane = __lane_id();
  s.rows = rows;
  s.per = (a.batch + 63) / 64;
  int units[Schedule::kPer];
  int sum = 0;
  int filled = 0;  // sequences with keys
#pragma unroll
  for (int i = 0; i < Schedule::kPer; ++i) {
    units[i] = s.keys[i] = 0;
    if (i < s.per) {
      const int b = lane * s.per + i;
      s.keys[i] = b < a.batch ? sequence_keys(a, b) : 0;
      units[i] = units_of(a, s.keys[i]);
    }
    sum += units[i];
    filled += units[i] > 0 ? 1 : 0;
    s.size[i] = units[i] > 0 ? units[i] + a.ramp_units : 0;
  }
  const int wgs = a.balanced_wgs;
  const float inv_wgs = reciprocal(wgs);
  const int all_units = __builtin_amdgcn_readlane(wave_inclusive_sum(sum), 63) * rows;
  const int all_filled = __builtin_amdgcn_readlane(wave_inclusive_sum(filled), 63) * rows;
  const int least = max(ceil_div(all_units, wgs, inv_wgs), a.min_units);
  s.chunk = max(ceil_div(all_units + all_filled * a.ramp_units, wgs, inv_wgs), a.min_units);
  s.inv_chunk = reciprocal(s.chunk);
  sum += filled * a.ramp_units;
  // The smallest chunk that the keys allow, then the line's own: each with rows padded to it.
  if (all_filled <= wgs) {
    for (int t = 0; t < 2; ++t) {
      const int c = t == 0 ? least : s.chunk;
      const float r = reciprocal(c);
      int chunks[Schedule::kPer];
      int mine = 0;
#pragma unroll
      for (int i = 0; i < Schedule::kPer; ++i) {
        chunks[i] = 0;
        if (i < s.per) chunks[i] = ceil_div(units[i], c, r);
        mine += chunks[i];
      }
      if (__builtin_amdgcn_readlane(wave_inclusive_sum(mine), 63) * rows <= wgs) {
#pragma unroll
        for (int i = 0; i < Schedule::kPer; ++i) s.size[i] = chunks[i] * c;
        sum = mine * c;
        s.chunk = c;
        s.inv_chunk = r;
        break;
      }
    }
  }
  s.through = wave_inclusive_sum(sum);
  s.before = s.through - sum;
  s.total = __builtin_amdgcn_readlane(s.through, 63) * rows;
  return s;
}

// The keys of a workgroup's segment that starts at position pos (in [0, total)) of the line, and where
// it leaves its partials. No keys (k_begin == k_end): only the positions of the row's start cost.
struct Segment {
  int b, head, k_begin, k_end;
  int64_t slot;
  int next;  // position after the segment
};
__device__ __forceinline__ Segment segment_at(const DecodeArgs& a, const Schedule& s, int wg, int pos, int end,
                                              bool writer) {
  const uint64_t mask = __builtin_amdgcn_ballot_w64(pos >= s.before * s.rows && pos < s.through * s.rows);
  const int owner = mask ? __builtin_ctzll(mask) : 0;
  int from = __builtin_amdgcn_readlane(s.before, owner) * s.rows;  // first row of the sequence
  int b = owner * s.per;
  int keys = __builtin_amdgcn_readlane(s.keys[0], owner);
  int size = __builtin_amdgcn_readlane(s.size[0], owner);
#pragma unroll
  for (int i = 1; i < Schedule::kPer; ++i) {
    if (i >= s.per || pos < from + size * s.rows) break;
    from += size * s.rows;
    b = owner * s.per + i;
    keys = __builtin_amdgcn_readlane(s.keys[i], owner);
    size = __builtin_amdgcn_readlane(s.size[i], owner);
  }
  Segment g;
  g.b = b;
  g.head = floor_div(pos - from, size, reciprocal(size));
  const int start = from + g.head * size;
  const int first = pos - start;
  g.next = min(end, start + size);
  g.k_begin = min(keys, first << a.unit_shift);
  g.k_end = min(keys, (first + g.next - pos) << a.unit_shift);
  const int row = b * s.rows + g.head;
  const int first_wg = floor_div(start, s.chunk, s.inv_chunk);
  const int split = wg - first_wg;
  g.slot = split < kRowSlots ? row * int64_t{kRowSlots} + split
                             : int64_t{a.batch} * s.rows * kRowSlots + wg + row;
  if (first == 0 && writer) {
    const int last_wg = floor_div(start + units_of(a, keys) - 1, s.chunk, s.inv_chunk);
    a.row_slots[row] = int2{last_wg - first_wg + 1, first_wg + row};
  }
  return g;
}

}  // namespace decode
}  // namespace fl
