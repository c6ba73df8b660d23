// What the two token-serial recurrences share (recurrence.hip: dense route
// vectors; route_recurrence.hip: sparse routes): a (bank, 32 columns) table in
// LDS, 8 lanes to a column, and the records that producer waves stage.

#pragma once

#include "common.h"

namespace cowsdm_impl {

constexpr int kRrCols = 8;                    // columns per compute wave
constexpr int kRrGroups = kWave / kRrCols;    // lanes per column
constexpr int kRrWaves = 4;                   // compute waves per workgroup, at most
constexpr int kRrProducers = 4 * kWave;       // threads that stage the tokens
constexpr int kRrThreads = kRrWaves * kWave + kRrProducers;
constexpr int kRrMaxChunk = 64;               // tokens staged at a time, at most
constexpr int kRrRowBytes = kRrCols * 4;      // a row in a wave's table
constexpr int kRrPad = 2;                     // records after a chunk that change nothing
constexpr int kRrRowsAhead = 8;               // initial rows a thread has in flight
constexpr int kRrLds = 160 * 1024;
constexpr int kRrMaxSlots = 1024;
constexpr int kXcds = 8;

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(
                 __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Sum over the 8 lanes of a column, the same in all of them: neighbours,
// pairs (quad_perm [1,0,3,2], [2,3,0,1]), then the other quad of the eight
// (row_half_mirror).
__device__ __forceinline__ float column_sum8(float v) {
  return dpp_add<0x141>(dpp_add<0x4E>(dpp_add<0xB1>(v)));
}

// One token's record in a chunk's staging area: its write entries, its read
// entries, exp(forget) and the input gate, the workgroup's columns of the
// value.  A chunk ends with kRrPad records that change nothing, for the loads
// that run ahead.
template <int WPL, int RPL>
struct RrRecord {
  static constexpr int kWrite = 0;
  static constexpr int kRead = 8 * kRrGroups * WPL;
  static constexpr int kGates = kRead + 8 * kRrGroups * RPL;
  static constexpr int kValue = kGates + 16;
  static constexpr int kBytes = kValue + 4 * kRrCols * kRrWaves;
};

}  // namespace cowsdm_impl
