// What the two halves of the prefill attention share: its parameters and constants.
#pragma once
#include <math.h>

#include "attn_common.h"

namespace jpt {
namespace prefill {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((address_space(3))) char* lds_char_ptr;

constexpr int kCols = 64;       // positions a tile
constexpr int kWaveRows = 32;   // query rows a wave
constexpr int kWavesPerGroup = 4;
constexpr int kRowsPerGroup = kWaveRows * kWavesPerGroup;
constexpr int kMaxTiles = 1024;  // tiles that fit the list in LDS: 65536 positions
constexpr int kOwnTiles = 32;   // of a workgroup that looks through the mask itself: 2048 positions
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int64_t kL2Bytes = 4 << 20;  // of an XCD
// Weights and sums are relative to a reference that starts 2^kAhead above a row's maximum and moves when the maximum has
// passed it: seldom (every step's move at heads of 256, 2000 rows: 84 -> 111 us; 4 -> 8: 85 -> 83), and no weight is ever above
// 1, so that sums over large values overflow no earlier than relative to the maximum itself.
constexpr float kAhead = 4.f;
constexpr float kFarBelow = -1e37f;  // times log2(e) finite

// what a mask block (32 rows x 64 positions) holds
constexpr int kLive = 1;     // some value that is not -inf
constexpr int kNonZero = 2;  // some value that is not 0

struct PrefillParams {
  jpt_attn_args a;
  const uint8_t* classes;   // per mask block, or NULL: every block may hold anything
  int64_t class_stride_b, class_stride_h;
  int32_t own_classes;      // bytes a load with which a workgroup looks through its rows of the mask itself (two key waves), or 0
  int32_t row_blocks, col_blocks;  // of one mask
  int32_t group_rows;       // query rows the row tiles of one group count through
  int32_t groups;           // groups a KV head
  int32_t tiles;            // row tiles a group
  int32_t key_waves;        // waves side by side over a tile's positions
  int32_t by_rows;          // workgroups in the order of their rows: the longest first
  int32_t xcd_units;        // compute units of an XCD, where two workgroups share one; or else more than there are
  int32_t mask_runs;        // runs of four mask values are aligned
};

// Defined in attn_prefill_<D>.hip.
template <int D>
void launch_prefill(const PrefillParams& p, dim3 grid, hipStream_t stream);

}  // namespace prefill
}  // namespace jpt
