// Attention of many query rows over bf16 keys and values (prefill, and any dense
// call whose query rows are too many for the streaming decode kernel), head_dim
// 64, 128 or 256, on the matrix cores.
//
// One workgroup of four waves takes 128 query rows of one KV head, or 64 (see
// key_waves_for), and walks the keys in tiles of 64 positions.  Tiles go from memory
// straight into LDS (two buffers); a wave holds 32 query rows and runs
//     S^T = K . Q^T     v_mfma_f32_32x32x16_bf16, positions on M, query rows on N
//     O^T = V^T . P^T   positions on the contraction index
// with the online softmax in between.  With positions on M the score
// accumulators of a lane belong to ONE query row (lane & 31) and are, in the
// order they lie, that lane's share of the second product's operand: softmax
// weights never cross lanes, a row's running maximum and factor are one
// register.  V^T comes out of the row-major tile by the transposing LDS read
// (ds_read_b64_tr_b16).
//
// Softmax weights go in as three bf16 numbers (the rounded weight, what the
// rounding left, and what rounding that left), whose sum is the float32 weight
// exactly.
//
// Matrix work: 4 . D flop per score, twice that with the weights' second and
// third numbers, and the vector ALU's exponentials and splits beside it, about as
// long.  So the two run side by side in every wave: the next tile's scores and this
// tile's products are matrix instructions with a few of the softmax's vector
// instructions between them, in an order that is pinned (a tile of 32 rows x 64
// positions: 64 matrix instructions of 32 clocks each, 450 vector ones of 4 or,
// exponentials, 16).  That holds for plain tiles, which all rows attend as they are;
// tiles that a mask changes, the diagonal of a causal one, come last and are done one
// step after the other.  3500 rows: matrix pipe busy in 47 % of the SIMD time (38 % one
// step after the other).
// Outputs are rescaled only when a row's maximum has grown by 2^4 since they last were (kAhead).
// What a causal mask leaves out is not computed: a pass over the mask (read
// once, not once a head) first writes down, for every 32 rows x 64 positions,
// whether anything there is live and whether anything there is not zero; dead
// tiles are neither loaded nor computed, and all-zero tiles need no mask reads.
//
// Measured, causal, 32 query heads over 8 KV heads of 128, a call with its pass over
// the mask, calls back to back, one step after the other -> side by side: 256 rows 21 ->
// 14 us, 1024 rows 46 -> 31, 2048 rows 93 -> 78, 3500 rows with scales 240 -> 218; 16 heads of
// 256, 2000 rows 157 -> 85 (12.3 ms for 1024 rows on the shape-generic kernel, one wave a
// row, scalar dot products).  Outputs that are not the rounded exact value: 0.021-0.042 % over eight
// shapes, 0.018-0.046 % before.
#include <math.h>

#include <type_traits>

#include "attn_common.h"

// Where the compiler's scheduler moves nothing across: it would gather the matrix instructions, the vector
// ALU's and the LDS reads each in a place, and hold more than there are registers.
#define JPT_PIN() __builtin_amdgcn_sched_barrier(0)

namespace jpt {
namespace {

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
  int32_t row_blocks, col_blocks;  // of one mask
  int32_t group_rows;       // query rows the row tiles of one group count through
  int32_t groups;           // groups a KV head
  int32_t tiles;            // row tiles a group
  int32_t key_waves;        // waves side by side over a tile's positions
  int32_t by_rows;          // workgroups in the order of their rows: the longest first
  int32_t mask_runs;        // runs of four mask values are aligned
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Value of the other half's lane with the same query row (lane ^ 32).
__device__ __forceinline__ float other_half(float v) {
  int a = __builtin_bit_cast(int, v), c = a;
  asm volatile("" : "+v"(c));  // the swap of a register with itself is not what the instruction does
  const auto s = __builtin_amdgcn_permlane32_swap(a, c, false, false);
  const int lo = s[0], hi = s[1];
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? lo : hi);
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  bf16x2 t = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, t);
}

// 0, which the compiler does not know.
__device__ __forceinline__ int nothing() {
  int x;
  asm volatile("s_mov_b32 %0, 0" : "=s"(x));
  return x;
}

// The same as one value: the compiler, which sees that half of it is one of the numbers, rounds that again.
__device__ __forceinline__ uint32_t pack_together(float lo, float hi) {
  uint32_t both = pack_bf16(lo, hi);
  asm("" : "+v"(both));
  return both;
}

// 16 bytes a lane from memory to LDS at `lds` + 16 * lane, not known to the
// compiler as an LDS write: it would make every later LDS read wait for all
// such loads, the next tile's among them.  A write of M0 needs one wait state
// before the load that uses it, which the compiler does not see to inside asm.
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t lane_off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_off), "s"(base), "s"(lds) : "memory");
}

// Where 16-byte piece p of row t lies in its row: p ^ swizzle(t).  Sixteen
// consecutive rows' pieces of one number are on sixteen different bank groups
// (the K operand's reads), and so are four consecutive rows' runs of 64 bytes
// (the V operand's).
template <int D>
__device__ __forceinline__ constexpr int swizzle(int t) {
  return D == 64 ? (((t >> 1) & 1) << 2) | ((t >> 2) & 3) : ((t & 3) << 2) | ((t >> 2) & 3);
}

template <int D, int SCALE, int MASK, int KEY_WAVES>
__global__ void __launch_bounds__(64 * kWavesPerGroup, D == 256 ? 1 : 2) attn_prefill_kernel(PrefillParams p) {
  const jpt_attn_args& a = p.a;
  constexpr int kRow = D * 2;                  // bytes of a row
  constexpr int kPieces = kRow / 16;
  constexpr int kTileBytes = kCols * kRow;     // keys or values of a tile
  constexpr int kRowsPerLoad = 1024 / kRow;    // rows of one wave-wide load
  constexpr int kLoads = kTileBytes / 1024 / kWavesPerGroup;  // loads a wave makes for the keys, and for the values
  constexpr int kSteps = D / 16;               // contraction steps of S^T
  constexpr int kBlocks = D / 32;              // row blocks of O^T
  constexpr int kRowWaves = kWavesPerGroup / KEY_WAVES;   // waves side by side over the query rows
  constexpr int kKeyBlocks = kCols / 32 / KEY_WAVES;      // blocks of 32 positions of a tile that are a wave's
  constexpr int kPvSteps = 2 * kKeyBlocks;                // 16 positions each
  __shared__ __attribute__((aligned(1024))) char sm[2][2 * kTileBytes];
  __shared__ float sm_scale[2][2][kCols];      // key and value scales of a tile
  __shared__ int sm_list[MASK ? kMaxTiles : 1];  // tiles to do: number << 8 | two class bits a row wave
  __shared__ int sm_count[2];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int row_wave = wave % kRowWaves, key0 = wave / kRowWaves * (32 * kKeyBlocks);
  const int T = a.q_rows, S = a.seq;
  const int rep = a.q_heads / a.kv_heads;

  // Workgroups go round the XCDs: all row tiles of one KV head on one XCD, whose
  // L2 then holds the head's keys and values; last rows first, which under a
  // causal mask have the most to do.
  const int pairs = a.batch * a.kv_heads, per_pair = p.groups * p.tiles;
  int pair, at;
  if (pairs % 8 == 0) {
    const int i = blockIdx.x >> 3;
    if (p.by_rows) {
      const int of_xcd = pairs / 8;
      pair = (blockIdx.x & 7) + 8 * (i % of_xcd);
      at = i / of_xcd;
    } else {
      pair = (blockIdx.x & 7) + 8 * (i / per_pair);
      at = i % per_pair;
    }
  } else {
    pair = blockIdx.x % pairs;
    at = blockIdx.x / pairs;
  }
  const int b = pair / a.kv_heads, hkv = pair % a.kv_heads;
  const int group = at % p.groups, tile_row = p.tiles - 1 - at / p.groups;
  const int hs = a.scale_heads == 1 ? 0 : hkv;

  int len = a.lengths ? a.lengths[b] : S;
  len = len < 0 ? 0 : (len > S ? S : len);

  // this lane's query row: index in its group, then (q head of the KV head, row of the head)
  const int row0 = (tile_row * kRowWaves + row_wave) * kWaveRows;
  const int row = row0 + n;
  const bool row_live = row < p.group_rows;
  const int row_in = row_live ? row : p.group_rows - 1;
  const int q_head = hkv * rep + (p.groups == 1 ? row_in / T : group);
  const int t = p.groups == 1 ? row_in % T : row_in;
  const int64_t q_row = (static_cast<int64_t>(b) * a.q_heads + q_head) * T + t;

  // ---- which tiles there are to do -------------------------------------------
  // Plain tiles, full ones that count for all rows of the workgroup as they are, come first; then those that a
  // mask changes or leaves rows out of, and the cache's last, partly filled one.
  const int n_tiles = (len + kCols - 1) / kCols;
  const bool listed = MASK && p.classes != nullptr;
  if (listed) {
    if (wave == 0) {
      // (the rows of one wave lie in one row block: row tiles start at multiples of a wave's rows)
      const uint8_t* cls = p.classes + b * p.class_stride_b + (hkv * rep + group) * p.class_stride_h +
                           static_cast<int64_t>(tile_row) * kRowWaves * p.col_blocks;
      const int row_waves = min(kRowWaves, p.row_blocks - tile_row * kRowWaves);
      int plain = 0, others = 0;  // plain tiles from the list's start on, the others from its end backwards
      for (int c0 = 0; c0 < n_tiles; c0 += 64) {
        const int c = c0 + lane;
        int bits = 0;
#pragma unroll
        for (int w = 0; w < kRowWaves; ++w)
          if (c < n_tiles && w < row_waves) bits |= cls[static_cast<int64_t>(w) * p.col_blocks + c] << (2 * w);
        const bool live = (bits & 0x55 * kLive) != 0;
        const bool is_plain = bits == (0x55 * kLive & ((1 << 2 * row_waves) - 1)) && (c + 1) * kCols <= len;
        const uint64_t set = __ballot(is_plain), rest = __ballot(live && !is_plain), below = (1ull << lane) - 1;
        if (is_plain) sm_list[plain + __popcll(set & below)] = c << 8 | bits;
        else if (live) sm_list[n_tiles - 1 - others - __popcll(rest & below)] = c << 8 | bits;
        plain += __popcll(set);
        others += __popcll(rest);
      }
      if (lane == 0) {
        sm_count[0] = plain;
        sm_count[1] = others;
      }
    }
    __syncthreads();
  }
  const int n_plain = listed ? sm_count[0] : MASK ? 0 : len / kCols;
  const int n_do = listed ? n_plain + sm_count[1] : n_tiles;
  // number << 8 | class for this wave (where nobody has looked: anything) of the i-th tile to do
  auto tile_at = [&](int i) -> int {
    if (!listed) return i << 8 | (MASK ? kLive | kNonZero : kLive);
    const int e = __builtin_amdgcn_readfirstlane(sm_list[i < n_plain ? i : n_tiles - 1 - (i - n_plain)]);
    return (e & ~255) | ((e >> (2 * row_wave)) & 3);
  };

  // ---- loads ------------------------------------------------------------------
  const int64_t kv0 = static_cast<int64_t>(pair) * S * kRow;
  const char* const k_base = static_cast<const char*>(a.k) + kv0;
  const char* const v_base = static_cast<const char*>(a.v) + kv0;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char_ptr)&sm[0][0]));
  // load j of a wave has rows load_row + j kStep; below kStep and above, the row number's bits go into the
  // swizzle each by itself
  constexpr int kStep = kWavesPerGroup * kRowsPerLoad;
  const int load_row = wave * kRowsPerLoad + lane / kPieces;
  const uint32_t load_piece = 16 * ((lane % kPieces) ^ swizzle<D>(load_row));
  auto issue = [&](const char* base, int tile, uint32_t to) {
    const int left = len - 1 - tile * kCols;
    const char* from = base + static_cast<int64_t>(tile) * kTileBytes;
    to = __builtin_amdgcn_readfirstlane(to + wave * 1024);
    if (left >= kCols - 1) {
#pragma unroll
      for (int j = 0; j < kLoads; ++j) load_to_lds(from + j * kStep * kRow, load_row * kRow + (load_piece ^ 16 * swizzle<D>(j * kStep)), to + j * kWavesPerGroup * 1024);
    } else {  // rows past the slot's end repeat its last: what lies there may be anything, and 0 times NaN is NaN
#pragma unroll 1
      for (int j = 0; j < kLoads; ++j)
        load_to_lds(from, static_cast<uint32_t>(min(load_row + j * kStep, left)) * kRow + (load_piece ^ 16 * swizzle<D>(j * kStep)),
                    to + j * kWavesPerGroup * 1024);
    }
  };
  auto issue_k = [&](int tile, int buf) { issue(k_base, tile, lds0 + buf * (2 * kTileBytes)); };
  auto issue_v = [&](int tile, int buf) { issue(v_base, tile, lds0 + buf * (2 * kTileBytes) + kTileBytes); };
  // scales: thread 64 m + c of the first two waves has position c's key (m = 0) or value scale
  float scale_next = 0.f;
  auto fetch_scale = [&](int tile) {
    if (SCALE && wave < 2) {
      const int at_pos = min(tile * kCols + lane, S - 1);
      scale_next = load_as_f32(wave == 0 ? a.k_scale : a.v_scale,
                               (static_cast<int64_t>(b) * a.scale_heads + hs) * S + at_pos, SCALE == 1 ? JPT_F32 : JPT_BF16);
    }
  };
  // entries of the list: this tile's, the next one's, the one after that
  int e0 = 0, e1 = 0, e2 = 0;
  if (n_do > 0) {
    e0 = tile_at(0);
    e1 = tile_at(min(1, n_do - 1));
    issue_k(e0 >> 8, 0);
    issue_v(e0 >> 8, 0);
    if (n_do > 1) issue_k(e1 >> 8, 1);
    fetch_scale(e0 >> 8);
  }

  // ---- query rows: the second operand of S^T, lane (n, h) holds q[n][16 kk + 8 h ..] ----
  // (with their signs flipped where sm_scale is negative, so that what scores are multiplied with is not)
  bf16x8 q[kSteps];
  {
    const uint4* src = reinterpret_cast<const uint4*>(static_cast<const char*>(a.q) + q_row * kRow) + h;
    const uint32_t flip = a.sm_scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
    for (int kk = 0; kk < kSteps; ++kk) {
      const uint4 w = src[2 * kk];
      q[kk] = __builtin_bit_cast(bf16x8, make_uint4(w.x ^ flip, w.y ^ flip, w.z ^ flip, w.w ^ flip));
    }
  }

  f32x16 o[kBlocks];
#pragma unroll
  for (int d = 0; d < kBlocks; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  // The row's maximum so far in log2 units, and as the scores are (what a mask may hold does not fit log2 units);
  // what weights and sums are relative to: 2^kAhead times an earlier maximum, until the row's is above that (rows whose
  // maximum is far below: the maximum).
  float ml_run = -INFINITY, m_run = -INFINITY, ml_ref = -INFINITY, m_ref = -INFINITY;
  float l_run = 0.f;  // this lane's share of the row sum
  const float c2 = fabsf(a.sm_scale), c2l = c2 * kLog2e;

  // lane's addresses inside a tile: keys - row n, piece h; values - the transposing
  // read's row 4 h + (lane & 15) / 4 (+ 8 for the second half of a step's positions)
  uint32_t k_lane = (key0 + n) * kRow + 16 * (h ^ swizzle<D>(n));
  uint32_t v_lane[2];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    const int r = 8 * jj + 4 * h + ((lane & 15) >> 2), c = lane & 3;
    const int piece = 2 * ((lane >> 4) & 1) + (c >> 1);
    v_lane[jj] = kTileBytes + key0 * kRow + r * kRow + 16 * (piece ^ swizzle<D>(r)) + 8 * (c & 1);
  }

  // S^T of the tile in buffer `buf`, contraction steps [k_first, k_end); `beside(kk, mb)` is work for the vector ALU
  // that the matrix instructions run beside.  Operands are read from LDS two steps ahead: `ahead` holds those of
  // k_first and k_first + 1, and in the end those of k_end and k_end + 1.
  using Ahead = bf16x8[2][kKeyBlocks];
  auto operand = [&](int buf, int kk, int mb) {
    return *reinterpret_cast<const bf16x8*>(&sm[buf][0] + (k_lane ^ (32 * kk)) + 32 * mb * kRow);
  };
  auto first_operands = [&](int buf, Ahead& ahead) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int mb = 0; mb < kKeyBlocks; ++mb) ahead[kk][mb] = operand(buf, kk, mb);
  };
  auto scores = [&](int buf, f32x16 (&s)[kKeyBlocks], int k_first, int k_end, Ahead& ahead, auto beside) {
#pragma unroll
    for (int kk = k_first; kk < k_end; ++kk) {
#pragma unroll
      for (int mb = 0; mb < kKeyBlocks; ++mb) {
        s[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ahead[kk & 1][mb], q[kk], s[mb], 0, 0, 0);
        if (kk + 2 < kSteps) ahead[kk & 1][mb] = operand(buf, kk + 2, mb);
        JPT_PIN();
        beside(kk, mb);
        JPT_PIN();
      }
    }
  };
  auto clear = [](f32x16 (&s)[kKeyBlocks]) {
#pragma unroll
    for (int mb = 0; mb < kKeyBlocks; ++mb)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[mb][e] = 0.f;
  };

  // ---- softmax and products with the values of the tile in buffer `buf` ----------
  // element e of block mb is position 32 mb + 8 (e / 4) + 4 h + e % 4 of the wave's part of the tile
  constexpr int kRuns = 4 * kKeyBlocks;
  auto scale_run = [&](int buf, int u, f32x16 (&s)[kKeyBlocks], float& tmax) {  // key scales and maximum of four elements
    const int mb = u / 4, g = u % 4;
    if (SCALE) {
      const float4 ks = *reinterpret_cast<const float4*>(&sm_scale[buf][0][key0 + 32 * mb + 8 * g + 4 * h]);
      s[mb][4 * g] *= ks.x; s[mb][4 * g + 1] *= ks.y; s[mb][4 * g + 2] *= ks.z; s[mb][4 * g + 3] *= ks.w;
    }
    tmax = fmaxf(fmaxf(tmax, s[mb][4 * g]), s[mb][4 * g + 1]);
    tmax = fmaxf(fmaxf(tmax, s[mb][4 * g + 2]), s[mb][4 * g + 3]);
  };
  // Softmax weights of four positions, as three bf16 numbers each, in six parts of six to twelve instructions: run u
  // of step st, into words 2 u and 2 u + 1 of part[0..2].  `left`: positions of the wave's lane that count from here on.
  constexpr int kSlices = 12;  // a step's
  float w[4];
  auto weight_slice = [&](int buf, int st, int slice, const f32x16 (&s)[kKeyBlocks], float to_log2, float ml_use, int left,
                          uint32_t (&part)[3][4]) {
    const int u = slice / 6, e = 8 * (st & 1) + 4 * u;
    auto next_part = [&](int i) {  // number i of the three, and what it leaves
#pragma unroll
      for (int j = 0; j < 2; ++j) part[i][2 * u + j] = pack_together(w[2 * j], w[2 * j + 1]);
    };
    auto take_off = [&](int i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        w[2 * j] -= __uint_as_float(part[i][2 * u + j] << 16);
        w[2 * j + 1] -= __uint_as_float(part[i][2 * u + j] & 0xffff0000u);
      }
    };
    switch (slice % 6) {
      case 0:
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = __builtin_fmaf(s[st >> 1][e + j], to_log2, -ml_use);
        w[0] = fast_exp2(w[0]);
        w[1] = fast_exp2(w[1]);
        break;
      case 1:
        w[2] = fast_exp2(w[2]);
        w[3] = fast_exp2(w[3]);
        l_run += w[0];
        l_run += w[1];
        break;
      case 2:
        l_run += w[2];
        l_run += w[3];
        if (SCALE) {
          const int at = 16 * st + 8 * u;
          const float4 vs = *reinterpret_cast<const float4*>(&sm_scale[buf][1][key0 + 4 * h + at]);
          w[0] *= vs.x; w[1] *= vs.y; w[2] *= vs.z; w[3] *= vs.w;
          if (left < kCols) {  // a position that does not count has weight 0 whatever its scale holds
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = at + j >= left ? 0.f : w[j];
          }
        }
        next_part(0);
        break;
      case 3: take_off(0); break;
      case 4: next_part(1); break;
      default:
        take_off(1);
#pragma unroll
        for (int j = 0; j < 2; ++j) part[2][2 * u + j] = pack_bf16(w[2 * j], w[2 * j + 1]);
    }
  };
  typedef __attribute__((address_space(3))) bf16x4* lds_b4;
  auto values = [&](int buf, int st, int d) {
    const char* const at = &sm[buf][0] + 16 * st * kRow;
    const bf16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b4)(at + (v_lane[0] ^ (64 * d))));
    const bf16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b4)(at + (v_lane[1] ^ (64 * d))));
    return __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  // O^T += V^T . P^T, with the next step's weights beside this step's products
  // (values are read from LDS two blocks ahead: v_ahead holds the first two)
  auto products = [&](int buf, bf16x8 (&v_ahead)[2], uint32_t (&part)[2][3][4], auto weights) {
#pragma unroll
    for (int st = 0; st < kPvSteps; ++st) {
      bf16x8 pw[3];
#pragma unroll
      for (int i = 0; i < 3; ++i)
        pw[i] = __builtin_bit_cast(bf16x8, make_uint4(part[st & 1][i][0], part[st & 1][i][1], part[st & 1][i][2], part[st & 1][i][3]));
#pragma unroll
      for (int d = 0; d < kBlocks; ++d) {
        const bf16x8 v = v_ahead[d & 1];
        if (d + 2 < kBlocks) v_ahead[d & 1] = values(buf, st, d + 2);
        else if (st + 1 < kPvSteps) v_ahead[d & 1] = values(buf, st + 1, d + 2 - kBlocks);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, pw[i], o[d], 0, 0, 0);
          JPT_PIN();
          if (st + 1 < kPvSteps) {
#pragma unroll
            for (int u = 0; u < kSlices; ++u)
              if (u * 3 * kBlocks / kSlices == 3 * d + i) weights(st + 1, u, part[(st + 1) & 1]);
          }
          JPT_PIN();
        }
      }
    }
  };

  // A plain tile, whose products of keys and queries are in s; the next tile's, from the other buffer into s_next,
  // run beside its softmax.  (Behind the last tile there are none, and what comes of the keys there is not looked at.)
  auto attend_plain = [&](int buf, f32x16 (&s)[kKeyBlocks], f32x16 (&s_next)[kKeyBlocks], Ahead& ahead) {
    constexpr int kHalf = kSteps / 2;
    float tmax = -INFINITY;
    clear(s_next);
    scores(buf ^ 1, s_next, 0, kHalf, ahead, [&](int kk, int mb) {
      const int at = kk * kKeyBlocks + mb, n_at = kHalf * kKeyBlocks;
#pragma unroll
      for (int u = 0; u < kRuns; ++u)
        if (u * n_at / kRuns == at) scale_run(buf, u, s, tmax);
    });
    tmax = fmaxf(tmax, other_half(tmax));
    ml_run = fmaxf(ml_run, tmax * c2l);
    if (MASK) m_run = fmaxf(m_run, tmax * c2);
    // (a loop of one turn: behind a branch the compiler would have o in two places, and move it at every tile)
    for (int turn = __any(ml_run > ml_ref) ? 1 : 0; turn; turn = nothing()) {
      const float alpha = fast_exp2(ml_ref - (ml_run == -INFINITY ? 0.f : ml_run + kAhead));
      ml_ref = ml_run + kAhead;
      m_ref = m_run;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < kBlocks; ++d) o[d] *= alpha;
    }
    const float ml_use = ml_ref == -INFINITY ? 0.f : ml_ref;
    uint32_t part[2][3][4];
    bf16x8 v_ahead[2] = {values(buf, 0, 0), values(buf, 0, 1)};
    // the first step's weights beside the rest of the next tile's scores
    scores(buf ^ 1, s_next, kHalf, kSteps, ahead, [&](int kk, int mb) {
      const int at = (kk - kHalf) * kKeyBlocks + mb, n_at = kHalf * kKeyBlocks;
#pragma unroll
      for (int u = 0; u < kSlices; ++u)
        if (u * n_at / kSlices == at) weight_slice(buf, 0, u, s, c2l, ml_use, kCols, part[0]);
    });
    products(buf, v_ahead, part, [&](int st, int u, uint32_t (&to)[3][4]) { weight_slice(buf, st, u, s, c2l, ml_use, kCols, to); });
  };

  // Any other tile.
  auto attend = [&](int entry, int buf, f32x16 (&s)[kKeyBlocks]) {
    const int tile = entry >> 8;
    const int pos0 = tile * kCols + key0 + 4 * h, left = len - pos0;
    const bool tail = tile * kCols + kCols > len;
    float tmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < kRuns; ++u) scale_run(buf, u, s, tmax);
    if (MASK && (entry & kNonZero)) {
      using M = std::conditional_t<MASK == 1, float, uint16_t>;
      const M* const mrow = static_cast<const M*>(a.mask) + b * a.mask_stride_b + q_head * a.mask_stride_h + t * a.mask_stride_t + pos0;
      auto as_f32 = [](M x) {
        if constexpr (MASK == 1) return x;
        else return bf16_bits_to_f32(x);
      };
#pragma unroll
      for (int mb = 0; mb < kKeyBlocks; ++mb) {
        float mk[16];
        if (tail) {
#pragma unroll
          for (int e = 0; e < 16; ++e) mk[e] = as_f32(mrow[min(32 * mb + 8 * (e / 4) + e % 4, S - 1 - pos0)]);
        } else if (p.mask_runs) {  // four positions a load
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            if constexpr (MASK == 1) {
              const float4 x = *reinterpret_cast<const float4*>(mrow + 32 * mb + 8 * g);
              mk[4 * g] = x.x; mk[4 * g + 1] = x.y; mk[4 * g + 2] = x.z; mk[4 * g + 3] = x.w;
            } else {
              const uint2 x = *reinterpret_cast<const uint2*>(mrow + 32 * mb + 8 * g);
              mk[4 * g] = __uint_as_float(x.x << 16); mk[4 * g + 1] = __uint_as_float(x.x & 0xffff0000u);
              mk[4 * g + 2] = __uint_as_float(x.y << 16); mk[4 * g + 3] = __uint_as_float(x.y & 0xffff0000u);
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 16; ++e) mk[e] = as_f32(mrow[32 * mb + 8 * (e / 4) + e % 4]);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) s[mb][e] = s[mb][e] * c2 + mk[e];
      }
    } else {
#pragma unroll
      for (int mb = 0; mb < kKeyBlocks; ++mb) s[mb] *= c2;
    }
    // s now holds scores as they are; positions past the end do not count
    tmax = -INFINITY;
#pragma unroll
    for (int mb = 0; mb < kKeyBlocks; ++mb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if (tail) s[mb][e] = 32 * mb + 8 * (e / 4) + e % 4 >= left ? -INFINITY : s[mb][e];
        tmax = fmaxf(tmax, s[mb][e]);
      }
    tmax = fmaxf(tmax, other_half(tmax));
    ml_run = fmaxf(ml_run, tmax * kLog2e);
    float ml_use = ml_ref == -INFINITY ? 0.f : ml_ref, to_log2 = kLog2e;
    bool move = ml_run > ml_ref;
    if (MASK) {
      m_run = fmaxf(m_run, tmax);
      move = move || m_run < kFarBelow;
    }
    if (__any(move)) {
      ml_use = ml_run == -INFINITY ? 0.f : ml_run + kAhead;
      float alpha = fast_exp2(ml_ref - ml_use);
      ml_ref = ml_run + kAhead;
      if (MASK) {
        // Rows whose largest score is near float32's lowest value (a mask may hold that): times log2(e) it may be
        // -infinity, and a row masked throughout would be empty instead of the mean of the values.
        if (__any(m_run < kFarBelow)) {
          const bool far = m_run < kFarBelow;
          const float m_use = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
          for (int mb = 0; mb < kKeyBlocks; ++mb)
#pragma unroll
            for (int e = 0; e < 16; ++e) s[mb][e] = far ? (s[mb][e] - m_use) * kLog2e : __builtin_fmaf(s[mb][e], kLog2e, -ml_use);
          alpha = far ? fast_exp2((m_ref - m_use) * kLog2e) : alpha;
          to_log2 = 1.f;
          ml_use = 0.f;
        }
        m_ref = m_run;
      }
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < kBlocks; ++d) o[d] *= alpha;
    }
    uint32_t part[2][3][4];
    const int counts = tail ? left : kCols;
    bf16x8 v_ahead[2] = {values(buf, 0, 0), values(buf, 0, 1)};
#pragma unroll
    for (int u = 0; u < kSlices; ++u) weight_slice(buf, 0, u, s, to_log2, ml_use, counts, part[0]);
    products(buf, v_ahead, part, [&](int st, int u, uint32_t (&to)[3][4]) { weight_slice(buf, st, u, s, to_log2, ml_use, counts, to); });
  };

  // While a plain tile's softmax runs in the vector ALU the matrix cores do the next tile's scores: tile i + 1's keys
  // and tile i's values are the ones that have to be there, and both have had a whole tile's time to come.
  f32x16 s[kKeyBlocks], s_next[kKeyBlocks];
  Ahead ahead;
  auto only_scores = [&](int buf, f32x16 (&to)[kKeyBlocks]) {
    first_operands(buf, ahead);
    clear(to);
    scores(buf, to, 0, kSteps, ahead, [](int, int) {});
  };
  clear(s);
  if (n_do > 0) {
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    __syncthreads();
    only_scores(0, s);
  }
  int i = 0;
  auto arrive = [&](int buf, bool plain) {
    asm volatile("" : "+v"(k_lane), "+v"(v_lane[0]), "+v"(v_lane[1]));  // addresses made of them are not to be kept across tiles
    if (SCALE && wave < 2) sm_scale[buf][wave][lane] = scale_next;
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wave's share of what was asked for is in LDS ...
    __syncthreads();                                    // ... and everybody's; what the last tile read is free
    if (plain) first_operands(buf ^ 1, ahead);
    if (i + 1 < n_do) {
      issue_v(e1 >> 8, buf ^ 1);
      fetch_scale(e1 >> 8);
      e2 = tile_at(min(i + 2, n_do - 1));
      if (i + 2 < n_do) issue_k(e2 >> 8, buf);
    }
    e0 = e1;
    e1 = e2;
    ++i;
  };
  while (i + 1 < n_plain) {  // two tiles a turn: s and s_next change places
    arrive(0, true);
    attend_plain(0, s, s_next, ahead);
    arrive(1, true);
    attend_plain(1, s_next, s, ahead);
  }
  if (i < n_plain) {
    arrive(0, true);
    attend_plain(0, s, s_next, ahead);
#pragma unroll
    for (int mb = 0; mb < kKeyBlocks; ++mb) s[mb] = s_next[mb];
  }
  while (i < n_do) {
    const int entry = e0, buf = i & 1;
    arrive(buf, false);
    if (entry & kLive) attend(entry, buf, s);  // or else nothing of this tile counts for this wave's rows
    if (i < n_do) only_scores(buf ^ 1, s);
  }

  float l = l_run + other_half(l_run);
  if constexpr (KEY_WAVES > 1) {
    // The waves of one row block, each with its part of every tile's positions, fold their parts: a wave
    // gets the others' accumulators of its own share of the O^T blocks.
    constexpr int kOwn = kBlocks / KEY_WAVES;
    static_assert(KEY_WAVES <= 2 && kBlocks % KEY_WAVES == 0 && sizeof(sm) >= kWavesPerGroup * kOwn * 4096 + kWavesPerGroup * 512, "");
    float* const parts = reinterpret_cast<float*>(&sm[0][0]);
    float* const stats = parts + kWavesPerGroup * kOwn * 1024;  // a wave's 32 references, maxima (both units) and sums
    const int me = wave / kRowWaves, other = wave ^ kRowWaves;
    __syncthreads();  // the tiles have been read
#pragma unroll
    for (int d = 0; d < kOwn; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = me == 0 ? o[kOwn + d][4 * g + i] : o[d][4 * g + i];
        *reinterpret_cast<float4*>(&parts[((wave * kOwn + d) * 4 + g) * 256 + 4 * lane]) = make_float4(x[0], x[1], x[2], x[3]);
      }
    if (h == 0) {
      stats[wave * 128 + n] = ml_ref;
      stats[wave * 128 + 32 + n] = ml_run;
      stats[wave * 128 + 64 + n] = m_run;
      stats[wave * 128 + 96 + n] = l;
    }
    __syncthreads();
    const float ref2 = stats[other * 128 + n], ml2 = stats[other * 128 + 32 + n], m2 = stats[other * 128 + 64 + n], l2 = stats[other * 128 + 96 + n];
    ml_run = fmaxf(ml_run, ml2);
    const float ml_use = ml_run == -INFINITY ? 0.f : ml_run;
    float f1 = fast_exp2(ml_ref - ml_use), f2 = fast_exp2(ref2 - ml_use);
    const float m_all = fmaxf(m_run, m2);
    if (MASK && m_all < kFarBelow) {
      const float m_use = m_all == -INFINITY ? 0.f : m_all;
      f1 = fast_exp2((m_run - m_use) * kLog2e);
      f2 = fast_exp2((m2 - m_use) * kLog2e);
    }
    m_run = m_all;
    l = l * f1 + l2 * f2;
#pragma unroll
    for (int d = 0; d < kOwn; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 x = *reinterpret_cast<const float4*>(&parts[((other * kOwn + d) * 4 + g) * 256 + 4 * lane]);
        const float theirs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)  // (a wave's own share is moved to the front)
          o[d][4 * g + i] = (me == 0 ? o[d][4 * g + i] : o[kOwn + d][4 * g + i]) * f1 + theirs[i] * f2;
      }
  }
  const float l_out = KEY_WAVES > 1 || (MASK && m_run < kFarBelow) || ml_run == -INFINITY ? l : l * fast_exp2(ml_ref - ml_run);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (!row_live) return;
  constexpr int kOut = kBlocks / KEY_WAVES;
  const int first = KEY_WAVES > 1 ? wave / kRowWaves * kOut : 0;
  char* dst = static_cast<char*>(a.out) + q_row * kRow + 64 * first + 8 * h;
#pragma unroll
  for (int d = 0; d < kOut; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2*>(dst + 64 * d + 16 * g) =
          make_uint2(pack_bf16(o[d][4 * g] * inv, o[d][4 * g + 1] * inv), pack_bf16(o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv));
  if (h == 0 && first == 0) {
    if (a.out_max) a.out_max[q_row] = MASK ? m_run : ml_run * kLn2;
    if (a.out_denom) a.out_denom[q_row] = l_out;
  }
}

// A wave takes one block of 32 mask rows x 64 positions, BYTES a load, every load asked for before the first is
// looked at; four blocks side by side a workgroup.  Bound by the trip to memory: 3500 rows
// of bf16 (8 bytes a load) 8.0 -> 6.4 us, 1024 rows (16) 4.6 -> 3.7, where a load was one value.
template <typename M, int BYTES>
__global__ void __launch_bounds__(256)
mask_class_kernel(const M* mask, int64_t stride_b, int64_t stride_h, int64_t stride_t, int rows, int cols, int heads,
                  uint8_t* classes, int row_blocks, int col_blocks) {
  constexpr int kEach = BYTES / static_cast<int>(sizeof(M));           // values a load
  constexpr int kLanes = kCols / kEach;                                // lanes a row
  constexpr int kLoads = kWaveRows * kLanes / 64;
  constexpr int kWords = BYTES < 4 ? 1 : BYTES / 4;
  // of a word of two bf16 values, one bf16 value or one float: -infinity everywhere, zero everywhere
  constexpr uint32_t kMinusInf = sizeof(M) == 4 ? 0xff800000u : BYTES < 4 ? 0xff80u : 0xff80ff80u;
  constexpr uint32_t kMagnitude = sizeof(M) == 4 ? 0x7fffffffu : BYTES < 4 ? 0x7fffu : 0x7fff7fffu;
  const int b = blockIdx.z / heads, hh = blockIdx.z % heads;
  const int lane = threadIdx.x & 63, cb = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (cb >= col_blocks) return;
  const int r0 = blockIdx.y * kWaveRows;
  const int c = cb * kCols + lane % kLanes * kEach;
  const M* const src = mask + b * stride_b + hh * stride_h + r0 * stride_t;
  auto row_of = [&](int j) { return static_cast<int64_t>(min(j * (64 / kLanes) + lane / kLanes, rows - 1 - r0)) * stride_t; };
  bool live = false, nonzero = false;
  if (c + kEach <= cols) {
    uint32_t w[kLoads][kWords];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const M* at = src + row_of(j) + c;
      if constexpr (BYTES == 16) {
        const uint4 x = *reinterpret_cast<const uint4*>(at);
        w[j][0] = x.x; w[j][1] = x.y; w[j][2] = x.z; w[j][3] = x.w;
      } else if constexpr (BYTES == 8) {
        const uint2 x = *reinterpret_cast<const uint2*>(at);
        w[j][0] = x.x; w[j][1] = x.y;
      } else {
        w[j][0] = static_cast<uint32_t>(*at);
      }
    }
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
#pragma unroll
      for (int i = 0; i < kWords; ++i) {
        live = live || w[j][i] != kMinusInf;  // a NaN counts
        nonzero = nonzero || (w[j][i] & kMagnitude) != 0;
      }
  } else {  // across the end of the row, or past it
    constexpr uint32_t kOneInf = sizeof(M) == 4 ? 0xff800000u : 0xff80u, kOneMagnitude = sizeof(M) == 4 ? 0x7fffffffu : 0x7fffu;
    for (int j = 0; j < kLoads; ++j)
      for (int i = 0; i < kEach && c + i < cols; ++i) {
        const uint32_t x = src[row_of(j) + c + i];
        live = live || x != kOneInf;
        nonzero = nonzero || (x & kOneMagnitude) != 0;
      }
  }
  const bool any_live = __any(live), any_nonzero = __any(nonzero);
  if (lane == 0)
    classes[(static_cast<int64_t>(blockIdx.z) * row_blocks + blockIdx.y) * col_blocks + cb] =
        static_cast<uint8_t>((any_live ? kLive : 0) | (any_nonzero ? kNonZero : 0));
}

// Mask blocks of a call: one mask a (batch, head) that has one of its own.
struct Classes {
  int64_t bytes;
  int32_t batches, heads, row_blocks, col_blocks;
};
Classes mask_classes(const jpt_attn_args& a) {
  Classes c;
  c.batches = a.mask_stride_b != 0 ? a.batch : 1;
  c.heads = a.mask_stride_h != 0 ? a.q_heads : 1;
  c.row_blocks = (a.q_rows + kWaveRows - 1) / kWaveRows;
  c.col_blocks = (a.seq + kCols - 1) / kCols;
  c.bytes = static_cast<int64_t>(c.batches) * c.heads * c.row_blocks * c.col_blocks;
  return c;
}

// Is a pass over the mask worth its launch (4 us for 1024 rows, 6 for 3500)?  Where it can leave out tiles: with one row
// tile and a handful of key tiles there is nothing to leave out that would pay for it.
bool classes_pay(const jpt_attn_args& a) {
  if (a.mask == nullptr || a.q_rows < kRowsPerGroup || a.seq < 256 || a.seq > kMaxTiles * kCols) return false;
  const Classes c = mask_classes(a);
  return c.row_blocks <= 65535 && static_cast<int64_t>(c.batches) * c.heads <= 65535;  // what a grid can count
}

// Four waves over 128 query rows, or two and two over 64 rows and the halves of a tile's positions: twice the
// workgroups, each half as long, but keys and values are read twice as often.  That is the faster way where workgroups of
// 128 would leave places empty (two a compute unit, one at heads of 256), or be a few more than there are: the longest
// workgroup, or the second round of them, is the launch.  Under a mask workgroups are of unequal length, and halves pay
// for longer.  us a call, 1 / 2 key waves, by workgroups of 128 over 256 compute units -
//   128, mask (causal): 128 23.7 / 18.9, 256 37.6 / 30.8, 384 55.3 / 53.5, 448 66.6 / 66.8 and 116.7 / 113.9 (8 and 16 KV
//     heads), 480 73.6 / 72.2, 512 79.1 / 80.5 (all places, once), 544 88.3 / 87.8 and 99 / 90 (8 and 32), 576 95.2 / 96.9 and
//     106.4 / 103.0, 608 111.3 / 113.2, 640 112 / 116;
//   128, none: 128 19.3 / 15.5, 256 39.7 / 40.6, 384 78.5 / 78.1, 448 94 / 109, 512 116 / 130, 544 164 / 162, 608 184 / 184;
//   64, mask: 256 28.9 / 23.0, 448 44.4 / 39.7, 512 53.5 / 49.7, 576 63.1 / 59.2, 640 72.5 / 69.2, 768 95.7 / 94.6;
//   64, none: 128 13.7 / 11.0, 384 50.8 / 46.7, 448 59.7 / 65.9, 512 70.8 / 76.4, 576 109 / 100, 640 122 / 114, 768 153 / 161;
//   256, mask: 128 58.4 / 41.8, 256 105 / 86, 288 118 / 116, 320 131 / 136, 448 205 / 232;
//   256, none: 128 56.2 / 41.1, 192 84 / 101, 256 121 / 138, 288 228 / 213, 320 252 / 235, 448 363 / 434.
// One block of 32 positions has no halves.
int32_t key_waves_for(const jpt_attn_args& a, int64_t workgroups) {
  const int64_t places = static_cast<int64_t>(a.dim == 256 ? 1 : 2) * compute_units();
  bool halves;
  if (workgroups > places) halves = a.dim == 128 ? 8 * workgroups <= 9 * places : 4 * workgroups <= 5 * places;
  else if (a.mask != nullptr) halves = a.dim != 128 || workgroups < places;
  else halves = a.dim == 256 ? 2 * workgroups <= places : 4 * workgroups <= 3 * places;
  return a.seq > 32 && halves ? 2 : 1;
}

template <int D, int SCALE, int MASK>
void launch_waves(const PrefillParams& p, dim3 grid, hipStream_t stream) {
  const dim3 block(64 * kWavesPerGroup);
  if (p.key_waves == 1) hipLaunchKernelGGL((attn_prefill_kernel<D, SCALE, MASK, 1>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((attn_prefill_kernel<D, SCALE, MASK, 2>), grid, block, 0, stream, p);
}

template <int D, int SCALE>
void launch_mask(const PrefillParams& p, dim3 grid, hipStream_t stream) {
  if (!p.a.mask) launch_waves<D, SCALE, 0>(p, grid, stream);
  else if (p.a.mask_dtype == JPT_F32) launch_waves<D, SCALE, 1>(p, grid, stream);
  else launch_waves<D, SCALE, 2>(p, grid, stream);
}

template <int D>
void launch_dim(const PrefillParams& p, dim3 grid, hipStream_t stream) {
  if (!p.a.k_scale) launch_mask<D, 0>(p, grid, stream);
  else if (p.a.scale_dtype == JPT_F32) launch_mask<D, 1>(p, grid, stream);
  else launch_mask<D, 2>(p, grid, stream);
}

// The mask's pass with the widest loads that its pointer and strides allow.
template <typename M>
void launch_classes(const PrefillParams& p, const Classes& c, uint8_t* classes, hipStream_t stream) {
  const jpt_attn_args& a = p.a;
  const dim3 grid((c.col_blocks + 3) / 4, c.row_blocks, c.batches * c.heads);
  auto fits = [&](int bytes) {
    const int each = bytes / static_cast<int>(sizeof(M));
    return aligned(a.mask, bytes) && a.mask_stride_b % each == 0 && a.mask_stride_h % each == 0 && a.mask_stride_t % each == 0;
  };
  const M* mask = static_cast<const M*>(a.mask);
#define JPT_CLASSES(BYTES)                                                                                              \
  hipLaunchKernelGGL((mask_class_kernel<M, BYTES>), grid, dim3(256), 0, stream, mask, a.mask_stride_b, a.mask_stride_h, \
                     a.mask_stride_t, a.q_rows, a.seq, c.heads, classes, c.row_blocks, c.col_blocks)
  if (fits(16)) JPT_CLASSES(16);
  else if (fits(8)) JPT_CLASSES(8);
  else JPT_CLASSES(static_cast<int>(sizeof(M)));
#undef JPT_CLASSES
}

}  // namespace

bool attn_prefill_supported(const jpt_attn_args& a, AttnMode mode) {
  if (a.force_generic || mode == kPaged || a.new_k) return false;
  if (a.q_dtype != JPT_BF16 || a.kv_dtype != JPT_BF16) return false;
  if (a.dim != 64 && a.dim != 128 && a.dim != 256) return false;
  if (!aligned(a.q, 16) || !aligned(a.k, 16) || !aligned(a.v, 16) || !aligned(a.out, 8)) return false;
  const int64_t rep = a.q_heads / a.kv_heads;
  if (rep * a.q_rows > (1ll << 30) || a.seq > (1ll << 24)) return false;
  return true;
}

int64_t attn_prefill_workspace_bytes(const jpt_attn_args& a) {
  if (!classes_pay(a)) return 0;
  return mask_classes(a).bytes;
}

int32_t attn_prefill_launch(const jpt_attn_args& a, hipStream_t stream) {
  PrefillParams p{};
  p.a = a;
  const int rep = a.q_heads / a.kv_heads;
  // short prompts: the rows of all query heads of a KV head side by side; else head by head
  const bool folded = a.q_rows < kRowsPerGroup;
  p.groups = folded ? 1 : rep;
  p.group_rows = folded ? rep * a.q_rows : a.q_rows;
  const int64_t pairs = static_cast<int64_t>(a.batch) * a.kv_heads;
  p.key_waves = key_waves_for(a, pairs * p.groups * ((p.group_rows + kRowsPerGroup - 1) / kRowsPerGroup));
  const int rows = kRowsPerGroup / p.key_waves;
  p.tiles = (p.group_rows + rows - 1) / rows;
  p.by_rows = pairs / 8 * 2 * a.seq * a.dim * 2 <= kL2Bytes;
  const int mask_run = a.mask_dtype == JPT_F32 ? 16 : 8;
  p.mask_runs = a.mask != nullptr && aligned(a.mask, mask_run) && a.mask_stride_b % 4 == 0 && a.mask_stride_h % 4 == 0 && a.mask_stride_t % 4 == 0;
  if (classes_pay(a)) {
    const Classes c = mask_classes(a);
    // without a workspace (it is the caller's to give) every block is taken to hold anything
    if (a.workspace != nullptr && a.workspace_bytes >= attn_partials_offset(a) + c.bytes) {
      uint8_t* classes = reinterpret_cast<uint8_t*>(attn_workspace_end(a, c.bytes));
      p.classes = classes;
      p.row_blocks = c.row_blocks;
      p.col_blocks = c.col_blocks;
      const int64_t one = static_cast<int64_t>(c.row_blocks) * c.col_blocks;
      p.class_stride_h = c.heads > 1 ? one : 0;
      p.class_stride_b = c.batches > 1 ? one * c.heads : 0;
      if (a.mask_dtype == JPT_F32) launch_classes<uint32_t>(p, c, classes, stream);
      else launch_classes<uint16_t>(p, c, classes, stream);
      const int32_t st = launch_status("mask_class_kernel");
      if (st != JPT_OK) return st;
    }
  }
  const int64_t blocks = static_cast<int64_t>(a.batch) * a.kv_heads * p.groups * p.tiles;
  JPT_REQUIRE(blocks < (1ll << 31), "too many query rows");
  const dim3 grid(static_cast<unsigned>(blocks));
  if (a.dim == 64) launch_dim<64>(p, grid, stream);
  else if (a.dim == 128) launch_dim<128>(p, grid, stream);
  else launch_dim<256>(p, grid, stream);
  return launch_status("attn_prefill_kernel");
}

}  // namespace jpt
