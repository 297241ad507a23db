// Attention of many query rows over bf16 keys and values (prefill, and any dense
// call whose query rows are too many for the streaming decode kernel), head_dim
// 64, 128 or 256, on the matrix cores.
//
// One workgroup of four waves takes 128 query rows of one KV head and walks the
// keys in tiles of 64 positions.  Tiles go from memory straight into LDS (two
// buffers: the next tile's loads are in flight while this one is worked on);
// a wave holds 32 query rows and runs
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
// third numbers, and the vector ALU's exponentials and splits beside it.  Neither
// is the bound: of 3500 rows' SIMD time the vector ALU issues in 53 %, the matrix
// pipe is busy in 38 %, and the waves of a workgroup meet at every tile; 1024 rows
// are 256 workgroups of unequal length, one wave a SIMD, which half the SIMD time
// have ended: 18 and 14 %.
// What a causal mask leaves out is not computed: a pass over the mask (read
// once, not once a head) first writes down, for every 32 rows x 64 positions,
// whether anything there is live and whether anything there is not zero; dead
// tiles are neither loaded nor computed, and all-zero tiles need no mask reads.
//
// Measured, causal, 32 query heads over 8 KV heads of 128, a call with its pass over
// the mask, calls back to back: 1024 rows 48 us (12.3 ms for the shape-generic
// kernel, one wave a row, scalar dot products), 3500 rows with scales 241 us (171 ms);
// with weights of two bf16 numbers, 16 bits, they would be 41 and 199 us.  Outputs
// that are not the rounded exact value: 0.025 % (shape-generic 0.034 %, 16 bits 0.21 %).
#include <math.h>

#include "attn_common.h"

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
__device__ __forceinline__ int swizzle(int t) {
  return D == 64 ? (((t >> 1) & 1) << 2) | ((t >> 2) & 3) : ((t & 3) << 2) | ((t >> 2) & 3);
}

template <int D, int SCALE, int MASK>
__global__ void __launch_bounds__(64 * kWavesPerGroup, D == 256 ? 1 : 2) attn_prefill_kernel(PrefillParams p) {
  const jpt_attn_args& a = p.a;
  constexpr int kRow = D * 2;                  // bytes of a row
  constexpr int kPieces = kRow / 16;
  constexpr int kTileBytes = kCols * kRow;     // keys or values of a tile
  constexpr int kRowsPerLoad = 1024 / kRow;    // rows of one wave-wide load
  constexpr int kLoads = kTileBytes / 1024 / kWavesPerGroup;  // loads a wave makes for the keys, and for the values
  constexpr int kSteps = D / 16;               // contraction steps of S^T
  constexpr int kBlocks = D / 32;              // row blocks of O^T
  __shared__ __attribute__((aligned(1024))) char sm[2][2 * kTileBytes];
  __shared__ float sm_scale[2][2][kCols];      // key and value scales of a tile
  __shared__ int sm_list[MASK ? kMaxTiles : 1];  // tiles to do: number << 8 | two class bits a wave
  __shared__ int sm_count;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int T = a.q_rows, S = a.seq;
  const int rep = a.q_heads / a.kv_heads;

  // Workgroups go round the XCDs: all row tiles of one KV head on one XCD, whose
  // L2 then holds the head's keys and values; last rows first, which under a
  // causal mask have the most to do.
  const int pairs = a.batch * a.kv_heads, per_pair = p.groups * p.tiles;
  int pair, at;
  if (pairs % 8 == 0) {
    const int i = blockIdx.x >> 3;
    pair = (blockIdx.x & 7) + 8 * (i / per_pair);
    at = i % per_pair;
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
  const int row0 = tile_row * kRowsPerGroup + wave * kWaveRows;
  const int row = row0 + n;
  const bool row_live = row < p.group_rows;
  const int row_in = row_live ? row : p.group_rows - 1;
  const int q_head = hkv * rep + (p.groups == 1 ? row_in / T : group);
  const int t = p.groups == 1 ? row_in % T : row_in;
  const int64_t q_row = (static_cast<int64_t>(b) * a.q_heads + q_head) * T + t;

  // ---- which tiles there are to do -------------------------------------------
  const int n_tiles = (len + kCols - 1) / kCols;
  const bool listed = MASK && p.classes != nullptr;
  if (listed) {
    if (wave == 0) {
      // (the rows of one wave lie in one row block: row tiles start at multiples of 128)
      const uint8_t* cls = p.classes + b * p.class_stride_b + (hkv * rep + group) * p.class_stride_h +
                           static_cast<int64_t>(tile_row) * kWavesPerGroup * p.col_blocks;
      int count = 0;
      for (int c0 = 0; c0 < n_tiles; c0 += 64) {
        const int c = c0 + lane;
        int bits = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerGroup; ++w)
          if (c < n_tiles && tile_row * kWavesPerGroup + w < p.row_blocks)
            bits |= cls[static_cast<int64_t>(w) * p.col_blocks + c] << (2 * w);
        const bool live = (bits & 0x55 * kLive) != 0;
        const uint64_t set = __ballot(live);
        if (live) sm_list[count + __popcll(set & ((1ull << lane) - 1))] = c << 8 | bits;
        count += __popcll(set);
      }
      if (lane == 0) sm_count = count;
    }
    __syncthreads();
  }
  const int n_do = listed ? sm_count : n_tiles;
  // tile number << 8 | its class for this wave (where nobody has looked: anything)
  auto tile_at = [&](int i) -> int {
    if (!listed) return i << 8 | (MASK ? kLive | kNonZero : kLive);
    const int e = __builtin_amdgcn_readfirstlane(sm_list[i]);
    return (e & ~255) | ((e >> (2 * wave)) & 3);
  };

  // ---- loads ------------------------------------------------------------------
  const int64_t kv0 = static_cast<int64_t>(pair) * S * kRow;
  const char* const k_base = static_cast<const char*>(a.k) + kv0;
  const char* const v_base = static_cast<const char*>(a.v) + kv0;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char_ptr)&sm[0][0]));
  auto issue = [&](int tile, int buf) {
    // rows past the slot's end repeat its last: what lies there may be anything, and 0 times NaN is NaN
    const int left = len - 1 - tile * kCols;
    const char* kt = k_base + static_cast<int64_t>(tile) * kTileBytes;
    const char* vt = v_base + static_cast<int64_t>(tile) * kTileBytes;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int c = j * kWavesPerGroup + wave;
      const int r = c * kRowsPerLoad + lane / kPieces;
      const uint32_t off = static_cast<uint32_t>(min(r, left)) * kRow + 16 * ((lane % kPieces) ^ swizzle<D>(r));
      const uint32_t to = lds0 + buf * (2 * kTileBytes) + c * 1024;
      load_to_lds(kt, off, to);
      load_to_lds(vt, off, to + kTileBytes);
    }
  };
  // scales: thread 64 m + c of the first two waves has position c's key (m = 0) or value scale
  float scale_next = 0.f;
  auto fetch_scale = [&](int tile) {
    if (SCALE && wave < 2) {
      const int at_pos = min(tile * kCols + lane, S - 1);
      scale_next = load_as_f32(wave == 0 ? a.k_scale : a.v_scale,
                               (static_cast<int64_t>(b) * a.scale_heads + hs) * S + at_pos, SCALE == 1 ? JPT_F32 : JPT_BF16);
    }
  };

  // ---- query rows: the second operand of S^T, lane (n, h) holds q[n][16 kk + 8 h ..] ----
  bf16x8 q[kSteps];
  {
    const uint4* src = reinterpret_cast<const uint4*>(static_cast<const char*>(a.q) + q_row * kRow) + h;
#pragma unroll
    for (int kk = 0; kk < kSteps; ++kk) q[kk] = __builtin_bit_cast(bf16x8, src[2 * kk]);
  }

  f32x16 o[kBlocks];
#pragma unroll
  for (int d = 0; d < kBlocks; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this lane's share of the row sum
  // Scores in log2 units - but where a mask is added, which may be float32's lowest value: that times
  // log2(e) would be -infinity, and a row masked throughout empty instead of the mean of the values.
  const float c2 = MASK ? a.sm_scale : a.sm_scale * kLog2e;
  auto weight_of = [](float above_max) { return fast_exp2(MASK ? above_max * kLog2e : above_max); };

  // lane's addresses inside a tile: keys - row n, piece h; values - the transposing
  // read's row 4 h + (lane & 15) / 4 (+ 8 for the second half of a step's positions)
  const uint32_t k_lane = n * kRow + 16 * (h ^ swizzle<D>(n));
  uint32_t v_lane[2];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    const int r = 8 * jj + 4 * h + ((lane & 15) >> 2), c = lane & 3;
    const int piece = 2 * ((lane >> 4) & 1) + (c >> 1);
    v_lane[jj] = kTileBytes + r * kRow + 16 * (piece ^ swizzle<D>(r)) + 8 * (c & 1);
  }

  if (n_do > 0) {
    const int first = tile_at(0) >> 8;
    issue(first, 0);
    fetch_scale(first);
  }
  for (int i = 0; i < n_do; ++i) {
    const int entry = tile_at(i), tile = entry >> 8, cls = entry & 255, buf = i & 1;
    if (SCALE && wave < 2) sm_scale[buf][wave][lane] = scale_next;
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wave's share of the tile is in LDS ...
    __syncthreads();                                    // ... and everybody's; the other buffer is free
    if (i + 1 < n_do) {
      const int next = tile_at(i + 1) >> 8;
      issue(next, buf ^ 1);
      fetch_scale(next);
    }
    if (!(cls & kLive)) continue;  // nothing of this tile counts for this wave's rows
    const char* const at_tile = &sm[buf][0];

    f32x16 s[2];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[mb][e] = 0.f;
    }
#pragma unroll
    for (int kk = 0; kk < kSteps; ++kk) {
      const char* src = at_tile + (k_lane ^ (32 * kk));
      const bf16x8 k0 = *reinterpret_cast<const bf16x8*>(src);
      const bf16x8 k1 = *reinterpret_cast<const bf16x8*>(src + 32 * kRow);
      s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k0, q[kk], s[0], 0, 0, 0);
      s[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k1, q[kk], s[1], 0, 0, 0);
    }
    // element e of block mb is position 32 mb + 8 (e / 4) + 4 h + e % 4 of the tile
    const int pos0 = tile * kCols + 4 * h;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[mb][e] *= c2;
    if (SCALE) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 ks = *reinterpret_cast<const float4*>(&sm_scale[buf][0][32 * mb + 8 * g + 4 * h]);
          s[mb][4 * g] *= ks.x; s[mb][4 * g + 1] *= ks.y; s[mb][4 * g + 2] *= ks.z; s[mb][4 * g + 3] *= ks.w;
        }
    }
    if (MASK && (cls & kNonZero)) {
      const int64_t mrow = b * a.mask_stride_b + q_head * a.mask_stride_h + t * a.mask_stride_t;
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int at_pos = min(pos0 + 32 * mb + 8 * (e / 4) + e % 4, S - 1);
          s[mb][e] += load_as_f32(a.mask, mrow + at_pos, MASK == 1 ? JPT_F32 : JPT_BF16);
        }
    }
    if (tile * kCols + kCols > len) {  // the last tile's positions past the end
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (pos0 + 32 * mb + 8 * (e / 4) + e % 4 >= len) s[mb][e] = -INFINITY;
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int e = 0; e < 16; ++e) tmax = fmaxf(tmax, s[mb][e]);
    tmax = fmaxf(tmax, other_half(tmax));
    const float m_new = fmaxf(m_run, tmax);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = weight_of(m_run - m_use);
    m_run = m_new;
    l_run *= alpha;
    if (__any(alpha != 1.f)) {
#pragma unroll
      for (int d = 0; d < kBlocks; ++d) o[d] *= alpha;
    }
#pragma unroll
    for (int st = 0; st < kCols / 16; ++st) {  // 16 positions a step
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        w[j] = weight_of(s[st >> 1][8 * (st & 1) + j] - m_use);
        l_run += w[j];
      }
      if (SCALE) {
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          const float4 vs = *reinterpret_cast<const float4*>(&sm_scale[buf][1][16 * st + 8 * jj + 4 * h]);
          w[4 * jj] *= vs.x; w[4 * jj + 1] *= vs.y; w[4 * jj + 2] *= vs.z; w[4 * jj + 3] *= vs.w;
        }
        if (tile * kCols + kCols > len) {  // a position that does not count has weight 0 whatever its scale holds
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (pos0 + 16 * st + 8 * (j / 4) + j % 4 >= len) w[j] = 0.f;
        }
      }
      uint32_t part[3][4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float x = w[2 * j], y = w[2 * j + 1];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const uint32_t both = part[i][j] = pack_bf16(x, y);
          x -= __uint_as_float(both << 16);
          y -= __uint_as_float(both & 0xffff0000u);
        }
      }
      bf16x8 pw[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) pw[i] = __builtin_bit_cast(bf16x8, make_uint4(part[i][0], part[i][1], part[i][2], part[i][3]));
#pragma unroll
      for (int d = 0; d < kBlocks; ++d) {
        typedef __attribute__((address_space(3))) bf16x4* lds_b4;
        const char* v0 = at_tile + 16 * st * kRow + (v_lane[0] ^ (64 * d));
        const char* v1 = at_tile + 16 * st * kRow + (v_lane[1] ^ (64 * d));
        const bf16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b4)v0);
        const bf16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_b4)v1);
        const bf16x8 v = __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int i = 0; i < 3; ++i) o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, pw[i], o[d], 0, 0, 0);
      }
    }
  }

  const float l = l_run + other_half(l_run);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (!row_live) return;
  char* dst = static_cast<char*>(a.out) + q_row * kRow + 8 * h;
#pragma unroll
  for (int d = 0; d < kBlocks; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2*>(dst + 64 * d + 16 * g) =
          make_uint2(pack_bf16(o[d][4 * g] * inv, o[d][4 * g + 1] * inv), pack_bf16(o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv));
  if (h == 0) {
    if (a.out_max) a.out_max[q_row] = MASK ? m_run : m_run * kLn2;
    if (a.out_denom) a.out_denom[q_row] = l;
  }
}

// One workgroup: 32 mask rows x 256 positions, a wave one block of 64 positions.
template <typename M>
__global__ void __launch_bounds__(256)
mask_class_kernel(const M* mask, int64_t stride_b, int64_t stride_h, int64_t stride_t, int rows, int cols, int heads,
                  uint8_t* classes, int row_blocks, int col_blocks) {
  const int b = blockIdx.z / heads, hh = blockIdx.z % heads;
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int r0 = blockIdx.y * kWaveRows;
  const M* src = mask + b * stride_b + hh * stride_h + r0 * stride_t + min(c, cols - 1);
  bool live = false, nonzero = false;
#pragma unroll 8
  for (int r = 0; r < kWaveRows; ++r) {
    const M raw = src[min(r, rows - 1 - r0) * stride_t];
    const float x = sizeof(M) == 2 ? bf16_bits_to_f32(static_cast<uint16_t>(raw)) : __uint_as_float(static_cast<uint32_t>(raw));
    live = live || x != -INFINITY;  // a NaN counts
    nonzero = nonzero || x != 0.f;
  }
  const bool inside = c < cols;
  const uint64_t any_live = __ballot(inside && live), any_nonzero = __ballot(inside && nonzero);
  const int cb = c / kCols;
  if ((threadIdx.x & 63) == 0 && cb < col_blocks)
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

// Is a pass over the mask worth its launch (4 us for 1024 rows, 8 for 3500)?  Where it can leave out tiles: with one row
// tile and a handful of key tiles there is nothing to leave out that would pay for it.
bool classes_pay(const jpt_attn_args& a) {
  if (a.mask == nullptr || a.q_rows < kRowsPerGroup || a.seq < 256 || a.seq > kMaxTiles * kCols) return false;
  const Classes c = mask_classes(a);
  return c.row_blocks <= 65535 && static_cast<int64_t>(c.batches) * c.heads <= 65535;  // what a grid can count
}

template <int D, int SCALE>
void launch_mask(const PrefillParams& p, dim3 grid, hipStream_t stream) {
  const dim3 block(64 * kWavesPerGroup);
  if (!p.a.mask) hipLaunchKernelGGL((attn_prefill_kernel<D, SCALE, 0>), grid, block, 0, stream, p);
  else if (p.a.mask_dtype == JPT_F32) hipLaunchKernelGGL((attn_prefill_kernel<D, SCALE, 1>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((attn_prefill_kernel<D, SCALE, 2>), grid, block, 0, stream, p);
}

template <int D>
void launch_dim(const PrefillParams& p, dim3 grid, hipStream_t stream) {
  if (!p.a.k_scale) launch_mask<D, 0>(p, grid, stream);
  else if (p.a.scale_dtype == JPT_F32) launch_mask<D, 1>(p, grid, stream);
  else launch_mask<D, 2>(p, grid, stream);
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
  p.tiles = (p.group_rows + kRowsPerGroup - 1) / kRowsPerGroup;
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
      const dim3 grid((a.seq + 255) / 256, c.row_blocks, c.batches * c.heads);
      if (a.mask_dtype == JPT_F32)
        hipLaunchKernelGGL(mask_class_kernel<uint32_t>, grid, dim3(256), 0, stream, static_cast<const uint32_t*>(a.mask),
                           a.mask_stride_b, a.mask_stride_h, a.mask_stride_t, a.q_rows, a.seq, c.heads, classes,
                           c.row_blocks, c.col_blocks);
      else
        hipLaunchKernelGGL(mask_class_kernel<uint16_t>, grid, dim3(256), 0, stream, static_cast<const uint16_t*>(a.mask),
                           a.mask_stride_b, a.mask_stride_h, a.mask_stride_t, a.q_rows, a.seq, c.heads, classes,
                           c.row_blocks, c.col_blocks);
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
