// Decode attention for what the streaming kernel (attn_decode_impl.h) is not built for: head_dim 64
// and 256, and head_dim 128 with a cache length or a mask it does not take.  Up to 16 query rows a
// KV head; int8 caches with scales, bf16 caches without; lengths or a mask; the step's new token as
// the cache holds it.
//
// Bound: HBM, each cache row is read once.  A group of four waves takes an equal share of all tiles
// (32 positions of one slot and KV head) of the batch, whatever the slots' lengths: shares are
// contiguous in (slot, head, tile) order, so a group cuts at most two sequences, and what it needs
// to know is worked out from the lengths at the head of the kernel - there is no planning launch.
// The four waves take the share's tiles in turn, straight from memory into registers in the
// matrix cores' layout (no LDS: with heads of 256 a ring of tiles in LDS would hold two): a row's
// keys 64 contiguous bytes at a time, a position's values as one contiguous row.  Keys of a wave's
// next tile are asked for when this tile's scores are done, values when its products are, also
// across the end of a sequence, so that a wave always has half a tile to a whole one in flight.
// Waves do not wait for each other: the one that delivers the last part of a sequence folds the
// parts.  (With barriers at every sequence's end and its tiles dealt to the waves anew, shares of equal
// tiles whatever the sequences' number, and the new token a tile of its own, 60 us where this took 48.)
//
// The arithmetic is the streaming kernel's (S^T = K . Q^T, O^T = V^T . P^T on 16x16x32 MFMAs), but keeps
// float32's bits: softmax weights are the sum of three 16-bit numbers, and int8 codes go in as float16 numbers
// of their own, not 1152 too high.  (The constant, carried through float32 sums and taken out at their end,
// costs ten bits of a sum of small terms: 1.4 % of the outputs of the case below were not the rounded exact
// value.  A packed subtraction a pair of codes takes it out; four layers of the case below 275 -> 287 us.)
// A weight times its value's scale is held against the row's largest so far, a power of two that rows carry
// along as they do their maximum: float16 alone would lose scales below 1e-3 bit by bit (0.3 % of the outputs
// of the case below, with scales of 0.03; all of them at 1e-7), and overflow above 65504.
//
// A sequence cut between groups: every group parks a float32 partial past the caches and counts
// itself; the last one folds them.  No group waits for another.
//
// Measured, calls back to back on caches that come from memory, int8, 16 heads of 256: 48 slots of 16..1024
// positions (201 MB a launch) 59 us, 3.4 TB/s; all 48 at 2048 positions 184 us, 4.4 TB/s (2.2 ms on the
// shape-generic kernel, one wave a query row).  With two-number weights, biased codes and raw scales 55 and
// 168 us.  A wave spends 54 % of its time waiting, for memory above all, and issues vector instructions in
// 21 % of it: 568 of them a tile of 32 x 128 int8, where the streaming kernel needs 321.
#include <algorithm>

#include "attn_decode_impl.h"

namespace jpt {
namespace decode {
namespace {

constexpr int kSplitWaves = 4;
constexpr int kSplitThreads = 64 * kSplitWaves;
constexpr int kMaxGroups = kSplitCounters;
constexpr int kLeastPart = 4;  // tiles, see where shares begin
constexpr int kSeqCost = 1;    // tiles a wave, likewise
constexpr int kLargestUp = 127 + 124;  // its inverse is a normal number too

struct SplitParams {
  jpt_attn_args a;
  float* partials;    // two records a group: (rows, D + 4)
  int32_t* counters;  // per group: parts of the sequence it began and did not end
  int32_t rows, rep;
};

template <int D, typename KV>
struct SplitTile;

// Operand of contraction step s of S^T: elements split_element<KV>(s, g) .. + 7 of the row, the
// elements of one 16-byte load lying side by side over the lanes g.
template <typename KV>
__device__ __forceinline__ int split_element(int s, int g) {
  return sizeof(KV) == 1 ? 64 * (s >> 1) + 16 * g + 8 * (s & 1) : 32 * s + 8 * g;
}

__device__ __forceinline__ uint4 load16_once(const char* p) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  return make_uint4(w.x, w.y, w.z, w.w);
}

// Keys of 32 positions: lane (r, g) has positions r and 16 + r, 16 bytes in every 64 of the row.
// Values: lane (r, g) has positions pos[i] = 4 g + i % 4 + 16 (i / 4), elements [D/16 r, D/16 (r + 1)).
template <int D, typename KV>
struct SplitTile {
  static constexpr int kRowBytes = D * sizeof(KV);
  static constexpr int kKeyLoads = kRowBytes / 64;                 // a position
  static constexpr int kValueWords = D / 16 * sizeof(KV) / 4;      // a position
  uint4 k[2][kKeyLoads];
  uint32_t v[8][kValueWords];

  // Rows base + min(position, top) rows: one scalar base and 32-bit offsets.  `fresh`: NULL, or the row of
  // position top_fresh, which lies elsewhere (the step's new token).
  __device__ __forceinline__ void load_keys(const char* base, int top, const char* fresh, int top_fresh, int r, int g) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const uint32_t off = static_cast<uint32_t>(min(r + 16 * half, top)) * kRowBytes + 16 * g;
#pragma unroll
      for (int j = 0; j < kKeyLoads; ++j) k[half][j] = load16_once(base + (off + 64 * j));
    }
    if (fresh != nullptr) {
#pragma unroll
      for (int half = 0; half < 2; ++half)
        if (r + 16 * half == top_fresh) {
#pragma unroll
          for (int j = 0; j < kKeyLoads; ++j) k[half][j] = load16_once(fresh + (static_cast<uint32_t>(16 * g) + 64 * j));
        }
    }
  }
  __device__ __forceinline__ void load_value_row(int i, const char* base, uint32_t off) {
    if constexpr (kValueWords == 1) {
      v[i][0] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(base + off));
    } else if constexpr (kValueWords == 2) {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(base + off));
      v[i][0] = w.x;
      v[i][1] = w.y;
    } else {
#pragma unroll
      for (int j = 0; j < kValueWords / 4; ++j) {
        const uint4 w = load16_once(base + (off + 16 * j));
        v[i][4 * j] = w.x; v[i][4 * j + 1] = w.y; v[i][4 * j + 2] = w.z; v[i][4 * j + 3] = w.w;
      }
    }
  }
  __device__ __forceinline__ void load_values(const char* base, int top, const char* fresh, int top_fresh, int r, int g) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      load_value_row(i, base, static_cast<uint32_t>(min(4 * g + (i & 3) + 16 * (i >> 2), top)) * kRowBytes + 4 * kValueWords * r);
    if (fresh != nullptr) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (4 * g + (i & 3) + 16 * (i >> 2) == top_fresh) load_value_row(i, fresh, 4 * kValueWords * r);
    }
  }
  using T = Tile<KV>;
  using Op = typename T::Op;
  // two float16 1152 + code as the codes, exactly
  static __device__ __forceinline__ uint32_t unbias(uint32_t both) {
    const f16x2 bias = {static_cast<_Float16>(T::kBias), static_cast<_Float16>(T::kBias)};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, both) - bias);
  }
  __device__ __forceinline__ Op k_op(int half, int s) const {
    if constexpr (sizeof(KV) == 1) {
      const uint4 x = k[half][s >> 1];
      const uint32_t w0 = ((s & 1) ? x.z : x.x) ^ 0x80808080u, w1 = ((s & 1) ? x.w : x.y) ^ 0x80808080u;
      return as_op<Op>(unbias(T::widen(w0, false)), unbias(T::widen(w0, true)), unbias(T::widen(w1, false)), unbias(T::widen(w1, true)));
    } else {
      return __builtin_bit_cast(Op, k[half][s]);
    }
  }
  // element j of the lane's for its eight positions
  __device__ __forceinline__ Op v_op(int j) const {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (sizeof(KV) == 1) {
        const uint32_t sel = 0x0c000c00u | static_cast<uint32_t>(j & 3) | (static_cast<uint32_t>(4 + (j & 3)) << 16);
        w[i] = unbias(__builtin_amdgcn_perm(v[2 * i + 1][j >> 2], v[2 * i][j >> 2], sel) ^ 0x64806480u);
      } else {
        w[i] = __builtin_amdgcn_perm(v[2 * i + 1][j >> 1], v[2 * i][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
      }
    }
    return as_op<Op>(w[0], w[1], w[2], w[3]);
  }
};

// A weight as the sum of three numbers of the operand's type, of each what rounding the ones before has
// left: float32's 24 bits (8 a number as bf16, 11 as float16).  Three packed pairs.
template <typename KV>
__device__ __forceinline__ void split_pack(float x, float y, uint32_t (&part)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const uint32_t both = part[i] = Tile<KV>::pack(x, y);
    if constexpr (sizeof(KV) == 1) {
      const f16x2 t = __builtin_bit_cast(f16x2, both);
      x -= static_cast<float>(t[0]);
      y -= static_cast<float>(t[1]);
    } else {
      x -= __uint_as_float(both << 16);
      y -= __uint_as_float(both & 0xffff0000u);
    }
  }
}

// Two waves a SIMD, but for bf16 rows of 256, whose tile is 128 registers.
template <int D, typename KV>
constexpr int split_waves_per_simd() { return D == 256 && sizeof(KV) == 2 ? 1 : 2; }

// 16 bytes a lane from memory to LDS at `lds` + 16 * lane, not known to the compiler as an LDS write
// (which would make every later LDS access wait for all loads in flight).  A write of M0 needs one
// wait state before the load that uses it, which the compiler does not see to inside asm.
__device__ __forceinline__ void stage_to_lds(const char* from, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(from), "s"(lds) : "memory");
}

template <int D, typename KV, int SCALE, bool MASK, int RC>
__global__ void __launch_bounds__(kSplitThreads, (split_waves_per_simd<D, KV>())) attn_split_kernel(SplitParams p) {
  using T = Tile<KV>;
  using Op = typename T::Op;
  using ST = SplitTile<D, KV>;
  constexpr int kSteps = D / 32, kJ = D / 16, kStride = D + 4;
  constexpr bool kQInLds = D == 256;  // the query operand's 32 registers are one tile's too many there
  constexpr int kParts = RC <= 4 ? 2 : 1;  // fold buffers: sequences that may be under way at once
  const jpt_attn_args& a = p.a;
  __shared__ __attribute__((aligned(16))) float so[kParts][kSplitWaves][RC][kStride];
  __shared__ float s_m[kParts][kSplitWaves][RC], s_l[kParts][kSplitWaves][RC];
  __shared__ __attribute__((aligned(16))) uint16_t s_q[kSplitWaves][RC * D];
  __shared__ int s_arrived[kParts], s_folded[kParts];
  __shared__ int s_jobs, s_job[2][4];  // cut sequences this group folds (it cuts two at most): slot, head, groups
  __shared__ int s_scan[kSplitWaves];
  __shared__ int s_found[2][2];  // for both ends of the share: slot, tiles of the batch before it
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int S = a.seq, H = a.kv_heads, R = p.rows;
  const int n_new = a.new_k != nullptr ? 1 : 0;  // the step's token: one more position behind the cache's

  auto length_of = [&](int b) {
    const int n = a.lengths ? a.lengths[b] : S;
    return n < 0 ? 0 : (n > S ? S : n);
  };
  // an empty slot has one tile, with nothing in it, so that somebody writes its output
  auto tiles_of = [&](int len) { return max((len + n_new + kTile - 1) / kTile, 1); };
  // What a sequence of nt tiles costs, in tiles: every wave that takes part in it (four at most) reads
  // and converts query rows and delivers a part.
  auto extra_of = [&](int nt) { return kSeqCost * min(nt, kSplitWaves); };
  auto cost_of = [&](int len) {
    const int nt = tiles_of(len);
    return nt + extra_of(nt);
  };

  // ---- this group's share --------------------------------------------------------
  const int per_thread = (a.batch + kSplitThreads - 1) / kSplitThreads;
  const int b_first = min(tid * per_thread, a.batch), b_end = min(b_first + per_thread, a.batch);
  int mine = 0;
  for (int b = b_first; b < b_end; ++b) mine += cost_of(length_of(b));
  int incl = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(incl, off);
    if (lane >= off) incl += y;
  }
  if (lane == 63) s_scan[wave] = incl;
  if (tid < kParts) s_arrived[tid] = s_folded[tid] = 0;
  if (tid == 0) s_jobs = 0;
  __syncthreads();
  int before = incl - mine, sum = 0;
#pragma unroll
  for (int w = 0; w < kSplitWaves; ++w) {
    if (w < wave) before += s_scan[w];
    sum += s_scan[w];
  }
  const int64_t total = static_cast<int64_t>(sum) * H;
  // How few tiles a share may have.  A sequence of n tiles in P parts takes about n / P * 0.45 us to
  // stream (four waves, 1.8 us a tile when memory is not the bound) and P / 4 trips to memory, a
  // microsecond each, for every 64 groups of four outputs to fold: both are even at
  // n / P = sqrt(n * rows * dim / 500) or so.  And a tile for each wave twice at least.
  const float mean = static_cast<float>(sum) / static_cast<float>(a.batch);
  const int64_t least = max(static_cast<int>(sqrtf(mean * static_cast<float>(R * D) * (1.f / 512.f))), 2 * kSplitWaves);
  const int groups = static_cast<int>(min(static_cast<int64_t>(gridDim.x), (total + least - 1) / least));
  const int me = blockIdx.x;
  if (me >= groups) return;
  // Share w begins at total * w / groups in the sequences laid end to end, each its cost long - but not
  // less than kLeastPart tiles inside a sequence: a cut costs its groups a partial, its count and a
  // fold.  (Ragged lengths as above, in one run: kLeastPart 4 and a sequence's cost of a tile a wave 47.5 us;
  // no such cost 49.8; kLeastPart 7 48.8 and, all slots at 512 positions, 51.1 for 46.7 us.)
  auto raw_begin = [&](int w) -> int64_t { return total * w / groups; };
  auto group_of = [&](int64_t at) -> int { return static_cast<int>(((at + 1) * groups - 1) / total); };  // before moving
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t edge = raw_begin(me + i);
    if (mine > 0 && static_cast<int64_t>(before) * H <= edge && edge < static_cast<int64_t>(before + mine) * H) {
      int b = b_first, at = before;
      for (;; ++b) {
        const int n = cost_of(length_of(b));
        if (edge < static_cast<int64_t>(at + n) * H) break;
        at += n;
      }
      s_found[i][0] = b;
      s_found[i][1] = at;
    }
  }
  __syncthreads();  // from here on every wave goes its own way

  // A sequence (one slot and KV head) of this group's share and the part of it in the share.
  struct Seq {
    int64_t first;  // where it begins
    int slot, h, len, nt, extra;
    int ta, tb;     // its tiles in the share
    int base;       // tiles of the share before tile ta
    int number;     // sequences of the share before it
  };
  auto seq_at = [&](int i, int64_t edge) {
    Seq s;
    s.slot = __builtin_amdgcn_readfirstlane(s_found[i][0]);
    s.len = __builtin_amdgcn_readfirstlane(length_of(s.slot));
    s.nt = tiles_of(s.len);
    s.extra = extra_of(s.nt);
    s.first = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(s_found[i][1])) * H;
    s.h = static_cast<int>((edge - s.first) / (s.nt + s.extra));
    s.first += static_cast<int64_t>(s.h) * (s.nt + s.extra);
    return s;
  };
  auto moved = [&](const Seq& s, int64_t edge) -> int64_t {
    const int64_t in = edge - s.first;
    return in < s.extra + kLeastPart ? s.first : s.nt + s.extra - in < kLeastPart ? s.first + s.nt + s.extra : edge;
  };
  Seq nxt = seq_at(0, raw_begin(me));
  const int64_t begin = moved(nxt, raw_begin(me));
  const int64_t end = me + 1 == groups ? total : moved(seq_at(1, raw_begin(me + 1)), raw_begin(me + 1));
  if (begin >= end) return;
  auto next_seq = [&]() {
    nxt.first += nxt.nt + nxt.extra;
    if (nxt.first >= end) return;
    if (++nxt.h == H) {
      nxt.h = 0;
      ++nxt.slot;
      nxt.len = __builtin_amdgcn_readfirstlane(length_of(nxt.slot));
      nxt.nt = tiles_of(nxt.len);
      nxt.extra = extra_of(nxt.nt);
    }
  };
  auto set_part = [&]() {
    nxt.ta = begin > nxt.first ? static_cast<int>(begin - nxt.first) - nxt.extra : 0;
    nxt.tb = end - nxt.first >= nxt.nt + nxt.extra ? nxt.nt : static_cast<int>(end - nxt.first) - nxt.extra;
  };
  if (begin >= nxt.first + nxt.nt + nxt.extra) next_seq();
  set_part();
  nxt.base = nxt.number = 0;
  // nxt: the sequence with tile x of the share, counted through the share's sequences; false: there is none
  auto move_to = [&](int x) -> bool {
    while (x >= nxt.base + nxt.tb - nxt.ta) {
      nxt.base += nxt.tb - nxt.ta;
      ++nxt.number;
      next_seq();
      if (nxt.first >= end) return false;
      set_part();
    }
    return true;
  };
  int x = wave;  // this wave's tiles: every fourth of the share
  bool more = move_to(x);

  int pos[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) pos[i] = 4 * g + (i & 3) + 16 * (i >> 2);
  // Scores in log2 units - but where a mask is added, which may be float32's lowest value: that times
  // log2(e) would be -infinity, and a row masked throughout empty instead of the mean of the values.
  const float c2 = MASK ? a.sm_scale : a.sm_scale * kLog2e;
  auto weight_of = [](float above_max) { return fast_exp2(MASK ? above_max * kLog2e : above_max); };
  const uint32_t q_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr)&s_q[wave][0]));
  auto q_row_of = [&](const Seq& s) { return (static_cast<int64_t>(s.slot) * a.q_heads + s.h * p.rep) * a.q_rows; };
  auto stage_q = [&](const Seq& s) {
    const char* from = static_cast<const char*>(a.q) + q_row_of(s) * (D * 2);
    for (int j = 0; j * 1024 < R * D * 2; ++j)
      if (j * 1024 + lane * 16 < R * D * 2) stage_to_lds(from + j * 1024 + lane * 16, q_lds + j * 1024);
  };

  ST tile;
  float ks[8], vs[8], mk[8];
  // positions of tile t that count (0: the tile of an empty slot)
  auto valid_of = [&](const Seq& s, int t) { return min(kTile, s.len + n_new - t * kTile); };
  // A tile's rows: its own from `base` on, the last of them row `top` (positions past the end repeat
  // it); in the tile with the position behind the cache's, the new token's row in its place.  An empty
  // slot has no row of its own: all are the token's (without one the tile's products are left out).
  // What lies past a slot's end may be anything, and 0 times NaN is NaN.
  struct Rows {
    const char *base, *fresh;
    int top, top_fresh;
  };
  auto rows_of = [&](const Seq& s, int t, const void* cache, const void* fresh) {
    const int left = s.len - t * kTile;  // cache rows from the tile's first position on
    const char* const token = static_cast<const char*>(fresh) + (static_cast<int64_t>(s.slot) * H + s.h) * ST::kRowBytes;
    Rows w;
    w.base = n_new && s.len == 0 ? token
                                 : static_cast<const char*>(cache) + ((static_cast<int64_t>(s.slot) * H + s.h) * S +
                                                                      min(t * kTile, max(s.len - 1, 0))) * ST::kRowBytes;
    w.top = min(max(left, 1), kTile) - 1;
    w.fresh = n_new && s.len > 0 && left < kTile ? token : nullptr;
    w.top_fresh = left;
    return w;
  };
  auto load_scales = [&](const Seq& s, int t, const void* cache, const void* fresh, float (&out)[8]) {
    if (!SCALE) return;
    constexpr int dt = SCALE == kScaleF32 ? JPT_F32 : JPT_BF16;
    const int hs = a.scale_heads == 1 ? 0 : s.h;
    const int64_t s0 = (static_cast<int64_t>(s.slot) * a.scale_heads + hs) * S + static_cast<int64_t>(t) * kTile;
    const int left = s.len - t * kTile;
    if (left >= kTile && S % 4 == 0) {  // runs of four, aligned (the scale tensors are, see the host's check)
      if (SCALE == kScaleF32) {
        const float4* src = reinterpret_cast<const float4*>(static_cast<const float*>(cache) + s0);
        const float4 u = src[g], w = src[4 + g];
        out[0] = u.x; out[1] = u.y; out[2] = u.z; out[3] = u.w; out[4] = w.x; out[5] = w.y; out[6] = w.z; out[7] = w.w;
      } else {
        const uint2* src = reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(cache) + s0);
        const uint2 u = src[g], w = src[4 + g];
        out[0] = __uint_as_float(u.x << 16); out[1] = __uint_as_float(u.x & 0xffff0000u);
        out[2] = __uint_as_float(u.y << 16); out[3] = __uint_as_float(u.y & 0xffff0000u);
        out[4] = __uint_as_float(w.x << 16); out[5] = __uint_as_float(w.x & 0xffff0000u);
        out[6] = __uint_as_float(w.y << 16); out[7] = __uint_as_float(w.y & 0xffff0000u);
      }
    } else {
      const int64_t sn = static_cast<int64_t>(s.slot) * a.scale_heads + hs;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        out[i] = pos[i] < left || !n_new ? load_as_f32(cache, s0 + max(min(pos[i], left - 1), 0), dt) : load_as_f32(fresh, sn, dt);
    }
  };
  auto load_mask = [&](const Seq& s, int t) {
    if (!MASK) return;
    const int rr = min(r, R - 1);
    const int64_t row = s.slot * a.mask_stride_b + (s.h * p.rep + rr / a.q_rows) * a.mask_stride_h + (rr % a.q_rows) * a.mask_stride_t;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int at = t * kTile + pos[i];
      mk[i] = at < s.len ? load_as_f32(a.mask, row + at, a.mask_dtype) : 0.f;
    }
  };
  auto load_k = [&](const Seq& s, int t) {
    const Rows w = rows_of(s, t, a.k, a.new_k);
    tile.load_keys(w.base, w.top, w.fresh, w.top_fresh, r, g);
    load_scales(s, t, a.k_scale, a.new_k_scale, ks);
    load_mask(s, t);
  };
  auto load_v = [&](const Seq& s, int t) {
    const Rows w = rows_of(s, t, a.v, a.new_v);
    tile.load_values(w.base, w.top, w.fresh, w.top_fresh, r, g);
    load_scales(s, t, a.v_scale, a.new_v_scale, vs);
  };
  auto write_out = [&](int64_t q_row, int d, const f32x4& o, float M, float l) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + q_row * D + d) =
        make_uint2(pack_bf16(o[0] * inv, o[1] * inv), pack_bf16(o[2] * inv, o[3] * inv));
    if (d == 0) {
      if (a.out_max) a.out_max[q_row] = MASK ? M : M * kLn2;
      if (a.out_denom) a.out_denom[q_row] = l;
    }
  };
  const int64_t record = static_cast<int64_t>(R) * kStride;
  typedef __attribute__((ext_vector_type(2))) float f32x2;

  // Folds the parts of sequence s that this group's waves left in buffer `buf`: one wave's work.  Where
  // the sequence is cut and this is its last part to arrive, the fold over the groups is left for the end.
  auto fold = [&](const Seq& s, int buf) {
    const bool begins = s.ta == 0, ends = s.tb == s.nt;
    const int64_t q_row0 = q_row_of(s);
    // waves that had tiles: those of the part's first (up to) four
    const int w0 = s.base % kSplitWaves, nw = min(kSplitWaves, s.tb - s.ta);
    // the part that begins a sequence is its group's second record, every other its group's first
    float* const part = p.partials + (2 * static_cast<int64_t>(me) + (begins ? 1 : 0)) * record;
    for (int u = lane; u < R * (D / 4); u += 64) {
      const int row = u / (D / 4), d = u % (D / 4) * 4;
      float M = -INFINITY;
#pragma unroll
      for (int i = 0; i < kSplitWaves; ++i)
        if (i < nw) M = fmaxf(M, s_m[buf][(w0 + i) % kSplitWaves][row]);
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      float l = 0.f;
#pragma unroll
      for (int i = 0; i < kSplitWaves; ++i) {
        if (i >= nw) continue;
        const int w = (w0 + i) % kSplitWaves;
        const float mw = s_m[buf][w][row];
        const float f = mw == -INFINITY ? 0.f : weight_of(mw - M);
        l += s_l[buf][w][row] * f;
        o += *reinterpret_cast<const f32x4*>(&so[buf][w][row][d]) * f;
      }
      if (begins && ends) {
        write_out(q_row0 + row, d, o, M, l);
      } else {  // past the caches: another XCD's group may fold it
        float* to = part + row * kStride;
        asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" : : "v"(to + d), "v"(o) : "memory");
        if (d == 0) {
          const f32x2 st = {M, l};
          asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" : : "v"(to + D), "v"(st) : "memory");
        }
      }
    }
    if (begins && ends) return;
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // the partial has arrived
    // the groups whose shares begin or end inside the sequence
    const int g_first = group_of(s.first + s.extra + kLeastPart - 1), g_last = group_of(s.first + s.extra + s.nt - kLeastPart), parts = g_last - g_first + 1;
    int seen = 0;
    if (lane == 0) seen = __hip_atomic_fetch_add(p.counters + g_first, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(seen) != parts - 1) return;
    if (lane == 0) {
      __hip_atomic_store(p.counters + g_first, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int i = __hip_atomic_fetch_add(&s_jobs, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      s_job[i][0] = s.slot;
      s_job[i][1] = s.h;
      s_job[i][2] = g_first;
      s_job[i][3] = g_last;
    }
  };

  if (more) {
    stage_q(nxt);
    load_k(nxt, nxt.ta + x - nxt.base);
    load_v(nxt, nxt.ta + x - nxt.base);
  }
  while (more) {
    const Seq cur = nxt;
    // ---- query rows, staged ahead of the sequence's first tile ----
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    Op qop[kQInLds ? 1 : kSteps];
    auto q_at = [&](int s) { return reinterpret_cast<Op*>(&s_q[wave][min(r, R - 1) * D + split_element<KV>(s, g)]); };
    float c2_row = c2;
    {
      uint4 raw[kSteps];
#pragma unroll
      for (int s = 0; s < kSteps; ++s)
        raw[s] = *reinterpret_cast<const uint4*>(q_at(s));
      if constexpr (sizeof(KV) == 1) {
        // as float16: the row times the power of two that puts its largest magnitude in [2^13, 2^14)
        float amax = 0.f;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
          const uint32_t w[4] = {raw[s].x, raw[s].y, raw[s].z, raw[s].w};
#pragma unroll
          for (int i = 0; i < 4; ++i)
            amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(w[i] << 16)), fabsf(__uint_as_float(w[i] & 0xffff0000u))));
        }
        amax = max_across_rows(amax);
        int e = 0;
        if (amax > 0.f && amax < INFINITY) frexpf(amax, &e);
        e = max(e, -100);
        const float up = ldexpf(1.f, 14 - e);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
          const uint32_t w[4] = {raw[s].x, raw[s].y, raw[s].z, raw[s].w};
          uint32_t f[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f[i] = pack_f16(__uint_as_float(w[i] << 16) * up, __uint_as_float(w[i] & 0xffff0000u) * up);
          }
          if constexpr (kQInLds) *q_at(s) = as_op<Op>(f[0], f[1], f[2], f[3]);
          else qop[s] = as_op<Op>(f[0], f[1], f[2], f[3]);
        }
        c2_row = c2 * ldexpf(1.f, e - 14);
      } else if constexpr (!kQInLds) {
#pragma unroll
        for (int s = 0; s < kSteps; ++s) qop[s] = __builtin_bit_cast(Op, raw[s]);
      }
    }
    f32x4 acc[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    // int8: the largest weight times value scale so far, and the exponent (biased as float32's) of the power
    // of two that puts it in [2^14, 2^15): float16's range is too short for what scales may be
    float w_run = 0.f;
    int up = kLargestUp;

    for (;;) {
      const int valid = valid_of(cur, cur.ta + x - cur.base);
      x += kSplitWaves;
      more = move_to(x);
      const int t_next = nxt.ta + x - nxt.base;
      f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = sa;
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        Op q;
        if constexpr (kQInLds) q = *q_at(s);
        else q = qop[s];
        sa = T::mfma(tile.k_op(0, s), q, sa);
        sb = T::mfma(tile.k_op(1, s), q, sb);
      }
      float sc[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sc[i] = (i < 4 ? sa[i] : sb[i - 4]) * (SCALE ? ks[i] * c2_row : c2_row);
        if (MASK) sc[i] += mk[i];
        if (valid != kTile) sc[i] = pos[i] < valid ? sc[i] : -INFINITY;
      }
      if (more) {
        if (nxt.number != cur.number) stage_q(nxt);
        load_k(nxt, t_next);
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) tmax = fmaxf(tmax, sc[i]);
      tmax = max_across_rows(tmax);
      const float m_new = fmaxf(m_run, tmax);
      const float m_use = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = weight_of(m_run - m_use);
      float w[8], psum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float pr = weight_of(sc[i] - m_use);
        psum += pr;
        w[i] = SCALE ? pr * vs[i] : pr;
        if (SCALE && valid != kTile) w[i] = pos[i] < valid ? w[i] : 0.f;  // whatever its scale holds
      }
      l_run = l_run * alpha + psum;
      m_run = m_new;
      float keep = alpha;  // what the products so far are multiplied with
      if (SCALE) {
        float w_max = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) w_max = fmaxf(w_max, fabsf(w[i]));
        w_run = fmaxf(w_run * alpha, max_across_rows(w_max));
        const int up_new = min(127 + 14 + 127 - static_cast<int>(__float_as_uint(w_run) >> 23), kLargestUp);
        keep = ldexpf(alpha, up_new - up);
        up = up_new;
        const float by = __uint_as_float(static_cast<uint32_t>(up) << 23);
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] *= by;
      }
      if (__any(keep != 1.f)) {
#pragma unroll
        for (int j = 0; j < kJ; ++j) acc[j] *= keep;
      }
      uint32_t part[4][3];
#pragma unroll
      for (int i = 0; i < 4; ++i) split_pack<KV>(w[2 * i], w[2 * i + 1], part[i]);
      Op pw[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) pw[i] = as_op<Op>(part[0][i], part[1][i], part[2][i], part[3][i]);
      if (valid > 0) {
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
          const Op v = tile.v_op(j);
#pragma unroll
          for (int i = 0; i < 3; ++i) acc[j] = T::mfma(v, pw[i], acc[j]);
        }
      }
      if (more) load_v(nxt, t_next);
      if (!more || nxt.number != cur.number) break;
    }

    // ---- deliver this wave's part; the last wave to do so folds them ----
    const int buf = cur.number % kParts;
    // the buffer's previous sequence is folded by the last of its waves, which needs nobody: the wait ends
    while (__hip_atomic_load(&s_folded[buf], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < cur.number / kParts)
      __builtin_amdgcn_s_sleep(1);
    const float l_row = sum_across_rows(l_run);
    if (r < R) {
      const float down = SCALE ? __uint_as_float(static_cast<uint32_t>(254 - up) << 23) : 1.f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < kJ; j += 4)
          *reinterpret_cast<float4*>(&so[buf][wave][r][kJ * (4 * g + i) + j]) =
              make_float4(acc[j][i] * down, acc[j + 1][i] * down, acc[j + 2][i] * down, acc[j + 3][i] * down);
      if (g == 0) {
        s_m[buf][wave][r] = m_run;
        s_l[buf][wave][r] = l_row;
      }
    }
    int arrived = 0;
    if (lane == 0) arrived = __hip_atomic_fetch_add(&s_arrived[buf], 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
    arrived = __builtin_amdgcn_readfirstlane(arrived);
    if (arrived == min(kSplitWaves, cur.tb - cur.ta) - 1) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      fold(cur, buf);
      if (lane == 0) {
        __hip_atomic_store(&s_arrived[buf], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_fetch_add(&s_folded[buf], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  }

  // Sequences whose last part this group delivered: all four waves fold their parts.
  __syncthreads();
  for (int i = 0; i < s_jobs; ++i) {
    const int g_first = s_job[i][2], g_last = s_job[i][3];
    const int64_t q_row0 = (static_cast<int64_t>(s_job[i][0]) * a.q_heads + s_job[i][1] * p.rep) * a.q_rows;
    for (int u = tid; u < R * (D / 4); u += kSplitThreads) {
      const int row = u / (D / 4), d = u % (D / 4) * 4;
      float M = -INFINITY, l = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      for (int c0 = g_first; c0 <= g_last; c0 += 4) {  // four parts a trip to memory
        const float* from[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = min(c0 + i, g_last);
          from[i] = p.partials + (2 * static_cast<int64_t>(c) + (c == g_first ? 1 : 0)) * record + row * kStride;
        }
        f32x4 y[4];
        f32x2 st[4];
        asm volatile("global_load_dwordx4 %0, %8, off sc0 sc1\n\t"
                     "global_load_dwordx4 %1, %9, off sc0 sc1\n\t"
                     "global_load_dwordx4 %2, %10, off sc0 sc1\n\t"
                     "global_load_dwordx4 %3, %11, off sc0 sc1\n\t"
                     "global_load_dwordx2 %4, %12, off sc0 sc1\n\t"
                     "global_load_dwordx2 %5, %13, off sc0 sc1\n\t"
                     "global_load_dwordx2 %6, %14, off sc0 sc1\n\t"
                     "global_load_dwordx2 %7, %15, off sc0 sc1\n\t"
                     "s_waitcnt vmcnt(0)"
                     : "=&v"(y[0]), "=&v"(y[1]), "=&v"(y[2]), "=&v"(y[3]), "=&v"(st[0]), "=&v"(st[1]), "=&v"(st[2]), "=&v"(st[3])
                     : "v"(from[0] + d), "v"(from[1] + d), "v"(from[2] + d), "v"(from[3] + d), "v"(from[0] + D), "v"(from[1] + D),
                       "v"(from[2] + D), "v"(from[3] + D)
                     : "memory");
        float Mb = M;
#pragma unroll
        for (int i = 0; i < 4; ++i) Mb = fmaxf(Mb, st[i][0]);
        const float keep = M == -INFINITY ? 0.f : weight_of(M - Mb);
        l *= keep;
        o *= keep;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = c0 + i > g_last || st[i][0] == -INFINITY ? 0.f : weight_of(st[i][0] - Mb);
          l += st[i][1] * f;
          o += y[i] * f;
        }
        M = Mb;
      }
      write_out(q_row0 + row, d, o, M, l);
    }
  }
}

constexpr int kMinGroups = 64;
int64_t group_bytes(const jpt_attn_args& a) {  // two records
  return 2ll * (a.q_heads / a.kv_heads) * a.q_rows * (a.dim + 4) * 4;
}
int64_t full_groups(const jpt_attn_args& a) {
  const int per_unit = a.dim == 256 && a.kv_dtype == JPT_BF16 ? 1 : 2;
  return std::min(compute_units() * per_unit, kMaxGroups);
}
// as many as the workspace has records for
int64_t split_groups(const jpt_attn_args& a) {
  return std::min(full_groups(a), (a.workspace_bytes - attn_partials_offset(a)) / group_bytes(a));
}

template <int D, typename KV, int SCALE>
void launch_split(const SplitParams& p, dim3 grid, hipStream_t stream) {
  const dim3 block(kSplitThreads);
  if (p.a.mask) {
    if (p.rows <= 4) hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, true, 4>), grid, block, 0, stream, p);
    else if (p.rows <= 8) hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, true, 8>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, true, kMaxRows>), grid, block, 0, stream, p);
  } else {
    if (p.rows <= 4) hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, false, 4>), grid, block, 0, stream, p);
    else if (p.rows <= 8) hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, false, 8>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, false, kMaxRows>), grid, block, 0, stream, p);
  }
}

template <int D>
void launch_split_dim(const SplitParams& p, dim3 grid, hipStream_t stream) {
  if (p.a.kv_dtype == JPT_BF16) launch_split<D, __bf16, kNoScale>(p, grid, stream);
  else if (p.a.scale_dtype == JPT_F32) launch_split<D, int8_t, kScaleF32>(p, grid, stream);
  else launch_split<D, int8_t, kScaleBF16>(p, grid, stream);
}

}  // namespace
}  // namespace decode

bool attn_split_supported(const jpt_attn_args& a, AttnMode mode) {
  if (a.force_generic || mode == kPaged || a.new_k_raw) return false;
  if (a.q_dtype != JPT_BF16 || (a.dim != 64 && a.dim != 128 && a.dim != 256)) return false;
  if (a.kv_dtype != JPT_I8 && a.kv_dtype != JPT_BF16) return false;
  if ((a.kv_dtype == JPT_I8) != (a.k_scale != nullptr)) return false;
  if (a.q_heads / a.kv_heads * static_cast<int64_t>(a.q_rows) > kMaxRows) return false;
  if (!aligned(a.q, 16) || !aligned(a.k, 16) || !aligned(a.v, 16) || !aligned(a.out, 8)) return false;
  if (a.k_scale && (!aligned(a.k_scale, 16) || !aligned(a.v_scale, 16))) return false;
  if (a.new_k && (!aligned(a.new_k, 16) || !aligned(a.new_v, 16))) return false;
  // tile numbers fit 32 bits, the sum over the batch before it is multiplied by the heads too
  return static_cast<int64_t>(a.batch) * (a.seq / kTile + 16) < (1ll << 31);
}

bool attn_split_has_room(const jpt_attn_args& a) {
  return a.workspace != nullptr && aligned(a.workspace, 256) && decode::split_groups(a) >= decode::kMinGroups;
}

int64_t attn_split_workspace_bytes(const jpt_attn_args& a) {
  return attn_partials_offset(a) + decode::full_groups(a) * decode::group_bytes(a);
}

int32_t attn_split_launch(const jpt_attn_args& a, hipStream_t stream) {
  decode::SplitParams p{};
  p.a = a;
  p.rep = a.q_heads / a.kv_heads;
  p.rows = p.rep * a.q_rows;
  p.counters = static_cast<int32_t*>(a.workspace) + kStateSplitCounters;
  const int64_t groups = decode::split_groups(a);
  p.partials = reinterpret_cast<float*>(attn_workspace_end(a, groups * decode::group_bytes(a)));
  const dim3 grid(static_cast<unsigned>(groups));
  if (a.dim == 64) decode::launch_split_dim<64>(p, grid, stream);
  else if (a.dim == 128) decode::launch_split_dim<128>(p, grid, stream);
  else decode::launch_split_dim<256>(p, grid, stream);
  return launch_status("attn_split_kernel");
}

}  // namespace jpt
