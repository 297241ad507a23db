// Decode attention for what the streaming kernel (attn_decode_impl.h) is not built for: head_dim 64
// and 256, and head_dim 128 with a cache length or a mask it does not take.  Up to 16 query rows a
// KV head; int8 caches with scales, bf16 caches without; lengths or a mask; the step's new token as
// the cache holds it.
//
// Bound: HBM, each cache row is read once.  A group of four waves takes an equal share of all tiles
// (32 positions of one slot and KV head) of the batch, whatever the slots' lengths: shares are
// contiguous in (slot, head, tile) order, so a group cuts at most two sequences, and what it needs
// to know is worked out from the lengths at the head of the kernel - there is no planning launch.
// The four waves take a sequence's tiles in turn, straight from memory into registers in the
// matrix cores' layout (no LDS: with heads of 256 a ring of tiles in LDS would hold two): a row's
// keys 64 contiguous bytes at a time, a position's values as one contiguous row.  Keys of the next
// tile are asked for when this tile's scores are done, values when its products are, so that a wave
// always has half a tile to a whole one in flight.
//
// The arithmetic is that of the streaming kernel (S^T = K . Q^T, O^T = V^T . P^T on 16x16x32 MFMAs,
// int8 codes as float16 1024 + 128 + code), with softmax weights as the sum of two 16-bit numbers:
// the matrix cores have the time, and the result keeps only its own rounding to bf16.
//
// A sequence cut between groups: every group parks a float32 partial past the caches and counts
// itself; the last one folds them.  Nobody waits for anybody.
//
// Measured, int8, 48 slots of 16..1024 positions, 16 heads of 256 (205 MB a launch): 62 us, 3.3 TB/s
// (2.2 ms on the shape-generic kernel, one wave a query row).
#include <algorithm>

#include "attn_decode_impl.h"

namespace jpt {
namespace decode {
namespace {

constexpr int kSplitWaves = 4;
constexpr int kSplitThreads = 64 * kSplitWaves;
constexpr int kMaxGroups = kSplitCounters;

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

  __device__ __forceinline__ void load_keys(const char* base, int valid, int r, int g) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const char* row = base + static_cast<uint32_t>(min(r + 16 * half, valid - 1)) * kRowBytes + 16 * g;
#pragma unroll
      for (int j = 0; j < kKeyLoads; ++j) k[half][j] = load16_once(row + 64 * j);
    }
  }
  __device__ __forceinline__ void load_values(const char* base, int valid, int r, int g) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const char* at = base + static_cast<uint32_t>(min(4 * g + (i & 3) + 16 * (i >> 2), valid - 1)) * kRowBytes + 4 * kValueWords * r;
      if constexpr (kValueWords == 1) {
        v[i][0] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(at));
      } else if constexpr (kValueWords == 2) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(at));
        v[i][0] = w.x;
        v[i][1] = w.y;
      } else {
#pragma unroll
        for (int j = 0; j < kValueWords / 4; ++j) {
          const uint4 w = load16_once(at + 16 * j);
          v[i][4 * j] = w.x; v[i][4 * j + 1] = w.y; v[i][4 * j + 2] = w.z; v[i][4 * j + 3] = w.w;
        }
      }
    }
  }
  using T = Tile<KV>;
  using Op = typename T::Op;
  __device__ __forceinline__ Op k_op(int half, int s) const {
    if constexpr (sizeof(KV) == 1) {
      const uint4 x = k[half][s >> 1];
      const uint32_t w0 = ((s & 1) ? x.z : x.x) ^ 0x80808080u, w1 = ((s & 1) ? x.w : x.y) ^ 0x80808080u;
      return as_op<Op>(T::widen(w0, false), T::widen(w0, true), T::widen(w1, false), T::widen(w1, true));
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
        w[i] = __builtin_amdgcn_perm(v[2 * i + 1][j >> 2], v[2 * i][j >> 2], sel) ^ 0x64806480u;
      } else {
        w[i] = __builtin_amdgcn_perm(v[2 * i + 1][j >> 1], v[2 * i][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
      }
    }
    return as_op<Op>(w[0], w[1], w[2], w[3]);
  }
};

// A weight as the sum of two numbers of the operand's type: two packed pairs.
template <typename KV>
__device__ __forceinline__ void split_pack(float x, float y, uint32_t& hi, uint32_t& lo) {
  hi = Tile<KV>::pack(x, y);
  float hx, hy;
  if constexpr (sizeof(KV) == 1) {
    const f16x2 t = __builtin_bit_cast(f16x2, hi);
    hx = static_cast<float>(t[0]);
    hy = static_cast<float>(t[1]);
  } else {
    hx = __uint_as_float(hi << 16);
    hy = __uint_as_float(hi & 0xffff0000u);
  }
  lo = Tile<KV>::pack(x - hx, y - hy);
}

// Two waves a SIMD, but for bf16 rows of 256, whose tile is 128 registers.
template <int D, typename KV>
constexpr int split_waves_per_simd() { return D == 256 && sizeof(KV) == 2 ? 1 : 2; }

template <int D, typename KV, int SCALE, bool MASK, int RC>
__global__ void __launch_bounds__(kSplitThreads, (split_waves_per_simd<D, KV>())) attn_split_kernel(SplitParams p) {
  using T = Tile<KV>;
  using Op = typename T::Op;
  using ST = SplitTile<D, KV>;
  constexpr int kSteps = D / 32, kJ = D / 16, kStride = D + 4;
  const jpt_attn_args& a = p.a;
  __shared__ __attribute__((aligned(16))) float so[kSplitWaves][RC][kStride];
  __shared__ float s_m[kSplitWaves][RC], s_l[kSplitWaves][RC];
  __shared__ int s_scan[kSplitWaves];
  __shared__ int s_found[3];  // slot, tiles of the batch before it, last part to arrive
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int S = a.seq, H = a.kv_heads, R = p.rows;
  const bool has_new = a.new_k != nullptr;

  auto length_of = [&](int b) {
    const int n = a.lengths ? a.lengths[b] : S;
    return n < 0 ? 0 : (n > S ? S : n);
  };
  // an empty slot has one tile, with nothing in it, so that somebody writes its output
  auto tiles_of = [&](int len) { return max((len + kTile - 1) / kTile + (has_new ? 1 : 0), 1); };

  // ---- this group's share --------------------------------------------------------
  const int per_thread = (a.batch + kSplitThreads - 1) / kSplitThreads;
  const int b_first = min(tid * per_thread, a.batch), b_end = min(b_first + per_thread, a.batch);
  int mine = 0;
  for (int b = b_first; b < b_end; ++b) mine += tiles_of(length_of(b));
  int incl = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(incl, off);
    if (lane >= off) incl += y;
  }
  if (lane == 63) s_scan[wave] = incl;
  __syncthreads();
  int before = incl - mine, sum = 0;
#pragma unroll
  for (int w = 0; w < kSplitWaves; ++w) {
    if (w < wave) before += s_scan[w];
    sum += s_scan[w];
  }
  const int64_t total = static_cast<int64_t>(sum) * H;
  // a group has four tiles at least, one for each of its waves
  const int groups = static_cast<int>(min(static_cast<int64_t>(gridDim.x), (total + kSplitWaves - 1) / kSplitWaves));
  const int me = blockIdx.x;
  if (me >= groups) return;
  auto share_begin = [&](int w) -> int64_t { return total * w / groups; };
  auto group_of = [&](int64_t tile) -> int { return static_cast<int>(((tile + 1) * groups - 1) / total); };
  const int64_t begin = share_begin(me), end = share_begin(me + 1);
  if (mine > 0 && static_cast<int64_t>(before) * H <= begin && begin < static_cast<int64_t>(before + mine) * H) {
    int b = b_first, at = before;
    for (;; ++b) {
      const int n = tiles_of(length_of(b));
      if (begin < static_cast<int64_t>(at + n) * H) break;
      at += n;
    }
    s_found[0] = b;
    s_found[1] = at;
  }
  __syncthreads();
  int slot = __builtin_amdgcn_readfirstlane(s_found[0]);
  int64_t slot_begin = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(s_found[1])) * H;  // the slot's first tile
  int len = __builtin_amdgcn_readfirstlane(length_of(slot));
  int nt = tiles_of(len);
  int h = static_cast<int>((begin - slot_begin) / nt);

  int pos[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) pos[i] = 4 * g + (i & 3) + 16 * (i >> 2);
  const float c2 = a.sm_scale * kLog2e;

  for (int64_t at = begin; at < end;) {
    const int64_t seq_begin = slot_begin + static_cast<int64_t>(h) * nt;  // of (slot, h)
    const int t_first = static_cast<int>(at - seq_begin);
    const int t_end = static_cast<int>(min(static_cast<int64_t>(nt), end - seq_begin));
    const int hs = a.scale_heads == 1 ? 0 : h;
    const int64_t kv0 = (static_cast<int64_t>(slot) * H + h) * S;
    const int64_t sc0 = SCALE ? (static_cast<int64_t>(slot) * a.scale_heads + hs) * S : 0;
    const int64_t new_row = static_cast<int64_t>(slot) * H + h;
    const int64_t q_row0 = (static_cast<int64_t>(slot) * a.q_heads + h * p.rep) * a.q_rows;
    const int n_new = has_new ? 1 : 0;  // the new token is tile 0 of its sequence

    // ---- query rows ----
    Op qop[kSteps];
    float c2_row = c2;
    f32x4 s_init = {0.f, 0.f, 0.f, 0.f};
    {
      uint4 raw[kSteps];
      const char* src = static_cast<const char*>(a.q) + (q_row0 + min(r, R - 1)) * (D * 2);
#pragma unroll
      for (int s = 0; s < kSteps; ++s) raw[s] = *reinterpret_cast<const uint4*>(src + 2 * split_element<KV>(s, g));
      if constexpr (sizeof(KV) == 1) {
        // as float16: the row times the power of two that puts its largest magnitude in [2^13, 2^14)
        float amax = 0.f, qs = 0.f;
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
            const float x = __uint_as_float(w[i] << 16) * up, y = __uint_as_float(w[i] & 0xffff0000u) * up;
            qs += x + y;
            f[i] = pack_f16(x, y);
          }
          qop[s] = as_op<Op>(f[0], f[1], f[2], f[3]);
        }
        qs = sum_across_rows(qs);
        c2_row = c2 * ldexpf(1.f, e - 14);
        const float bias = -T::kBias * qs;
        s_init = f32x4{bias, bias, bias, bias};
      } else {
#pragma unroll
        for (int s = 0; s < kSteps; ++s) qop[s] = __builtin_bit_cast(Op, raw[s]);
      }
    }
    int64_t mask_row = 0;  // of this lane's query row
    if (MASK) {
      const int rr = min(r, R - 1);
      mask_row = slot * a.mask_stride_b + (h * p.rep + rr / a.q_rows) * a.mask_stride_h + (rr % a.q_rows) * a.mask_stride_t;
    }

    f32x4 acc[kJ], accw = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    ST tile;
    float ks[8], vs[8], mk[8];
    auto base_of = [&](int t, const void* cache, const void* fresh) -> const char* {
      return t < n_new ? static_cast<const char*>(fresh) + new_row * ST::kRowBytes
                       : static_cast<const char*>(cache) + (kv0 + static_cast<int64_t>(t - n_new) * kTile) * ST::kRowBytes;
    };
    auto valid_of = [&](int t) { return t < n_new ? 1 : min(kTile, len - (t - n_new) * kTile); };
    // scales of the lane's positions; past the end: of the last position
    auto load_scales = [&](int t, const void* cache, const void* fresh, float (&out)[8]) {
      if (!SCALE) return;
      const int dt = SCALE == kScaleF32 ? JPT_F32 : JPT_BF16;
      if (t < n_new) {
        const float x = load_as_f32(fresh, static_cast<int64_t>(slot) * a.scale_heads + hs, dt);
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = x;
        return;
      }
      const int64_t s0 = sc0 + static_cast<int64_t>(t - n_new) * kTile;
      const int valid = valid_of(t);
      if (valid == kTile && S % 4 == 0) {  // runs of four, aligned (the scale tensors are, see the host's check)
        if (SCALE == kScaleF32) {
          const float4* src = reinterpret_cast<const float4*>(static_cast<const float*>(cache) + s0);
          const float4 x = src[g], y = src[4 + g];
          out[0] = x.x; out[1] = x.y; out[2] = x.z; out[3] = x.w; out[4] = y.x; out[5] = y.y; out[6] = y.z; out[7] = y.w;
        } else {
          const uint2* src = reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(cache) + s0);
          const uint2 x = src[g], y = src[4 + g];
          out[0] = __uint_as_float(x.x << 16); out[1] = __uint_as_float(x.x & 0xffff0000u);
          out[2] = __uint_as_float(x.y << 16); out[3] = __uint_as_float(x.y & 0xffff0000u);
          out[4] = __uint_as_float(y.x << 16); out[5] = __uint_as_float(y.x & 0xffff0000u);
          out[6] = __uint_as_float(y.y << 16); out[7] = __uint_as_float(y.y & 0xffff0000u);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = load_as_f32(cache, s0 + max(min(pos[i], valid - 1), 0), dt);
      }
    };
    auto load_mask = [&](int t) {
      if (!MASK) return;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        mk[i] = t < n_new ? 0.f : load_as_f32(a.mask, mask_row + min((t - n_new) * kTile + pos[i], S - 1), a.mask_dtype);
    };
    auto load_k = [&](int t) {
      tile.load_keys(base_of(t, a.k, a.new_k), max(valid_of(t), 1), r, g);
      load_scales(t, a.k_scale, a.new_k_scale, ks);
      load_mask(t);
    };
    auto load_v = [&](int t) {
      tile.load_values(base_of(t, a.v, a.new_v), max(valid_of(t), 1), r, g);
      load_scales(t, a.v_scale, a.new_v_scale, vs);
    };

    const int t0 = t_first + wave;
    if (t0 < t_end) {
      load_k(t0);
      load_v(t0);
    }
    for (int t = t0; t < t_end; t += kSplitWaves) {
      const int valid = valid_of(t), next = t + kSplitWaves;
      f32x4 sa = s_init, sb = s_init;
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        sa = T::mfma(tile.k_op(0, s), qop[s], sa);
        sb = T::mfma(tile.k_op(1, s), qop[s], sb);
      }
      float sc[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sc[i] = (i < 4 ? sa[i] : sb[i - 4]) * (SCALE ? ks[i] * c2_row : c2_row);
        if (MASK) sc[i] += mk[i] * kLog2e;
        if (valid != kTile) sc[i] = pos[i] < valid ? sc[i] : -INFINITY;
      }
      if (next < t_end) load_k(next);
      float tmax = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) tmax = fmaxf(tmax, sc[i]);
      tmax = max_across_rows(tmax);
      const float m_new = fmaxf(m_run, tmax);
      const float m_use = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = fast_exp2(m_run - m_use);
      float w[8], psum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float pr = fast_exp2(sc[i] - m_use);
        psum += pr;
        w[i] = SCALE ? pr * vs[i] : pr;
        if (SCALE && valid != kTile) w[i] = pos[i] < valid ? w[i] : 0.f;  // whatever its scale holds
      }
      l_run = l_run * alpha + psum;
      m_run = m_new;
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int j = 0; j < kJ; ++j) acc[j] *= alpha;
        if (T::kBias != 0.f) accw *= alpha;
      }
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) split_pack<KV>(w[2 * i], w[2 * i + 1], hi[i], lo[i]);
      const Op p_hi = as_op<Op>(hi[0], hi[1], hi[2], hi[3]), p_lo = as_op<Op>(lo[0], lo[1], lo[2], lo[3]);
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        const Op v = tile.v_op(j);
        acc[j] = T::mfma(v, p_hi, acc[j]);
        acc[j] = T::mfma(v, p_lo, acc[j]);
      }
      if (T::kBias != 0.f) {
        accw = T::mfma(T::ones(), p_hi, accw);
        accw = T::mfma(T::ones(), p_lo, accw);
      }
      if (next < t_end) load_v(next);
    }

    // ---- fold the four waves' parts ----
    const float l_row = sum_across_rows(l_run);
    __syncthreads();  // the previous sequence's parts have been read
    if (r < R) {
      const float bias = T::kBias * accw[0];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < kJ; j += 4)
          *reinterpret_cast<float4*>(&so[wave][r][kJ * (4 * g + i) + j]) =
              make_float4(acc[j][i] - bias, acc[j + 1][i] - bias, acc[j + 2][i] - bias, acc[j + 3][i] - bias);
      if (g == 0) {
        s_m[wave][r] = m_run;
        s_l[wave][r] = l_row;
      }
    }
    __syncthreads();
    const bool whole = t_first == 0 && t_end == nt;
    const int64_t seq_end = seq_begin + nt;
    const int g_first = whole ? me : group_of(seq_begin), g_last = whole ? me : group_of(seq_end - 1);
    const int64_t record = static_cast<int64_t>(R) * kStride;
    // the part that begins the sequence is its group's second record, every other its group's first
    float* const part = p.partials + (2 * static_cast<int64_t>(me) + (t_first == 0 ? 1 : 0)) * record;
    auto write_out = [&](int row, int d, const f32x4& o, float M, float l) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + (q_row0 + row) * D + d) =
          make_uint2(pack_bf16(o[0] * inv, o[1] * inv), pack_bf16(o[2] * inv, o[3] * inv));
      if (d == 0) {
        if (a.out_max) a.out_max[q_row0 + row] = M * kLn2;
        if (a.out_denom) a.out_denom[q_row0 + row] = l;
      }
    };
    for (int x = tid; x < R * (D / 4); x += kSplitThreads) {
      const int row = x / (D / 4), d = x % (D / 4) * 4;
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < kSplitWaves; ++w) M = fmaxf(M, s_m[w][row]);
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      float l = 0.f;
#pragma unroll
      for (int w = 0; w < kSplitWaves; ++w) {
        const float mw = s_m[w][row];
        const float f = mw == -INFINITY ? 0.f : fast_exp2(mw - M);
        l += s_l[w][row] * f;
        o += *reinterpret_cast<const f32x4*>(&so[w][row][d]) * f;
      }
      if (whole) {
        write_out(row, d, o, M, l);
      } else {  // past the caches: another XCD's group may fold it
        float* to = part + row * kStride;
        asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" : : "v"(to + d), "v"(o) : "memory");
        if (d == 0) {
          typedef __attribute__((ext_vector_type(2))) float f32x2;
          const f32x2 st = {M, l};
          asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" : : "v"(to + D), "v"(st) : "memory");
        }
      }
    }
    if (!whole) {
      asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wave's stores have arrived
      __syncthreads();
      const int parts = g_last - g_first + 1;
      if (tid == 0) {
        const int seen = __hip_atomic_fetch_add(p.counters + g_first, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (seen == parts - 1) __hip_atomic_store(p.counters + g_first, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_found[2] = seen == parts - 1;
      }
      __syncthreads();
      if (s_found[2]) {
        for (int x = tid; x < R * (D / 4); x += kSplitThreads) {
          const int row = x / (D / 4), d = x % (D / 4) * 4;
          float M = -INFINITY, l = 0.f;
          f32x4 o = {0.f, 0.f, 0.f, 0.f};
          for (int c = g_first; c <= g_last; ++c) {
            const float* from = p.partials + (2 * static_cast<int64_t>(c) + (c == g_first ? 1 : 0)) * record + row * kStride;
            f32x4 x4;
            __attribute__((ext_vector_type(2))) float st;
            asm volatile("global_load_dwordx4 %0, %2, off sc0 sc1\n\t"
                         "global_load_dwordx2 %1, %3, off sc0 sc1\n\t"
                         "s_waitcnt vmcnt(0)"
                         : "=&v"(x4), "=&v"(st) : "v"(from + d), "v"(from + D) : "memory");
            const float Mb = fmaxf(M, st[0]);
            const float keep = M == -INFINITY ? 0.f : fast_exp2(M - Mb);
            const float f = st[0] == -INFINITY ? 0.f : fast_exp2(st[0] - Mb);
            l = l * keep + st[1] * f;
            o = o * keep + x4 * f;
            M = Mb;
          }
          write_out(row, d, o, M, l);
        }
      }
    }
    // ---- the next sequence ----
    at = seq_begin + t_end;
    if (t_end == nt && at < end) {
      if (++h == H) {
        h = 0;
        ++slot;
        slot_begin = at;
        len = __builtin_amdgcn_readfirstlane(length_of(slot));
        nt = tiles_of(len);
      }
    }
  }
}

int32_t compute_units() {
  static const int32_t v = [] {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
    return cus;
  }();
  return v;
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
  const bool small = p.rows <= 4;
  if (p.a.mask) {
    if (small) hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, true, 4>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, true, kMaxRows>), grid, block, 0, stream, p);
  } else {
    if (small) hipLaunchKernelGGL((attn_split_kernel<D, KV, SCALE, false, 4>), grid, block, 0, stream, p);
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
  if (static_cast<int64_t>(a.batch) * (a.seq / kTile + 2) >= (1ll << 31)) return false;
  // the partials lie where a plan's do, behind its entries: a workspace that holds a plan keeps it
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
  p.partials = reinterpret_cast<float*>(static_cast<char*>(a.workspace) + attn_partials_offset(a));
  const dim3 grid(static_cast<unsigned>(decode::split_groups(a)));
  if (a.dim == 64) decode::launch_split_dim<64>(p, grid, stream);
  else if (a.dim == 128) decode::launch_split_dim<128>(p, grid, stream);
  else decode::launch_split_dim<256>(p, grid, stream);
  return launch_status("attn_split_kernel");
}

}  // namespace jpt
