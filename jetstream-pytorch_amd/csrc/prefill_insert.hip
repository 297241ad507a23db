// Prefill -> decode insert: a prompt's K and V rows (heads, tokens, dim) written
// into one slot of a dense cache (with ring wrap) or into the slot's pages,
// either copied or quantised per token to int8 with the insert quantiser.
//
// HBM-bound data movement: the prompt is read once, codes (or rows) and scales
// are written.  Rows of whole, aligned 16-byte pieces are copied by
// prefill_copy_kernel and, from bf16, quantised by prefill_insert_rows_kernel;
// any other dtype, shape or alignment takes prefill_insert_kernel.
#include "common.h"

namespace jpt {
namespace {

constexpr int kPieces = 4;
// How a workgroup's threads are laid out: heads x tokens x 2^lanes_log lanes of a row, `passes` heads a thread; `along`:
// `passes` tokens a thread instead, of the one head.
struct RowSplit {
  int lanes_log, tokens_log, passes;
  bool along = false;
  constexpr int tokens_a_block() const { return (along ? passes : 1) << tokens_log; }
};
constexpr RowSplit kLlamaRows = {4, 3, 4}, kOneWideRow = {7, 1, kPieces, true};  // 8 heads of 128 elements; one of 1024
// False: the shape is not taken (a row is a power of two of pieces up to 64, a token's pieces four a thread).
bool split_rows(int heads, int dim, RowSplit* s) {
  const int lanes = dim / 8;
  if (heads == 1 && lanes == 128 && dim % 8 == 0) {
    *s = kOneWideRow;
    return true;
  }
  if (dim < 8 || dim % 8 != 0 || lanes > 64 || (lanes & (lanes - 1)) != 0 || heads < 1 || heads * lanes > 256 * kPieces) return false;
  s->lanes_log = 0;
  while ((1 << s->lanes_log) < lanes) ++s->lanes_log;
  // as many tokens as leave a thread four heads: long runs of one head
  for (s->tokens_log = 8 - s->lanes_log;; --s->tokens_log) {
    const int heads_a_pass = 256 >> (s->tokens_log + s->lanes_log);
    s->passes = (heads + heads_a_pass - 1) / heads_a_pass;
    if (s->passes <= kPieces) return true;
  }
}

// Layers that are tensors of their own (no common stride) come as a table of
// pointers inside the kernel arguments.
constexpr int kTableLayers = 64;
struct InsertParams {
  jpt_prefill_insert_args a;
  jpt_insert_state_row state;  // (no mask and no rows: nothing to write)
  RowSplit split;  // of the rows kernel
  int32_t use_table;
  const void* src_k[kTableLayers];
  const void* src_v[kTableLayers];
  void* dst_k[kTableLayers];
  void* dst_v[kTableLayers];
  void* k_scale[kTableLayers];
  void* v_scale[kTableLayers];
};

// A copy's: no scales, and the ids of the pages, where they came from the host.
struct CopyParams {
  jpt_prefill_insert_args a;
  jpt_insert_state_row state;
  int32_t use_table, host_pages;
  const void* src_k[kTableLayers];
  const void* src_v[kTableLayers];
  void* dst_k[kTableLayers];
  void* dst_v[kTableLayers];
  int32_t ids[JPT_INSERT_HOST_PAGES];
};
static_assert(sizeof(InsertParams) <= 4096 && sizeof(CopyParams) <= 4096, "what kernel arguments may be");

// The slot's row of the decode state, by the workgroups of one layer and tensor that lie along x.
__device__ __forceinline__ void state_row(const jpt_insert_state_row& s, int slot) {
  const int64_t first = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x, step = static_cast<int64_t>(gridDim.x) * blockDim.x;
  if (s.mask) {
    for (int64_t x = first; x < s.seq; x += step) {
      const bool live = s.wrap ? (x >= s.lo || x < s.hi) : (x >= s.lo && x < s.hi);
      if (s.mask_dtype == JPT_BF16) static_cast<uint16_t*>(s.mask)[slot * s.seq + x] = live ? 0 : 0xff80u;
      else static_cast<uint32_t*>(s.mask)[slot * s.seq + x] = live ? 0 : 0xff800000u;
    }
  }
  if (first == 0) {
    if (s.start) s.start[slot] = s.first;
    if (s.input_pos) s.input_pos[slot] = s.position;
    if (s.lens) s.lens[slot] = s.length;
  }
}

// Source, destination and scale tensor of (layer, K|V): the table's, or the
// first layer's moved on by the layer strides.
__device__ __forceinline__ void layer_tensors(const InsertParams& p, int layer, bool is_v, int esz_in, int esz_out,
                                              int esz_scale, const void** src, char** dst, void** scale) {
  const jpt_prefill_insert_args& a = p.a;
  if (p.use_table) {
    *src = is_v ? p.src_v[layer] : p.src_k[layer];
    *dst = static_cast<char*>(is_v ? p.dst_v[layer] : p.dst_k[layer]);
    *scale = is_v ? p.v_scale[layer] : p.k_scale[layer];
    return;
  }
  *src = static_cast<const char*>(is_v ? a.src_v : a.src_k) + layer * a.src_layer_stride * esz_in;
  *dst = static_cast<char*>(is_v ? a.dst_v : a.dst_k) + layer * a.dst_layer_stride * esz_out;
  void* s0 = is_v ? a.v_scale : a.k_scale;
  *scale = s0 == nullptr ? nullptr : static_cast<char*>(s0) + layer * a.scale_layer_stride * esz_scale;
}

template <bool ROUND_BF16>
__device__ __forceinline__ float rnd(float x) {
  return ROUND_BF16 ? round_to_bf16(x) : x;
}

// four consecutive elements of the source row as float
__device__ __forceinline__ void load4(const void* src, int64_t i, int dtype, float* x) {
  if (dtype == JPT_BF16) {
    const uint2 raw = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(src) + i);
    x[0] = __uint_as_float(raw.x << 16);
    x[1] = __uint_as_float(raw.x & 0xffff0000u);
    x[2] = __uint_as_float(raw.y << 16);
    x[3] = __uint_as_float(raw.y & 0xffff0000u);
  } else {
    const float4 raw = *reinterpret_cast<const float4*>(static_cast<const float*>(src) + i);
    x[0] = raw.x; x[1] = raw.y; x[2] = raw.z; x[3] = raw.w;
  }
}

// A workgroup a (token, K|V, layer).  dim % 4 == 0.  The op order of the quantiser is that of
// jpt_kv_append_quant_i8 (each op rounded to the scale dtype):
//   trunc: a = absmax; s = a / 127;             q = x / s;      code = trunc(q)
//   rne:   a = max(absmax, eps); s = a / 127; r = 1 / s; q = x * r;
//          code = clamp(rint(q), -128, 127)
template <bool BF16_MATH>
__global__ void __launch_bounds__(256) prefill_insert_kernel(InsertParams p) {
  const jpt_prefill_insert_args& a = p.a;
  const int t = blockIdx.x;
  const bool is_v = blockIdx.y == 1;
  const int layer = blockIdx.z;
  const bool paged = a.page_ids != nullptr;
  const bool quant = a.dst_dtype == JPT_I8 && a.in_dtype != JPT_I8;
  const int H = a.heads, D = a.dim, HD = H * D;
  const int esz_in = a.in_dtype == JPT_F32 ? 4 : a.in_dtype == JPT_BF16 ? 2 : 1;
  const int esz_out = quant ? 1 : esz_in;
  const int esz_scale = a.scale_dtype == JPT_F32 ? 4 : 2;
  const void* src;
  char* dst;
  void* scale_out;
  layer_tensors(p, layer, is_v, esz_in, esz_out, esz_scale, &src, &dst, &scale_out);

  // destination row of (this token, head h): element index row * D
  int64_t pool_row = 0;  // dense: position in the slot's row; paged: row in the pool
  if (paged) {
    const int page = a.page_ids[t / a.page_size];
    if (page < 0 || page >= a.total_pages) return;
    pool_row = static_cast<int64_t>(page) * a.page_size + t % a.page_size;
  } else {
    int at = (a.start + t) % a.seq;
    pool_row = at < 0 ? at + a.seq : at;
  }
  auto row_of = [&](int h) -> int64_t {
    return paged ? static_cast<int64_t>(h) * a.total_pages * a.page_size + pool_row
                 : (static_cast<int64_t>(a.slot) * H + h) * a.seq + pool_row;
  };
  auto scale_index = [&](int g) -> int64_t {
    return paged ? static_cast<int64_t>(g) * a.total_pages * a.page_size + pool_row
                 : (static_cast<int64_t>(a.slot) * a.scale_heads + g) * a.seq + pool_row;
  };

  if (t >= a.tokens) {  // paged only: the tail of the last page is zero-filled
    for (int i = 4 * threadIdx.x; i < HD; i += 4 * blockDim.x) {
      const int h = i / D, d = i - h * D;
      char* out = dst + (row_of(h) * D + d) * esz_out;
      if (esz_out == 1) *reinterpret_cast<uint32_t*>(out) = 0u;
      else if (esz_out == 2) *reinterpret_cast<uint2*>(out) = make_uint2(0u, 0u);
      else *reinterpret_cast<uint4*>(out) = make_uint4(0u, 0u, 0u, 0u);
    }
    return;
  }
  const int64_t head_stride = a.src_head_stride > 0 ? a.src_head_stride : static_cast<int64_t>(a.tokens) * D;
  auto src_index = [&](int h, int d) -> int64_t { return h * head_stride + static_cast<int64_t>(t) * D + d; };

  if (!quant) {  // copy
    for (int i = 4 * threadIdx.x; i < HD; i += 4 * blockDim.x) {
      const int h = i / D, d = i - h * D;
      const char* in = static_cast<const char*>(src) + src_index(h, d) * esz_in;
      char* out = dst + (row_of(h) * D + d) * esz_in;
      if (esz_in == 1) *reinterpret_cast<uint32_t*>(out) = *reinterpret_cast<const uint32_t*>(in);
      else if (esz_in == 2) *reinterpret_cast<uint2*>(out) = *reinterpret_cast<const uint2*>(in);
      else *reinterpret_cast<uint4*>(out) = *reinterpret_cast<const uint4*>(in);
    }
    return;
  }

  __shared__ float s_red[4];
  __shared__ float s_scale[64];
  const int groups = a.scale_heads;  // 1 or H
  const int per_group = HD / groups;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int g = 0; g < groups; ++g) {
    float m = 0.f;
    for (int i = 4 * threadIdx.x; i < per_group; i += 4 * blockDim.x) {
      const int e = g * per_group + i, h = e / D, d = e - h * D;
      float x[4];
      load4(src, src_index(h, d), a.in_dtype, x);
      m = fmaxf(m, fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))));
    }
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (lane == 0) s_red[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
      float amax = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
      if (a.rounding == JPT_ROUND_RNE) amax = fmaxf(amax, rnd<BF16_MATH>(1e-5f));
      s_scale[g] = rnd<BF16_MATH>(amax / 127.0f);
    }
    __syncthreads();
  }
  for (int i = 4 * threadIdx.x; i < HD; i += 4 * blockDim.x) {
    const int h = i / D, d = i - h * D;
    const float s = s_scale[groups == 1 ? 0 : h];
    float x[4];
    load4(src, src_index(h, d), a.in_dtype, x);
    int code[4];
    if (a.rounding == JPT_ROUND_TRUNC) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float q = rnd<BF16_MATH>(x[j] / s);
        code[j] = (q != q) ? 0 : static_cast<int>(q);
      }
    } else {
      const float r = rnd<BF16_MATH>(1.0f / s);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float q = rnd<BF16_MATH>(x[j] * r);
        code[j] = static_cast<int>(fminf(fmaxf(rintf(q), -128.f), 127.f));
      }
    }
    const uint32_t packed = (static_cast<uint32_t>(code[0]) & 0xffu) | ((static_cast<uint32_t>(code[1]) & 0xffu) << 8) |
                            ((static_cast<uint32_t>(code[2]) & 0xffu) << 16) | (static_cast<uint32_t>(code[3]) << 24);
    *reinterpret_cast<uint32_t*>(dst + row_of(h) * D + d) = packed;
  }
  if (threadIdx.x < groups) store_from_f32(scale_out, scale_index(threadIdx.x), a.scale_dtype, s_scale[threadIdx.x]);
}

// bf16 prompts quantised, laid out for memory: a workgroup takes a few consecutive tokens in all heads.  A thread keeps
// one 16-byte piece of one token's row in up to four heads, so that the lanes of a wave read consecutive rows of one head
// (1 KiB in one piece at 128 elements a row and four tokens or more) and write contiguous codes, the token's position or
// page is worked out once, and the prompt is read once: the pieces stay in registers, all asked for before the first wait,
// between the absmax pass and the quantise pass.  A token's absmax: over the lanes that share its row, then (one scale a
// token) over the thread's heads and, in LDS, the waves that have the others.  Same op order as the general kernel.
// Measured, 16 layers into a slot with bf16 scales, heads x dim, tokens; prefill_insert_kernel -> this, us a call: 32x128,
// 1000: 154.5 -> 78 (5.0 TB/s read and written); 8x256, 1200: 106 -> 46; 4x128, 1500: 70.6 -> 18.6; 8x64, 1000: 50 ->
// 14.3; 1x128, 900: 35.5 -> 7.4.  Four heads a thread and not fewer: one a thread takes 93.5, 71, 23, 18 and 6.7 there, two
// 94, 52, 18.5, 14 and 6.7 (the prompts out of memory; out of the caches one a thread is the fastest by far).
// The `block`-th workgroup's tokens of the prompt `a` describes (tokens, page_ids, n_pages,
// src_head_stride), read from src, written to dst / scale_out.
template <bool BF16_MATH, int PASSES, bool ALONG = false>
__device__ __forceinline__ void quant_insert_rows(const jpt_prefill_insert_args& a, const RowSplit split, const int H, const int D,
                                                  const uint16_t* src, char* dst, void* scale_out, int block) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  const int lanes = 1 << split.lanes_log, tokens = 1 << split.tokens_log;
  const bool paged = a.page_ids != nullptr;
  const int rows = paged ? a.n_pages * a.page_size : a.tokens;
  const int groups = a.scale_heads;
  const int64_t head_stride = a.src_head_stride > 0 ? a.src_head_stride : static_cast<int64_t>(a.tokens) * D;
  const int piece = threadIdx.x & (lanes - 1), tq = (threadIdx.x >> split.lanes_log) & (tokens - 1);
  const int d = 8 * piece;
  // the thread's heads: h0 .. h0 + PASSES - 1, of one token; ALONG: its tokens, of one head
  const int h0 = (threadIdx.x >> (split.lanes_log + split.tokens_log)) * (ALONG ? 1 : PASSES);
  constexpr int kTokens = ALONG ? PASSES : 1;
  int t[kTokens];
#pragma unroll
  for (int j = 0; j < kTokens; ++j) t[j] = (block * kTokens + j) * tokens + tq;

  // addresses clamped into the prompt, results masked afterwards
  u32x4 raw[PASSES];
#pragma unroll
  for (int j = 0; j < PASSES; ++j) {
    const uint16_t* const from = src + static_cast<int64_t>(min(t[ALONG ? j : 0], a.tokens - 1)) * D + d;
    raw[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(from + min(ALONG ? h0 : h0 + j, H - 1) * head_stride));  // read once
  }
  int64_t pool_row[kTokens];  // dense: position in the slot's row; paged: row in the pool; -1: nothing to write
#pragma unroll
  for (int j = 0; j < kTokens; ++j) {
    const int page = paged ? a.page_ids[min(t[j], rows - 1) / a.page_size] : 0;
    pool_row[j] = -1;
    if (t[j] < rows) {
      if (paged) {
        if (page >= 0 && page < a.total_pages) pool_row[j] = static_cast<int64_t>(page) * a.page_size + t[j] % a.page_size;
      } else {
        const int at = (a.start + t[j]) % a.seq;
        pool_row[j] = at < 0 ? at + a.seq : at;
      }
    }
  }
  float m[PASSES];
#pragma unroll
  for (int j = 0; j < PASSES; ++j) {
    m[j] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      m[j] = fmaxf(m[j], fmaxf(fabsf(__uint_as_float(raw[j][i] << 16)), fabsf(__uint_as_float(raw[j][i] & 0xffff0000u))));
  }
  __shared__ float s_max[256];  // by (the threads' heads, token); ALONG: by (pass, token, wave of the row)
  if constexpr (ALONG) {  // a row is two waves'
#pragma unroll
    for (int j = 0; j < PASSES; ++j) {
      for (int off = 32; off > 0; off >>= 1) m[j] = fmaxf(m[j], __shfl_xor(m[j], off));
      if ((piece & 63) == 0) s_max[4 * j + (threadIdx.x >> 6)] = m[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PASSES; ++j) m[j] = fmaxf(s_max[4 * j + 2 * tq], s_max[4 * j + 2 * tq + 1]);
  } else if (groups == 1) {
    // (a head clamped above is one that counts anyway)
#pragma unroll
    for (int j = 1; j < PASSES; ++j) m[0] = fmaxf(m[0], m[j]);
    for (int off = lanes / 2; off > 0; off >>= 1) m[0] = fmaxf(m[0], __shfl_xor(m[0], off));
    if (piece == 0) s_max[threadIdx.x >> split.lanes_log] = m[0];
    __syncthreads();
    for (int i = tq; i < (256 >> split.lanes_log); i += tokens) m[0] = fmaxf(m[0], s_max[i]);
#pragma unroll
    for (int j = 1; j < PASSES; ++j) m[j] = m[0];
  } else {
#pragma unroll
    for (int j = 0; j < PASSES; ++j)
      for (int off = lanes / 2; off > 0; off >>= 1) m[j] = fmaxf(m[j], __shfl_xor(m[j], off));
  }
  if (!ALONG && pool_row[0] < 0) return;
  const int64_t head_rows = paged ? static_cast<int64_t>(a.total_pages) * a.page_size : a.seq;
  const int64_t row0 = paged ? 0 : static_cast<int64_t>(a.slot) * H * a.seq;
#pragma unroll
  for (int j = 0; j < PASSES; ++j) {
    const int h = ALONG ? h0 : h0 + j, i_t = ALONG ? j : 0;
    if (!ALONG && h >= H) break;
    if (ALONG && (h >= H || pool_row[j] < 0)) continue;
    u32x2* out = reinterpret_cast<u32x2*>(dst + (row0 + pool_row[i_t] + h * head_rows) * D + d);
    if (t[i_t] >= a.tokens) {  // paged only: the tail of the last page is zero-filled
      *out = u32x2{0u, 0u};
      continue;
    }
    float amax = m[j];
    if (a.rounding == JPT_ROUND_RNE) amax = fmaxf(amax, rnd<BF16_MATH>(1e-5f));
    const float s = rnd<BF16_MATH>(amax / 127.0f);
    uint32_t code[8];
    const float inv = a.rounding == JPT_ROUND_TRUNC ? 0.f : rnd<BF16_MATH>(1.0f / s);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = __uint_as_float((i & 1) ? raw[j][i / 2] & 0xffff0000u : raw[j][i / 2] << 16);
      if (a.rounding == JPT_ROUND_TRUNC) {
        const float q = rnd<BF16_MATH>(x / s);
        code[i] = static_cast<uint32_t>((q != q) ? 0 : static_cast<int>(q)) & 0xffu;
      } else {
        const float q = rnd<BF16_MATH>(x * inv);
        code[i] = static_cast<uint32_t>(static_cast<int>(fminf(fmaxf(rintf(q), -128.f), 127.f))) & 0xffu;
      }
    }
    // written once, read by later launches only: keep it out of the way of the prompt being read
    const u32x2 packed = {code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24),
                          code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24)};
    __builtin_nontemporal_store(packed, out);
    if (d == 0 && (groups != 1 || h == 0)) {
      const int64_t idx = (paged ? 0 : static_cast<int64_t>(a.slot) * groups * a.seq) + (groups == 1 ? 0 : h) * head_rows + pool_row[i_t];
      store_from_f32(scale_out, idx, a.scale_dtype, s);
    }
  }
}

// Two shapes have numbers that the compiler knows, in kernels of their own (both compared while a rounding to bf16 took six
// instructions; with one, kOneWide takes 23.5 and 61).  kLlama: 1500 tokens, 16 layers 50.6 us a call, 52.8 through the
// other branch.  kOneWide, whose threads would have one piece each: 900 and 3000 tokens, 16 layers 30 and 79 us
// (prefill_insert_kernel 57 and 176; this layout in the other branch 36 and 93, which cost that branch's shapes 3 % too).
enum RowShape { kAnyShape, kLlama, kOneWide };
template <bool BF16_MATH, RowShape SHAPE>
__device__ __forceinline__ void quant_insert_block(const jpt_prefill_insert_args& a, const RowSplit& split, const uint16_t* src,
                                                   char* dst, void* scale_out, int block) {
  if constexpr (SHAPE == kLlama) {
    quant_insert_rows<BF16_MATH, 4>(a, kLlamaRows, 8, 128, src, dst, scale_out, block);
  } else if constexpr (SHAPE == kOneWide) {
    quant_insert_rows<BF16_MATH, kPieces, true>(a, kOneWideRow, 1, 1024, src, dst, scale_out, block);
  } else {
    if (split.passes == 4) quant_insert_rows<BF16_MATH, 4>(a, split, a.heads, a.dim, src, dst, scale_out, block);
    else if (split.passes == 3) quant_insert_rows<BF16_MATH, 3>(a, split, a.heads, a.dim, src, dst, scale_out, block);
    else if (split.passes == 2) quant_insert_rows<BF16_MATH, 2>(a, split, a.heads, a.dim, src, dst, scale_out, block);
    else quant_insert_rows<BF16_MATH, 1>(a, split, a.heads, a.dim, src, dst, scale_out, block);
  }
}
RowShape row_shape(const jpt_prefill_insert_args& a, const RowSplit& split) {
  return split.along ? kOneWide : a.heads == 8 && a.dim == 128 ? kLlama : kAnyShape;
}

template <bool BF16_MATH, RowShape SHAPE>
__global__ void __launch_bounds__(256) prefill_insert_rows_kernel(InsertParams p) {
  const jpt_prefill_insert_args& a = p.a;
  const bool is_v = blockIdx.y == 1;
  const void* src;
  char* dst;
  void* scale_out;
  layer_tensors(p, blockIdx.z, is_v, 2, 1, a.scale_dtype == JPT_F32 ? 4 : 2, &src, &dst, &scale_out);
  if (blockIdx.z == 0 && !is_v) state_row(p.state, a.slot);
  quant_insert_block<BF16_MATH, SHAPE>(a, p.split, static_cast<const uint16_t*>(src), dst, scale_out, blockIdx.x);
}

// Rows copied as they are, 16 bytes a piece: a workgroup takes 1024 consecutive pieces of one head's rows (16 KiB: 64
// rows of 128 bf16), four a thread, asked for before the first is written.  The ordinary kernel
// moves 2 KiB a workgroup with one load in flight a thread.  Measured, 16 layers of bf16 rows, us a call, before -> now:
// pages of 64, 8x128, 1500 tokens 75 -> 56; pages of 32, 8x128, 4000 tokens 158 -> 113 (4.6 TB/s); 1x128, 2000 tokens 69
// -> 23; 32x128, 1500 tokens 166 -> 165 (4.8 TB/s before, too); a slot, 8x128, 1000 tokens 34.5 -> 27.
// `HOST_PAGES`: the pages' ids are among the arguments (uploaded ahead of the launch, from pageable memory, they held the
// host up for 40 us: the first case above from the allocator's ids 54.5 -> 38.8 us a call, 5.1 TB/s).
template <bool HOST_PAGES>
__global__ void __launch_bounds__(256) prefill_copy_kernel(CopyParams p, int esz, int pieces_a_row) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const jpt_prefill_insert_args& a = p.a;
  const int h = blockIdx.y >> 1, layer = blockIdx.z;
  const bool is_v = blockIdx.y & 1;
  const char* src = static_cast<const char*>(is_v ? a.src_v : a.src_k) + layer * a.src_layer_stride * esz;
  char* dst = static_cast<char*>(is_v ? a.dst_v : a.dst_k) + layer * a.dst_layer_stride * esz;
  if (p.use_table) {
    src = static_cast<const char*>(is_v ? p.src_v[layer] : p.src_k[layer]);
    dst = static_cast<char*>(is_v ? p.dst_v[layer] : p.dst_k[layer]);
  }
  if (layer == 0 && blockIdx.y == 0) state_row(p.state, a.slot);
  const int32_t* const ids = HOST_PAGES ? p.ids : a.page_ids;
  const bool paged = HOST_PAGES || ids != nullptr;
  const int rows = paged ? a.n_pages * a.page_size : a.tokens;
  const int64_t row_bytes = 16ll * pieces_a_row;
  const int64_t head_bytes = a.src_head_stride > 0 ? a.src_head_stride * esz : a.tokens * row_bytes;
  const char* const from = src + h * head_bytes;
  u32x4 x[kPieces];
  int t[kPieces], off[kPieces], page[kPieces];
#pragma unroll
  for (int j = 0; j < kPieces; ++j) {
    const int i = (static_cast<int>(blockIdx.x) * kPieces + j) * 256 + static_cast<int>(threadIdx.x);
    t[j] = i / pieces_a_row;
    off[j] = 16 * (i - t[j] * pieces_a_row);
    // pieces of the zero-filled tail, and past it, read nothing
    x[j] = u32x4{0u, 0u, 0u, 0u};
    if (t[j] < a.tokens) x[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(from + t[j] * row_bytes + off[j]));
  }
#pragma unroll
  for (int j = 0; j < kPieces; ++j) page[j] = paged ? ids[min(t[j], rows - 1) / a.page_size] : 0;
#pragma unroll
  for (int j = 0; j < kPieces; ++j) {
    if (t[j] >= rows || (paged && (page[j] < 0 || page[j] >= a.total_pages))) continue;
    int64_t row;
    if (paged) {
      row = (static_cast<int64_t>(h) * a.total_pages + page[j]) * a.page_size + t[j] % a.page_size;
    } else {
      const int at = (a.start + t[j]) % a.seq;
      row = (static_cast<int64_t>(a.slot) * a.heads + h) * a.seq + (at < 0 ? at + a.seq : at);
    }
    __builtin_nontemporal_store(x[j], reinterpret_cast<u32x4*>(dst + row * row_bytes + off[j]));
  }
}

// Several prompts into the pages of one stacked pool in one launch: the
// workgroups of all prompts side by side (prompt r owns those from
// first_block[r] on), layers along z by the layer strides.
constexpr int kLaunchPrompts = 32;
struct PromptsParams {
  RowSplit split;
  jpt_prefill_insert_args a;  // destination, geometry, dtypes; its source and page fields are unused
  int32_t n_prompts;
  int32_t first_block[kLaunchPrompts + 1];
  jpt_insert_prompt prompt[kLaunchPrompts];
};

template <bool BF16_MATH, RowShape SHAPE>
__global__ void __launch_bounds__(256) prefill_insert_prompts_kernel(PromptsParams p) {
  int r = 0;
  while (r + 1 < p.n_prompts && static_cast<int>(blockIdx.x) >= p.first_block[r + 1]) ++r;
  const jpt_insert_prompt& pr = p.prompt[r];
  jpt_prefill_insert_args a = p.a;
  a.tokens = pr.tokens;
  a.n_pages = pr.n_pages;
  a.page_ids = pr.page_ids;
  a.src_head_stride = pr.src_head_stride;
  const bool is_v = blockIdx.y == 1;
  const int layer = blockIdx.z;
  const uint16_t* src = static_cast<const uint16_t*>(is_v ? pr.src_v : pr.src_k) + layer * pr.src_layer_stride;
  char* dst = static_cast<char*>(is_v ? a.dst_v : a.dst_k) + layer * a.dst_layer_stride;
  const int esz_scale = a.scale_dtype == JPT_F32 ? 4 : 2;
  void* scale_out = static_cast<char*>(is_v ? a.v_scale : a.k_scale) + layer * a.scale_layer_stride * esz_scale;
  quant_insert_block<BF16_MATH, SHAPE>(a, p.split, src, dst, scale_out, static_cast<int>(blockIdx.x) - p.first_block[r]);
}

}  // namespace
}  // namespace jpt

namespace jpt {
namespace {

// Checks and launches.  layers == nullptr: the tensors of args, n_layers of them
// a layer stride apart; else a table of at most kTableLayers layers.  `state`: NULL, or the slot's row to write beside,
// `*wrote` says whether it was.  `host_ids`: the pages' ids, and nothing but the copy kernel, or 1.
int32_t insert_launch(const jpt_prefill_insert_args& a, const jpt_insert_layer* layers, int32_t n_table, void* stream,
                      const jpt_insert_state_row* state = nullptr, bool* wrote = nullptr, const int32_t* host_ids = nullptr) {
  const bool paged = a.page_ids != nullptr || host_ids != nullptr;
  JPT_REQUIRE(a.tokens >= 0 && a.heads > 0 && a.dim > 0, "tokens, heads, dim out of range");
  JPT_REQUIRE(a.dim % 4 == 0, "dim must be a multiple of 4");
  JPT_REQUIRE(a.in_dtype == JPT_BF16 || a.in_dtype == JPT_F32 || a.in_dtype == JPT_I8, "bad in_dtype");
  const bool quant = a.dst_dtype == JPT_I8 && a.in_dtype != JPT_I8;
  JPT_REQUIRE(quant || a.dst_dtype == a.in_dtype, "dst_dtype must be in_dtype (copy) or int8 (quantise)");
  if (quant && host_ids) return 1;  // the quantising kernels read ids from the device
  const int esz = a.in_dtype == JPT_F32 ? 4 : a.in_dtype == JPT_BF16 ? 2 : 1;
  const int esz_out = quant ? 1 : esz;
  JPT_REQUIRE(a.src_head_stride == 0 || (a.src_head_stride >= static_cast<int64_t>(a.tokens) * a.dim && a.src_head_stride % 4 == 0),
              "src_head_stride must cover the tokens and be a multiple of 4");
  if (quant) {
    JPT_REQUIRE(a.scale_dtype == a.in_dtype || a.scale_dtype == JPT_F32, "scale_dtype must equal in_dtype or be f32");
    JPT_REQUIRE(a.scale_heads == 1 || a.scale_heads == a.heads, "scale_heads must be 1 or heads");
    JPT_REQUIRE(a.scale_heads <= 64, "per-head scales support at most 64 heads");
    JPT_REQUIRE(a.rounding == JPT_ROUND_TRUNC || a.rounding == JPT_ROUND_RNE, "bad rounding mode");
  }
  InsertParams p{};
  p.a = a;
  bool wide_ok = true, pieces_ok = true;  // every tensor is aligned for the wide quantising kernel, for 16-byte copies
  auto check_layer = [&](const void* sk, const void* sv, const void* dk, const void* dv, const void* ks,
                         const void* vs) -> int32_t {
    JPT_REQUIRE(sk && sv && dk && dv, "NULL tensor argument");
    JPT_REQUIRE(aligned(sk, 4 * esz) && aligned(sv, 4 * esz), "source rows must be aligned to four elements");
    JPT_REQUIRE(aligned(dk, 4 * esz_out) && aligned(dv, 4 * esz_out), "destination must be aligned to four elements");
    if (quant) JPT_REQUIRE(ks && vs, "k_scale/v_scale are NULL");
    wide_ok = wide_ok && aligned(sk, 16) && aligned(sv, 16) && aligned(dk, 8) && aligned(dv, 8);
    pieces_ok = pieces_ok && aligned(sk, 16) && aligned(sv, 16) && aligned(dk, 16) && aligned(dv, 16);
    return JPT_OK;
  };
  if (layers) {
    JPT_REQUIRE(n_table >= 1 && n_table <= kTableLayers, "1..%d layers a table", kTableLayers);
    p.use_table = 1;
    p.a.n_layers = n_table;
    for (int l = 0; l < n_table; ++l) {
      const jpt_insert_layer& t = layers[l];
      const int32_t st = check_layer(t.src_k, t.src_v, t.dst_k, t.dst_v, t.k_scale, t.v_scale);
      if (st != JPT_OK) return st;
      p.src_k[l] = t.src_k; p.src_v[l] = t.src_v;
      p.dst_k[l] = t.dst_k; p.dst_v[l] = t.dst_v;
      p.k_scale[l] = t.k_scale; p.v_scale[l] = t.v_scale;
    }
  } else {
    const int32_t st = check_layer(a.src_k, a.src_v, a.dst_k, a.dst_v, a.k_scale, a.v_scale);
    if (st != JPT_OK) return st;
    JPT_REQUIRE(a.src_layer_stride % 4 == 0 && a.dst_layer_stride % 4 == 0, "layer strides must be multiples of 4");
    if (p.a.n_layers <= 0) p.a.n_layers = 1;
    JPT_REQUIRE(p.a.n_layers <= 65535, "n_layers out of range");
    wide_ok = wide_ok && a.src_layer_stride % 8 == 0 && a.dst_layer_stride % 8 == 0;
    pieces_ok = pieces_ok && a.src_layer_stride * esz % 16 == 0 && a.dst_layer_stride * esz % 16 == 0;
  }
  int32_t rows = a.tokens;
  if (paged) {
    JPT_REQUIRE(a.total_pages > 0 && a.page_size > 0 && a.n_pages >= 0, "paged geometry out of range");
    JPT_REQUIRE(static_cast<int64_t>(a.n_pages) * a.page_size >= a.tokens, "too few pages for %d tokens", a.tokens);
    rows = a.n_pages * a.page_size;
  } else {
    JPT_REQUIRE(a.seq > 0 && a.batch > 0 && a.slot >= 0 && a.slot < a.batch, "slot or seq out of range");
    JPT_REQUIRE(a.tokens <= a.seq, "%d tokens do not fit a cache of %d positions", a.tokens, a.seq);
  }
  if (rows == 0) return JPT_OK;
  if (state) p.state = *state;
  if (quant && wide_ok && a.tokens > 0 && a.in_dtype == JPT_BF16 && split_rows(a.heads, a.dim, &p.split) &&
      (a.src_head_stride == 0 || a.src_head_stride % 8 == 0)) {
    const int tb = p.split.tokens_a_block();
    const dim3 blocks((rows + tb - 1) / tb, 2, p.a.n_layers);
    using Kernel = decltype(&prefill_insert_rows_kernel<true, kAnyShape>);
    static constexpr Kernel kernels[2][3] = {
        {prefill_insert_rows_kernel<false, kAnyShape>, prefill_insert_rows_kernel<false, kLlama>, prefill_insert_rows_kernel<false, kOneWide>},
        {prefill_insert_rows_kernel<true, kAnyShape>, prefill_insert_rows_kernel<true, kLlama>, prefill_insert_rows_kernel<true, kOneWide>}};
    const Kernel kernel = kernels[a.scale_dtype != JPT_F32][row_shape(a, p.split)];
    hipLaunchKernelGGL(kernel, blocks, dim3(256), 0, static_cast<hipStream_t>(stream), p);
    if (wrote) *wrote = true;
    return launch_status("prefill_insert_rows_kernel");
  }
  // rows of whole 16-byte pieces, all of them aligned, in numbers that 32 bits and a grid count: never slower above
  const int64_t row_pieces = static_cast<int64_t>(a.dim) * esz / 16;
  if (!quant && pieces_ok && a.dim * esz % 16 == 0 && a.src_head_stride * esz % 16 == 0 &&
      rows * row_pieces < (1ll << 31) - 256 * kPieces && a.heads < 32768) {
    const dim3 blocks(static_cast<unsigned>((rows * row_pieces + 256 * kPieces - 1) / (256 * kPieces)), 2 * a.heads, p.a.n_layers);
    CopyParams c{};
    c.a = p.a;
    c.state = p.state;
    c.use_table = p.use_table;
    for (int l = 0; p.use_table && l < kTableLayers; ++l) {
      c.src_k[l] = p.src_k[l]; c.src_v[l] = p.src_v[l];
      c.dst_k[l] = p.dst_k[l]; c.dst_v[l] = p.dst_v[l];
    }
    if (host_ids) {
      for (int i = 0; i < a.n_pages; ++i) c.ids[i] = host_ids[i];
      hipLaunchKernelGGL(prefill_copy_kernel<true>, blocks, dim3(256), 0, static_cast<hipStream_t>(stream), c, esz, static_cast<int>(row_pieces));
    } else {
      hipLaunchKernelGGL(prefill_copy_kernel<false>, blocks, dim3(256), 0, static_cast<hipStream_t>(stream), c, esz, static_cast<int>(row_pieces));
    }
    if (wrote) *wrote = true;
    return launch_status("prefill_copy_kernel");
  }
  if (host_ids) return 1;
  dim3 grid(rows, 2, p.a.n_layers);
  if (quant && a.scale_dtype == JPT_BF16)
    hipLaunchKernelGGL(prefill_insert_kernel<true>, grid, dim3(256), 0, static_cast<hipStream_t>(stream), p);
  else
    hipLaunchKernelGGL(prefill_insert_kernel<false>, grid, dim3(256), 0, static_cast<hipStream_t>(stream), p);
  return launch_status("prefill_insert_kernel");
}

}  // namespace
}  // namespace jpt

extern "C" {

int32_t jpt_prefill_insert(const jpt_prefill_insert_args* args, void* stream) {
  using namespace jpt;
  JPT_REQUIRE(args != nullptr, "args is NULL");
  return insert_launch(*args, nullptr, 0, stream);
}

static int32_t insert_layers(const jpt_prefill_insert_args* args, const jpt_insert_layer* layers, int32_t n_layers,
                             const jpt_insert_state_row* state, bool* wrote, void* stream) {
  using namespace jpt;
  JPT_REQUIRE(args != nullptr && layers != nullptr, "NULL argument");
  JPT_REQUIRE(n_layers >= 1, "n_layers must be positive");
  for (int32_t l0 = 0; l0 < n_layers; l0 += kTableLayers) {
    const int32_t n = n_layers - l0 < kTableLayers ? n_layers - l0 : kTableLayers;
    const int32_t st = insert_launch(*args, layers + l0, n, stream, l0 == 0 ? state : nullptr, l0 == 0 ? wrote : nullptr);
    if (st != JPT_OK) return st;
  }
  return JPT_OK;
}

int32_t jpt_prefill_insert_layers(const jpt_prefill_insert_args* args, const jpt_insert_layer* layers,
                                  int32_t n_layers, void* stream) {
  return insert_layers(args, layers, n_layers, nullptr, nullptr, stream);
}

// (The state's own launch took 2 us behind the insert's: 1000 tokens into 32 layers of 8x128 int8 48.1 -> 46.3 us.)
int32_t jpt_prefill_insert_layers_state(const jpt_prefill_insert_args* args, const jpt_insert_layer* layers, int32_t n_layers,
                                        const jpt_insert_state_row* state, void* stream) {
  using namespace jpt;
  JPT_REQUIRE(args != nullptr && state != nullptr && args->page_ids == nullptr, "a dense slot and its state are needed");
  JPT_REQUIRE(args->slot >= 0, "slot %d out of range", args->slot);
  JPT_REQUIRE(!state->mask || (state->seq > 0 && state->seq < (1ll << 31)), "seq out of range");
  JPT_REQUIRE(!state->mask || state->mask_dtype == JPT_F32 || state->mask_dtype == JPT_BF16, "mask_dtype must be f32 or bf16");
  bool wrote = false;
  const int32_t st = insert_layers(args, layers, n_layers, state, &wrote, stream);
  if (st != JPT_OK || wrote) return st;
  return jpt_insert_state(state->mask, state->mask_dtype, state->seq, state->start, state->input_pos, state->lens, args->slot, state->first,
                          state->position, state->length, state->lo, state->hi, state->wrap, stream);
}

int32_t jpt_prefill_insert_layers_host_pages(const jpt_prefill_insert_args* args, const int32_t* ids, const jpt_insert_layer* layers,
                                             int32_t n_layers, void* stream) {
  using namespace jpt;
  JPT_REQUIRE(args != nullptr && ids != nullptr && layers != nullptr, "NULL argument");
  JPT_REQUIRE(n_layers >= 1, "n_layers must be positive");
  if (n_layers > kTableLayers || args->n_pages > JPT_INSERT_HOST_PAGES) return 1;
  jpt_prefill_insert_args a = *args;
  a.page_ids = nullptr;
  return insert_launch(a, layers, n_layers, stream, nullptr, nullptr, ids);
}

int32_t jpt_prefill_insert_prompts(const jpt_prefill_insert_args* args, const jpt_insert_prompt* prompts,
                                   int32_t n_prompts, void* stream) {
  using namespace jpt;
  JPT_REQUIRE(args != nullptr && prompts != nullptr, "NULL argument");
  JPT_REQUIRE(n_prompts >= 1, "n_prompts must be positive");
  const jpt_prefill_insert_args& a = *args;
  const int n_layers = a.n_layers > 0 ? a.n_layers : 1;
  // the shapes the one-launch kernel takes; anything else goes prompt by prompt
  RowSplit split;
  bool wide = a.dst_dtype == JPT_I8 && a.in_dtype == JPT_BF16 && split_rows(a.heads, a.dim, &split) &&
              // (more than 64 scales a token: what this call has always taken beside what jpt_prefill_insert takes)
              (a.scale_heads == 1 || (a.scale_heads == a.heads && (a.scale_heads <= 64 || a.heads * a.dim == 1024))) &&
              a.dst_k && a.dst_v && a.k_scale && a.v_scale && aligned(a.dst_k, 8) && aligned(a.dst_v, 8) &&
              a.dst_layer_stride % 8 == 0 && a.total_pages > 0 && a.page_size > 0 && n_layers <= 65535 &&
              (a.scale_dtype == JPT_BF16 || a.scale_dtype == JPT_F32) &&
              (a.rounding == JPT_ROUND_TRUNC || a.rounding == JPT_ROUND_RNE);
  for (int32_t r = 0; r < n_prompts && wide; ++r) {
    const jpt_insert_prompt& pr = prompts[r];
    wide = pr.src_k && pr.src_v && pr.page_ids && pr.tokens > 0 && pr.n_pages > 0 &&
           static_cast<int64_t>(pr.n_pages) * a.page_size >= pr.tokens && aligned(pr.src_k, 16) &&
           aligned(pr.src_v, 16) && pr.src_layer_stride % 8 == 0 &&
           (pr.src_head_stride == 0 || (pr.src_head_stride % 8 == 0 &&
                                        pr.src_head_stride >= static_cast<int64_t>(pr.tokens) * a.dim));
  }
  if (!wide) {
    for (int32_t r = 0; r < n_prompts; ++r) {
      jpt_prefill_insert_args one = a;
      one.src_k = prompts[r].src_k;
      one.src_v = prompts[r].src_v;
      one.page_ids = prompts[r].page_ids;
      one.tokens = prompts[r].tokens;
      one.n_pages = prompts[r].n_pages;
      one.src_head_stride = prompts[r].src_head_stride;
      one.src_layer_stride = prompts[r].src_layer_stride;
      const int32_t st = insert_launch(one, nullptr, 0, stream);
      if (st != JPT_OK) return st;
    }
    return JPT_OK;
  }
  for (int32_t r0 = 0; r0 < n_prompts; r0 += kLaunchPrompts) {
    PromptsParams p{};
    p.a = a;
    p.split = split;
    p.a.n_layers = n_layers;
    p.n_prompts = n_prompts - r0 < kLaunchPrompts ? n_prompts - r0 : kLaunchPrompts;
    const int tb = split.tokens_a_block();
    int blocks = 0;
    for (int r = 0; r < p.n_prompts; ++r) {
      p.prompt[r] = prompts[r0 + r];
      p.first_block[r] = blocks;
      blocks += (prompts[r0 + r].n_pages * a.page_size + tb - 1) / tb;
    }
    p.first_block[p.n_prompts] = blocks;
    const dim3 grid(blocks, 2, n_layers);
    using Kernel = decltype(&prefill_insert_prompts_kernel<true, kAnyShape>);
    static constexpr Kernel kernels[2][3] = {
        {prefill_insert_prompts_kernel<false, kAnyShape>, prefill_insert_prompts_kernel<false, kLlama>, prefill_insert_prompts_kernel<false, kOneWide>},
        {prefill_insert_prompts_kernel<true, kAnyShape>, prefill_insert_prompts_kernel<true, kLlama>, prefill_insert_prompts_kernel<true, kOneWide>}};
    const Kernel kernel = kernels[a.scale_dtype != JPT_F32][row_shape(a, split)];
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), p);
    const int32_t st = launch_status("prefill_insert_prompts_kernel");
    if (st != JPT_OK) return st;
  }
  return JPT_OK;
}

}  // extern "C"
