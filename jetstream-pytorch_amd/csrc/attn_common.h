// Argument checks and addressing shared by the decode-attention kernels.
#pragma once

#include "common.h"

namespace jpt {

enum AttnMode { kRagged = 0, kDense = 1, kPaged = 2 };

int32_t check_attn_args(const jpt_attn_args& a, AttnMode mode);

// The MFMA kernel's own entry; returns JPT_OK after enqueueing, or
// JPT_E_BADARG (without setting the message) when the shape is outside what
// it handles and the generic kernel must run.
bool attn_fast_supported(const jpt_attn_args& a, AttnMode mode);
// stash_k, stash_v and the line: see FastParams
struct StepLine {
  const void *k = nullptr, *v = nullptr;
  const int32_t* pos = nullptr;
  const float* rope = nullptr;
  int32_t count = 0, rounding = 0;
};
int32_t attn_fast_launch(const jpt_attn_args& a, AttnMode mode, hipStream_t stream, void* stash_k = nullptr, void* stash_v = nullptr,
                         const StepLine& line = StepLine());
int64_t attn_fast_workspace_bytes(const jpt_attn_args& a);
int64_t attn_partials_offset(const jpt_attn_args& a);  // in the workspace: behind the plan
// Where kernels that need no plan put what they need: the last `bytes` of the workspace, from a multiple of
// 256 on, so that a plan for other calls that the workspace holds stays (bytes from attn_partials_offset(a)
// on are there to have: a plan for this call's slots and heads lies below it, and one for more of them has
// its partials, which no launch leaves for the next, between its records and the end).
inline char* attn_workspace_end(const jpt_attn_args& a, int64_t bytes) {
  return static_cast<char*>(a.workspace) + (a.workspace_bytes - bytes) / 256 * 256;
}
int32_t attn_plan_launch(const jpt_attn_args& a, bool paged, bool fresh, hipStream_t stream);

// Few query rows over caches the streaming kernel is not built for: attn_split.hip.  Needs a workspace
// (its state block zero before the first use; the rest need not be cleared).
bool attn_split_supported(const jpt_attn_args& a, AttnMode mode);
bool attn_split_has_room(const jpt_attn_args& a);  // in its workspace
int64_t attn_split_workspace_bytes(const jpt_attn_args& a);
int32_t attn_split_launch(const jpt_attn_args& a, hipStream_t stream);

// Many query rows (prefill) over bf16 keys and values: attn_prefill.hip.  Bytes of workspace it can use,
// which need not be cleared.
bool attn_prefill_supported(const jpt_attn_args& a, AttnMode mode);
int64_t attn_prefill_workspace_bytes(const jpt_attn_args& a);
int32_t attn_prefill_launch(const jpt_attn_args& a, hipStream_t stream);

// Of the current device (all of a process are alike).
inline int32_t compute_units() {
  static const int32_t v = [] {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
    return cus;
  }();
  return v;
}

int32_t attn_generic_launch(const jpt_attn_args& a, AttnMode mode, hipStream_t stream);

}  // namespace jpt
