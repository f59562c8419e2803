// Entry points that the library's own host code shares across sources (the
// public ones are in nnops_amd.h).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>

#include "nnops_amd.h"

namespace nnops_amd {

// The workspace that is enough for a call of nnops_hip_gemm_i8: its plan's, or
// that of the plan by its rows alone, whichever is less.
size_t gemm_i8_least_workspace(const NnopsGemmI8Args& g);

// nnops_hip_gemm_i8 with whatever workspace there is, without K splits if need
// be: for callers whose buffer was sized before the operands were known (the
// operators' workspace query sees descriptors only).
int gemm_i8_in(const NnopsGemmI8Args& g, void* workspace, size_t ws_bytes, hipStream_t stream);

// The Q4_1 GEMM as K splits whose partials, in the workspace, the output pass
// sums (one launch and one staging fewer than the product and then the pass);
// NNOPS_UNSUPPORTED, nothing launched, where another route is the call's.
int gemm_q4_1_split_pass(const NnopsGemmQ41Args& g, const NnopsFpOutArgs& pass, void* workspace, size_t ws_bytes,
                         hipStream_t stream);

}  // namespace nnops_amd
