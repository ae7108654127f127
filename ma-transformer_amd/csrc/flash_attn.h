// flash_attn.h -- host interface of the banded MFMA kernels of flash_kernel.h
// (head_dims 8 to 128), for the dispatch in ma_attn.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/ma_attn.h"

namespace ma_flash {

// Whether the kernels can take desc with these tensors: SLIDING with left,
// right >= 0 or DENSE, head_dim a multiple of 8 up to 128, 16-byte aligned
// tensors, one (batch, residue class)'s rows within 2^31 bytes.
bool applies(const ma_attn_desc* d, const void* const* ptrs, int n);

// Launches the forward; lse (optional): each row's statistic, as
// ma_attn_forward_lse writes it.  Non-zero on failure.
int forward(const ma_attn_desc* d, const void* q, const void* k, const void* v, void* o, float* lse, hipStream_t st);

// The forward of d (float32 SLIDING, dilation 1, head_dim 64) with the keys
// 0..num_global-1 (1 to 16) joined to every row's window; rows below num_global
// are left alone.  Non-zero on failure.
int forward_globals(const ma_attn_desc* d, int64_t num_global, const void* q, const void* k, const void* v, void* o,
                    hipStream_t st);

// Launches the backward (ptrs: q, k, v, dout, dq, dk, dv); stats: 2 floats per
// row of workspace.  fo, lse: the forward's O and statistics
// (ma_attn_backward_saved; head_dim 64), or null.  Non-zero on
// failure.
int backward(const ma_attn_desc* d, const void* const* ptrs, float* stats, const void* fo, const float* lse,
             hipStream_t st);

}  // namespace ma_flash
