// host_common.h -- what the library's translation units share on the host:
// the error channel, kernel launches with the timed calls' events, and the
// dynamic-LDS reservation.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace ma_host {

// Sets the message of ma_attn_last_error() and returns 1.
int set_error(const char* msg);
int fail(const char* fmt, ...);
void clear_error();

// Events of the current ma_attn_*_timed call (null otherwise): the call's
// first kernel takes the start event and its last kernel the stop event, so
// they bracket the kernels' own execution (hipExtLaunchKernel stamps them on
// the dispatch packets; no extra queue packets).
extern thread_local hipEvent_t g_ev_start;
extern thread_local hipEvent_t g_ev_stop;

template <typename F, typename... Args>
void launch(bool last, F kernel, dim3 grid, dim3 block, uint32_t shm, hipStream_t st, Args... args) {
  hipEvent_t e0 = g_ev_start, e1 = last ? g_ev_stop : nullptr;
  if (e0 || e1) {
    g_ev_start = nullptr;
    if (last) g_ev_stop = nullptr;
    hipExtLaunchKernelGGL(kernel, grid, block, shm, st, e0, e1, 0u, args...);
  } else {
    hipLaunchKernelGGL(kernel, grid, block, shm, st, args...);
  }
}

// Raises a kernel's dynamic-LDS limit to `shm` bytes once per (kernel,
// device), with that device current; safe from any number of threads.
int reserve_lds(const void* kern, size_t shm, hipStream_t st);

}  // namespace ma_host
