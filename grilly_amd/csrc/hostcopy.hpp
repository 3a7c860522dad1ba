// Host-side copies of large arrays, spread over a few threads (hostcopy.cpp).
#pragma once
#include <stddef.h>

enum { GRL_COPY_F32 = 0,          // float -> float
       GRL_COPY_F32_BF16 = 1,     // float -> bf16 bits, round to nearest even, NaN stays NaN (as f32_to_bf16_bits on the device)
       GRL_COPY_BF16_F32 = 2 };   // bf16 bits -> float
// n values from src to dst; returns when they are there.  past_caches: float values are stored without reading their lines first
void grl_host_copy(int kind, void* dst, const void* src, size_t n, bool past_caches = false);
// a call that will copy more than once begins (+1) or is over (-1): the helpers look for its next job ten times as long
void grl_host_call(int change);
struct grl_host_calling {
    grl_host_calling() { grl_host_call(1); }
    ~grl_host_calling() { grl_host_call(-1); }
};
// unmaps the result memory that no array stands in
void grl_host_trim();
