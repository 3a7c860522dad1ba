// Host-side copies of large arrays, spread over a few threads (hostcopy.cpp).
#pragma once
#include <stddef.h>

enum { GRL_COPY_F32 = 0,          // float -> float
       GRL_COPY_F32_BF16 = 1,     // float -> bf16 bits, round to nearest even, NaN stays NaN (as f32_to_bf16_bits on the device)
       GRL_COPY_BF16_F32 = 2 };   // bf16 bits -> float
// n values from src to dst; returns when they are there
void grl_host_copy(int kind, void* dst, const void* src, size_t n);
// writes one byte of every 4 KiB page, so that the process has all of them mapped
void grl_host_touch(void* p, size_t bytes);
