// scratch.h -- per (device, stream) scratch of the kernels whose results leave in parts (qgemm_prefill.hip): lives until exl2_release_scratch
#pragma once
#include "hw.h"
#include <mutex>

// kind 0 = staged activation rows, 1 = decoded weight fragments, 2 = split-K partial tiles, 3 = a sparse block's lists and expert rows,
// 4 = attention's key splits (two buffers of one call must not alias)
int prefill_scratch(size_t bytes, void* stream, int kind, f16** out);
// the same for a route that only wants it: null (and no error) where it cannot be had -- inside a graph capture that would grow it, out of
// memory -- and the caller takes the route that needs none
f16* prefill_scratch_try(size_t bytes, void* stream, int kind);
// Held from a call's first launch that writes a stream's scratch to its last that reads it: host threads that launch on one stream take turns.
// Without it another thread's launches come between the two and this call reads that one's parts.  Once per thread or nested.
std::unique_lock<std::recursive_mutex> scratch_turn(void* stream);
