// Dynamic LDS beyond the default 64 KB of a workgroup has to be asked for once
// per kernel AND device: a process that works on a second device asks again.
// `asked` is one word for each kernel (a function-local static next to its
// launch); two threads that meet here ask twice, which does no harm.
#pragma once

#include <atomic>

static inline void lds_limit(const void* kernel, int bytes,
                             std::atomic<unsigned long long>& asked) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) device = 64;
  const unsigned long long bit = device < 64 ? 1ull << device : 0ull;
  if (asked.load(std::memory_order_relaxed) & bit) return;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                          bytes) == hipSuccess)
    asked.fetch_or(bit, std::memory_order_relaxed);
}
