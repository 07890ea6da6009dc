// Address arithmetic of a run of consecutive pages (prefill_body), in a file of its own so that it also compiles
// for the host.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define KVQ_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define KVQ_HOST_DEVICE static inline
#endif

// Byte offset of key `key` from the run's key 0: 64 bits, a run may be longer than 4 GiB (524,288 keys of 32 kv
// heads in the bf16 cache) and its key 0 may lie before the cache (the base of a piece whose pages have low ids).
KVQ_HOST_DEVICE uint64_t run_offset(uint32_t key, uint32_t row_bytes) { return (uint64_t)key * row_bytes; }
