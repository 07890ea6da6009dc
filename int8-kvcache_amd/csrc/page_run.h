// Address arithmetic of a run of consecutive pages (prefill_body), in a file of its own so that it also compiles
// for the host.
#pragma once
#include <stdbool.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define KVQ_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define KVQ_HOST_DEVICE static inline
#endif

// Whether the run of a request's pages 0 .. pages - 1 (page_bytes each) ends within 4 GiB of its key 0: the offset of
// each of its keys is then a 32-bit product. (524,288 keys of 32 kv heads in the bf16 cache are the most; the product
// formed in 64 bits for every tile instead made shorter runs' steps 0.35% slower on average, up to 3% at d64.)
KVQ_HOST_DEVICE bool run_fits(uint32_t pages, uint32_t page_bytes) { return (uint64_t)pages * page_bytes <= 1ull << 32; }
