// trace_cursors.h -- the work split of the traversal kernel's launches:
// the rays are cut into 8 regions (one per XCD), every wave takes a fixed
// first chunk of its region, and the rest of each region is claimed through
// an atomic cursor that counts from 0.  Shared by the kernel, the kernel that
// clears the cursors before a launch, and wavefront loops whose own kernels
// clear them for the next launch.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#ifndef LMX_CLAIM_CHUNK
#define LMX_CLAIM_CHUNK 64     // rays claimed from a region cursor per atomic
#endif
// words between two region cursors: each cursor sits in a 256-byte line of
// its own, so the atomics of different regions do not serialise on one line
#ifndef LMX_CURSOR_STRIDE
#define LMX_CURSOR_STRIDE 64
#endif
#define CURSOR_STRIDE LMX_CURSOR_STRIDE
// counter block of one trace launch: 8 region cursors, an unused line, and a
// sticky stack-overflow flag, each on a line of its own
#define LMX_TRACE_COUNTER_WORDS (10 * CURSOR_STRIDE)

__host__ __device__ __forceinline__ uint32_t region_start(uint32_t j, uint32_t n)
{
    return (uint32_t)(((uint64_t)n * j) / 8u);
}

__host__ __device__ __forceinline__ uint32_t region_end(uint32_t j, uint32_t n)
{
    return (uint32_t)(((uint64_t)n * (j + 1u)) / 8u);
}

// Rays per claim: LMX_CLAIM_CHUNK for full queues; short queues (the tail of
// a wavefront render) are spread over every wave of the grid, so that their
// time is that of a few rays per wave, not of whole chunks in turn.
__host__ __device__ __forceinline__ uint32_t trace_claim(uint32_t n, uint32_t grid)
{
    const uint32_t even = (uint32_t)(((uint64_t)n + grid - 1u) / grid);
    return even < 1u ? 1u : even > LMX_CLAIM_CHUNK ? LMX_CLAIM_CHUNK : even;
}

// Every wave's first chunk is fixed by its index (wave b, of XCD region
// r = b mod 8, takes chunk b / 8 of its region); the region's cursor counts
// from the end of those chunks, so a launch claims with atomics only what is left,
// and one with few rays (the tail of a wavefront render) with none.
__host__ __device__ __forceinline__ uint32_t region_dyn_start(uint32_t r, uint32_t n, uint32_t grid, uint32_t claim)
{
    const uint64_t waves = (grid + 7u - r) / 8u;          // waves b < grid with b mod 8 = r
    const uint64_t s = (uint64_t)region_start(r, n) + waves * claim;
    const uint64_t e = region_end(r, n);
    return (uint32_t)(s < e ? s : e);
}

// Whether any ray of a launch is left to the cursors.
__host__ __device__ __forceinline__ bool trace_has_dynamic(uint32_t n, uint32_t grid)
{
    const uint32_t claim = trace_claim(n, grid);
    bool any = false;
    for (uint32_t r = 0; r < 8; r++) any |= region_dyn_start(r, n, grid, claim) < region_end(r, n);
    return any;
}

// Thread j of a workgroup, on a stream where no trace launch is running:
// clears the cursors for the next one.
__device__ __forceinline__ void trace_cursors_clear(uint32_t* cursors, uint32_t j)
{
    if (j < 8) cursors[j * CURSOR_STRIDE] = 0u;
}
