// Single-pass scans: each workgroup ("tile") publishes the sum of its elements
// and finds the sum of all tiles before it by looking back over what they
// published (Merrill and Garland, Single-pass Parallel Prefix Scan with
// Decoupled Look-back, 2016), so a scan is one launch.  A scan as reduce, scan
// of the tile sums and apply is three launches of about 4 us each whatever
// they do, and reads its input twice.
//
// A tile's word holds its state and value together, so relaxed device-scope
// atomics carry it without a fence (a device-scope release writes back the
// XCD's L2).  Tiles are numbered by a ticket in the order they start, so a
// tile only waits for tiles that run already.  Words are tagged with an epoch
// that the last tile to finish advances (and resets the ticket): the state
// needs no clearing between launches, only once when it is allocated.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"

namespace prg {
namespace {

// Device state of a stream's scans: ticket, finished tiles, epoch; then the tiles' words.
constexpr int kLookHeader = 8;  // 64-bit words
constexpr uint32_t kLookSum = 1, kLookPrefix = 2;  // state of a word: the tile's own sum; the sum up to and with it

struct LookTile {
    uint32_t tile, tag;
};

// A tile that cannot do its part: the launch's results are wrong, and the
// host, which looks at the flag where it waits for them (look_check), says so.
__device__ __forceinline__ void look_failed(const LookState& state) {
    __hip_atomic_store(state.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The calling workgroup's tile number and the launch's tag (every thread).  A
// number past the launch's tiles (only if the state was damaged from outside)
// is reported; the workgroup returns.
__device__ __forceinline__ LookTile look_begin(const LookState& state, uint32_t tiles) {
    __shared__ LookTile t;
    if (threadIdx.x == 0) {
        if (tiles == 1) {
            t = LookTile{0, 0};
        } else {
            uint32_t* h = reinterpret_cast<uint32_t*>(state.words);
            const uint32_t e = __hip_atomic_load(h + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            t.tile = __hip_atomic_fetch_add(h, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            t.tag = e + 1 < 0x3fffffffu ? e + 1 : 1;  // (never 0, the cleared words' tag)
            if (t.tile >= tiles) look_failed(state);
        }
    }
    __syncthreads();
    return t;
}

// Called by one whole wave: publishes the tile's sum and returns the sum of
// the tiles before it (every lane).  `row`: which of the launch's sums, each
// with `tiles` words of its own.
__device__ __forceinline__ int32_t look_back(const LookState& state, int row, LookTile t, uint32_t tiles, int32_t sum) {
    if (tiles == 1) return 0;
    uint64_t* words = state.words + kLookHeader + int64_t(row) * tiles;
    const int lane = threadIdx.x & 63;
    const uint64_t tag = uint64_t(t.tag) << 34;
    if (lane == 0)
        __hip_atomic_store(words + t.tile, tag | (uint64_t(t.tile == 0 ? kLookPrefix : kLookSum) << 32) | uint32_t(sum),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t.tile == 0) return 0;
    int32_t before = 0;
    int64_t top = int64_t(t.tile) - 1;  // the nearest tile not yet added
    // (bounded: every tile looked at has started, so its word comes; the bound
    // ends the wave, and reports it, if the state was damaged from outside)
    bool found = false;
    for (uint32_t spin = 0; spin < state.spins; spin++) {
        const int64_t i = top - lane;
        const uint64_t w =
            i >= 0 ? __hip_atomic_load(words + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                   : tag | (uint64_t(kLookPrefix) << 32);
        const bool ready = (w >> 34) == (tag >> 34);
        const bool prefix = ready && uint32_t((w >> 32) & 3u) == kLookPrefix;
        const uint64_t rm = __ballot(ready), pm = __ballot(prefix);
        // lanes up to the nearest prefix, or all 64
        const int last = pm ? int(__builtin_ctzll(pm)) : 63;
        const uint64_t need = last == 63 ? ~uint64_t(0) : (uint64_t(1) << (last + 1)) - 1;
        if ((rm & need) != need) continue;
        int32_t v = lane <= last ? int32_t(uint32_t(w)) : 0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        before += v;
        if (pm) {
            found = true;
            break;
        }
        top -= 64;
    }
    if (!found && lane == 0) look_failed(state);
    if (lane == 0)
        __hip_atomic_store(words + t.tile, tag | (uint64_t(kLookPrefix) << 32) | uint32_t(before + sum),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return before;
}

// After every look_back of the workgroup (a barrier in between): the last
// tile to finish readies the state for the next launch.
__device__ __forceinline__ void look_end(const LookState& state, LookTile t, uint32_t tiles) {
    if (tiles == 1 || threadIdx.x != 0) return;
    uint32_t* h = reinterpret_cast<uint32_t*>(state.words);
    if (__hip_atomic_fetch_add(h + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == tiles - 1) {
        __hip_atomic_store(h, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(h + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(h + 2, t.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// exclusive scan of one value per thread over the workgroup, and its total
__device__ __forceinline__ int32_t block_exclusive_scan(int32_t v, int32_t* lds_waves, int32_t& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds_waves[wave] = x;
    __syncthreads();
    int32_t before = 0, tot = 0;
    for (int w = 0; w < int(blockDim.x >> 6); w++) {
        const int32_t t = lds_waves[w];
        if (w < wave) before += t;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return before + x - v;
}

}  // namespace
}  // namespace prg
