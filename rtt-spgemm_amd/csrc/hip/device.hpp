// Device helpers shared by the kernels (wave64 primitives, tile bit algebra).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace rtt {

constexpr int kWave = 64;

// Orders the LDS traffic of one wavefront: every store issued before the
// barrier is visible to every lane after it.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// Workgroups are dispatched to the 8 XCDs round-robin (workgroup b runs on
// XCD b % 8).  The row kernels keep the rows in flight on the chip one
// window of consecutive rows spread over every XCD: measured against giving
// each XCD a contiguous eighth of the rows, the stencil A*A^T numeric pass
// ran 3 % and the banded batch 6 % faster.
constexpr int kXcds = 8;

// Row of workgroup b of n: chunks of C consecutive rows dealt to the XCDs
// round-robin (XCD x takes chunks x, x + 8, ...), so that the rows one L2
// holds come in runs of C; rows past the last whole round of 8 C rows map
// to themselves.  A bijection of [0, n).
template <int C>
__device__ __forceinline__ int xcd_chunk_row(int b, int n)
{
    if (b >= n / (kXcds * C) * (kXcds * C))
        return b;
    const int x = b % kXcds, i = b / kXcds;
    return ((i / C) * kXcds + x) * C + i % C;
}

// Gathers bits k, k+4, ..., k+28 of a 32-bit tile mask into 8 bits.  For an
// A tile (bit r*4+k) this is the set of rows present in column k; for a B
// tile (bit c*4+k) the set of columns present in row k.
__device__ __forceinline__ uint32_t stride4_bits(uint32_t mask, int k)
{
    uint32_t x = (mask >> k) & 0x11111111u;
    x = (x | (x >> 3)) & 0x03030303u;
    x = (x | (x >> 6)) & 0x000F000Fu;
    x = (x | (x >> 12)) & 0x000000FFu;
    return x;
}

// Bit r of `rows` -> byte r of the result is 0xFF.
__device__ __forceinline__ uint64_t rows_to_bytes(uint32_t rows)
{
    auto nibble = [](uint32_t x) {
        x = (x | (x << 14)) & 0x00030003u;
        x = (x | (x << 7)) & 0x01010101u;
        return (x << 8) - x;
    };
    return (static_cast<uint64_t>(nibble(rows >> 4)) << 32) | nibble(rows & 15u);
}

// Payload slot of physical position `phys` of a hybrid tile.
__device__ __forceinline__ int payload_slot(uint32_t mask, int span, int phys)
{
    return span == 32 ? phys : __popc(mask & ((1u << phys) - 1u));
}

__device__ __forceinline__ uint32_t hash_tile_col(int j)
{
    return static_cast<uint32_t>(j) * 0x9E3779B1u;
}

template <typename T>
__device__ __forceinline__ T wave_inclusive_scan(T v)
{
    const int lane = lane_id();
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const T u = __shfl_up(v, o, kWave);
        if (lane >= o)
            v += u;
    }
    return v;
}

// The same for ints by data-parallel moves: shifts within the rows of 16
// lanes, then each row's last lane into the rows after it.  Six adds, where
// the form above takes six trips through the LDS.
__device__ __forceinline__ int wave_inclusive_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15, rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31, rows 2 and 3
    return v;
}

__device__ __forceinline__ int last_lane(int v) { return __builtin_amdgcn_readlane(v, kWave - 1); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1)
        v += __shfl_xor(v, o, kWave);
    return v;
}

// Largest index i in [0, n) with pre[i] <= p (pre non-decreasing, pre[0] = 0).
__device__ __forceinline__ int upper_index(const int *pre, int n, int p)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= p)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Decoupled look-back over workgroups, two sums (below 2^62) each: the words
// of workgroup b are look[2 b] and look[2 b + 1], state in the top two bits (0
// nothing yet, 1 the workgroup's own sums, 2 sums up to and with it).  All
// words start at zero.
constexpr unsigned long long kOwn = 1ull << 62, kUpTo = 2ull << 62, kSums = kOwn - 1ull;

__device__ __forceinline__ void publish(unsigned long long *look, int64_t b,
                                        unsigned long long state, unsigned long long x,
                                        unsigned long long y)
{
    __hip_atomic_store(look + 2 * b, state | x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(look + 2 * b + 1, state | y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sums of the workgroups before b, by one wave, 64 of them at a time.
// Workgroups take their numbers from a ticket, so every workgroup before b
// has started and publishes its own sums without waiting for anything: the
// wait ends.
__device__ __forceinline__ void look_back(const unsigned long long *look, int64_t b,
                                          unsigned long long *x, unsigned long long *y)
{
    unsigned long long sx = 0, sy = 0;
    for (int64_t hi = b; hi > 0; hi -= kWave) {
        const int64_t i = hi - 1 - lane_id();
        unsigned long long wx = kUpTo, wy = kUpTo;
        if (i >= 0) {
            for (;;) {
                wx = __hip_atomic_load(look + 2 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                wy = __hip_atomic_load(look + 2 * i + 1, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                if ((wx >> 62) != 0 && (wx >> 62) == (wy >> 62))
                    break;
                __builtin_amdgcn_s_sleep(1);
            }
        }
        const unsigned long long done = __ballot((wx >> 62) == 2);
        const int last = done ? __builtin_ctzll(done) : kWave - 1;
        const bool take = lane_id() <= last;
        sx += wave_sum(take ? wx & kSums : 0ull);
        sy += wave_sum(take ? wy & kSums : 0ull);
        if (done)
            break;
    }
    *x = sx;
    *y = sy;
}

} // namespace rtt
