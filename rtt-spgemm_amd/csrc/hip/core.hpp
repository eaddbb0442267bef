// Device code shared by the SpGEMM core's files: C's structure, workgroup
// scans and the slab rows' entry points.
#pragma once

#include "device.hpp"
#include "internal.hpp"

namespace rtt {

struct COut {
    const int64_t *__restrict__ tile_ptr;     // tilem + 1
    const int64_t *__restrict__ row_nnz_off;  // tilem + 1
    int *__restrict__ col;
    uint64_t *__restrict__ mask;
    int64_t *__restrict__ tile_nnz;
    uint8_t *__restrict__ csr_ptr;
    uint8_t *__restrict__ csr_col;
    double *__restrict__ val;
};

// Byte r of the result is the number of set bits in bytes 0..r-1 of m (the
// u8 row offsets of a C tile): per-byte popcounts, then an exclusive byte
// prefix sum by multiplication (sums stay below 256, so no byte carries).
__device__ __forceinline__ uint64_t packed_row_offsets(uint64_t m)
{
    uint64_t x = m - ((m >> 1) & 0x5555555555555555ull);
    x = (x & 0x3333333333333333ull) + ((x >> 2) & 0x3333333333333333ull);
    x = (x + (x >> 4)) & 0x0F0F0F0F0F0F0F0Full;
    return (x * 0x0101010101010101ull) << 8;
}

// C tile t's structure; put takes its entries' local columns in order.
template <class Put>
__device__ __forceinline__ void write_tile_structure(const COut &c, int64_t t, int j,
                                                     uint64_t m, int64_t off, Put &&put)
{
    c.col[t] = j;
    c.mask[t] = m;
    c.tile_nnz[t] = off;
    reinterpret_cast<uint64_t *>(c.csr_ptr)[t] = packed_row_offsets(m);
    while (m) {
        const int pos = __builtin_ctzll(m);
        m &= m - 1;
        put(static_cast<uint8_t>(pos & 7));
    }
}

__device__ __forceinline__ void write_tile_structure(const COut &c, int64_t t, int j,
                                                     uint64_t m, int64_t off)
{
    uint8_t *bytes = c.csr_col + off;
    write_tile_structure(c, t, j, m, off, [&](uint8_t col) { *bytes++ = col; });
}

// Exclusive scans of two values over a workgroup of NW waves with one
// barrier; s2 (2 * NW ints) must not be reused without a barrier between.
template <int NW>
__device__ __forceinline__ void dual_exclusive_scan(int a, int b, int *s2, int *pa, int *pb,
                                                    int *ta, int *tb)
{
    const int w = threadIdx.x / kWave;
    const int ia = wave_inclusive_scan(a);
    const int ib = wave_inclusive_scan(b);
    if (lane_id() == kWave - 1) {
        s2[w] = ia;
        s2[NW + w] = ib;
    }
    __syncthreads();
    int ba = 0, bb = 0, sa = 0, sb = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int x = s2[i], y = s2[NW + i];
        ba += i < w ? x : 0;
        bb += i < w ? y : 0;
        sa += x;
        sb += y;
    }
    *pa = ba + ia - a;
    *pb = bb + ib - b;
    *ta = sa;
    *tb = sb;
}

// Exclusive scan over a workgroup of NW waves; *total receives the sum.
template <int NW>
__device__ __forceinline__ int block_exclusive_scan(int v, int *s_tmp, int *total)
{
    const int w = threadIdx.x / kWave;
    const int incl = wave_inclusive_scan(v);
    if (lane_id() == kWave - 1)
        s_tmp[w] = incl;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int t = s_tmp[i];
        before += i < w ? t : 0;
        all += t;
    }
    __syncthreads();
    *total = all;
    return before + incl - v;
}

// ---- rows beyond the LDS tables (slab.hip) ------------------------------------
// A's slot codes and B's entries by scalar row for a call with such rows, `n`
// tile rows listed in `rows` and n_more in `more` (device): of all of A and B, or
// where the rows are few of these and the B rows they select (one host wait).
// longest: most slots of A's payload in one of them.
int slab_prepare(const DevTiles &a, const DevTiles &b, BuildWork *bw, SpgemmWork *w,
                 const int *rows, int n, const int *more, int n_more, int64_t longest);
// Slab rows in the order they are taken, tasks base[i] .. base[i + 1] of row
// i: as many as its pairs hold slab_target.  most: at least all of them.
struct SlabTasks {
    const int *__restrict__ rows = nullptr;
    const int *__restrict__ base = nullptr;
    int nrows = 0;
    int64_t most = 0;
};
constexpr int kSlabParts = 256;   // most tasks of a row
int64_t slab_target(unsigned long long pairs);
// Workgroups of a slab pass whose longest row has `longest` slots, with `held`
// bytes of cursors there and `free_bytes` of device memory free.
unsigned slab_cursor_blocks(int64_t longest, size_t held, size_t free_bytes);
// Counts the listed rows' tiles and entries into w->row_tiles / row_nnz and
// stages their tile lists; *cursor sums what the staging needs.  longest:
// most slots of A's payload in one of the rows.
int slab_symbolic(const DevTiles &a, SpgemmWork *w, const SlabTasks &tasks, int *queue,
                  int static_rows, unsigned long long *cursor, int64_t longest);
// Writes the structure of the rows slab_symbolic counted.
int slab_structure(const DevTiles &a, SpgemmWork *w, const SlabTasks &tasks, int *queue,
                   int static_rows, const COut &c);
// Values of the listed rows, whose structure is written.
int slab_numeric(const DevTiles &a, SpgemmWork *w, const SlabTasks &tasks, int *queue,
                 int static_rows, const COut &c, int64_t longest);

} // namespace rtt
