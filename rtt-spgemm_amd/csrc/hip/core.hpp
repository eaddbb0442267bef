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

__device__ __forceinline__ uint32_t byte_of(uint32_t v, int k) { return (v >> (8 * k)) & 0xFFu; }

// Byte k is nonzero where byte k of v is (its bit 7 set).
__device__ __forceinline__ uint32_t nonzero_tops(uint32_t v)
{
    return (((v & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | v) & 0x80808080u;
}

// An A tile spread for products with many B tiles: word k of lo (hi) is 0xFF
// in byte r where row r (row 4 + r) has an entry in column k.
__device__ __forceinline__ void spread_tile(uint32_t ab, uint4 *lo, uint4 *hi)
{
    uint64_t s[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        s[k] = rows_to_bytes(byte_of(ab, k));
    *lo = make_uint4(static_cast<uint32_t>(s[0]), static_cast<uint32_t>(s[1]),
                     static_cast<uint32_t>(s[2]), static_cast<uint32_t>(s[3]));
    *hi = make_uint4(static_cast<uint32_t>(s[0] >> 32), static_cast<uint32_t>(s[1] >> 32),
                     static_cast<uint32_t>(s[2] >> 32), static_cast<uint32_t>(s[3] >> 32));
}

// Structural product of a spread A tile and the per-k column bytes of a B
// tile: byte k of b_bytes to every byte of a word, then a bitwise select each.
__device__ __forceinline__ uint64_t spread_product(const uint4 &lo, const uint4 &hi,
                                                   uint32_t b_bytes)
{
    const uint32_t b0 = __builtin_amdgcn_perm(b_bytes, b_bytes, 0x00000000u);
    const uint32_t b1 = __builtin_amdgcn_perm(b_bytes, b_bytes, 0x01010101u);
    const uint32_t b2 = __builtin_amdgcn_perm(b_bytes, b_bytes, 0x02020202u);
    const uint32_t b3 = __builtin_amdgcn_perm(b_bytes, b_bytes, 0x03030303u);
    const uint32_t l = (lo.x & b0) | (lo.y & b1) | (lo.z & b2) | (lo.w & b3);
    const uint32_t h = (hi.x & b0) | (hi.y & b1) | (hi.z & b2) | (hi.w & b3);
    return (static_cast<uint64_t>(h) << 32) | l;
}

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
// Rows listed: most slots of A's payload and most tiles of A in one of them, and
// those of all.
struct SlabSizes {
    int64_t longest = 0, most_tiles = 0, slots = 0, tiles = 0;
};
// Whether the symbolic passes of such rows go by tiles: they then need no
// slab_prepare.
bool slab_by_tiles(const DevTiles &b, const SlabSizes &rows);
// Counts the listed rows' tiles and entries into w->row_tiles / row_nnz and
// stages their tile lists; *cursor sums what the staging needs.
int slab_symbolic(const DevTiles &a, const DevTiles &b, SpgemmWork *w, const SlabTasks &tasks,
                  int *queue, int static_rows, unsigned long long *cursor, const SlabSizes &rows);
// Writes the structure of the rows slab_symbolic counted.
int slab_structure(const DevTiles &a, const DevTiles &b, SpgemmWork *w, const SlabTasks &tasks,
                   int *queue, int static_rows, const COut &c);
// Values of the listed rows, whose structure is written.
int slab_numeric(const DevTiles &a, SpgemmWork *w, const SlabTasks &tasks, int *queue,
                 int static_rows, const COut &c, int64_t longest);

} // namespace rtt
