// SpGEMM core: symbolic -> allocate -> numeric for C = A * B with A in 8x4
// row-major tiles, B in 4x8 column-major tiles and C in 8x8 tiles.
//
// Work unit: one A tile row I (8 scalar rows), one 256-thread workgroup.
// Its (A tile, B tile) pairs are A(I,K) x B(K,J) for every A tile of row I
// and every B tile of B's tile row K -- a tile-level Gustavson expansion, so
// no K-list merge or candidate sort is needed (the reference reaches the same
// pairs through Super16 candidates + exact intersection,
// src/super16_symbolic.cuh:2406-2774, and a K-merge per C tile,
// src/dmma_spgemm.h:4307-4410).
//
// Pairs are enumerated per chunk of up to kChunk A tiles: every A tile's
// B-row extent comes from a per-A-tile table built with B, the pair count is
// scanned, and an LDS segment table maps pair index -> A tile, so a thread
// reaches its (A tile, B tile) with two LDS reads.
//
//  * symbolic: the 8x8 masks of the row's C tiles are ORed into an LDS hash
//    table, compacted, ranked by tile column and staged; after the size scan
//    a light pass writes the final structure.  Rows whose tile set outgrows
//    the table go to the slab kernels (slab.hip).
//  * numeric: the row's C layout (tile columns, masks, value offsets) and
//    its A payload (column-major per tile) are loaded into LDS.  Each thread
//    takes a pair, loads its 80-byte B record (packed meta + the first eight
//    values in k-major order), walks B's entries row by row with A's column
//    in registers, and adds each scalar product into an LDS FP64 accumulator
//    laid out exactly like the row's output segment, which is finally
//    streamed to HBM.  Rows that exceed the LDS budgets go to the slab
//    kernels (slab.hip).
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "core.hpp"

namespace rtt {

namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;

constexpr int kChunk = 128;        // A tiles per enumeration step
constexpr int kSeg = 1024;         // pairs per segment-table window

constexpr int kSymSlots = 1024;    // LDS hash slots (power of 2)
constexpr int kSymSlotBits = 10;
constexpr int kSymPerThread = kSymSlots / kThreads;
constexpr int kSymProbe = 32;      // longest probe before a row goes to the slab path
constexpr int kSymBatch = 4;       // pairs whose loads a thread issues together

constexpr int kWSlots = 256;       // hash slots of the one-wave symbolic table
constexpr int kWSlotBits = 8;
static_assert(kWSlots == 1 << kWSlotBits, "one-wave table size");
constexpr int kWStage = 3 * kWSlots / 4;   // C tiles a row may have there
constexpr int kWChunk = kWave;     // A tiles per one-wave enumeration step
constexpr int kWSeg = 512;         // pairs per one-wave segment window
constexpr int kWBatch = 6;         // pairs whose loads a lane of that kernel issues together

constexpr int kColRegs = 3;         // values of an A column a numeric lane holds in registers
constexpr int kOneVals = 3;         // B values a lane loads of the one row of a light pair
constexpr int kSkew = 32;           // SpreadRow: accumulator slots between two unused ones
constexpr int kExtVals = 3;         // B values past the record a numeric lane prefetches

// The numeric instances: threads per workgroup (four pair runs of kChunk A
// tiles each), pairs per segment-table window, and LDS budgets:
// accumulator slots, staged A values, C tiles, hash slots (at least twice
// the tiles).  TinyRow is one wave with 3 KB of LDS against SmallRow's
// 20 KB, so that a CU holds four times as many of the short rows of sparse
// operands (prolongators, Galerkin products) in flight.  A second one-wave
// instance with a 512-value accumulator measured no faster than SmallRow
// on the rows between the two.
struct TinyRow {
    static constexpr int kThreads = kWave, kChunk = kWave / 4, kSeg = 128;
    static constexpr bool kLeavesTiny = false, kSpread = false;
    static constexpr int kWavesPerSimd = 7;
    static constexpr int kAcc = 128, kAStage = 64, kTiles = 16, kSlots = 32, kSlotBits = 5;
};
// SmallRow leaves the rows within TinyRow's budgets to that instance.  (Its
// launch goes over its own rows' list, or over every row where all are its own
// and in the traced form.)
struct SmallRow {
    static constexpr int kThreads = 256, kChunk = 64, kSeg = 1024;
    static constexpr bool kLeavesTiny = true, kSpread = false;
    static constexpr int kWavesPerSimd = 7;
    static constexpr int kAcc = 1024, kAStage = 256, kTiles = 128, kSlots = 256, kSlotBits = 8;
};
// SmallRow for products whose C tiles hold kSpreadFill entries or fewer on
// average: the lanes of a wave then add to the same few places of many C
// tiles at once.  The accumulator has an unused slot after every kSkew, which
// takes the tiles' like places to different LDS banks (the tiles of eight
// equal C rows, stencils', otherwise lie a multiple of eight slots apart: an
// add took 17 ns a wave and CU, with the slots 8), and a pair with a light
// tile, of which such products have many, takes the one row it needs of B's
// record instead of walking all of it.  The LDS pipe was busy 75 % of the
// kernel's time and is now 55 %, vector instructions 74 %: 128^3 box stencil,
// A*A^T (14 entries a C tile), 2.83 -> 2.29 ms.  With more to a C tile the extra
// index work costs more than the conflicts: bands of 400000 rows with 21, 23,
// 26, 30 and 38 entries a C tile take 0.46, 0.48, 0.50, 0.53 and 0.75 ms a step
// with it, 0.43, 0.46, 0.49, 0.51 and 0.73 without.  (It is the rows' likeness
// that counts, which the fill only hints at: block FEM on this path, 31 entries,
// takes 1.31 ms with it and 1.44 without.)
struct SpreadRow : SmallRow {
    static constexpr bool kSpread = true;
};
constexpr int kSpreadFill = 18;
// MediumRow takes rows past SmallRow's accumulator with few C tiles and A
// values (narrow bands squared) at a third of LargeRow's LDS.
struct MediumRow {
    static constexpr int kThreads = 256, kChunk = 64, kSeg = 1024;
    static constexpr bool kLeavesTiny = false, kSpread = false;
    static constexpr int kWavesPerSimd = 6;
    static constexpr int kAcc = 2048, kAStage = 256, kTiles = 64, kSlots = 128, kSlotBits = 7;
};
struct LargeRow {
    static constexpr int kThreads = 256, kChunk = 64, kSeg = 1024;
    static constexpr bool kLeavesTiny = false, kSpread = false;
    static constexpr int kWavesPerSimd = 2;
    static constexpr int kAcc = 4096, kAStage = 2048, kTiles = 512, kSlots = 1024, kSlotBits = 10;
};
static_assert(LargeRow::kAcc <= 65536 && LargeRow::kTiles <= 32768, "packed tile slots");
static_assert(TinyRow::kAcc <= SmallRow::kAcc && TinyRow::kAStage <= SmallRow::kAStage &&
                  TinyRow::kTiles <= SmallRow::kTiles,
              "nested row budgets");

// Whether a row of the LDS level with these sizes fits the instance Cfg.
template <class Cfg>
__device__ __forceinline__ bool fits_row(int64_t nt, int64_t nnz, int64_t a_len)
{
    return nt <= Cfg::kTiles && nnz <= Cfg::kAcc && a_len <= Cfg::kAStage;
}

constexpr int kWriteBuf = 2048;    // column bytes staged per row in the write pass

constexpr int kEmpty = -1;
constexpr uint32_t kDenseBit = 0x80000000u;

// kLevelLarge: the row outgrew the wave table and waits for the workgroup
// table; kLevelSlab: it outgrew that too.
enum RowLevel : int { kLevelEmpty = 0, kLevelLds = 1, kLevelLarge = 2, kLevelSlab = 3 };

// The numeric kernel that takes a row of the LDS level, by its sizes: the
// smallest instance that holds it, the slab kernel when none does.
enum RowClass : int { kRowTiny, kRowSmall, kRowMid, kRowLarge, kRowSlab, kRowClasses };

// Counters the host reads back after the symbolic pass, and the state of the
// kernels that fill them (zeroed with them).
enum Counter : int {
    kCtrPairs,       // (A tile, B tile) pairs
    kCtrTiles,       // C tiles
    kCtrNnz,         // nnz(C)
    kCtrOutgrown,    // rows that outgrew the wave table
    kCtrSymSlab,     // rows that outgrew the workgroup table too
    kCtrSlabTiles,   // slab tiles the staging cursor handed out
    kCtrLongest,     // most A payload slots in a slab row
    kCtrMostTiles,   // most A tiles in one
    kCtrSymSizes,    // A tiles (upper half) and payload slots of the symbolic pass's
    kCtrRows,        // rows of each RowClass, kRowClasses of them
    kCtrWide = kCtrRows + kRowClasses,   // tile-pair rows of many C tiles: the rows (upper 28
                                         // bits) and their C tiles
    kCtrTicket,
    kCtrDone,
    kCounters
};

constexpr int kWideRowShift = 36;

struct Operands {
    const int *__restrict__ a_trp;
    const int4 *__restrict__ a_meta;
    const int4 *__restrict__ a_brange;   // per A tile: first B tile, heavy, count
    const int2 *__restrict__ a_blight;   // per A tile: the light B tiles it can meet
    const double *__restrict__ a_vals_cm;   // A payload, each tile column-major
    const int *__restrict__ a_row_off;      // A payload offset of each tile row
    const double *__restrict__ b_vals_km;   // B payload, each tile k-major
    const int4 *__restrict__ b_meta;        // B records' plane 0
    float tile_fill;   // rows whose A tiles hold this many values on average go to the
                       // tile-pair kernel (+inf: none)
};

// The tile-pair kernel takes the tile rows whose A tiles hold at least
// `fill` stored values on average; the LDS-accumulator kernels the others.
__device__ __forceinline__ bool tile_routed(float fill, int tiles, int payload)
{
    return tiles > 0 && static_cast<float>(payload) >= fill * static_cast<float>(tiles);
}

struct Stage {
    int *__restrict__ j;
    unsigned long long *__restrict__ m;
    int stride;
};


// The look-back words and the counters from `first` on to be zeroed before a
// sizes pass; with a pair total, also that counter to be set and the queue
// heads to be zeroed.  The symbolic pass before it does so on the side: a
// launch of its own took 1.3 us of the smallest product's 122.
struct SizesInit {
    unsigned long long *ctr;
    int first;
    unsigned long long *look;
    int64_t words;
    const unsigned long long *pair_total;
    int *queue;
    int n_queue;
};

__device__ __forceinline__ void sizes_init(const SizesInit &z)
{
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
         i < max<int64_t>(z.words, kCounters); i += stride) {
        if (i < z.words)
            z.look[i] = 0ull;
        if (i < kCounters && i >= z.first)
            z.ctr[i] = i == kCtrPairs && z.pair_total ? *z.pair_total : 0ull;
        if (z.pair_total && i < z.n_queue)
            z.queue[i] = 0;
    }
}

__device__ __forceinline__ uint32_t slot_of(int j, int bits)
{
    return hash_tile_col(j) >> (32 - bits);
}

template <typename T>
__device__ __forceinline__ T block_sum(T v, T *s_tmp)
{
    v = wave_sum(v);
    if (lane_id() == 0)
        s_tmp[threadIdx.x / kWave] = v;
    __syncthreads();
    T all = 0;
#pragma unroll
    for (int i = 0; i < kWavesPerBlock; ++i)
        all += s_tmp[i];
    __syncthreads();
    return all;
}

// Segment table of pairs [r0, r1): s_seg[p - r0] = chunk-local A tile.
// Thread t < n owns A tile t with pairs [pre_t, pre_t + nb_t).
__device__ __forceinline__ void fill_segments(unsigned char *s_seg, int pre, int nb, int r0,
                                              int r1)
{
    const int lo = max(pre, r0), hi = min(pre + nb, r1);
    for (int p = lo; p < hi; ++p)
        s_seg[p - r0] = static_cast<unsigned char>(threadIdx.x);
}

// ---------------------------------------------------------------------------
// Symbolic, one wave per row: the same hash -> compact -> rank -> stage as the
// workgroup kernel below, with a kWSlots table, so that a CU holds four times
// as many rows and their load latencies overlap.  Pairs come in two runs per
// chunk of kWChunk A tiles, the heavy and then the light tiles of the B
// rows; lane t owns both runs of tile t.  A row that outgrows the table is
// marked kLevelLarge for the workgroup kernel.
// Vector instructions bound it (88 % of its cycles on the 128^3 stencil), so
// they were cut: a pair's mask without a loop over its k or a multiply,
// scans by data-parallel moves, two entries ranked at a time: 0.73 -> 0.61 ms
// there, 0.42 -> 0.33 on the AMG batch, 0.28 -> 0.21 on the 500k-node FEM
// square.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kWave) void symbolic_wave_kernel(
    Operands g, Stage st, int64_t *__restrict__ row_tiles, int64_t *__restrict__ row_nnz,
    int *__restrict__ row_level, SizesInit init)
{
    sizes_init(init);
    __shared__ __align__(16) int s_key[kWSlots];
    __shared__ unsigned long long s_msk[kWSlots];
    __shared__ uint4 s_lo[kWChunk], s_hi[kWChunk];   // spread_tile of the chunk's tiles
    __shared__ int s_pw[2 * kWChunk]; // per (run, tile): first B tile minus first pair
    __shared__ unsigned char s_seg[kWSeg];
    static_assert(2 * kWChunk <= 256, "segment entries are bytes");

    const int row = static_cast<int>(blockIdx.x);
    const int lane = threadIdx.x;
    const int a0 = g.a_trp[row], a1 = g.a_trp[row + 1];
    for (int i = lane; i < kWSlots; i += kWave) {
        s_key[i] = kEmpty;
        s_msk[i] = 0ull;
    }
    bool ovf = false;
    for (int c0 = a0; c0 < a1 && !ovf; c0 += kWChunk) {
        const int n = min(kWChunk, a1 - c0);
        int nh = 0, bh = 0, nl = 0, bls = 0;
        if (lane < n) {
            const int4 am = g.a_meta[c0 + lane];
            const int4 br = g.a_brange[c0 + lane];
            const int2 bl = g.a_blight[c0 + lane];
            spread_tile(static_cast<uint32_t>(am.z), &s_lo[lane], &s_hi[lane]);
            nh = br.y;
            bh = br.x;
            nl = bl.y;
            bls = bl.x;
        }
        // Pair offsets: the heavy runs of all tiles, then the light runs.
        const int ih = wave_inclusive_scan(nh), il = wave_inclusive_scan(nl);
        const int heavy_total = last_lane(ih);
        const int total = heavy_total + last_lane(il);
        const int ph = ih - nh, pl = heavy_total + il - nl;
        s_pw[lane] = bh - ph;
        s_pw[kWChunk + lane] = bls - pl;
        for (int r0 = 0; r0 < total && !ovf; r0 += kWSeg) {
            const int r1 = min(total, r0 + kWSeg);
            for (int p = max(ph, r0); p < min(ph + nh, r1); ++p)
                s_seg[p - r0] = static_cast<unsigned char>(lane);
            for (int p = max(pl, r0); p < min(pl + nl, r1); ++p)
                s_seg[p - r0] = static_cast<unsigned char>(kWChunk + lane);
            __syncthreads();
            bool lane_ovf = false;
            for (int p0 = r0 + lane; p0 < r1; p0 += kWBatch * kWave) {
                int4 bm[kWBatch];
                int ai[kWBatch];
#pragma unroll
                for (int u = 0; u < kWBatch; ++u) {
                    const int p = p0 + u * kWave;
                    ai[u] = -1;
                    bm[u] = make_int4(0, 0, 0, 0);
                    if (p < r1) {
                        const int v = s_seg[p - r0];
                        ai[u] = v % kWChunk;
                        bm[u] = g.b_meta[s_pw[v] + p];
                    }
                }
#pragma unroll
                for (int u = 0; u < kWBatch; ++u) {
                    if (ai[u] < 0)
                        continue;
                    const uint64_t pm = spread_product(s_lo[ai[u]], s_hi[ai[u]],
                                                       static_cast<uint32_t>(bm[u].z));
                    if (!pm)
                        continue;
                    const int j = bm[u].x;
                    uint32_t h = slot_of(j, kWSlotBits);
                    for (int probe = 0; probe < kSymProbe; ++probe) {
                        int k = s_key[h];
                        if (k == kEmpty) {
                            k = atomicCAS(&s_key[h], kEmpty, j);
                            if (k == kEmpty) {
                                atomicOr(&s_msk[h], static_cast<unsigned long long>(pm));
                                break;
                            }
                        }
                        if (k == j) {
                            atomicOr(&s_msk[h], static_cast<unsigned long long>(pm));
                            break;
                        }
                        h = (h + 1) & (kWSlots - 1);
                        if (probe == kSymProbe - 1)
                            lane_ovf = true;
                    }
                }
            }
            ovf = __any(lane_ovf);
            __syncthreads();
        }
    }
    // Compact the occupied slots to the front; the scan total is the tile count.
    constexpr int kPer = kWSlots / kWave;
    int rk[kPer];
    unsigned long long rm[kPer];
    int mine = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        rk[i] = s_key[lane * kPer + i];
        rm[i] = s_msk[lane * kPer + i];
        mine += rk[i] != kEmpty ? 1 : 0;
    }
    const int incl = wave_inclusive_scan(mine);
    const int nt = last_lane(incl);
    if (ovf || nt > kWStage) {
        if (lane == 0)
            row_level[row] = kLevelLarge;
        return;
    }
    __syncthreads();
    int pos = incl - mine;
    int nz = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
        if (rk[i] != kEmpty) {
            s_key[pos] = rk[i];
            s_msk[pos] = rm[i];
            nz += __popcll(rm[i]);
            ++pos;
        }
    static_assert(kWStage + 4 <= kWSlots, "padding of the key list");
    if (lane < 4)
        s_key[nt + lane] = INT_MAX;   // to whole groups of four
    __syncthreads();
    // Rank by counting: entry t goes to the number of smaller columns.  Two
    // entries a lane share the reads of the list.
    const int64_t sb = static_cast<int64_t>(row) * st.stride;
    const int4 *k4 = reinterpret_cast<const int4 *>(s_key);
    auto below = [](const int4 &kk, int mj) {
        return (kk.x < mj ? 1 : 0) + (kk.y < mj ? 1 : 0) + (kk.z < mj ? 1 : 0) +
               (kk.w < mj ? 1 : 0);
    };
    auto place = [&](int t, int mj, int rank) {
        st.j[sb + rank] = mj;
        st.m[sb + rank] = s_msk[t];
    };
    for (int t = lane, left = nt; left > 0; t += 2 * kWave, left -= 2 * kWave) {
        const int t1 = t + kWave;
        const int j0 = t < nt ? s_key[t] : INT_MIN, j1 = t1 < nt ? s_key[t1] : INT_MIN;
        int r0 = 0, r1 = 0;
        if (left <= kWave) {
            for (int f = 0; f < (nt + 3) / 4; ++f)
                r0 += below(k4[f], j0);
        } else {
            for (int f = 0; f < (nt + 3) / 4; ++f) {
                const int4 kk = k4[f];
                r0 += below(kk, j0);
                r1 += below(kk, j1);
            }
        }
        if (t < nt)
            place(t, j0, r0);
        if (t1 < nt)
            place(t1, j1, r1);
    }
    nz = last_lane(wave_inclusive_scan(nz));
    if (lane == 0) {
        row_level[row] = nt > 0 ? kLevelLds : kLevelEmpty;
        row_tiles[row] = nt;
        row_nnz[row] = nz;
    }
}

// ---------------------------------------------------------------------------
// Symbolic: per-row hash of C tile masks, compaction, ranking, staging.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void symbolic_count_kernel(
    Operands g, int stage_limit, Stage st, const int *__restrict__ rows,
    int64_t *__restrict__ row_tiles, int64_t *__restrict__ row_nnz, int *__restrict__ row_level,
    int *__restrict__ slab_rows, unsigned long long *__restrict__ ctr, SizesInit init)
{
    sizes_init(init);   // (the counters below `first` are in use here)
    __shared__ __align__(16) int s_key[kSymSlots];
    __shared__ unsigned long long s_msk[kSymSlots];
    __shared__ uint4 s_lo[kChunk], s_hi[kChunk];   // spread_tile of the chunk's tiles
    __shared__ int s_b0[kChunk];
    __shared__ int s_pre[kChunk];
    __shared__ unsigned char s_seg[kSeg];
    __shared__ int s_tmp[kWavesPerBlock];
    __shared__ long long s_tmp64[kWavesPerBlock];
    __shared__ int s_ovf;

    const int row = rows[blockIdx.x];
    const int tid = threadIdx.x;
    for (int i = tid; i < kSymSlots; i += kThreads) {
        s_key[i] = kEmpty;
        s_msk[i] = 0ull;
    }
    if (tid == 0)
        s_ovf = 0;
    const int a0 = g.a_trp[row], a1 = g.a_trp[row + 1];
    for (int c0 = a0; c0 < a1; c0 += kChunk) {
        const int n = min(kChunk, a1 - c0);
        int nb = 0;
        if (tid < n) {
            const uint32_t ab = static_cast<uint32_t>(g.a_meta[c0 + tid].z);
            const int4 br = g.a_brange[c0 + tid];
            nb = br.z;
            s_b0[tid] = br.x;
            spread_tile(ab, &s_lo[tid], &s_hi[tid]);
        }
        int total = 0;
        const int pre = block_exclusive_scan<kWavesPerBlock>(nb, s_tmp, &total);
        if (tid < n)
            s_pre[tid] = pre;
        for (int r0 = 0; r0 < total; r0 += kSeg) {
            const int r1 = min(total, r0 + kSeg);
            if (tid < n)
                fill_segments(s_seg, pre, nb, r0, r1);
            __syncthreads();
            // Each thread takes kSymBatch pairs and issues their B-meta loads
            // together before using any of them.
            for (int p0 = r0 + tid; p0 < r1; p0 += kSymBatch * kThreads) {
                int4 bm[kSymBatch];
                int ai[kSymBatch];
#pragma unroll
                for (int u = 0; u < kSymBatch; ++u) {
                    const int p = p0 + u * kThreads;
                    ai[u] = -1;
                    bm[u] = make_int4(0, 0, 0, 0);
                    if (p < r1) {
                        ai[u] = s_seg[p - r0];
                        bm[u] = g.b_meta[s_b0[ai[u]] + (p - s_pre[ai[u]])];
                    }
                }
#pragma unroll
                for (int u = 0; u < kSymBatch; ++u) {
                    if (ai[u] < 0)
                        continue;
                    const uint64_t pm = spread_product(s_lo[ai[u]], s_hi[ai[u]],
                                                       static_cast<uint32_t>(bm[u].z));
                    if (!pm)
                        continue;
                    const int j = bm[u].x;
                    uint32_t h = slot_of(j, kSymSlotBits);
                    // A probe longer than kSymProbe means the table is close
                    // to full: the row is sent to the slab path, which is
                    // always correct, instead of probing on.
                    for (int probe = 0; probe < kSymProbe; ++probe) {
                        int k = s_key[h];
                        if (k == kEmpty) {
                            k = atomicCAS(&s_key[h], kEmpty, j);
                            if (k == kEmpty) {
                                atomicOr(&s_msk[h], static_cast<unsigned long long>(pm));
                                break;
                            }
                        }
                        if (k == j) {
                            atomicOr(&s_msk[h], static_cast<unsigned long long>(pm));
                            break;
                        }
                        h = (h + 1) & (kSymSlots - 1);
                        if (probe == kSymProbe - 1)
                            s_ovf = 1;
                    }
                }
            }
            __syncthreads();
            if (s_ovf)
                break;
        }
        if (s_ovf)
            break;
    }
    __syncthreads();
    // Compact the occupied slots to the front; the scan total is the row's
    // tile count.  A probe that ran out (a table close to full) or more tiles
    // than the staging holds sends the row to the slab path.
    int rk[kSymPerThread];
    unsigned long long rm[kSymPerThread];
    int mine = 0;
#pragma unroll
    for (int i = 0; i < kSymPerThread; ++i) {
        rk[i] = s_key[tid * kSymPerThread + i];
        rm[i] = s_msk[tid * kSymPerThread + i];
        mine += rk[i] != kEmpty ? 1 : 0;
    }
    int nt = 0;
    int pos = block_exclusive_scan<kWavesPerBlock>(mine, s_tmp, &nt);
    if (s_ovf || nt > stage_limit) {
        if (tid == 0) {
            row_level[row] = kLevelSlab;
            row_tiles[row] = 0;
            row_nnz[row] = 0;
            slab_rows[atomicAdd(&ctr[kCtrSymSlab], 1ull)] = row;
        }
        return;
    }
    long long nz = 0;
#pragma unroll
    for (int i = 0; i < kSymPerThread; ++i)
        if (rk[i] != kEmpty) {
            s_key[pos] = rk[i];
            s_msk[pos] = rm[i];
            nz += __popcll(rm[i]);
            ++pos;
        }
    __syncthreads();
    const int64_t sb = static_cast<int64_t>(row) * st.stride;
    if (nt <= kThreads) {
        // Rank by counting: entry t goes to the number of smaller columns.
        // The keys are read four at a time, the last nt % 4 one by one.
        if (tid < nt) {
            const int mj = s_key[tid];
            const int4 *k4 = reinterpret_cast<const int4 *>(s_key);
            int rank = 0;
            const int full = nt & ~3;
            for (int f = 0; f < full / 4; ++f) {
                const int4 kk = k4[f];
                rank += (kk.x < mj ? 1 : 0) + (kk.y < mj ? 1 : 0) + (kk.z < mj ? 1 : 0) +
                        (kk.w < mj ? 1 : 0);
            }
            for (int f = full; f < nt; ++f)
                rank += s_key[f] < mj ? 1 : 0;
            st.j[sb + rank] = mj;
            st.m[sb + rank] = s_msk[tid];
        }
    } else {
        int npow = 1;
        while (npow < nt)
            npow <<= 1;
        for (int i = nt + tid; i < npow; i += kThreads)
            s_key[i] = INT_MAX;
        __syncthreads();
        for (int k = 2; k <= npow; k <<= 1) {
            for (int jj = k >> 1; jj > 0; jj >>= 1) {
                for (int i = tid; i < npow; i += kThreads) {
                    const int ixj = i ^ jj;
                    if (ixj > i) {
                        const int ki = s_key[i], kx = s_key[ixj];
                        const bool up = (i & k) == 0;
                        if ((ki > kx) == up) {
                            s_key[i] = kx;
                            s_key[ixj] = ki;
                            const unsigned long long t = s_msk[i];
                            s_msk[i] = s_msk[ixj];
                            s_msk[ixj] = t;
                        }
                    }
                }
                __syncthreads();
            }
        }
        for (int i = tid; i < nt; i += kThreads) {
            st.j[sb + i] = s_key[i];
            st.m[sb + i] = s_msk[i];
        }
    }
    const long long row_nz = block_sum(nz, s_tmp64);
    if (tid == 0) {
        row_level[row] = nt > 0 ? kLevelLds : kLevelEmpty;
        row_tiles[row] = nt;
        row_nnz[row] = row_nz;
    }
}

// Staged (column, mask) lists -> final C structure; one wave per row.  The
// row's local-column bytes are assembled in LDS and written coalesced: a
// table gives, for a row byte x of a tile mask, the columns of its set bits
// packed in increasing order, and each tile row ORs them into the zeroed
// buffer with at most two 64-bit LDS ORs.
__global__ __launch_bounds__(kThreads) void symbolic_write_kernel(
    const int *__restrict__ rows, int count, Stage st, const int *__restrict__ row_level, COut c,
    float tile_fill = 0.f, const int *__restrict__ a_trp = nullptr,
    const int *__restrict__ a_row_off = nullptr)
{
    __shared__ unsigned long long s_buf[kWavesPerBlock][kWriteBuf / 8];
    __shared__ unsigned long long s_cols[256];
    const int w = threadIdx.x / kWave;
    const int lane = lane_id();
    {
        const int x = threadIdx.x;
        unsigned long long v = 0;
        int nset = 0;
#pragma unroll
        for (int cl = 0; cl < 8; ++cl)
            if ((x >> cl) & 1)
                v |= static_cast<unsigned long long>(cl) << (8 * nset++);
        s_cols[x] = v;
    }
    __syncthreads();
    const int idx = blockIdx.x * kWavesPerBlock + w;
    if (idx >= count)
        return;
    const int row = rows ? rows[idx] : idx;
    if (row_level[row] != kLevelLds)
        return;
    // Without a list: the rows the tile-pair kernel takes.
    if (!rows && !tile_routed(tile_fill, a_trp[row + 1] - a_trp[row],
                              a_row_off[row + 1] - a_row_off[row]))
        return;
    const int64_t tb = c.tile_ptr[row];
    const int nt = static_cast<int>(c.tile_ptr[row + 1] - tb);
    const int64_t zb = c.row_nnz_off[row];
    const int64_t nnz_row = c.row_nnz_off[row + 1] - zb;
    const bool staged = nnz_row <= kWriteBuf;
    const int64_t sb = static_cast<int64_t>(row) * st.stride;
    unsigned long long *buf = s_buf[w];
    if (staged) {
        for (int i = lane; i < kWriteBuf / 8; i += kWave)
            buf[i] = 0ull;
        wave_sync();
    }
    int64_t carry = 0;
    for (int q0 = 0; q0 < nt; q0 += kWave) {
        const int q = q0 + lane;
        uint64_t m = q < nt ? st.m[sb + q] : 0ull;
        const int pc = __popcll(m);
        const int incl = wave_inclusive_scan(pc);
        if (q < nt) {
            const int64_t off = carry + (incl - pc);
            const int64_t t = tb + q;
            const uint64_t ro = packed_row_offsets(m);
            c.col[t] = st.j[sb + q];
            c.mask[t] = m;
            c.tile_nnz[t] = zb + off;
            reinterpret_cast<uint64_t *>(c.csr_ptr)[t] = ro;
            if (staged) {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const uint32_t x = static_cast<uint32_t>(m >> (8 * r)) & 0xFFu;
                    if (!x)
                        continue;
                    const int p = static_cast<int>(off) + static_cast<int>((ro >> (8 * r)) & 0xFFu);
                    const unsigned long long v = s_cols[x];
                    const int sh = (p & 7) * 8;
                    atomicOr(&buf[p >> 3], v << sh);
                    if (sh && __popc(x) * 8 + sh > 64)
                        atomicOr(&buf[(p >> 3) + 1], v >> (64 - sh));
                }
            } else {
                int i = 0;
                while (m) {
                    const int pos = __builtin_ctzll(m);
                    m &= m - 1;
                    c.csr_col[zb + off + i] = static_cast<uint8_t>(pos & 7);
                    ++i;
                }
            }
        }
        carry += last_lane(incl);
    }
    if (staged) {
        wave_sync();
        const unsigned char *bytes = reinterpret_cast<const unsigned char *>(buf);
        for (int64_t i = lane; i < nnz_row; i += kWave)
            c.csr_col[zb + i] = bytes[i];
    }
}

// Cost of each listed row: the (A tile, B tile) pairs it visits.  One wave
// per row.
__global__ __launch_bounds__(kThreads) void row_pairs_kernel(const int *__restrict__ rows, int n,
                                                             const int *__restrict__ a_trp,
                                                             const int4 *__restrict__ a_brange,
                                                             unsigned int *__restrict__ cost)
{
    const int i = blockIdx.x * kWavesPerBlock + static_cast<int>(threadIdx.x) / kWave;
    if (i >= n)
        return;
    const int row = rows[i];
    unsigned long long sum = 0;
    for (int t = a_trp[row] + lane_id(); t < a_trp[row + 1]; t += kWave)
        sum += static_cast<unsigned int>(a_brange[t].z);
    sum = wave_sum(sum);
    if (lane_id() == 0)
        cost[i] = static_cast<unsigned int>(sum < 0xffffffffull ? sum : 0xffffffffull);
}

// ---------------------------------------------------------------------------
// Numeric, LDS path: one workgroup per row, LDS accumulator.
// ---------------------------------------------------------------------------
// The row's output segment is an FP64 accumulator in LDS, every C tile of
// the row is in a hash table, and each thread takes the pairs p,
// p + kThreads, ... of a window.  A pair walks its B tile's entries in
// k-major order (its record holds them so): when the walk reaches row k of
// B, the lane loads the first values of column k of the A tile (staged
// column-major in LDS) into registers, and B entry (k, cl) adds
// A(r, k) * B(k, cl) into C(r, cl) for every row r of that column.
//
// The accumulator has the output's layout: a tile's entries row by row,
// columns ascending.  When every row of the C tile is one contiguous run of
// columns and every column of the A tile one contiguous run of rows, the
// slot of C(r, cl) is (first slot of row r - its first column) + cl: the
// lane takes those bases for the rows of A column k once per k, and each
// product costs one add.  Other tiles take the slot from a popcount of the
// tile mask.
// Hash slot of a C tile: {tile column or kEmpty, first value slot | local
// tile index << 16, row_runs low word, row_runs high word}, so that one
// LDS read gives a pair everything the walk needs of its C tile.
__device__ __forceinline__ int4 make_tile_slot(int j, int base, int q, uint64_t runs)
{
    return make_int4(j, base | (q << 16), static_cast<int>(static_cast<uint32_t>(runs)),
                     static_cast<int>(static_cast<uint32_t>(runs >> 32)));
}

// Byte value of a row whose columns are not one contiguous run.
constexpr uint32_t kNoRun = 0x80u;

__device__ __forceinline__ bool is_run(uint32_t bits)
{
    const uint32_t x = bits >> __builtin_ctz(bits);
    return (x & (x + 1)) == 0;
}

// Byte r: (slot of row r's first entry within the tile) - (its first
// column) + kTileN, which is 1 to 64, when the row's columns are contiguous,
// kNoRun when they are not, 0 for an empty row (never addressed).
__device__ __forceinline__ uint64_t row_runs(uint64_t m)
{
    uint64_t out = 0;
    int first = 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const uint32_t bits = static_cast<uint32_t>(m >> (8 * r)) & 0xFFu;
        uint32_t b = 0;
        if (bits)
            b = is_run(bits) ? static_cast<uint32_t>(first + kTileN - __builtin_ctz(bits)) : kNoRun;
        out |= static_cast<uint64_t>(b) << (8 * r);
        first += __popc(bits);
    }
    return out;
}

__device__ __forceinline__ int run_base(uint64_t runs, int r)
{
    return static_cast<int>((runs >> (8 * r)) & 0xFFu) - kTileN;
}

// Byte k: rows of A column k as count | first row << 4, with bit 7 set when
// they are not one contiguous run of at most kColRegs rows.
__device__ __forceinline__ uint32_t a_column_runs(uint32_t ab)
{
    uint32_t out = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t rk = byte_of(ab, k);
        if (rk) {
            const bool regs = is_run(rk) && __popc(rk) <= kColRegs;
            out |= ((__popc(rk) | (__builtin_ctz(rk) << 4) | (regs ? 0u : kNoRun)) << (8 * k));
        }
    }
    return out;
}

// Place of a C row's i-th value in the accumulator.
template <class Cfg>
__device__ __forceinline__ int acc_place(int i)
{
    return Cfg::kSpread ? i + i / kSkew : i;
}

// Sampled start/end times of the numeric kernel's waves (the timeline
// trace): workgroups b with b mod 2^shift == phase record, per wave, the
// compute unit and the device's constant-rate wall clock at entry and exit.
// Null pointers switch it off.
struct Timeline {
    unsigned long long *start = nullptr, *end = nullptr;
    unsigned int *cu = nullptr;
    unsigned int shift = 0, phase = 0;
};

__device__ __forceinline__ void trace_mark(const Timeline &tl, bool at_end)
{
    if (!tl.start || lane_id() != 0)
        return;
    const unsigned int b = blockIdx.x;
    if ((b & ((1u << tl.shift) - 1u)) != tl.phase)
        return;
    const size_t slot = static_cast<size_t>((b - tl.phase) >> tl.shift) * kWavesPerBlock +
                        threadIdx.x / kWave;
    const unsigned long long t = static_cast<unsigned long long>(wall_clock64());
    if (at_end) {
        tl.end[slot] = t;
    } else {
        tl.cu[slot] = __smid();
        tl.start[slot] = t;
    }
}

template <class Cfg, bool TRACE = false>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kWavesPerSimd) void numeric_row_kernel(
    Operands g, const int4 *__restrict__ recs, int64_t rec_n, const int *__restrict__ rows,
    const int *__restrict__ row_level, Stage st, COut c, Timeline tl)
{
    constexpr int kT = Cfg::kThreads, kCh = Cfg::kChunk, kSg = Cfg::kSeg, kNW = kT / kWave;
    static_assert(kT == 4 * kCh && kT % kWave == 0, "one thread per (pair run, chunk tile)");
    __shared__ double s_acc[Cfg::kAcc + (Cfg::kSpread ? Cfg::kAcc / kSkew : 0)];
    __shared__ double s_acol[Cfg::kAStage + kColRegs];
    __shared__ unsigned long long s_cmask[Cfg::kTiles];   // C tile masks, bit r * 8 + cl
    __shared__ int s_cbase[Cfg::kTiles];   // first slot of each tile within the row's segment
    __shared__ int4 s_slot[Cfg::kSlots];   // hash of the row's C tiles (make_tile_slot)
    // Per chunk A tile: its staged info and B runs (see stage_tile), and per
    // (run, tile) the first B record minus the run's first pair.
    __shared__ int4 s_at[kCh];
    __shared__ int4 s_br[kCh];
    __shared__ int s_pw[kT];
    __shared__ unsigned char s_seg[kSg];
    __shared__ int s_tmp[kNW];
    __shared__ int s_dual[2 * kNW];

    const int tid = threadIdx.x;
    if constexpr (TRACE)
        trace_mark(tl, false);
    // Rows (or list entries) in 64-row chunks per XCD: the B records that
    // neighbouring rows share stay in one L2 for a run of 64 rows, and the
    // window of rows in flight still spans the chip.  Against row b in
    // workgroup b: the same speed or 1 % better on the stencil step, a
    // third less L2 fetch traffic, and 0.5 % on the batched forms' lists.
    const int bx = xcd_chunk_row<64>(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
    const int row = rows ? rows[bx] : bx;
    // The row's inputs come in two rounds of independent loads: its level,
    // C's row extents, A's tile and payload extents (the payload base per
    // tile row is precomputed); then the first staged C tile, A value and A
    // tile of each thread, before the first barrier.
    const int level = row_level[row];
    const int64_t t0 = c.tile_ptr[row];
    const int nt = static_cast<int>(c.tile_ptr[row + 1] - t0);
    const int64_t zb = c.row_nnz_off[row];
    const int64_t nnz_row = c.row_nnz_off[row + 1] - zb;
    const int a0 = g.a_trp[row], a1 = g.a_trp[row + 1];
    const int a_base = g.a_row_off[row];
    const int a_len = g.a_row_off[row + 1] - a_base;
    bool skip = (level != kLevelLds) | (nt > Cfg::kTiles) | (nnz_row > Cfg::kAcc) |
                (a_len > Cfg::kAStage) | tile_routed(g.tile_fill, a1 - a0, a_len);
    if constexpr (Cfg::kLeavesTiny)
        skip |= fits_row<TinyRow>(nt, nnz_row, a_len);
    if (skip) {
        if constexpr (TRACE)
            trace_mark(tl, true);
        return;
    }
    const int64_t sb = static_cast<int64_t>(row) * st.stride;
    int j0 = 0;
    uint64_t m0 = 0;
    if (tid < nt) {
        j0 = st.j[sb + tid];
        m0 = st.m[sb + tid];
    }
    double av0 = 0.0;
    if (tid < a_len)
        av0 = g.a_vals_cm[a_base + tid];
    int4 am0 = make_int4(0, 0, 0, 0), br0 = make_int4(0, 0, 0, 0);
    int2 bl0 = make_int2(0, 0);
    if (tid < min(kCh, a1 - a0)) {
        am0 = g.a_meta[a0 + tid];
        br0 = g.a_brange[a0 + tid];
        bl0 = g.a_blight[a0 + tid];
    }
    for (int i = tid; i < Cfg::kSlots; i += kT)
        s_slot[i] = make_int4(kEmpty, 0, 0, 0);
    for (int i = tid; i < acc_place<Cfg>(static_cast<int>(nnz_row)); i += kT)
        s_acc[i] = 0.0;
    if (tid < a_len)
        s_acol[tid] = av0;
    for (int i = tid + kT; i < a_len; i += kT)
        s_acol[i] = g.a_vals_cm[a_base + i];
    if (tid < kColRegs)
        s_acol[a_len + tid] = 0.0;   // the register loads of a column may run past it
    // Chunk tile info: {rows present in column k (byte k), heavy (bit 0) and
    // first staged value of column k (byte k, k > 0), first staged value,
    // row runs of the columns (a_column_runs)} and its B runs {first heavy
    // tile, heavy count, first light tile, light count}.
    auto stage_tile = [&](const int4 &am, const int4 &br, const int2 &bl) {
        const uint32_t ab = static_cast<uint32_t>(am.z);
        const uint32_t p1 = __popc(byte_of(ab, 0));
        const uint32_t p2 = p1 + __popc(byte_of(ab, 1));
        const uint32_t p3 = p2 + __popc(byte_of(ab, 2));
        const uint32_t heavy = __popc(static_cast<uint32_t>(am.y)) >= kHeavyMin ||
                                       __popc(nonzero_tops(ab)) > 1
                                   ? 1u
                                   : 0u;
        s_at[tid] = make_int4(static_cast<int>(ab),
                              static_cast<int>(heavy | (p1 << 8) | (p2 << 16) | (p3 << 24)),
                              static_cast<int>(static_cast<uint32_t>(am.w) & ~kDenseBit) - a_base,
                              static_cast<int>(a_column_runs(ab)));
        s_br[tid] = make_int4(br.x, br.y, bl.x, bl.y);
    };
    // The chunk's pairs come in four runs, one per (A class, B class): heavy
    // and light A tiles times the heavy and light runs of their B rows, so
    // that the lanes of a wave take pairs of like cost.  Thread v stands for
    // run v / kCh of tile v % kCh.
    const int run = tid / kCh, vt = tid % kCh;
    auto chunk_runs = [&](int n, int &nb, int &bstart) {
        nb = 0;
        bstart = 0;
        if (vt < n && (s_at[vt].y & 1) == ((run & 1) == 0 ? 1 : 0)) {
            const int4 br = s_br[vt];
            nb = run < 2 ? br.y : br.w;
            bstart = run < 2 ? br.x : br.z;
        }
    };
    // C's structure for the row from the staged (column, mask) list, in
    // column order, with value offsets from a scan of the tile popcounts;
    // the row's tiles also go into LDS and the hash table.
    auto insert_tile = [&](int q, int j, uint64_t m, int base) {
        const int64_t t = t0 + q;
        c.col[t] = j;
        c.mask[t] = m;
        c.tile_nnz[t] = zb + base;
        reinterpret_cast<uint64_t *>(c.csr_ptr)[t] = packed_row_offsets(m);
        s_cmask[q] = m;
        s_cbase[q] = base;
        uint32_t h = slot_of(j, Cfg::kSlotBits);
        while (atomicCAS(&s_slot[h].x, kEmpty, j) != kEmpty)
            h = (h + 1) & (Cfg::kSlots - 1);
        s_slot[h] = make_tile_slot(j, base, q, row_runs(m));
    };
    if (tid < min(kCh, a1 - a0))
        stage_tile(am0, br0, bl0);
    __syncthreads();   // chunk 0 staged, table cleared
    // One scan gives the value offsets of the first kT tiles (one per
    // thread) and chunk 0's pair offsets.
    int nb = 0, bstart = 0, pre = 0, total = 0, base = 0, carry = 0;
    chunk_runs(min(kCh, a1 - a0), nb, bstart);
    dual_exclusive_scan<kNW>(tid < nt ? __popcll(m0) : 0, nb, s_dual, &base, &pre, &carry, &total);
    if (tid < nt)
        insert_tile(tid, j0, m0, base);
    for (int q0 = kT; q0 < nt; q0 += kT) {
        const int q = q0 + tid;
        int j = 0;
        uint64_t m = 0;
        if (q < nt) {
            j = st.j[sb + q];
            m = st.m[sb + q];
        }
        int tot = 0;
        const int qb = carry + block_exclusive_scan<kNW>(q < nt ? __popcll(m) : 0, s_tmp, &tot);
        carry += tot;
        if (q < nt)
            insert_tile(q, j, m, qb);
    }
    for (int c0 = a0; c0 < a1; c0 += kCh) {
        const int n = min(kCh, a1 - c0);
        if (c0 != a0) {
            if (tid < n)
                stage_tile(g.a_meta[c0 + tid], g.a_brange[c0 + tid], g.a_blight[c0 + tid]);
            __syncthreads();
            chunk_runs(n, nb, bstart);
            pre = block_exclusive_scan<kNW>(nb, s_tmp, &total);
        }
        s_pw[tid] = bstart - pre;
        {
            for (int r0 = 0; r0 < total; r0 += kSg) {
                const int r1 = min(total, r0 + kSg);
                if (nb > 0)
                    fill_segments(s_seg, pre, nb, r0, r1);
                __syncthreads();
                // Consecutive lanes take consecutive pairs, so a wave's record
                // loads are one contiguous stretch of B's records.
                for (int p = r0 + tid; p < r1; p += kT) {
                    const int v = s_seg[p - r0];
                    const int4 at = s_at[v % kCh];
                    // The pair's B record, part by part from the planes.
                    const int64_t rb_idx = s_pw[v] + p;
                    BRecord rec;
                    rec.meta = recs[rb_idx];
                    // Runs 2 and 3 hold the light B tiles (fewer than
                    // kHeavyMin entries, one row): their values fit in the
                    // first part.
                    static_assert(kHeavyMin - 1 <= 2, "light values fill one record part");
                    const bool light_b = v >= 2 * kCh;
                    const bool one = Cfg::kSpread && v >= kCh;
#pragma unroll
                    for (int i = 0; i < kRecVals / 2; ++i) {
                        double2 d = make_double2(0.0, 0.0);
                        if (one ? i < 1 && light_b : i < 1 || !light_b)
                            d = reinterpret_cast<const double2 *>(recs + (i + 1) * rec_n)[rb_idx];
                        rec.v[2 * i] = d.x;
                        rec.v[2 * i + 1] = d.y;
                    }
                    const uint32_t ab = static_cast<uint32_t>(at.x);
                    const uint32_t bb = static_cast<uint32_t>(rec.meta.z);
                    const uint32_t boff = static_cast<uint32_t>(rec.meta.w) & ~kDenseBit;
                    const uint32_t ks = nonzero_tops(ab) & nonzero_tops(bb);
                    if (!ks)
                        continue;
                    // One of the tiles is light: the pair is column k1 of A times
                    // row k1 of B alone, whose values a light B tile has in its
                    // first part.
                    const int k1 = __builtin_ctz(ks) >> 3;
                    const int j1 = __popc(bb & ((1u << (8 * k1)) - 1u));
                    auto value = [&](int j) {
                        return j < kRecVals ? reinterpret_cast<const double *>(
                                                  recs + (1 + (j >> 1)) * rec_n + rb_idx)[j & 1]
                                            : g.b_vals_km[boff + j];
                    };
                    if (one && !light_b) {
                        const int n1 = __popc(byte_of(bb, k1));
#pragma unroll
                        for (int i = 0; i < kOneVals; ++i)
                            if (i < n1)
                                rec.v[i] = value(j1 + i);
                    }
                    // C tile of the pair; every tile of the row is in the table and
                    // at least half of its slots are empty, so the probe ends.
                    uint32_t h = slot_of(rec.meta.x, Cfg::kSlotBits);
                    int4 sl;
                    for (;;) {
                        sl = s_slot[h];
                        if (sl.x == rec.meta.x || sl.x == kEmpty)
                            break;
                        h = (h + 1) & (Cfg::kSlots - 1);
                    }
                    if (sl.x != rec.meta.x)
                        continue;
                    const int q = sl.y >> 16;
                    const unsigned long long cruns =
                        (static_cast<unsigned long long>(static_cast<uint32_t>(sl.w)) << 32) |
                        static_cast<uint32_t>(sl.z);
                    const int acc = sl.y & 0xFFFF;   // first slot of the tile
                    const uint32_t apf = static_cast<uint32_t>(at.y) & ~0xFFu;
                    const uint32_t aruns = static_cast<uint32_t>(at.w);
                    const double *acol = s_acol + at.z;
                    // B entries in k-major order: the record's values, then the
                    // payload's.  The first kExtVals payload values are loaded once
                    // kExtVals record values have been used, into the registers
                    // those held, and arrive while the rest of the record is walked.
                    auto walk = [&](auto &&entry) {
                        uint32_t mz = bb;
                        if (one) {
                            mz &= 0xFFu << (8 * k1);
#pragma unroll
                            for (int j = 0; j < kOneVals; ++j) {
                                if (mz) {
                                    const int pos = __builtin_ctz(mz);
                                    mz &= mz - 1;
                                    entry(pos, rec.v[j]);
                                }
                            }
                            for (int j = j1 + kOneVals; mz; ++j) {
                                const int pos = __builtin_ctz(mz);
                                mz &= mz - 1;
                                entry(pos, value(j));
                            }
                            return;
                        }
                        const int nbv = __popc(mz);
                        double ext[kExtVals > 0 ? kExtVals : 1];
#pragma unroll
                        for (int j = 0; j < kRecVals; ++j) {
                            if (j == kExtVals) {
#pragma unroll
                                for (int i = 0; i < kExtVals; ++i)
                                    ext[i] = kRecVals + i < nbv ? g.b_vals_km[boff + kRecVals + i]
                                                                : 0.0;
                            }
                            if (mz) {
                                const int pos = __builtin_ctz(mz);
                                mz &= mz - 1;
                                entry(pos, rec.v[j]);
                            }
                        }
#pragma unroll
                        for (int i = 0; i < kExtVals; ++i) {
                            if (mz) {
                                const int pos = __builtin_ctz(mz);
                                mz &= mz - 1;
                                entry(pos, ext[i]);
                            }
                        }
                        int j = kRecVals + kExtVals;
                        while (mz) {
                            const int pos = __builtin_ctz(mz);
                            mz &= mz - 1;
                            entry(pos, g.b_vals_km[boff + j]);
                            ++j;
                        }
                    };
                    // The wave takes one way together: with lanes on both it
                    // would run both (banded batch: 0.60 and 0.46 ms against
                    // 0.57 and 0.42 in the two instances it uses).
                    if (__all(((cruns & 0x8080808080808080ull) | (aruns & 0x80808080u)) == 0)) {
                        // All runs, and no A column longer than kColRegs: at each
                        // new k the lane takes the values and the row bases of the
                        // rows r0, r0 + 1, ... of A column k into registers.
                        static_assert(kColRegs <= 4, "row bases of one dword");
                        int kcur = -1;
                        uint32_t kd = 0;   // a_column_runs byte of column kcur
                        uint32_t rb = 0;   // byte i: row base of row r0 + i
                        double av[kColRegs];
#pragma unroll
                        for (int i = 0; i < kColRegs; ++i)
                            av[i] = 0.0;
                        walk([&](int pos, double vb) {
                            const int k = pos >> 3, cl = pos & 7;
                            if (k != kcur) {
                                kcur = k;
                                kd = byte_of(aruns, k);
                                rb = static_cast<uint32_t>(cruns >> (8 * (kd >> 4)));
                                const double *ap = acol + byte_of(apf, k);
#pragma unroll
                                for (int i = 0; i < kColRegs; ++i)
                                    av[i] = ap[i];
                            }
                            const int pc = acc + cl;
                            const int na = static_cast<int>(kd & 15u);
#pragma unroll
                            for (int i = 0; i < kColRegs; ++i)
                                if (i < na)
                                    atomicAdd(s_acc + acc_place<Cfg>(pc + run_base(rb, i)), av[i] * vb);
                        });
                    } else {
                        // Slots from popcounts of the tile mask.
                        const uint64_t cm = s_cmask[q];
                        walk([&](int pos, double vb) {
                            const int k = pos >> 3, cl = pos & 7;
                            const double *ap = acol + byte_of(apf, k);
                            uint32_t rr = byte_of(ab, k);
                            int i = 0;
                            while (rr) {
                                const int r = __builtin_ctz(rr);
                                rr &= rr - 1;
                                const int slot =
                                    acc + __popcll(cm & ((1ull << (r * 8 + cl)) - 1ull));
                                atomicAdd(s_acc + acc_place<Cfg>(slot), ap[i++] * vb);
                            }
                        });
                    }
                }
                __syncthreads();
            }
        }
    }
    __syncthreads();
    // Column bytes of the row's entries, staged in the A buffer (free now),
    // then values and column bytes stream out together.
    // They are staged at the output's byte alignment, zb mod 4, so that
    // whole words go out as words.
    const int shift = static_cast<int>(zb & 3);
    unsigned char *s_colb = reinterpret_cast<unsigned char *>(s_acol);
    static_assert(sizeof(s_acol) >= Cfg::kAcc + 3, "column byte staging");
    for (int it = tid; it < nt * 8; it += kT) {
        const int q = it >> 3, r = it & 7;
        const uint64_t m = s_cmask[q];
        uint32_t x = static_cast<uint32_t>(m >> (8 * r)) & 0xFFu;
        int o = shift + s_cbase[q] + __popcll(m & ((1ull << (8 * r)) - 1ull));
        while (x) {
            s_colb[o++] = static_cast<unsigned char>(__builtin_ctz(x));
            x &= x - 1;
        }
    }
    __syncthreads();
    for (int64_t i = tid; i < nnz_row; i += kT)
        c.val[zb + i] = s_acc[acc_place<Cfg>(static_cast<int>(i))];
    // Words [0, nw) of the row's column bytes from the aligned word at zb -
    // shift; the first and last may hold bytes of the neighbouring rows and
    // are written byte by byte.
    unsigned char *colw = c.csr_col + (zb - shift);
    const int nw = static_cast<int>((shift + nnz_row + 3) >> 2);
    for (int i = tid; i < nw; i += kT) {
        const uint32_t v = reinterpret_cast<const uint32_t *>(s_colb)[i];
        if (i > 0 && i < nw - 1) {
            reinterpret_cast<uint32_t *>(colw)[i] = v;
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int idx = 4 * i + b;
                if (idx >= shift && idx < shift + nnz_row)
                    colw[idx] = static_cast<unsigned char>(v >> (8 * b));
            }
        }
    }
    if constexpr (TRACE)
        trace_mark(tl, true);
}

struct RowLists {
    int *__restrict__ rows[kRowClasses];
    int *__restrict__ outgrown;
};

// 1024 rows a workgroup: the look-back moves 64 workgroups a step, and at 256
// rows the pass took 95 us of the AMG batch's two products, now 42 us.
constexpr int kSizeThreads = 1024;
constexpr int kSizeWaves = kSizeThreads / kWave;

// Sizes of C and the numeric routing from the rows' counts, in one launch:
// every workgroup sums its rows, takes the rows' offsets by a decoupled
// look-back, lists its rows for the numeric kernels, and the last one to
// finish writes the counters to the host's buffer.  Rows that still wait
// for another symbolic pass (outgrown, or slab rows before theirs) count as
// empty; the host then runs that pass and this kernel again.  It replaces
// two row-listing passes, two scans, a gather and a copy: eight launches of
// 2 to 10 us each, most of what a product of a few thousand rows spent
// between its symbolic and its numeric pass.
__global__ __launch_bounds__(kSizeThreads) void row_sizes_kernel(
    int n, const int *__restrict__ level, bool slab_done, const int64_t *__restrict__ tiles,
    const int64_t *__restrict__ nnz, const int *__restrict__ a_trp,
    const int *__restrict__ a_row_off, float tile_fill, bool list, int64_t *__restrict__ tile_ptr,
    int64_t *__restrict__ nnz_off, int64_t *__restrict__ tile_nnz, int64_t tile_nnz_len,
    RowLists out, unsigned long long *__restrict__ ctr, unsigned long long *__restrict__ look,
    unsigned long long *__restrict__ host)
{
    __shared__ unsigned int s_block;
    __shared__ unsigned long long s_x[kSizeWaves + 1], s_y[kSizeWaves + 1];
    __shared__ int s_count[kRowClasses + 1][kSizeWaves];
    __shared__ int s_base[kRowClasses + 1];
    const int tid = threadIdx.x, w = tid / kWave;
    if (tid == 0)
        s_block = static_cast<unsigned int>(atomicAdd(&ctr[kCtrTicket], 1ull));
    __syncthreads();
    const int64_t b = s_block;
    const int64_t i = b * kSizeThreads + tid;
    unsigned long long nt = 0, nz = 0;
    int cls = -1;   // list the row goes to, kRowClasses for an outgrown row
    bool slab = false, sym_slab = false;
    int slots_of = 0, tiles_of = 0;
    unsigned long long wide = 0;
    if (i < n) {
        const int lv = level[i];
        const bool sized = lv == kLevelLds || (lv == kLevelSlab && slab_done);
        if (sized) {
            nt = static_cast<unsigned long long>(tiles[i]);
            nz = static_cast<unsigned long long>(nnz[i]);
        }
        const int a_tiles = a_trp[i + 1] - a_trp[i];
        const int64_t alen = a_row_off[i + 1] - a_row_off[i];
        if (lv == kLevelLarge) {
            cls = kRowClasses;
        } else if (sized && list && !tile_routed(tile_fill, a_tiles, static_cast<int>(alen))) {
            const int64_t t = static_cast<int64_t>(nt), z = static_cast<int64_t>(nz);
            cls = lv == kLevelSlab                ? kRowSlab
                  : fits_row<TinyRow>(t, z, alen)   ? kRowTiny
                  : fits_row<SmallRow>(t, z, alen)  ? kRowSmall
                  : fits_row<MediumRow>(t, z, alen) ? kRowMid
                  : fits_row<LargeRow>(t, z, alen)  ? kRowLarge
                                                    : kRowSlab;
        }
        if (sized && nt > kWideTiles && tile_routed(tile_fill, a_tiles, static_cast<int>(alen)))
            wide = (1ull << kWideRowShift) + nt;
        slab = (lv == kLevelSlab && !slab_done) || cls == kRowSlab;
        sym_slab = lv == kLevelSlab && !slab_done;
        if (slab)
            slots_of = static_cast<int>(alen), tiles_of = a_tiles;
    }
    // Sizes of the slab rows, an atomic each for a wave that has some: one for
    // every row took 20 us of a pass over 2000 of them.
    if (__any(slab)) {
        unsigned long long sum =
            sym_slab ? (static_cast<unsigned long long>(tiles_of) << 32) |
                           static_cast<unsigned int>(slots_of)
                     : 0ull;
        sum = wave_sum(sum);
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) {
            slots_of = max(slots_of, __shfl_xor(slots_of, o, kWave));
            tiles_of = max(tiles_of, __shfl_xor(tiles_of, o, kWave));
        }
        if (lane_id() == 0) {
            atomicMax(&ctr[kCtrLongest], static_cast<unsigned long long>(slots_of));
            atomicMax(&ctr[kCtrMostTiles], static_cast<unsigned long long>(tiles_of));
            if (sum)
                atomicAdd(&ctr[kCtrSymSizes], sum);
        }
        // There before the workgroup counts as done, whichever wave this is.
        __threadfence();
    }
    if (__any(wide != 0)) {
        wide = wave_sum(wide);
        if (lane_id() == 0)
            atomicAdd(&ctr[kCtrWide], wide);
        __threadfence();   // (likewise)
    }
    const unsigned long long ix = wave_inclusive_scan(nt), iy = wave_inclusive_scan(nz);
    if (lane_id() == kWave - 1) {
        s_x[w] = ix;
        s_y[w] = iy;
    }
    int rank = 0;
#pragma unroll
    for (int c = 0; c <= kRowClasses; ++c) {
        const unsigned long long m = __ballot(cls == c);
        if (cls == c)
            rank = __popcll(m & ((1ull << lane_id()) - 1ull));
        if (lane_id() == 0)
            s_count[c][w] = __popcll(m);
    }
    __syncthreads();
    unsigned long long bx = 0, by = 0, all_x = 0, all_y = 0;
#pragma unroll
    for (int k = 0; k < kSizeWaves; ++k) {
        bx += k < w ? s_x[k] : 0ull;
        by += k < w ? s_y[k] : 0ull;
        all_x += s_x[k];
        all_y += s_y[k];
    }
    if (tid <= kRowClasses) {
        // One atomic per list and workgroup that has rows for it.
        int sum = 0;
#pragma unroll
        for (int k = 0; k < kSizeWaves; ++k)
            sum += s_count[tid][k];
        unsigned long long *at = tid == kRowClasses ? &ctr[kCtrOutgrown] : &ctr[kCtrRows + tid];
        s_base[tid] = sum ? static_cast<int>(atomicAdd(at, static_cast<unsigned long long>(sum))) : 0;
    }
    if (w == 0) {
        if (lane_id() == 0)
            publish(look, b, b == 0 ? kUpTo : kOwn, all_x, all_y);
        unsigned long long px = 0, py = 0;
        if (b > 0) {
            look_back(look, b, &px, &py);
            if (lane_id() == 0)
                publish(look, b, kUpTo, px + all_x, py + all_y);
        }
        if (lane_id() == 0) {
            s_x[kSizeWaves] = px;
            s_y[kSizeWaves] = py;
        }
    }
    __syncthreads();
    const unsigned long long px = s_x[kSizeWaves], py = s_y[kSizeWaves];
    if (i < n) {
        tile_ptr[i] = static_cast<int64_t>(px + bx + ix - nt);
        nnz_off[i] = static_cast<int64_t>(py + by + iy - nz);
        if (cls >= 0) {
            int at = s_base[cls] + rank;
#pragma unroll
            for (int k = 0; k < kSizeWaves; ++k)
                at += k < w ? s_count[cls][k] : 0;
            (cls == kRowClasses ? out.outgrown : out.rows[cls])[at] = static_cast<int>(i);
        }
    }
    if ((b + 1) * kSizeThreads >= n && tid == 0) {   // the workgroup of the last row
        const int64_t t = static_cast<int64_t>(px + all_x), z = static_cast<int64_t>(py + all_y);
        tile_ptr[n] = t;
        nnz_off[n] = z;
        if (t < tile_nnz_len)
            tile_nnz[t] = z;
        __hip_atomic_store(&ctr[kCtrTiles], px + all_x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ctr[kCtrNnz], py + all_y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (w == 0) {
        int last = 0;
        if (tid == 0) {
            __threadfence();
            last = atomicAdd(&ctr[kCtrDone], 1ull) + 1 == gridDim.x ? 1 : 0;
        }
        if (__shfl(last, 0, kWave) && tid < kCtrTicket) {
            __threadfence();
            host[tid] = __hip_atomic_load(&ctr[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

__global__ void sizes_init_kernel(SizesInit z)
{
    sizes_init(z);
}

__global__ void fill_i32_kernel(int *p, int64_t n, int v)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

__global__ void fill_u64_kernel(unsigned long long *p, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0ull;
}

__global__ void set_last_kernel(int64_t *p, const int64_t *v) { *p = *v; }

double event_ms(hipEvent_t a, hipEvent_t b)
{
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, a, b) != hipSuccess) {
        (void)hipGetLastError();
        return 0.0;
    }
    return ms;
}

} // namespace

// Timeline trace of the main numeric launch, switched on by the reference's
// environment variables: DMMA_TRACE_FILE (output path), DMMA_TRACE_SHIFT
// (sample every 2^shift-th workgroup, default 4, at most 10) and
// DMMA_TRACE_PHASE (which one, default min(7, 2^shift - 1)).
static unsigned int trace_env(const char *name, unsigned int fallback, unsigned int maximum)
{
    const char *text = std::getenv(name);
    if (!text || !*text)
        return fallback;
    char *end = nullptr;
    const unsigned long v = std::strtoul(text, &end, 10);
    return (end == text || *end || v > maximum) ? fallback : static_cast<unsigned int>(v);
}

// The reference's DMTL0001 layout (dmma_write_timeline_trace,
// src/dmma_spgemm.h:95-164): magic, version, compute units, waves per
// workgroup, shift, phase, output tiles, workgroups, slots, then the slot
// start times, end times (ns) and compute unit ids.
static int write_timeline(const char *path, const Timeline &tl, size_t slots, uint64_t blocks,
                          uint64_t output_tiles, int num_cus)
{
    std::vector<unsigned long long> start(slots), end(slots);
    std::vector<uint32_t> cu(slots);
    RTT_HIP(hipMemcpy(start.data(), tl.start, slots * sizeof(start[0]), hipMemcpyDeviceToHost));
    RTT_HIP(hipMemcpy(end.data(), tl.end, slots * sizeof(end[0]), hipMemcpyDeviceToHost));
    RTT_HIP(hipMemcpy(cu.data(), tl.cu, slots * sizeof(cu[0]), hipMemcpyDeviceToHost));
    int rate_khz = 0;
    RTT_HIP(hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, ctx().device));
    const double ns_per_tick = rate_khz > 0 ? 1e6 / rate_khz : 1.0;
    for (size_t i = 0; i < slots; ++i) {
        start[i] = static_cast<unsigned long long>(static_cast<double>(start[i]) * ns_per_tick);
        end[i] = static_cast<unsigned long long>(static_cast<double>(end[i]) * ns_per_tick);
    }
    FILE *f = std::fopen(path, "wb");
    if (!f)
        return fail(RTT_ERR_INVALID, "cannot open timeline output %s", path);
    const char magic[8] = {'D', 'M', 'T', 'L', '0', '0', '0', '1'};
    const uint32_t head[5] = {1u, static_cast<uint32_t>(num_cus),
                              static_cast<uint32_t>(kWavesPerBlock), tl.shift, tl.phase};
    const uint64_t tail[3] = {output_tiles, blocks, static_cast<uint64_t>(slots)};
    bool ok = std::fwrite(magic, sizeof(magic), 1, f) == 1 &&
              std::fwrite(head, sizeof(head), 1, f) == 1 &&
              std::fwrite(tail, sizeof(tail), 1, f) == 1;
    if (slots)
        ok = ok && std::fwrite(start.data(), sizeof(start[0]), slots, f) == slots &&
             std::fwrite(end.data(), sizeof(end[0]), slots, f) == slots &&
             std::fwrite(cu.data(), sizeof(cu[0]), slots, f) == slots;
    ok = (std::fclose(f) == 0) && ok;
    if (!ok)
        return fail(RTT_ERR_INVALID, "write of timeline %s failed", path);
    return RTT_OK;
}

__global__ void slab_parts_kernel(int n, const unsigned int *__restrict__ cost, unsigned int target,
                                  int *__restrict__ parts)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        parts[i] = 1 + static_cast<int>(min(cost[i] / target, static_cast<unsigned int>(kSlabParts - 1)));
    else if (i == n)
        parts[i] = 0;
}

// The tasks of a slab row list: its rows heaviest first (most pairs) with
// `sorted`, so that the work queue hands out the long rows before the short
// ones, and the tasks of every row.  Stream-ordered: the previous user of
// the arrays has been queued.
static int plan_slab_tasks(const int *rows, int n, bool sorted, unsigned long long pairs,
                           const Operands &g, SpgemmWork *w, hipStream_t s, SlabTasks *out)
{
    const size_t bytes_n = (static_cast<size_t>(n) + 1) * sizeof(unsigned int);
    RTT_TRY(w->row_cost.ensure(bytes_n));
    RTT_TRY(w->row_cost2.ensure(bytes_n));
    RTT_TRY(w->rows_sorted.ensure(bytes_n));
    RTT_TRY(w->slab_base.ensure(bytes_n));
    unsigned int *cost = w->row_cost.as<unsigned int>();
    unsigned int *cost2 = w->row_cost2.as<unsigned int>();
    hipLaunchKernelGGL(row_pairs_kernel, dim3(blocks_for(n, kWavesPerBlock)), dim3(kThreads), 0,
                       s, rows, n, g.a_trp, g.a_brange, cost);
    RTT_HIP(hipGetLastError());
    size_t bytes = 0;
    if (sorted) {
        int *to = w->rows_sorted.as<int>();
        RTT_HIP(hipcub::DeviceRadixSort::SortPairsDescending(nullptr, bytes, cost, cost2, rows, to,
                                                             n, 0, 32, s));
        RTT_TRY(w->scan_tmp.ensure(bytes));
        RTT_HIP(hipcub::DeviceRadixSort::SortPairsDescending(w->scan_tmp.ptr, bytes, cost, cost2,
                                                             rows, to, n, 0, 32, s));
        rows = to;
        std::swap(cost, cost2);
    }
    const int64_t target = slab_target(pairs);
    int *parts = reinterpret_cast<int *>(cost2), *base = w->slab_base.as<int>();
    hipLaunchKernelGGL(slab_parts_kernel, dim3(blocks_for(n + 1, kThreads)), dim3(kThreads), 0, s,
                       n, cost, static_cast<unsigned int>(std::min<int64_t>(target, UINT_MAX)),
                       parts);
    RTT_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, parts, base, n + 1, s));
    RTT_TRY(w->scan_tmp.ensure(bytes));
    RTT_HIP(hipcub::DeviceScan::ExclusiveSum(w->scan_tmp.ptr, bytes, parts, base, n + 1, s));
    out->rows = rows;
    out->base = base;
    out->nrows = n;
    out->most = n + static_cast<int64_t>(pairs / static_cast<unsigned long long>(target));
    return RTT_OK;
}

int spgemm_core(const DevTiles &a, DevTiles &b, BuildWork *b_work, DevC *c, SpgemmWork *w,
                Events *ev, CoreTimes *times, int lb_mode, const TileOpts *tile)
{
    // tile: rows routed to the tile-pair kernel (all when fill is 0);
    // vector: rows left to the LDS-accumulator kernels.
    const bool any_tile = tile != nullptr;
    const bool any_vector = !tile || tile->fill > 0.f;
    RTT_TRY(require_ctx());
    RTT_TRY(ev->create());
    hipStream_t s = ctx().stream;
    const int R = a.tile_row_count;
    const int BC = b.tile_col_count;
    w->tail_ran = false;   // until the tail queue admits for this call
    c->tilem = R;
    c->tilen = BC;
    c->rows = a.rows;
    c->cols = b.cols;

    Operands g;
    g.a_trp = a.tile_row_ptr.as<int>();
    g.a_meta = a.meta.as<int4>();
    g.a_brange = b.a_brange.as<int4>();
    g.a_blight = b.a_blight.as<int2>();
    g.a_vals_cm = a.values_cm.as<double>();
    g.a_row_off = a.row_payload_off.as<int>();
    g.b_vals_km = b.payload_kmajor();
    g.b_meta = b.records.as<int4>();   // part 0 of every record is the tile's meta
    g.tile_fill = tile ? tile->fill : INFINITY;

    const int num_cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    // The counters and the look-back words of the sizes pass; the host's copy
    // of the counters is written by the pass itself.
    const int64_t size_blocks = std::max<int64_t>(1, blocks_for(R, kSizeThreads));
    const int64_t words = 2 * size_blocks;
    RTT_TRY(w->counters.ensure(static_cast<size_t>(kCounters + words) * sizeof(unsigned long long)));
    RTT_TRY(w->host_counters.ensure((kCounters + 1) * sizeof(unsigned long long)));
    unsigned long long *ctr = w->counters.as<unsigned long long>();
    unsigned long long *look = ctr + kCounters;
    const unsigned long long *hctr = w->host_counters.as<unsigned long long>();

    auto t_sym = Clock::now();
    // ---- symbolic: per-row tile sets, staged ------------------------------
    const int stage_limit = 3 * kSymSlots / 4;
    const size_t row_ints = (static_cast<size_t>(R) + 1) * sizeof(int);
    RTT_TRY(w->row_tiles.ensure((R + 1) * sizeof(int64_t)));
    RTT_TRY(w->row_nnz.ensure((R + 1) * sizeof(int64_t)));
    RTT_TRY(w->row_level.ensure(row_ints));
    RTT_TRY(w->l3_rows.ensure(row_ints));
    RTT_TRY(w->sym_slab_rows.ensure(row_ints));
    RowLists lists;
    for (int c = 0; c < kRowClasses; ++c) {
        RTT_TRY(w->class_rows[c].ensure(row_ints));
        lists.rows[c] = w->class_rows[c].as<int>();
    }
    lists.outgrown = w->l3_rows.as<int>();
    RTT_TRY(w->stage_j.ensure(static_cast<size_t>(R) * stage_limit * sizeof(int)));
    RTT_TRY(w->stage_m.ensure(static_cast<size_t>(R) * stage_limit * sizeof(uint64_t)));
    RTT_TRY(c->tile_ptr.ensure((R + 1) * sizeof(int64_t)));
    RTT_TRY(w->c_row_nnz_off.ensure((R + 1) * sizeof(int64_t)));
    Stage st{w->stage_j.as<int>(), w->stage_m.as<unsigned long long>(), stage_limit};
    // Queue heads: [0] symbolic slab count, [1] symbolic slab fill, [2] numeric slab.
    RTT_TRY(w->queue.ensure(3 * sizeof(int)));
    int *queue = w->queue.as<int>();
    // The pair total was summed by the B update's pair-extent pass.
    const SizesInit start{ctr, 0, look, words, b.pair_total.as<unsigned long long>(), queue, 3};
    const SizesInit again{ctr, static_cast<int>(kCtrRows), look, words, nullptr, nullptr, 0};
    // The tail queue needs B's tile columns only if some C tile can clear its
    // threshold: told from B's tile rows where that is enough, else from its
    // longest tile column (for B = A^T at tile level A's longest tile row),
    // read with the sizes.
    bool tail = any_tile && tile->tail && tail_possible(tile->longest_a, b.tile_row_count, tile->threshold);
    const bool count_columns = tail && !b.transpose_of;
    if (tail && b.transpose_of)
        tail = tail_possible(tile->longest_a, tile->longest_a, tile->threshold);
    if (count_columns)
        RTT_TRY(longest_b_column(b, &b_work->keys_in,
                                 w->host_counters.as<unsigned long long>() + kCounters));
    // One wave per row first; rows that outgrow its table go to the
    // workgroup table, and rows that outgrow that to the slab.
    RTT_HIP(hipEventRecord(ev->ev[0], s));
    if (R > 0)
        hipLaunchKernelGGL(symbolic_wave_kernel, dim3(R), dim3(kWave), 0, s, g, st,
                           w->row_tiles.as<int64_t>(), w->row_nnz.as<int64_t>(),
                           w->row_level.as<int>(), start);
    else
        hipLaunchKernelGGL(sizes_init_kernel, dim3(1), dim3(kThreads), 0, s, start);
    RTT_HIP(hipGetLastError());
    RTT_HIP(hipEventRecord(ev->ev[1], s));
    int n_slab = 0;
    // Sizes of C from the per-row counts, the numeric routing lists and
    // every counter, in one launch and one wait.  Rows of the tile-pair
    // kernel are not listed.
    auto finish_sizes = [&](bool slab_done) -> int {
        hipLaunchKernelGGL(row_sizes_kernel, dim3(static_cast<unsigned>(size_blocks)),
                           dim3(kSizeThreads), 0, s, R, w->row_level.as<int>(), slab_done,
                           w->row_tiles.as<int64_t>(), w->row_nnz.as<int64_t>(), g.a_trp,
                           g.a_row_off, g.tile_fill, any_vector, c->tile_ptr.as<int64_t>(),
                           w->c_row_nnz_off.as<int64_t>(), c->tile_nnz.as<int64_t>(),
                           static_cast<int64_t>(c->tile_nnz.bytes / sizeof(int64_t)), lists, ctr,
                           look, w->host_counters.as<unsigned long long>());
        RTT_HIP(hipGetLastError());
        RTT_HIP(hipStreamSynchronize(s));
        return RTT_OK;
    };
    // Sized at once, as if every row fit the wave table: one wait when none
    // outgrew it (the usual case), redone when some did.
    RTT_TRY(finish_sizes(false));
    const int n_large = static_cast<int>(hctr[kCtrOutgrown]);
    if (n_large > 0) {
        hipLaunchKernelGGL(symbolic_count_kernel, dim3(n_large), dim3(kThreads), 0, s, g,
                           stage_limit, st, w->l3_rows.as<int>(), w->row_tiles.as<int64_t>(),
                           w->row_nnz.as<int64_t>(), w->row_level.as<int>(),
                           w->sym_slab_rows.as<int>(), ctr, again);
        RTT_HIP(hipGetLastError());
        RTT_HIP(hipEventRecord(ev->ev[1], s));
        RTT_TRY(finish_sizes(false));
        n_slab = static_cast<int>(hctr[kCtrSymSlab]);
    }
    const int static_rows = lb_mode == RTT_LB_STATIC ? 1 : 0;
    const bool by_cost = lb_mode == RTT_LB_ADAPTIVE_TAIL;
    SlabTasks tasks;
    // Entry by entry, the symbolic passes need the rows' operands, and those of
    // the rows whose C outgrows the numeric kernels' come with them.
    const SlabSizes sym_rows{static_cast<int64_t>(hctr[kCtrLongest]),
                             static_cast<int64_t>(hctr[kCtrMostTiles]),
                             static_cast<int64_t>(hctr[kCtrSymSizes] & 0xFFFFFFFFull),
                             static_cast<int64_t>(hctr[kCtrSymSizes] >> 32)};
    const bool entries_first = n_slab > 0 && !slab_by_tiles(b, sym_rows);
    if (entries_first)
        RTT_TRY(slab_prepare(a, b, b_work, w, w->sym_slab_rows.as<int>(), n_slab,
                             lists.rows[kRowSlab], static_cast<int>(hctr[kCtrRows + kRowSlab]),
                             static_cast<int64_t>(hctr[kCtrLongest])));
    if (n_slab > 0) {
        RTT_TRY(plan_slab_tasks(w->sym_slab_rows.as<int>(), n_slab, by_cost, hctr[kCtrPairs], g, w,
                                s, &tasks));
        RTT_TRY(slab_symbolic(a, b, w, tasks, queue, static_rows, ctr + kCtrSlabTiles, sym_rows));
        hipLaunchKernelGGL(sizes_init_kernel, dim3(blocks_for(words, kThreads)), dim3(kThreads), 0,
                               s, again);
        RTT_TRY(finish_sizes(true));
    }
    w->slab_stage_need = std::max<uint64_t>(w->slab_stage_need, hctr[kCtrSlabTiles]);
    const unsigned long long pairs = hctr[kCtrPairs];
    int n_rows[kRowClasses];
    for (int k = 0; k < kRowClasses; ++k)
        n_rows[k] = static_cast<int>(hctr[kCtrRows + k]);
    const int n_num_slab = n_rows[kRowSlab];
    if (n_num_slab > 0 && !entries_first)
        RTT_TRY(slab_prepare(a, b, b_work, w, lists.rows[kRowSlab], n_num_slab, nullptr, 0,
                             static_cast<int64_t>(hctr[kCtrLongest])));
    const int64_t total_tiles = static_cast<int64_t>(hctr[kCtrTiles]);
    const int64_t total_nnz = static_cast<int64_t>(hctr[kCtrNnz]);
    const double sym_count_ms = ms_since(t_sym);

    // ---- allocate C -----------------------------------------------------
    auto t_alloc = Clock::now();
    c->num_tiles = total_tiles;
    c->nnz = total_nnz;
    RTT_TRY(c->tile_col.ensure(c->num_tiles * sizeof(int)));
    RTT_TRY(c->tile_mask.ensure(c->num_tiles * sizeof(uint64_t)));
    // The sizes pass wrote the last offset where the array was long enough.
    const bool ended = (c->num_tiles + 1) * sizeof(int64_t) <= c->tile_nnz.bytes;
    RTT_TRY(c->tile_nnz.ensure((c->num_tiles + 1) * sizeof(int64_t)));
    RTT_TRY(c->tile_csr_ptr.ensure(c->num_tiles * 8));
    RTT_TRY(c->tile_csr_col.ensure(c->nnz));
    RTT_TRY(c->tile_csr_val.ensure(c->nnz * sizeof(double)));
    times->allocation_ms = ms_since(t_alloc);

    // ---- symbolic: final structure -------------------------------------------
    auto t_fill = Clock::now();
    COut co;
    co.tile_ptr = c->tile_ptr.as<int64_t>();
    co.row_nnz_off = w->c_row_nnz_off.as<int64_t>();
    co.col = c->tile_col.as<int>();
    co.mask = c->tile_mask.as<uint64_t>();
    co.tile_nnz = c->tile_nnz.as<int64_t>();
    co.csr_ptr = c->tile_csr_ptr.as<uint8_t>();
    co.csr_col = c->tile_csr_col.as<uint8_t>();
    co.val = c->tile_csr_val.as<double>();
    RTT_HIP(hipEventRecord(ev->ev[2], s));
    // The numeric LDS kernels write the structure of their own rows from the
    // staged lists; this pass writes it for the staged rows they cannot hold
    // (the numeric fallback list, whose slab rows it skips), and for the rows of
    // the tile-pair kernels, which need their structure first.
    if (any_tile && R > 0 && c->num_tiles > 0)
        hipLaunchKernelGGL(symbolic_write_kernel, dim3(blocks_for(R, kWavesPerBlock)),
                           dim3(kThreads), 0, s, nullptr, R, st, w->row_level.as<int>(), co,
                           g.tile_fill, g.a_trp, g.a_row_off);
    if (n_num_slab > 0 && c->num_tiles > 0)
        hipLaunchKernelGGL(symbolic_write_kernel, dim3(blocks_for(n_num_slab, kWavesPerBlock)),
                           dim3(kThreads), 0, s, lists.rows[kRowSlab], n_num_slab, st,
                           w->row_level.as<int>(), co, 0.f, nullptr, nullptr);
    RTT_HIP(hipGetLastError());
    RTT_HIP(hipEventRecord(ev->ev[3], s));
    if (n_slab > 0)
        RTT_TRY(slab_structure(a, b, w, tasks, queue + 1, static_rows, co));
    if (!ended)
        hipLaunchKernelGGL(set_last_kernel, dim3(1), dim3(1), 0, s,
                           c->tile_nnz.as<int64_t>() + c->num_tiles,
                           w->c_row_nnz_off.as<int64_t>() + R);
    RTT_HIP(hipGetLastError());
    RTT_HIP(hipEventRecord(ev->ev[6], s));
    // ---- numeric ----------------------------------------------------------
    if (count_columns)
        tail = tail_possible(tile->longest_a, static_cast<int64_t>(hctr[kCounters]),
                             tile->threshold);
    TileColumns columns;
    if (tail) {
        auto tc = Clock::now();
        RTT_TRY(build_b_columns(&b, b_work));
        RTT_HIP(hipStreamSynchronize(s));
        times->b_columns_ms = ms_since(tc);
        columns = b_columns(b);
    }
    Timeline tl;
    size_t trace_slots = 0;
    const char *trace_path = std::getenv("DMMA_TRACE_FILE");
    if (trace_path && *trace_path && R > 0 && c->nnz > 0) {
        tl.shift = trace_env("DMMA_TRACE_SHIFT", 4, 10);
        const unsigned int stride = 1u << tl.shift;
        tl.phase = trace_env("DMMA_TRACE_PHASE", std::min(7u, stride - 1u), stride - 1u);
        const size_t sampled = static_cast<unsigned int>(R) <= tl.phase
                                   ? 0
                                   : (static_cast<size_t>(R) - 1 - tl.phase) / stride + 1;
        trace_slots = sampled * kWavesPerBlock;
        if (trace_slots) {
            RTT_TRY(w->trace_start.ensure(trace_slots * sizeof(unsigned long long)));
            RTT_TRY(w->trace_end.ensure(trace_slots * sizeof(unsigned long long)));
            RTT_TRY(w->trace_cu.ensure(trace_slots * sizeof(unsigned int)));
            tl.start = w->trace_start.as<unsigned long long>();
            tl.end = w->trace_end.as<unsigned long long>();
            tl.cu = w->trace_cu.as<unsigned int>();
            hipLaunchKernelGGL(fill_u64_kernel, dim3(blocks_for(trace_slots, kThreads)),
                               dim3(kThreads), 0, s, tl.start, static_cast<int64_t>(trace_slots));
            hipLaunchKernelGGL(fill_u64_kernel, dim3(blocks_for(trace_slots, kThreads)),
                               dim3(kThreads), 0, s, tl.end, static_cast<int64_t>(trace_slots));
            hipLaunchKernelGGL(fill_i32_kernel, dim3(blocks_for(trace_slots, kThreads)),
                               dim3(kThreads), 0, s, reinterpret_cast<int *>(tl.cu),
                               static_cast<int64_t>(trace_slots), 0);
        }
    }
    RTT_HIP(hipEventRecord(ev->ev[4], s));
    if (any_tile) {
        const unsigned long long wide = hctr[kCtrWide];
        RTT_TRY(plan_wide_rows(a, *c, tile->fill, static_cast<int64_t>(wide >> kWideRowShift),
                               static_cast<int64_t>(wide & ((1ull << kWideRowShift) - 1ull)), w, s));
        RTT_TRY(tile_numeric(a, b, *c, *tile, tail ? &columns : nullptr, w, s));
    }
    auto rows_launch = [&](auto kernel, int cls, int threads, bool every) {
        if (n_rows[cls] > 0)
            hipLaunchKernelGGL(kernel, dim3(n_rows[cls]), dim3(threads), 0, s, g,
                               b.records.as<int4>(), b.num_tiles,
                               every ? nullptr : lists.rows[cls], w->row_level.as<int>(), st, co,
                               Timeline{});
    };
    // SmallRow takes the rows of its list, or every row when all of them are
    // its own (a list entry is one more dependent load per row).  Launched
    // over every row whatever its class, as the traced form still is, the
    // workgroups that leave at once took 0.3 of the AMG batch's 3.0 ms.
    auto small_launch = [&](auto cfg) {
        using Cfg = decltype(cfg);
        if (trace_slots && any_vector)
            hipLaunchKernelGGL((numeric_row_kernel<Cfg, true>), dim3(R), dim3(kThreads), 0, s, g,
                               b.records.as<int4>(), b.num_tiles, nullptr, w->row_level.as<int>(),
                               st, co, tl);
        else
            rows_launch(numeric_row_kernel<Cfg>, kRowSmall, Cfg::kThreads, n_rows[kRowSmall] == R);
    };
    if (c->nnz <= kSpreadFill * c->num_tiles)
        small_launch(SpreadRow{});
    else
        small_launch(SmallRow{});
    RTT_HIP(hipGetLastError());
    rows_launch(numeric_row_kernel<TinyRow>, kRowTiny, TinyRow::kThreads, false);
    rows_launch(numeric_row_kernel<MediumRow>, kRowMid, MediumRow::kThreads, false);
    rows_launch(numeric_row_kernel<LargeRow>, kRowLarge, LargeRow::kThreads, false);
    if (n_num_slab > 0) {
        // The structure pass above is queued before this plan reuses its arrays.
        RTT_TRY(plan_slab_tasks(lists.rows[kRowSlab], n_num_slab, by_cost, pairs, g, w, s, &tasks));
        RTT_TRY(slab_numeric(a, w, tasks, queue + 2, static_rows, co,
                             static_cast<int64_t>(hctr[kCtrLongest])));
    }
    RTT_HIP(hipEventRecord(ev->ev[5], s));   // behind the numeric kernels of every class
    RTT_HIP(hipStreamSynchronize(s));
    if (any_tile && c->num_tiles > 0) {
        // Written by the last of the tile-pair path's kernels.
        const unsigned long long *st = w->host_tile_stats.as<unsigned long long>();
        times->mfma_pairs = st[0];
        times->tail_reason = static_cast<int>(st[1]);
        times->tail_records = st[2];
        times->tail_chunks = st[3];
    }
    if (trace_slots)
        RTT_TRY(write_timeline(trace_path, tl, trace_slots, static_cast<uint64_t>(R),
                               static_cast<uint64_t>(c->num_tiles), num_cus));
    // Structure write and numeric share the stream without a host wait
    // between them; their split comes from the device events.
    const double fill_ms = event_ms(ev->ev[2], ev->ev[6]);
    const double tail_ms = ms_since(t_fill);
    times->symbolic_ms = sym_count_ms + fill_ms;
    times->numeric_ms = std::max(0.0, tail_ms - fill_ms);
    times->sym_count_kernel_ms = event_ms(ev->ev[0], ev->ev[1]);
    times->sym_fill_kernel_ms = event_ms(ev->ev[2], ev->ev[3]);
    times->numeric_kernel_ms = event_ms(ev->ev[4], ev->ev[5]);
    times->pairs = pairs;
    times->heavy_rows = static_cast<unsigned long long>(n_num_slab + n_rows[kRowLarge] + n_rows[kRowMid]);
    return RTT_OK;
}

} // namespace rtt
