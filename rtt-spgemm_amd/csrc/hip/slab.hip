// Rows beyond the LDS tables (hub rows of graphs, scattered wide rows): their
// tiles hold one or two entries each, so they are multiplied entry by entry
// (row-wise Gustavson on scalars) instead of tile by tile.
//
// A row of more work than its share is cut into tasks by columns (the hub row
// of R-MAT 2^18 held one workgroup for 88 ms).
//
// Operands: every slot of A's payload gets its column and its row within the
// tile, and B's entries are laid out by scalar row, columns ascending, from its
// tiles.  Where a product has many such rows this is done for all of A (once
// per prepared A) and all of B; where it has few, for the rows themselves and
// the rows of B they select (slab_prepare).  A workgroup owns one tile row of C, or a
// part of it, at a time.  A thread owns one slot of the row's A payload, with a
// cursor into the B row it selects, for chunks of as many slots as the workgroup
// has threads.
//
// The row is walked in windows of C columns.  In a window, every thread
// gallops its cursor to the window's end; the products are numbered by a
// scan, a bit word per 64 products marks where a thread's products begin, and
// product p of the window finds its thread with one word and one count.
// Consecutive lanes so take consecutive entries of a B row.
//  * symbolic: the window's C tile masks are ORed in LDS, then counted and
//    appended to the staged lists, or written to C's structure.  Operands whose
//    tiles are well filled go tile by tile here (slab_by_tiles).
//  * numeric: the window's C tiles (masks and first values) lie in LDS, found
//    by a bit per tile column and a count of those before each word, and their
//    values accumulate in LDS in C's order, to be stored once, whatever the
//    number of A entries.
//
// On R-MAT 2^18 (2.9e9 products, a pair of tiles carries 1.3) the count takes
// 7.7 ms and the numeric pass 16.9 ms, waiting for short pieces of B rows, of
// which the L2s reuse little: the wider the window, the longer the pieces.
// With tables directly mapped by column, 2048 tile columns and 4096 values a
// window, and two workgroups of 512 threads on a CU it took 23.8 ms (twice the
// L2 reads); mapped tables of 4096 columns for one workgroup of 1024 took 19.6.
// Searching a cursor's next stop by eight probes at a time was slower (18.8).
// Tile by tile, with a binary search over 1280 runs and a 16-byte table entry
// from HBM per pair, the two passes took 35 and 108 ms, waiting on dependent
// loads.
#include <algorithm>
#include <climits>

#include "core.hpp"

namespace rtt {

namespace {

constexpr int kSymThreads = 512;               // symbolic pass: two workgroups fit a CU
constexpr int kNumThreads = 1024;              // numeric pass: one, with all of its LDS
constexpr int kSubProducts = 16384;            // products numbered by the bit words at once
constexpr int kSubWords = kSubProducts / 64;
constexpr int kSymWin = 8192;                  // C tile columns of a symbolic window,
constexpr int kTileWin = 4096;                 // of one by tiles
constexpr double kTileProducts = 2.0;          // products a pair of tiles from which it does
constexpr int kFillBytes = 8192;               // column bytes of C staged at a time
constexpr int kNumSpan = 32768;                // C tile columns a numeric window may span,
constexpr int kNumTiles = 3072;                // C tiles it may hold,
constexpr int kNumVals = 13312;                // and C values
constexpr int kNumWords = kNumSpan / 64;
constexpr int kLookTiles = kNumTiles / kNumThreads;   // C tiles a thread looks at per window
constexpr int kRuns = 5;                       // classes of a row of B: heavy, light k = 0..3
constexpr int kUnroll = 4;                     // products a thread loads together
static_assert(kSubWords <= 4 * kWave, "one wave ranks the bit words");
static_assert(kNumVals <= 65536 - 64 && kNumTiles <= 65536, "16-bit value and tile positions");
static_assert(kNumTiles % kNumThreads == 0 && kNumWords % kWave == 0 &&
                  kNumWords / kWave * kWave <= kNumThreads,
              "shares of a window's tables");

// Column (-1: an absent slot of a dense tile) and row of every slot of the A
// tile with meta m, from slot `at` of the codes on.
__device__ __forceinline__ void write_slot_codes(const int4 &m, int64_t at, int *__restrict__ k,
                                                 uint8_t *__restrict__ r)
{
    const uint32_t mask = static_cast<uint32_t>(m.y);
    const bool dense = m.w < 0;
    for (int phys = 0, j = 0; phys < 32; ++phys) {
        const bool has = (mask >> phys) & 1u;
        if (!has && !dense)
            continue;
        k[at + j] = has ? 4 * m.x + (phys & 3) : -1;
        r[at + j] = static_cast<uint8_t>(phys >> 2);
        ++j;
    }
}

// For every slot of A's payload; a thread per tile.
__global__ void slot_codes_kernel(int64_t n, const int4 *__restrict__ meta, int *__restrict__ k,
                                  uint8_t *__restrict__ r)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < n)
        write_slot_codes(meta[t], meta[t].w & 0x7FFFFFFF, k, r);
}

// ---- the rows of a few slab rows ------------------------------------------------
// The B tile rows that the listed rows select, and those rows' entries.
struct Picked {
    unsigned long long rows, entries;
};

// Listed rows of two lists; workgroups x, y take every gridDim.y-th 256 A tiles
// of row x: the slot codes and values of its A payload, `stride` slots from the
// row before it, and a flag for every B tile row it selects.
__global__ __launch_bounds__(256) void pick_rows_kernel(
    const int *__restrict__ rows, int n, const int *__restrict__ more, int64_t stride,
    const int *__restrict__ a_trp, const int4 *__restrict__ a_meta,
    const int *__restrict__ a_row_off, const double *__restrict__ a_vals, int *__restrict__ flag,
    int *__restrict__ code_off, int *__restrict__ k, uint8_t *__restrict__ r,
    double *__restrict__ v)
{
    const int i = blockIdx.x;
    const int row = i < n ? rows[i] : more[i - n];
    if (code_off && blockIdx.y == 0 && threadIdx.x == 0)
        code_off[row] = static_cast<int>(i * stride);
    const int64_t shift = i * stride - a_row_off[row];
    const int t1 = a_trp[row + 1];
    for (int t = a_trp[row] + static_cast<int>(blockIdx.y * 256 + threadIdx.x); t < t1;
         t += static_cast<int>(gridDim.y) * 256) {
        const int4 m = a_meta[t];
        flag[m.x] = 1;
        if (k) {
            const int off = m.w & 0x7FFFFFFF;
            write_slot_codes(m, shift + off, k, r);
            const int slots = m.w < 0 ? 32 : __popc(static_cast<uint32_t>(m.y));
            for (int j = 0; j < slots; ++j)
                v[shift + off + j] = a_vals[off + j];
        }
    }
}

// B's tile rows (the listed ones, or without a list all R) and where their
// entries go.
struct BRows {
    int R;
    const int *__restrict__ list;              // null: all rows
    const unsigned long long *__restrict__ n;  // rows listed
    const int *__restrict__ trp;
    const int *__restrict__ groups;            // start of each (row, class) run
    const int4 *__restrict__ meta;             // rows in class order
    const int *__restrict__ order;             // per row, its tiles by column; null: the arrays are
    const int *__restrict__ tcol;
    const uint32_t *__restrict__ masks;
    const int *__restrict__ offs;
    const double *__restrict__ vals;
    int *__restrict__ start;                   // see scalar_rows_kernel
    int *__restrict__ col;
    double *__restrict__ val;
};

// The tile row of threads [i T, i T + T), -1 past the last.
template <int T>
__device__ __forceinline__ int b_row(const BRows &g)
{
    const int i = static_cast<int>(blockIdx.x) * (256 / T) + static_cast<int>(threadIdx.x) / T;
    if (!g.list)
        return i < g.R ? i : -1;
    return i < static_cast<int>(*g.n) ? g.list[i] : -1;
}

// Exclusive sum of n over the workgroup's 256 threads and the workgroups that
// have added to *total (one atomic a workgroup: on one address they take 7 ns
// each, one a row took 0.45 ms of 65000 rows).
__device__ __forceinline__ int64_t grid_place(int n, unsigned long long *total)
{
    __shared__ int s_tmp[256 / kWave];
    __shared__ unsigned long long s_base;
    int all = 0;
    const int before = block_exclusive_scan<256 / kWave>(n, s_tmp, &all);
    if (threadIdx.x == 0)
        s_base = all ? atomicAdd(total, static_cast<unsigned long long>(all)) : 0ull;
    __syncthreads();
    return static_cast<int64_t>(s_base) + before;
}

// The flagged rows' list; a thread per row of B.
__global__ __launch_bounds__(256) void list_rows_kernel(int R, const int *__restrict__ flag,
                                                        Picked *picked, int *__restrict__ list)
{
    const int K = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    const int has = K < R && flag[K] ? 1 : 0;
    const int64_t at = grid_place(has, &picked->rows);
    if (has)
        list[at] = K;
}

// Entries of every row, for place_rows_kernel.
template <int T>
__global__ __launch_bounds__(256) void count_rows_kernel(BRows g)
{
    const int K = b_row<T>(g);
    if (K < 0)
        return;   // a whole wave or workgroup
    __shared__ int s_sum[256 / kWave];
    int n = 0;
    for (int t = g.trp[K] + static_cast<int>(threadIdx.x) % T; t < g.trp[K + 1]; t += T)
        n += __popc(static_cast<uint32_t>(g.meta[t].y));
    n = wave_sum(n);
    if constexpr (T > kWave) {
        if (lane_id() == 0)
            s_sum[threadIdx.x / kWave] = n;
        __syncthreads();
        n = 0;
        for (int w = 0; w < T / kWave; ++w)
            n += s_sum[w];
    }
    if (threadIdx.x % T == 0)
        g.start[5 * static_cast<int64_t>(K) + 4] = n;
}

// The place of every row's entries; a thread per row.  Rows built from a CSR
// get the slots of their payload.
__global__ __launch_bounds__(256) void place_rows_kernel(BRows g, Picked *picked)
{
    const int K = b_row<1>(g);
    int n = 0;
    if (K >= 0)
        n = g.order ? g.start[5 * static_cast<int64_t>(K) + 4]
                    : g.offs[g.trp[K + 1]] - g.offs[g.trp[K]];
    const int64_t at = grid_place(n, &picked->entries);
    if (K >= 0)
        g.start[5 * static_cast<int64_t>(K)] = static_cast<int>(at);
}

// A row's tiles by column, from its class runs, each of which has ascending
// columns: a tile's place is its own run's before it and, of the other runs,
// those with smaller columns.
template <int T>
__global__ __launch_bounds__(256) void order_tiles_kernel(BRows g, int *__restrict__ order)
{
    const int K = b_row<T>(g);
    if (K < 0)
        return;
    const int *gp = g.groups + static_cast<int64_t>(kClassSlots) * K;
    int at[kRuns + 1];
#pragma unroll
    for (int c = 0; c <= kRuns; ++c)
        at[c] = gp[c];
    for (int t = at[0] + static_cast<int>(threadIdx.x) % T; t < at[kRuns]; t += T) {
        const int j = g.meta[t].x;
        int rank = 0;
#pragma unroll
        for (int c = 0; c < kRuns; ++c) {
            if (t >= at[c] && t < at[c + 1]) {
                rank += t - at[c];
                continue;
            }
            int lo = at[c], hi = at[c + 1];
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (g.meta[mid].x < j)
                    lo = mid + 1;
                else
                    hi = mid;
            }
            rank += lo - at[c];
        }
        order[at[0] + rank] = t;
    }
}

// B's entries by scalar row: the entries of tile row K lie together, row 4K
// first, columns ascending; row 4K + k is start[5K + k] .. start[5K + k + 1].
// They begin at start[5K] where the rows were placed (PLACED), else at the
// row's place in the payload.  T threads per tile row (a wave, or a workgroup).
template <int T, bool PLACED>
__global__ __launch_bounds__(256) void scalar_rows_kernel(BRows g)
{
    __shared__ unsigned long long s_sum[256 / kWave];
    const int lt = threadIdx.x % T;
    const int K = b_row<T>(g);
    if (K < 0)
        return;   // a whole wave or workgroup
    const int t0 = g.trp[K], t1 = g.trp[K + 1];
    // Entries per k in 16-bit fields (at most 8 per tile and k).
    auto count = [&](uint32_t m) {
        unsigned long long c = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            c |= static_cast<unsigned long long>(__popc(m & (0x11111111u << k))) << (16 * k);
        return c;
    };
    auto mask_of = [&](int t) {
        return g.order ? static_cast<uint32_t>(g.meta[g.order[t]].y) : g.masks[t];
    };
    // Sum over the row's threads of c, and before[]: the threads below.
    auto scan = [&](unsigned long long c, unsigned long long *before) {
        const unsigned long long incl = wave_inclusive_scan(c);
        unsigned long long all = __shfl(incl, kWave - 1, kWave);
        *before = incl - c;
        if constexpr (T > kWave) {
            const int w = threadIdx.x / kWave;
            if (lane_id() == 0)
                s_sum[w] = all;
            __syncthreads();
            all = 0;
            for (int i = 0; i < T / kWave; ++i) {
                *before += i < w ? s_sum[i] : 0ull;
                all += s_sum[i];
            }
            __syncthreads();
        }
        return all;
    };
    int total[4] = {0, 0, 0, 0};
    for (int t = t0; t < t1; t += T) {
        unsigned long long before;
        const unsigned long long all = scan(t + lt < t1 ? count(mask_of(t + lt)) : 0ull, &before);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            total[k] += static_cast<int>(all >> (16 * k) & 0xFFFFull);
    }
    int at[4];
    int run = PLACED ? g.start[5 * static_cast<int64_t>(K)] : g.offs[t0];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        at[k] = run;
        run += total[k];
    }
    if (lt > 0 && lt < 5)
        g.start[5 * static_cast<int64_t>(K) + lt] =
            lt == 1 ? at[1] : (lt == 2 ? at[2] : (lt == 3 ? at[3] : run));
    if (!PLACED && lt == 0)
        g.start[5 * static_cast<int64_t>(K)] = at[0];
    for (int t = t0; t < t1; t += T) {
        uint32_t m = 0;
        int off = 0, c0 = 0;
        bool dense = false;
        if (t + lt < t1) {
            if (g.order) {
                const int4 e = g.meta[g.order[t + lt]];
                m = static_cast<uint32_t>(e.y);
                off = e.w & 0x7FFFFFFF;
                dense = e.w < 0;
                c0 = 8 * e.x;
            } else {
                m = g.masks[t + lt];
                off = g.offs[t + lt];
                dense = g.offs[t + lt + 1] - off == 32;
                c0 = 8 * g.tcol[t + lt];
            }
        }
        unsigned long long before;
        const unsigned long long all = scan(count(m), &before);
        int j = 0;
        for (uint32_t x = m; x; x &= x - 1, ++j) {
            const int phys = __builtin_ctz(x), k = phys & 3;
            const int below = __popc(m & (0x11111111u << k) & ((1u << phys) - 1u));
            const int base = k == 0 ? at[0] : (k == 1 ? at[1] : (k == 2 ? at[2] : at[3]));
            const int p = base + static_cast<int>(before >> (16 * k) & 0xFFFFull) + below;
            g.col[p] = c0 + (phys >> 2);
            g.val[p] = g.vals[off + (dense ? phys : j)];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            at[k] += static_cast<int>(all >> (16 * k) & 0xFFFFull);
    }
}

__global__ void zero_ints_kernel(int *__restrict__ p, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0;
}

struct SlabOps {
    const int *__restrict__ a_trp;       // A's and B's tiles, for the pass by tiles
    const int4 *__restrict__ a_meta;
    const int4 *__restrict__ b_meta;
    const int *__restrict__ b_groups;
    const int *__restrict__ a_row_off;   // A payload offset of each tile row
    const int *__restrict__ a_code_off;  // first slot code of each tile row
    const int *__restrict__ a_k;         // per slot code: column, -1 absent
    const uint8_t *__restrict__ a_r;     // per slot code: row within the tile
    const double *__restrict__ a_vals;   // per slot code
    const int *__restrict__ b_start;     // scalar_rows_kernel's layout
    const int *__restrict__ b_col;
    const double *__restrict__ b_val;
    SlabTasks tasks;
    int *__restrict__ queue;
    int static_rows;
    int2 *__restrict__ cursors;          // per workgroup: a run per slot of a long row
    int64_t cursor_stride;
};

// What a thread takes of a tile row, [first, first + count) of them, and the run
// of B it selects, by ascending column: a slot of A's payload with a scalar row
// of B (BY_TILES false), or a tile of A with one class of the tiles of its row of
// B.  at(e) is the column of B's entry (tile) e.
template <bool BY_TILES>
struct Slots;

template <>
struct Slots<false> {
    static constexpr int kToTile = 3;   // at(e) >> kToTile: its tile column
    __device__ static int first(const SlabOps &o, int row) { return o.a_code_off[row]; }
    __device__ static int count(const SlabOps &o, int row)
    {
        return o.a_row_off[row + 1] - o.a_row_off[row];
    }
    __device__ static int at(const SlabOps &o, int64_t e) { return o.b_col[e]; }
    __device__ static void run(const SlabOps &o, int, int x, int *lo, int *hi)
    {
        const int k = o.a_k[x];
        *lo = *hi = 0;
        if (k >= 0) {
            const int *p = o.b_start + 5 * static_cast<int64_t>(k >> 2) + (k & 3);
            *lo = p[0];
            *hi = p[1];
        }
    }
};

template <>
struct Slots<true> {
    static constexpr int kToTile = 0;
    __device__ static int first(const SlabOps &, int) { return 0; }
    __device__ static int count(const SlabOps &o, int row)
    {
        return kRuns * (o.a_trp[row + 1] - o.a_trp[row]);
    }
    __device__ static int at(const SlabOps &o, int64_t e) { return o.b_meta[e].x; }
    __device__ static int4 tile(const SlabOps &o, int row, int x)
    {
        return o.a_meta[o.a_trp[row] + x / kRuns];
    }
    __device__ static void run(const SlabOps &o, int row, int x, int *lo, int *hi)
    {
        const int4 m = tile(o, row, x);
        const int c = x % kRuns;
        const int *p = o.b_groups + static_cast<int64_t>(kClassSlots) * m.x + c;
        *lo = *hi = p[0];
        // A light tile of row k meets the tiles with entries in column k alone.
        if (c == 0 || byte_of(static_cast<uint32_t>(m.z), c - 1))
            *hi = p[1];
    }
};

// A workgroup's task: part `part` of `parts` of a tile row, cut by columns.
struct Task {
    int id, row, part, parts;
    int64_t lo, hi;   // its columns [lo, hi), multiples of 8
};

// The next task: round robin, or from the queue.  The cuts of a row in parts
// are quantiles of the longest B row it selects: hub columns hold most of a
// power-law row's products, and equal stretches of columns would leave most
// of them in the first part.
template <int T, class S>
__device__ __forceinline__ bool next_task(const SlabOps &o, int step, int *s_task,
                                          unsigned long long *s_long, Task *t)
{
    __syncthreads();   // the previous task's readers of s_task
    if (threadIdx.x == 0) {
        const int i = o.static_rows
                          ? static_cast<int>(blockIdx.x) + step * static_cast<int>(gridDim.x)
                          : atomicAdd(o.queue, 1);
        s_task[0] = i;
        if (i < o.tasks.base[o.tasks.nrows]) {
            const int r = upper_index(o.tasks.base, o.tasks.nrows, i);
            s_task[1] = o.tasks.rows[r];
            s_task[2] = i - o.tasks.base[r];
            s_task[3] = o.tasks.base[r + 1] - o.tasks.base[r];
        } else {
            s_task[1] = -1;
        }
        *s_long = 0ull;
    }
    __syncthreads();
    // The same in every lane: scalar registers.
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    t->id = uniform(s_task[0]);
    t->row = uniform(s_task[1]);
    if (t->row < 0)
        return false;
    t->part = uniform(s_task[2]);
    t->parts = uniform(s_task[3]);
    t->lo = 0;
    t->hi = INT64_MAX;
    if (t->parts > 1) {
        // {entries, slot from the end}: the longest, the first of equals.
        unsigned long long best = 0;
        const int s0 = S::first(o, t->row), s1 = s0 + S::count(o, t->row);
        for (int x = s0 + static_cast<int>(threadIdx.x); x < s1; x += T) {
            int lo, hi;
            S::run(o, t->row, x, &lo, &hi);
            if (lo < hi)
                best = max(best, (static_cast<unsigned long long>(hi - lo) << 32) |
                                     static_cast<uint32_t>(s1 - x));
        }
#pragma unroll
        for (int d = kWave / 2; d > 0; d >>= 1)
            best = max(best, __shfl_xor(best, d, kWave));
        if (lane_id() == 0)
            atomicMax(s_long, best);
        __syncthreads();
        if (*s_long != 0) {
            int lo, hi;
            S::run(o, t->row, s1 - static_cast<int>(*s_long & 0xFFFFFFFFull), &lo, &hi);
            const int64_t len = hi - lo;
            auto cut = [&](int q) {
                return static_cast<int64_t>(S::at(o, lo + static_cast<int>(len * q / t->parts)) >>
                                            S::kToTile) * 8;
            };
            if (t->part > 0)
                t->lo = cut(t->part);
            if (t->part + 1 < t->parts)
                t->hi = cut(t->part + 1);
        }
    }
    return true;
}

// First entry of [lo, hi) with at(entry) >= lim.
template <class At>
__device__ __forceinline__ int first_at(At &&at, int lo, int hi, int64_t lim)
{
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (at(mid) < lim)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// Entries [*lo, *hi) of the B row that slot x of A selects, within the task.
template <class S>
__device__ __forceinline__ void slot_run(const SlabOps &o, const Task &t, int x, int *lo, int *hi)
{
    S::run(o, t.row, x, lo, hi);
    auto at = [&](int64_t e) { return S::at(o, e); };
    if (t.part > 0)
        *lo = first_at(at, *lo, *hi, t.lo >> (3 - S::kToTile));
    if (t.part + 1 < t.parts)
        *hi = first_at(at, *lo, *hi, t.hi >> (3 - S::kToTile));
}

// First entry at or after a, below end, with at(entry) >= lim: doubling
// steps, then a binary search in the last one.
template <class At>
__device__ __forceinline__ int gallop(At &&at, int a, int end, int64_t lim)
{
    int lo = a;
    int64_t step = 1;
    while (lo + step <= end && at(lo + step - 1) < lim) {
        lo += static_cast<int>(step);
        step <<= 1;
    }
    return first_at(at, lo, static_cast<int>(min<int64_t>(lo + step - 1, end)), lim);
}

// *at = min(*at, v) over the workgroup's threads (one LDS atomic per wave).
__device__ __forceinline__ void lds_min(int *at, int v)
{
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1)
        v = min(v, __shfl_xor(v, d, kWave));
    if (lane_id() == 0)
        atomicMin(at, v);
}

// A window's runs in LDS: run i (one per thread with products) covers the
// products from s_pre on, entry = pw + product.
template <int T>
struct Runs {
    int pw[T];
    uint8_t r[T];
    unsigned long long bits[kSubWords];   // bit p: a run begins with product p
    int rank[kSubWords];                  // runs that begin before the word
    int scan[2 * (T / kWave)];
};

// The products of the workgroup's threads, cnt each from entry `first` of B
// on.  stage(i) stores the thread's operands as those of run i; load(e)
// fetches what product needs of B's entry e, use(i, x) consumes it.  Every
// thread calls it; it ends with a barrier.
template <class X, int T, class StageF, class LoadF, class UseF>
__device__ __forceinline__ void for_products(Runs<T> &s, int cnt, int first, int r, StageF &&stage,
                                             LoadF &&load, UseF &&use)
{
    const int tid = threadIdx.x;
    int pre, run, total, nrun;
    dual_exclusive_scan<T / kWave>(cnt, cnt > 0 ? 1 : 0, s.scan, &pre, &run, &total, &nrun);
    if (cnt > 0) {
        s.pw[run] = first - pre;
        s.r[run] = static_cast<uint8_t>(r);
        stage(run);
    }
    for (int q0 = 0; q0 < total; q0 += kSubProducts) {
        const int begun = q0 ? __syncthreads_count(cnt > 0 && pre < q0) : 0;
        if (tid < kSubWords)
            s.bits[tid] = 0ull;
        __syncthreads();
        if (cnt > 0 && pre >= q0 && pre < q0 + kSubProducts)
            atomicOr(&s.bits[(pre - q0) >> 6], 1ull << ((pre - q0) & 63));
        __syncthreads();
        if (tid < kWave) {
            constexpr int kPer = kSubWords / kWave;
            int c[kPer], sum = 0;
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                c[i] = __popcll(s.bits[tid * kPer + i]);
                sum += c[i];
            }
            int at = begun + wave_inclusive_scan(sum) - sum;
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                s.rank[tid * kPer + i] = at;
                at += c[i];
            }
        }
        __syncthreads();
        const int n = min(total - q0, kSubProducts);
        for (int p0 = tid; p0 < n; p0 += kUnroll * T) {
            X x[kUnroll];
            int id[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int p = p0 + u * T;
                id[u] = -1;
                if (p < n) {
                    // The run that begins last at or before p.
                    const unsigned long long upto = ~0ull >> (63 - (p & 63));
                    id[u] = s.rank[p >> 6] + __popcll(s.bits[p >> 6] & upto) - 1;
                    x[u] = load(s.pw[id[u]] + q0 + p);
                }
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
                if (id[u] >= 0)
                    use(id[u], x[u]);
        }
        __syncthreads();
    }
    if (total == 0)
        __syncthreads();   // the scan's buffer is reused
}

// Staged tile lists of slab rows: a task's list is a chain of segments, one
// per window, each a header entry (j: its tiles, m: the next segment's
// header, ~0 at the end) and its tiles in column order; a chain per task.
// task[id] holds {first header or -1 when the task did not fit, tiles,
// entries}.  cursor sums what every task needs, fitted or not, so that the
// caller learns the capacity.
struct TaskSize {
    long long head, tiles, nnz;
};
struct SlabStage {
    int *j = nullptr;
    unsigned long long *m = nullptr;
    TaskSize *task = nullptr;
    unsigned long long *cursor = nullptr;
    unsigned long long capacity = 0;
};

template <bool FILL, bool BY_TILES>
__global__ __launch_bounds__(kSymThreads, 4) void symbolic_slab_kernel(SlabOps o,
                                                                     int64_t *__restrict__ row_tiles,
                                                                     int64_t *__restrict__ row_nnz,
                                                                     SlabStage ss, COut c)
{
    using S = Slots<BY_TILES>;
    constexpr int kWin = BY_TILES ? kTileWin : kSymWin;
    __shared__ unsigned long long s_wm[kWin];
    __shared__ uint4 s_tile[2 * (BY_TILES ? kSymThreads : 1)];   // spread_tile of every run's A tile
    __shared__ Runs<kSymThreads> s;
    __shared__ int s_min[2];
    __shared__ long long s_base;
    __shared__ int s_task[4];
    __shared__ unsigned long long s_long;
    __shared__ __align__(4) unsigned char s_bytes[FILL ? kFillBytes + 4 : 4];
    const int tid = threadIdx.x;
    constexpr int kPer = kWin / kSymThreads;
    for (int i = tid; i < kWin; i += kSymThreads)
        s_wm[i] = 0ull;
    for (int step = 0;; ++step) {
        Task task;
        if (!next_task<kSymThreads, S>(o, step, s_task, &s_long, &task))
            break;
        const int row = task.row;
        int64_t tb = 0, zb = 0;
        if constexpr (FILL) {
            tb = c.tile_ptr[row];
            zb = c.row_nnz_off[row];
            for (int q = task.id - task.part; q < task.id; ++q) {
                tb += ss.task[q].tiles;
                zb += ss.task[q].nnz;
            }
            int64_t seg = ss.task[task.id].head;
            if (seg >= 0) {
                while (seg >= 0) {
                    const int n = ss.j[seg];
                    for (int q0 = 0; q0 < n; q0 += kSymThreads) {
                        const int q = q0 + tid;
                        unsigned long long m = 0;
                        int j = 0;
                        if (q < n) {
                            j = ss.j[seg + 1 + q];
                            m = ss.m[seg + 1 + q];
                        }
                        int npc = 0;
                        const int zpos = block_exclusive_scan<kSymThreads / kWave>(__popcll(m), s.scan, &npc);
                        // The tiles' column bytes lie one behind the other:
                        // through LDS they go out a word at a time.  A lane
                        // writing its own tile's to memory byte by byte took
                        // 4.7 ms on R-MAT 2^18; now 4.1.
                        const bool stage = npc <= kFillBytes;
                        const int shift = static_cast<int>(zb & 3);
                        if (q < n) {
                            int at = shift + zpos;
                            if (stage)
                                write_tile_structure(c, tb + q, j, m, zb + zpos,
                                                     [&](uint8_t col) { s_bytes[at++] = col; });
                            else
                                write_tile_structure(c, tb + q, j, m, zb + zpos);
                        }
                        if (stage) {
                            __syncthreads();
                            unsigned char *to = c.csr_col + (zb - shift);
                            for (int i = tid; i < (shift + npc + 3) >> 2; i += kSymThreads) {
                                const uint32_t v = reinterpret_cast<const uint32_t *>(s_bytes)[i];
                                if (4 * i >= shift && 4 * i + 4 <= shift + npc) {
                                    reinterpret_cast<uint32_t *>(to)[i] = v;
                                    continue;
                                }
                                for (int x = max(4 * i, shift); x < min(4 * i + 4, shift + npc); ++x)
                                    to[x] = s_bytes[x];
                            }
                        }
                        zb += npc;
                    }
                    tb += n;
                    seg = static_cast<int64_t>(ss.m[seg]);
                }
                continue;
            }
        }
        const int s0 = S::first(o, row), s1 = s0 + S::count(o, row);
        const bool one = s1 - s0 <= kSymThreads;   // one chunk: cursors in registers
        int2 *cursors = o.cursors + static_cast<int64_t>(blockIdx.x) * o.cursor_stride;
        int cur = 0, end = 0;
        if (tid == 0)
            s_min[0] = INT_MAX;
        __syncthreads();
        for (int c0 = s0; c0 < s1; c0 += kSymThreads) {
            cur = end = 0;
            if (c0 + tid < s1)
                slot_run<S>(o, task, c0 + tid, &cur, &end);
            lds_min(&s_min[0], cur < end ? S::at(o, cur) : INT_MAX);
            if (!one && c0 + tid < s1)
                cursors[c0 - s0 + tid] = make_int2(cur, end);
        }
        __syncthreads();
        int64_t tiles = 0, nz = 0;
        int64_t head = -1;    // header of the task's last staged segment
        long long first_seg = -1;   // thread 0: the first segment's
        bool fits = ss.capacity > 0;
        for (int w = 0;; w ^= 1) {
            // The window starts at the lowest column left (none: done).
            const int first = s_min[w];
            if (first == INT_MAX)
                break;
            if (tid == 0)
                s_min[w ^ 1] = INT_MAX;
            __syncthreads();
            const int wlo = first >> S::kToTile;
            const int64_t lim = (static_cast<int64_t>(wlo) + kWin) << S::kToTile;
            for (int c0 = s0; c0 < s1; c0 += kSymThreads) {
                int r = 0;
                if (!one) {
                    cur = end = 0;
                    if (c0 + tid < s1) {
                        const int2 run = cursors[c0 - s0 + tid];
                        cur = run.x;
                        end = run.y;
                    }
                }
                if constexpr (!BY_TILES) {
                    if (c0 + tid < s1)
                        r = o.a_r[c0 + tid];
                }
                const int from = cur;
                if (cur < end)
                    cur = gallop([&](int64_t e) { return S::at(o, e); }, cur, end, lim);
                lds_min(&s_min[w ^ 1], cur < end ? S::at(o, cur) : INT_MAX);
                if (!one && c0 + tid < s1)
                    cursors[c0 - s0 + tid].x = cur;
                if constexpr (BY_TILES) {
                    uint4 lo{}, hi{};
                    if (from < cur)
                        spread_tile(static_cast<uint32_t>(S::tile(o, row, c0 + tid).z), &lo, &hi);
                    for_products<int4>(
                        s, cur - from, from, 0,
                        [&](int i) {
                            s_tile[i] = lo;
                            s_tile[kSymThreads + i] = hi;
                        },
                        [&](int e) { return o.b_meta[e]; },
                        [&](int i, const int4 &m) {
                            const uint64_t pm = spread_product(s_tile[i], s_tile[kSymThreads + i],
                                                               static_cast<uint32_t>(m.z));
                            if (pm)
                                atomicOr(&s_wm[m.x - wlo], static_cast<unsigned long long>(pm));
                        });
                } else {
                    for_products<int>(
                        s, cur - from, from, r, [](int) {}, [&](int e) { return o.b_col[e]; },
                        [&](int i, int col) {
                            const int t = (col >> 3) - wlo;
                            const int rr = s.r[i];
                            atomicOr(reinterpret_cast<unsigned int *>(&s_wm[t]) + (rr >> 2),
                                     1u << ((rr & 3) * 8 + (col & 7)));
                        });
                }
            }
            // A wave's stretch of the window's masks, 64 at a time, counted
            // and cleared.
            unsigned long long m[kPer];
            int nt = 0, npc = 0;
            const int i0 = (tid / kWave) * (kPer * kWave) + lane_id();
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                m[i] = s_wm[i0 + i * kWave];
                s_wm[i0 + i * kWave] = 0ull;
                nt += __popcll(__ballot(m[i] != 0));
                npc += __popcll(m[i]);
            }
            npc = wave_sum(npc);
            if (lane_id() == 0) {
                s.scan[tid / kWave] = nt;
                s.scan[kSymThreads / kWave + tid / kWave] = npc;
            }
            __syncthreads();
            int tpos = 0, zpos = 0, all = 0, zall = 0;
#pragma unroll
            for (int i = 0; i < kSymThreads / kWave; ++i) {
                const int x = s.scan[i], y = s.scan[kSymThreads / kWave + i];
                tpos += i < tid / kWave ? x : 0;
                zpos += i < tid / kWave ? y : 0;
                all += x;
                zall += y;
            }
            const unsigned long long below = (1ull << lane_id()) - 1ull;
            if constexpr (FILL) {
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    const unsigned long long has = __ballot(m[i] != 0);
                    const int pc = __popcll(m[i]);
                    const int incl = wave_inclusive_scan(pc);
                    if (m[i])
                        write_tile_structure(c, tb + tiles + tpos + __popcll(has & below),
                                             wlo + i0 + i * kWave, m[i], zb + nz + zpos + incl - pc);
                    tpos += __popcll(has);
                    zpos += __shfl(incl, kWave - 1, kWave);
                }
            } else {
                if (tid == 0) {
                    long long b = -1;
                    if (ss.cursor) {
                        const unsigned long long need = static_cast<unsigned long long>(all) + 1;
                        const unsigned long long at = atomicAdd(ss.cursor, need);
                        if (at + need <= ss.capacity)
                            b = static_cast<long long>(at);
                    }
                    s_base = b;
                }
                __syncthreads();
                const long long b = s_base;
                fits = fits && b >= 0;
                if (fits) {
                    if (tid == 0) {
                        ss.j[b] = all;
                        ss.m[b] = ~0ull;
                        if (head >= 0)
                            ss.m[head] = static_cast<unsigned long long>(b);
                        else
                            first_seg = b;
                    }
                    head = b;
#pragma unroll
                    for (int i = 0; i < kPer; ++i) {
                        const unsigned long long has = __ballot(m[i] != 0);
                        if (m[i]) {
                            const long long at = b + 1 + tpos + __popcll(has & below);
                            ss.j[at] = wlo + i0 + i * kWave;
                            ss.m[at] = m[i];
                        }
                        tpos += __popcll(has);
                    }
                }
            }
            tiles += all;
            nz += zall;
            __syncthreads();   // the scan's buffer, s_base and s_min are reused
        }
        if constexpr (!FILL) {
            if (tid == 0) {
                ss.task[task.id] = TaskSize{fits && head >= 0 ? first_seg : -1ll, tiles, nz};
                if (tiles > 0) {
                    atomicAdd(reinterpret_cast<unsigned long long *>(row_tiles + row),
                              static_cast<unsigned long long>(tiles));
                    atomicAdd(reinterpret_cast<unsigned long long *>(row_nnz + row),
                              static_cast<unsigned long long>(nz));
                }
            }
        }
    }
}

struct Product {
    int col;
    double val;
};

__global__ __launch_bounds__(kNumThreads, 4) void numeric_slab_kernel(SlabOps o, COut c)
{
    __shared__ double s_acc[kNumVals];
    __shared__ unsigned long long s_mask[kNumTiles];  // of the window's C tiles
    __shared__ unsigned short s_at[kNumTiles];        // their first values
    // Bit j: a C tile lies j tile columns into the window; tiles before a word.
    __shared__ unsigned long long s_col[kNumWords];
    __shared__ unsigned short s_rank[kNumWords];
    __shared__ double s_a[kNumThreads];
    __shared__ Runs<kNumThreads> s;
    constexpr int kNumWaves = kNumThreads / kWave;
    __shared__ int s_fit[kNumWaves], s_last[kNumWaves], s_vals[kNumWaves];
    __shared__ int s_task[4];
    __shared__ unsigned long long s_long;
    const int tid = threadIdx.x, w = tid / kWave;
    for (int i = tid; i < kNumVals; i += kNumThreads)
        s_acc[i] = 0.0;
    for (int step = 0;; ++step) {
        Task task;
        if (!next_task<kNumThreads, Slots<false>>(o, step, s_task, &s_long, &task))
            break;
        const int row = task.row;
        int64_t t0 = c.tile_ptr[row];
        int64_t nt = c.tile_ptr[row + 1] - t0;
        if (task.parts > 1) {
            // The part's C tiles.
            auto cols = [at = c.col + t0](int t) { return at[t]; };
            const int n = static_cast<int>(nt);
            const int from = task.part > 0 ? first_at(cols, 0, n, task.lo >> 3) : 0;
            const int to = task.part + 1 < task.parts ? first_at(cols, from, n, task.hi >> 3) : n;
            t0 += from;
            nt = to - from;
        }
        const int s0 = o.a_code_off[row];
        const int s1 = s0 + o.a_row_off[row + 1] - o.a_row_off[row];
        const bool one = s1 - s0 <= kNumThreads;
        int2 *cursors = o.cursors + static_cast<int64_t>(blockIdx.x) * o.cursor_stride;
        int cur = 0, end = 0, r = 0;
        double av = 0.0;
        for (int c0 = s0; c0 < s1; c0 += kNumThreads) {
            cur = end = 0;
            if (c0 + tid < s1) {
                slot_run<Slots<false>>(o, task, c0 + tid, &cur, &end);
                r = o.a_r[c0 + tid];
                av = o.a_vals[c0 + tid];
                if (!one)
                    cursors[c0 - s0 + tid] = make_int2(cur, end);
            }
        }
        for (int64_t t_lo = 0; t_lo < nt;) {
            // The window: as many tiles from t_lo on as the tables and the
            // accumulator hold (at least one: a tile has at most 64 values).
            // A thread looks at kLookTiles of the next kNumTiles.
            for (int i = tid; i < kNumWords; i += kNumThreads)
                s_col[i] = 0ull;
            __syncthreads();
            const int wlo = c.col[t0 + t_lo];
            const int64_t v0 = c.tile_nnz[t0 + t_lo];
            int fit = 0, last = 0, vals = 0;
#pragma unroll
            for (int i = 0; i < kLookTiles; ++i) {
                const int x = i * kNumThreads + tid;
                const int64_t t = t_lo + x;
                if (t < nt) {
                    const int j = c.col[t0 + t] - wlo;
                    const uint64_t m = c.mask[t0 + t];
                    const int64_t at = c.tile_nnz[t0 + t] - v0;
                    const int64_t to = at + __popcll(m);
                    if (j >= 0 && j < kNumSpan && to <= kNumVals) {
                        s_mask[x] = m;
                        s_at[x] = static_cast<unsigned short>(at);
                        atomicOr(&s_col[j >> 6], 1ull << (j & 63));
                        ++fit;
                        last = max(last, j);
                        vals = max(vals, static_cast<int>(to));
                    }
                }
            }
            fit = wave_sum(fit);
#pragma unroll
            for (int d = kWave / 2; d > 0; d >>= 1) {
                last = max(last, __shfl_xor(last, d, kWave));
                vals = max(vals, __shfl_xor(vals, d, kWave));
            }
            if (lane_id() == 0) {
                s_fit[w] = fit;
                s_last[w] = last;
                s_vals[w] = vals;
            }
            __syncthreads();
            if (tid < kWave) {
                constexpr int kPer = kNumWords / kWave;
                int n[kPer], sum = 0;
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    n[i] = __popcll(s_col[tid * kPer + i]);
                    sum += n[i];
                }
                int at = wave_inclusive_scan(sum) - sum;
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    s_rank[tid * kPer + i] = static_cast<unsigned short>(at);
                    at += n[i];
                }
            }
            fit = last = vals = 0;
#pragma unroll
            for (int i = 0; i < kNumWaves; ++i) {
                fit += s_fit[i];
                last = max(last, s_last[i]);
                vals = max(vals, s_vals[i]);
            }
            const int64_t lim = (static_cast<int64_t>(wlo) + last + 1) * 8;
            for (int c0 = s0; c0 < s1; c0 += kNumThreads) {
                if (!one) {
                    cur = end = 0;
                    if (c0 + tid < s1) {
                        const int2 run = cursors[c0 - s0 + tid];
                        cur = run.x;
                        end = run.y;
                        r = o.a_r[c0 + tid];
                        av = o.a_vals[c0 + tid];
                    }
                }
                const int from = cur;
                if (cur < end)
                    cur = gallop([&](int64_t e) { return o.b_col[e]; }, cur, end, lim);
                if (!one && c0 + tid < s1)
                    cursors[c0 - s0 + tid].x = cur;
                for_products<Product>(
                    s, cur - from, from, r, [&](int i) { s_a[i] = av; },
                    [&](int e) { return Product{o.b_col[e], o.b_val[e]}; },
                    [&](int i, const Product &x) {
                        // Every product's tile lies in the window; the bounds
                        // keep a damaged structure inside the LDS.
                        const int j = (x.col >> 3) - wlo;
                        if (j < 0 || j >= kNumSpan)
                            return;
                        const int t = s_rank[j >> 6] +
                                      __popcll(s_col[j >> 6] & ((1ull << (j & 63)) - 1ull));
                        if (t >= kNumTiles)
                            return;
                        const int bit = s.r[i] * 8 + (x.col & 7);
                        const int at = s_at[t] + __popcll(s_mask[t] & ((1ull << bit) - 1ull));
                        if (at < kNumVals)
                            atomicAdd(&s_acc[at], s_a[i] * x.val);
                    });
            }
            for (int i = tid; i < vals; i += kNumThreads) {
                c.val[v0 + i] = s_acc[i];
                s_acc[i] = 0.0;
            }
            t_lo += fit > 0 ? fit : nt;   // (a first tile always fits)
            __syncthreads();   // the window's tables are rewritten
        }
    }
}

} // namespace

static SlabOps slab_ops(const DevTiles &a, const DevTiles *b, const SpgemmWork *w, const SlabTasks &tasks, int *queue,
                        int static_rows)
{
    SlabOps o{};
    if (b) {
        o.a_trp = a.tile_row_ptr.as<int>();
        o.a_meta = a.meta.as<int4>();
        o.b_meta = b->records.as<int4>();
        o.b_groups = b->row_groups.as<int>();
    }
    o.a_row_off = a.row_payload_off.as<int>();
    if (w->slot_codes_ready) {
        o.a_code_off = o.a_row_off;
        o.a_k = w->slot_k.as<int>();
        o.a_r = w->slot_r.as<uint8_t>();
    } else {
        o.a_code_off = w->code_off.as<int>();
        o.a_k = w->row_slot_k.as<int>();
        o.a_r = w->row_slot_r.as<uint8_t>();
    }
    o.a_vals = w->slot_codes_ready ? a.values.as<double>() : w->row_slot_v.as<double>();
    o.b_start = w->b_start.as<int>();
    o.b_col = w->b_col.as<int>();
    o.b_val = w->b_val.as<double>();
    o.tasks = tasks;
    o.queue = queue;
    o.static_rows = static_rows;
    o.cursors = w->slab_cursors.as<int2>();
    o.cursor_stride = w->slab_cursor_stride;
    return o;
}

// Workgroups of the symbolic passes; the numeric pass has half as many.
static unsigned slab_blocks()
{
    return 2u * static_cast<unsigned>(ctx().num_cus > 0 ? ctx().num_cus : 256);
}

int64_t slab_target(unsigned long long pairs)
{
    // Sixteen tasks per workgroup of the symbolic passes on average, and at least the work that
    // pays for a task's search of its cuts.
    return static_cast<int64_t>(std::max<unsigned long long>(65536, pairs / (16ull * slab_blocks())));
}

// A workgroup's cursors take 8 bytes a slot of the longest row: 128 MB for a
// hub of 16 million entries, 67 GB for all workgroups.  Fewer workgroups then
// take the tasks, as many as a quarter of the free memory (and what is held)
// has room for, rather than none for want of memory.
unsigned slab_cursor_blocks(int64_t longest, size_t held, size_t free_bytes)
{
    const uint64_t per = static_cast<uint64_t>(longest) * sizeof(int2);
    return static_cast<unsigned>(
        std::max<uint64_t>(1, std::min<uint64_t>(slab_blocks(), (free_bytes / 4 + held) / per)));
}

// Cursors in memory for rows of more slots than a workgroup may have threads,
// and the workgroups they serve.
static int slab_cursors(SpgemmWork *w, int64_t longest)
{
    constexpr size_t kUnasked = size_t(1) << 30;   // taken without a look at the free memory
    const DevBuf &buf = w->slab_cursors;
    w->slab_cursor_stride = 0;   // (no buffer behind it, should its allocation fail)
    w->slab_cursor_blocks = slab_blocks();
    if (longest <= kSymThreads)
        return RTT_OK;
    const size_t per = static_cast<size_t>(longest) * sizeof(int2);
    if (buf.bytes < slab_blocks() * per) {
        unsigned blocks = slab_blocks();
        const bool large = blocks * per > kUnasked;
        size_t free_b = 0, total_b = 0;
        if (large && hipMemGetInfo(&free_b, &total_b) == hipSuccess)
            blocks = slab_cursor_blocks(longest, buf.bytes, free_b);
        // A large buffer is kept while it serves half of what there is room for.
        if (!large || buf.bytes / per < (blocks + 1) / 2)
            RTT_TRY(w->slab_cursors.ensure(blocks * per));
        w->slab_cursor_blocks =
            static_cast<unsigned>(std::min<uint64_t>(slab_blocks(), buf.bytes / per));
    }
    w->slab_cursor_stride = longest;
    return RTT_OK;
}

int slab_prepare(const DevTiles &a, const DevTiles &b, BuildWork *bw, SpgemmWork *w,
                 const int *rows, int n, const int *more, int n_more, int64_t longest)
{
    hipStream_t s = ctx().stream;
    const int R = b.tile_row_count;
    const int listed = n + n_more;
    if (R == 0 || listed == 0)
        return RTT_OK;
    // Few rows are served by their own slots and the rows of B they select, for
    // a host wait; many select most of B.  64^3 box stencil (6.9e6 entries, 32768
    // tile rows) with 64, 512, 2048 and 4096 wide rows, A*A: 1.12, 1.32, 1.88
    // and 2.33 ms with all of B, 1.01, 1.25, 1.86 and 2.35 ms with the rows
    // selected; A*A^T: 1.07, 1.45, 2.01, 2.55 and 0.85, 1.33, 2.02, 2.60.  One
    // row of 60 entries more in the 128^3 stencil, A*A^T: 6.78 -> 3.75 ms (3.52
    // without it).  By slots, a hub of 10000, 100000 and 300000 entries in a
    // 1000^2 Laplacian: 2.81, 7.94, 15.3 and 2.70, 7.79, 15.4 ms.
    const bool few = static_cast<int64_t>(listed) * 16 < a.tile_row_count &&
                     listed * longest * 16 < a.payload;
    const bool transposed = b.transpose_of != nullptr;
    const size_t rows_b = static_cast<size_t>(R), rows_a = static_cast<size_t>(a.tile_row_count);
    RTT_TRY(w->b_start.ensure((rows_b * 5 + 1) * sizeof(int)));
    BRows g{};
    g.R = R;
    g.trp = b.tile_row_ptr.as<int>();
    g.groups = b.row_groups.as<int>();
    g.meta = b.records.as<int4>();
    g.tcol = b.tile_col_idx.as<int>();
    g.masks = b.masks.as<uint32_t>();
    g.offs = b.value_offsets.as<int>();
    g.vals = b.payload_values();
    g.start = w->b_start.as<int>();
    if (transposed) {
        // B = A^T at tile level has its rows in class order alone.
        RTT_TRY(bw->keys_in.ensure(static_cast<size_t>(std::max<int64_t>(1, b.num_tiles)) *
                                   sizeof(int)));
        g.order = bw->keys_in.as<int>();
    }
    // A workgroup per tile row where rows average past 16 tiles (a hub row
    // holds thousands), a wave otherwise: R-MAT 2^13, 2^16 and 2^18 took 19, 69 and
    // 370 us in workgroups, 37, 154 and 745 in waves; a 64^3 box stencil with 4096
    // wide rows 185 and 99, a band of 40 entries a row 16 and 13.
    const bool wide = b.num_tiles > 16 * static_cast<int64_t>(R);
    auto over_rows = [&](auto wave_kernel, auto block_kernel, int64_t count, auto... args) {
        if (wide)
            hipLaunchKernelGGL(block_kernel, dim3(static_cast<unsigned>(count)), dim3(256), 0, s, g,
                               args...);
        else
            hipLaunchKernelGGL(wave_kernel, dim3(blocks_for(count, 256 / kWave)), dim3(256), 0, s, g,
                               args...);
    };
    int64_t count = R;             // B rows laid out (to be looked at, while it isn't known)
    int64_t entries = b.payload;   // at most
    Picked *picked = nullptr;
    if (few || transposed) {
        constexpr size_t kHeadInts = sizeof(Picked) / sizeof(int);
        RTT_TRY(w->slab_pick.ensure((kHeadInts + 2 * rows_b) * sizeof(int)));
        picked = w->slab_pick.as<Picked>();
        int *flag = w->slab_pick.as<int>() + kHeadInts, *list = flag + R;
        const int64_t clear = static_cast<int64_t>(kHeadInts) + (few ? R : 0);
        hipLaunchKernelGGL(zero_ints_kernel, dim3(blocks_for(clear, 256)), dim3(256), 0, s,
                           w->slab_pick.as<int>(), clear);
        if (few) {
            const size_t slots = static_cast<size_t>(listed * longest);
            const bool codes = !w->slot_codes_ready;
            if (codes) {
                RTT_TRY(w->code_off.ensure(rows_a * sizeof(int)));
                RTT_TRY(w->row_slot_k.ensure(slots * sizeof(int)));
                RTT_TRY(w->row_slot_r.ensure(slots));
                RTT_TRY(w->row_slot_v.ensure(slots * sizeof(double)));
            }
            hipLaunchKernelGGL(pick_rows_kernel, dim3(static_cast<unsigned>(listed), 4), dim3(256),
                               0, s, rows, n, more, longest, a.tile_row_ptr.as<int>(),
                               a.meta.as<int4>(), a.row_payload_off.as<int>(), a.values.as<double>(), flag,
                               codes ? w->code_off.as<int>() : nullptr,
                               codes ? w->row_slot_k.as<int>() : nullptr,
                               codes ? w->row_slot_r.as<uint8_t>() : nullptr,
                               codes ? w->row_slot_v.as<double>() : nullptr);
            hipLaunchKernelGGL(list_rows_kernel, dim3(blocks_for(R, 256)), dim3(256), 0, s, R, flag,
                               picked, list);
            g.list = list;
            g.n = &picked->rows;
            count = std::min<int64_t>(R, listed * longest);
        }
        if (transposed)
            over_rows(count_rows_kernel<kWave>, count_rows_kernel<256>, count);
        hipLaunchKernelGGL(place_rows_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, s, g,
                           picked);
        RTT_HIP(hipGetLastError());
    }
    if (few) {
        RTT_TRY(w->host_pick.ensure(sizeof(Picked)));
        RTT_HIP(hipMemcpyAsync(w->host_pick.ptr, picked, sizeof(Picked), hipMemcpyDeviceToHost, s));
        RTT_HIP(hipStreamSynchronize(s));
        count = static_cast<int64_t>(w->host_pick.as<Picked>()->rows);
        entries = static_cast<int64_t>(w->host_pick.as<Picked>()->entries);
    } else if (!w->slot_codes_ready) {
        RTT_TRY(w->slot_k.ensure(static_cast<size_t>(std::max<int64_t>(1, a.payload)) * sizeof(int)));
        RTT_TRY(w->slot_r.ensure(static_cast<size_t>(std::max<int64_t>(1, a.payload))));
        hipLaunchKernelGGL(slot_codes_kernel, dim3(blocks_for(a.num_tiles, 256)), dim3(256), 0, s,
                           a.num_tiles, a.meta.as<int4>(), w->slot_k.as<int>(),
                           w->slot_r.as<uint8_t>());
        RTT_HIP(hipGetLastError());
        w->slot_codes_ready = true;
    }
    RTT_TRY(w->b_col.ensure(static_cast<size_t>(std::max<int64_t>(1, entries)) * sizeof(int)));
    RTT_TRY(w->b_val.ensure(static_cast<size_t>(std::max<int64_t>(1, entries)) * sizeof(double)));
    g.col = w->b_col.as<int>();
    g.val = w->b_val.as<double>();
    if (count == 0)
        return RTT_OK;
    if (transposed)
        over_rows(order_tiles_kernel<kWave>, order_tiles_kernel<256>, count, bw->keys_in.as<int>());
    if (picked)
        over_rows(scalar_rows_kernel<kWave, true>, scalar_rows_kernel<256, true>, count);
    else
        over_rows(scalar_rows_kernel<kWave, false>, scalar_rows_kernel<256, false>, count);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

static SlabStage slab_stage(const SpgemmWork *w, unsigned long long *cursor)
{
    SlabStage ss;
    ss.task = w->slab_task_size.as<TaskSize>();
    ss.cursor = cursor;
    if (w->slab_stage_cap > 0) {
        ss.j = w->slab_stage_j.as<int>();
        ss.m = w->slab_stage_m.as<unsigned long long>();
        ss.capacity = w->slab_stage_cap;
    }
    return ss;
}

// Whether the symbolic passes go by tiles: where an A tile of the rows and a B
// tile carry several products on average (spread evenly, a quarter of the
// product of their entries), one select of their masks does for all of them,
// and where it has no more runs to start than entries (kRuns a tile: a hub of
// 1.7 entries a tile in a 1000^2 Laplacian took 10.5 ms by tiles, 3.4 by entries).  All but the
// numeric pass of 16384 rows of 100 random full 8x8 blocks a tile row, 256
// products a pair: 18.6 ms by entries, 2.3 by tiles (their first call 60 and 28
// ms, 44 with the passes before these); 40 such blocks at 8 % (1.9): 0.55 and
// 0.52 ms; R-MAT 2^18 (0.5): 16.2 and 19.6; a band of 8000 at 2 % (0.5): 9.3
// and 11.7.
bool slab_by_tiles(const DevTiles &b, const SlabSizes &rows)
{
    const double fa = static_cast<double>(rows.slots) / static_cast<double>(rows.tiles);
    const double fb = static_cast<double>(b.payload) / static_cast<double>(b.num_tiles);
    return fa * fb / 4.0 >= kTileProducts && fa >= kRuns && rows.most_tiles <= INT_MAX / kRuns;
}

int slab_symbolic(const DevTiles &a, const DevTiles &b, SpgemmWork *w, const SlabTasks &tasks,
                  int *queue, int static_rows, unsigned long long *cursor, const SlabSizes &rows)
{
    w->slab_by_tiles = slab_by_tiles(b, rows);
    RTT_TRY(slab_cursors(w, w->slab_by_tiles ? kRuns * rows.most_tiles : rows.longest));
    // Staging of the rows' tile lists: grown to what the previous calls
    // needed, within a quarter of the free device memory; without it every
    // row is recomputed by the fill pass.
    if (w->slab_stage_need > w->slab_stage_cap) {
        size_t free_b = 0, total_b = 0;
        const uint64_t per = sizeof(int) + sizeof(unsigned long long);
        uint64_t want = w->slab_stage_need + w->slab_stage_need / 16;
        if (hipMemGetInfo(&free_b, &total_b) == hipSuccess)
            want = std::min<uint64_t>(want, free_b / 4 / per);
        w->slab_stage_cap = 0;
        if (want > 0 && w->slab_stage_j.ensure(want * sizeof(int)) == RTT_OK &&
            w->slab_stage_m.ensure(want * sizeof(unsigned long long)) == RTT_OK)
            w->slab_stage_cap = want;
        clear_error();
    }
    RTT_TRY(w->slab_task_size.ensure(static_cast<size_t>(tasks.most) * sizeof(TaskSize)));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(w->slab_cursor_blocks), dim3(kSymThreads), 0, ctx().stream,
                           slab_ops(a, &b, w, tasks, queue, static_rows), w->row_tiles.as<int64_t>(),
                           w->row_nnz.as<int64_t>(), slab_stage(w, cursor), COut{});
    };
    if (w->slab_by_tiles)
        launch(symbolic_slab_kernel<false, true>);
    else
        launch(symbolic_slab_kernel<false, false>);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int slab_structure(const DevTiles &a, const DevTiles &b, SpgemmWork *w, const SlabTasks &tasks,
                   int *queue, int static_rows, const COut &c)
{
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(w->slab_cursor_blocks), dim3(kSymThreads), 0, ctx().stream,
                           slab_ops(a, &b, w, tasks, queue, static_rows), nullptr, nullptr,
                           slab_stage(w, nullptr), c);
    };
    if (w->slab_by_tiles)
        launch(symbolic_slab_kernel<true, true>);
    else
        launch(symbolic_slab_kernel<true, false>);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int slab_numeric(const DevTiles &a, SpgemmWork *w, const SlabTasks &tasks, int *queue,
                 int static_rows, const COut &c, int64_t longest)
{
    RTT_TRY(slab_cursors(w, longest));
    hipLaunchKernelGGL(numeric_slab_kernel, dim3(std::max(1u, w->slab_cursor_blocks / 2)), dim3(kNumThreads), 0,
                       ctx().stream, slab_ops(a, nullptr, w, tasks, queue, static_rows), c);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

} // namespace rtt
