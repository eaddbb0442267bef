// CSR -> hybrid tile builder.
//
// Tiles are formed without a global sort: rows are kept column-sorted (they
// are sorted once at upload when they arrive unsorted), so the tiles of one
// tile row are the ordered merge of its TR row streams.  This replaces the
// reference's 64-bit key radix sort + reduce_by_key
// (src/gpu_dmma_tiles.h:1117-1395) and its 4-lane ordered-warp B path
// (src/gpu_dmma_tiles.h:313-560).
//
// One launch counts, scans and fills.  A workgroup stages the columns of its
// 512 rows in LDS, counts its tile rows' tiles, gets the totals of the
// workgroups before it by a decoupled look-back, and fills its part of the
// arrays.  The host does not know the totals beforehand: a workgroup whose
// part lies past the arrays' capacity fills nothing, and the host, which
// reads the totals once at the end, grows the arrays and launches again when
// they did not fit (the first build of a handle; a rebuild in place fits).
//
// Tile rows with more than kLongRow entries per scalar row on average would
// hold one lane each for thousands of steps; a workgroup each counts and
// fills those, parallel over entries (the hub rows of R-MAT 2^18 held the
// rebuild to 37 ms; now 1.8 ms).  That takes longer than a lane each where most
// rows are like that, and less where few are: a step of block FEM with 124
// entries a row (240000 rows) takes 6.2 ms with the limit at 128, 6.5 at 96, and
// 84 entries 3.0 and 3.4; 40 rows of 400 entries in a 500^2 Laplacian 1.37 and
// 0.65 ms, a band of 150 entries in 4000 rows 0.49 and 0.37.
#include <algorithm>
#include <climits>

#include "device.hpp"
#include "internal.hpp"

namespace rtt {

namespace {

constexpr int kThreads = 256;     // long rows and small kernels
// The build kernel: 512 threads at 6 waves per SIMD.  256 took the AMG
// batch's first build from 317 to 324 us (twice the workgroups to look back
// over), 1024 to 470 us (its staging, walks and copy hardly overlap).
constexpr int kBuild = 512;
constexpr int kBuildWaves = kBuild / kWave;
constexpr int kWaves = kThreads / kWave;

// Columns a workgroup stages: the average of its rows and a tenth, at most
// kStageMax (entries past the stage are walked in global memory; 79 KB with
// the skew, two workgroups per CU).  A stage cut to 64 KB, short of
// block-FEM's rows, took its build from 0.53 to 0.8 ms.
constexpr int kStageMax = 19200;
constexpr int kLoads = 8;   // entries whose loads a thread issues together
constexpr int kLongRow = 128;

// LDS word of staged column x: lanes walk rows of like length, so equal
// strides of a multiple of 32 words are skewed over the banks.
__host__ __device__ constexpr int staged(int x) { return x + (x >> 5); }
constexpr int kLongWin = 4096;   // tile columns a long row's window covers

// Fields of a tile row's class counts: five classes of 12 bits.  Tile rows
// counted this way have at most kLongRow * kTileK tiles.
constexpr int kClassBits = 12;
constexpr int kClassesUsed = 5;
static_assert(kLongRow * kTileK < (1 << kClassBits), "class fields");

// Sizes and classes of a long tile row.
struct LongRow {
    int tiles = 0, dense = 0;
    long long payload = 0;
    long long first = 0;   // the row's first payload slot, set by the build kernel
    int cls[kClassesUsed] = {};
};

// Head of the builder's scratch; the look-back words follow it.  Cleared
// before every launch.
struct BuildHead {
    unsigned int ticket;
    unsigned int n_long;
    unsigned int dups;
    unsigned int fits;     // the whole build lies within the arrays
};

struct BuildArgs {
    int R = 0;                 // tile rows
    int active_rows = 0, active_cols = 0;
    const int *__restrict__ rp = nullptr;
    const int *__restrict__ ci = nullptr;
    const double *__restrict__ val = nullptr;
    const int *__restrict__ row_map = nullptr;
    int dense_threshold = 0;
    int stage = 0;             // columns staged per workgroup
    BuildHead *head = nullptr;
    unsigned long long *look = nullptr;   // two words per workgroup
    const int *__restrict__ long_rows = nullptr;
    LongRow *long_of = nullptr;   // per tile row; null: no long rows
    long long cap_tiles = 0, cap_payload = 0;
    int *__restrict__ tile_row_ptr = nullptr;
    int *__restrict__ groups = nullptr;   // B: class runs of every row
    int *__restrict__ tile_col_idx = nullptr;
    uint32_t *__restrict__ masks = nullptr;
    int *__restrict__ value_offsets = nullptr;
    double *__restrict__ values = nullptr;
    int4 *__restrict__ meta = nullptr;    // B: in class order within a row
    int *__restrict__ src_slot = nullptr; // per source entry, null: not wanted
    long long *totals = nullptr;          // pinned host memory: tiles, payload, dense, dups
};

// DPP reductions over groups of TR = 4 or 8 lanes.
template <int TR>
__device__ __forceinline__ int group_min(int v)
{
    v = min(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false));   // lane ^ 1
    v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false));   // lane ^ 2
    if constexpr (TR == 8)   // row_half_mirror: the other four lanes
        v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false));
    return v;
}

template <int TR>
__device__ __forceinline__ uint32_t group_or(uint32_t u)
{
    int v = static_cast<int>(u);
    v |= __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false);
    v |= __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false);
    if constexpr (TR == 8)
        v |= __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false);
    return static_cast<uint32_t>(v);
}

template <int TR>
__device__ __forceinline__ int group_sum(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false);
    if constexpr (TR == 8)
        v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false);
    return v;
}

// Class of a B tile (bit c*4+k) within its row: 0 heavy, 1 + k light in row k.
__device__ __forceinline__ int mask_class(uint32_t mask)
{
    if (__popc(mask) >= kHeavyMin)
        return 0;
    const int k = __builtin_ctz(mask) & 3;
    return (mask & ~(0x11111111u << k)) ? 0 : 1 + k;
}

__device__ __forceinline__ int4 tile_meta(int col, uint32_t mask, int64_t off, bool dense)
{
    uint32_t bytes = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        bytes |= stride4_bits(mask, k) << (8 * k);
    return make_int4(col, static_cast<int>(mask), static_cast<int>(bytes),
                     static_cast<int>(off) | (dense ? INT_MIN : 0));
}

// Look-back words of the build: word 0 holds tiles (31 bits) over dense tiles
// (31 bits), word 1 payload slots.  Both fields of word 0 stay below 2^31:
// there are at most nnz <= INT_MAX tiles.
__global__ void build_init_kernel(unsigned long long *p, int64_t n, unsigned long long *q)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0ull;
    if (i == 0 && q)
        *q = 0ull;
}

// One group of TR lanes per tile row, lane r on scalar row r of it.  The
// group repeatedly takes the smallest tile column among its lanes' heads and
// ORs the lanes' bits into the tile's mask, once to count and once to fill.
// The fill walk replaces every staged column by its payload slot (kDup: a
// duplicate of the entry before it; kOut: past the tiled columns; kDone:
// stored by the walk itself), and one pass over the stage then moves the
// values: whole-line loads and stores that lie close together, against one
// dependent load and store per entry and lane in the walk.  Duplicates
// (adjacent equal columns in a sorted row) are summed in row order.
// Bound by latency, a workgroup at a time: block-FEM 500k 0.53 ms (2.6 TB/s),
// 0.66 ms with the stage unskewed and one load per thread in flight, 1.20 ms
// for separate count and fill passes, their scans and a copy (AMG batch of
// 8, two builds: 0.65 against 1.1 ms).
constexpr int kDup = -1, kOut = -2, kDone = -3;

template <int TR, int TC, bool B>
__global__ __launch_bounds__(kBuild, 6) void tile_build_kernel(BuildArgs g)
{
    static_assert(TR * TC == 32, "tiles hold 32 elements");
    static_assert(kWave % TR == 0, "a wave holds whole tile rows");
    extern __shared__ int s_stage[];
    __shared__ unsigned int s_block;
    __shared__ unsigned long long s_x[kBuildWaves + 1], s_y[kBuildWaves + 1];
    const int tid = threadIdx.x;
    if (tid == 0)
        s_block = atomicAdd(&g.head->ticket, 1u);
    __syncthreads();
    const int64_t b = s_block;
    const int64_t row0 = b * kBuild;
    const int64_t row = row0 + tid;
    const int64_t tr = row / TR;
    const int r = static_cast<int>(row % TR);
    const int64_t lim = min<int64_t>(static_cast<int64_t>(g.R) * TR, g.active_rows);
    // Without a row map the workgroup's rows are one stretch of the CSR.
    int e0 = 0, ns = 0;
    if (!g.row_map && row0 < lim) {
        e0 = g.rp[row0];
        ns = min(g.rp[min<int64_t>(row0 + kBuild, lim)] - e0, g.stage);
    }
    for (int x0 = tid; x0 < ns; x0 += kLoads * kBuild) {
        int v[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
            v[u] = x0 + u * kBuild < ns ? g.ci[e0 + x0 + u * kBuild] : 0;
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
            if (x0 + u * kBuild < ns)
                s_stage[staged(x0 + u * kBuild)] = v[u];
    }
    int p = 0, end = 0;
    if (row < lim) {
        const int src = g.row_map ? g.row_map[row] : static_cast<int>(row);
        p = g.rp[src];
        end = g.rp[src + 1];
    }
    __syncthreads();
    auto col = [&](int x) { return x - e0 < ns ? s_stage[staged(x - e0)] : g.ci[x]; };
    // Long tile rows are counted and filled by their own kernels.
    const bool is_long = g.long_of && group_sum<TR>(end - p) > kLongRow * TR;
    if (g.long_of) {
        for (unsigned long long m = __ballot(is_long); m; m &= m - 1) {
            const int l = __builtin_ctzll(m);
            const int lp = __shfl(p, l, kWave), le = __shfl(end, l, kWave);
            for (int x = lp - e0 + lane_id(); x < min(le - e0, ns); x += kWave)
                s_stage[staged(x)] = kDone;
        }
        if (is_long)
            end = p;
    }
    // Columns at or beyond active_cols are outside the tiled extent.
    while (end > p && col(end - 1) >= g.active_cols) {
        --end;
        if (end - e0 < ns)
            s_stage[staged(end - e0)] = kOut;
        else if (g.src_slot)
            g.src_slot[end] = -1;
    }
    // Next tile of the group from its lanes' positions x: its column, its
    // mask, this lane's bits and the lane's entries [x, q) in it.  (Unsigned
    // column arithmetic throughout: a shift and a mask each.)
    constexpr unsigned kTC = TC;
    auto bit_of = [&](unsigned c) { return 1u << (B ? (c % kTC) * TR + r : r * TC + c % kTC); };
    auto next_tile = [&](int x, int *head, uint32_t *bits, int *q, int (&cb)[TC]) {
        const int h = group_min<TR>(x < end ? static_cast<int>(static_cast<unsigned>(col(x)) / kTC)
                                            : INT_MAX);
        *head = h;
        uint32_t v = 0;
        int y = x;
        // The first TC columns from x, when staged, are read together;
        // without duplicates a row has at most TC entries in a tile.
        if (x + TC - e0 <= ns) {
#pragma unroll
            for (int u = 0; u < TC; ++u)
                cb[u] = x + u < end ? s_stage[staged(x + u - e0)] : INT_MIN;
            bool in = true;
#pragma unroll
            for (int u = 0; u < TC; ++u) {
                const unsigned c = static_cast<unsigned>(cb[u]);
                in = in && c / kTC == static_cast<unsigned>(h);
                v |= in ? bit_of(c) : 0u;
                y += in ? 1 : 0;
            }
        }
        while (y < end) {
            const unsigned c = static_cast<unsigned>(col(y));
            if (c / kTC != static_cast<unsigned>(h))
                break;
            v |= bit_of(c);
            ++y;
        }
        *bits = v;
        *q = y;
        return group_or<TR>(v);
    };

    // ---- count ------------------------------------------------------------
    int nt = 0, nd = 0;
    long long pay = 0;
    unsigned long long cls = 0;   // kClassBits per class
    {
        int x = p;
        int cb[TC];
        for (;;) {
            int h, q;
            uint32_t bits;
            const uint32_t mask = next_tile(x, &h, &bits, &q, cb);
            if (h == INT_MAX)
                break;
            const int cnt = __popc(mask);
            const bool dense = cnt >= g.dense_threshold;
            ++nt;
            nd += dense ? 1 : 0;
            pay += dense ? 32 : cnt;
            if constexpr (B)
                cls += 1ull << (kClassBits * mask_class(mask));
            x = q;
        }
    }
    if (is_long) {
        nt = g.long_of[tr].tiles;
        nd = g.long_of[tr].dense;
        pay = g.long_of[tr].payload;
    }
    // ---- offsets -------------------------------------------------------------
    const unsigned long long mine =
        r == 0 ? (static_cast<unsigned long long>(nt) << 31) | static_cast<unsigned int>(nd) : 0ull;
    const unsigned long long my_pay = r == 0 ? static_cast<unsigned long long>(pay) : 0ull;
    const unsigned long long ix = wave_inclusive_scan(mine), iy = wave_inclusive_scan(my_pay);
    const int w = tid / kWave;
    if (lane_id() == kWave - 1) {
        s_x[w] = ix;
        s_y[w] = iy;
    }
    __syncthreads();
    unsigned long long all_x = 0, all_y = 0, bx = 0, by = 0;
#pragma unroll
    for (int i = 0; i < kBuildWaves; ++i) {
        bx += i < w ? s_x[i] : 0ull;
        by += i < w ? s_y[i] : 0ull;
        all_x += s_x[i];
        all_y += s_y[i];
    }
    if (w == 0) {
        if (lane_id() == 0)
            publish(g.look, b, b == 0 ? kUpTo : kOwn, all_x, all_y);
        unsigned long long px = 0, py = 0;
        if (b > 0) {
            look_back(g.look, b, &px, &py);
            if (lane_id() == 0)
                publish(g.look, b, kUpTo, px + all_x, py + all_y);
        }
        if (lane_id() == 0) {
            s_x[kBuildWaves] = px;
            s_y[kBuildWaves] = py;
        }
    }
    __syncthreads();
    const unsigned long long px = s_x[kBuildWaves], py = s_y[kBuildWaves];
    const long long end_tiles = static_cast<long long>((px + all_x) >> 31);
    const long long end_pay = static_cast<long long>(py + all_y);
    const bool fits = end_tiles <= g.cap_tiles && end_pay <= g.cap_payload;
    // The group's first lane holds its exclusive sums.
    const int lead = lane_id() & ~(TR - 1);
    const int t0 = __shfl(static_cast<int>((px + bx + ix - mine) >> 31), lead, kWave);
    const long long o0 = __shfl(static_cast<long long>(py + by + iy - my_pay), lead, kWave);
    const bool last = (b + 1) * kBuild >= static_cast<int64_t>(g.R) * TR;
    unsigned long long at = 0;   // tiles of the classes below each class, kClassBits each
    if constexpr (B) {
#pragma unroll
        for (int c = 1; c < kClassesUsed; ++c)
            at |= ((at >> (kClassBits * (c - 1)) & ((1u << kClassBits) - 1)) +
                   (cls >> (kClassBits * (c - 1)) & ((1u << kClassBits) - 1)))
                  << (kClassBits * c);
    }
    if (tr < g.R) {
        if (r == 0)
            g.tile_row_ptr[tr] = t0;
        if (r == 0 && is_long)
            g.long_of[tr].first = o0;
        if constexpr (B) {
            static_assert(TR * 2 == kClassSlots, "two class slots per lane");
            int s[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int c = 2 * r + i;
                if (c >= kClassesUsed) {
                    s[i] = t0 + nt;
                } else if (is_long) {
                    s[i] = t0;
                    for (int k = 0; k < c; ++k)
                        s[i] += g.long_of[tr].cls[k];
                } else {
                    s[i] = t0 + static_cast<int>(at >> (kClassBits * c) & ((1u << kClassBits) - 1));
                }
            }
            *reinterpret_cast<int2 *>(g.groups + kClassSlots * tr + 2 * r) = make_int2(s[0], s[1]);
        }
    }
    if (last && tid == 0) {
        g.tile_row_ptr[g.R] = static_cast<int>(end_tiles);
        if constexpr (B)
            g.groups[static_cast<int64_t>(kClassSlots) * g.R] = static_cast<int>(end_tiles);
        if (fits) {
            g.value_offsets[end_tiles] = static_cast<int>(end_pay);
            g.values[end_pay] = 0.0;   // the zero that absent entries read
        }
        g.head->fits = fits ? 1u : 0u;
        g.totals[0] = end_tiles;
        g.totals[1] = end_pay;
        g.totals[2] = static_cast<long long>((px + all_x) & ((1ull << 31) - 1ull));
    }
    if (!fits)
        return;
    // ---- fill -----------------------------------------------------------------
    {
        int x = p, t = t0;
        long long o = o0;
        int cb[TC];
        for (;;) {
            int h, q;
            uint32_t bits;
            const uint32_t mask = next_tile(x, &h, &bits, &q, cb);
            if (h == INT_MAX)
                break;
            const int cnt = __popc(mask);
            const bool dense = cnt >= g.dense_threshold;
            int tm = t;   // where the tile's meta goes
            if constexpr (B) {
                const int sh = kClassBits * mask_class(mask);
                tm = t0 + static_cast<int>(at >> sh & ((1u << kClassBits) - 1));
                at += 1ull << sh;
            }
            if (r == 0) {
                g.meta[tm] = tile_meta(h, mask, o, dense);
            } else if (r < 4) {
                // One store for the three arrays, lanes 1 to 3.
                int *dst = r == 1 ? g.tile_col_idx
                                  : (r == 2 ? reinterpret_cast<int *>(g.masks) : g.value_offsets);
                dst[t] = r == 1 ? h : (r == 2 ? static_cast<int>(mask) : static_cast<int>(o));
            }
            if (dense) {
                // Absent slots of this lane's row are explicit zeros.
#pragma unroll
                for (int lc = 0; lc < TC; ++lc) {
                    const int phys = B ? lc * TR + r : r * TC + lc;
                    if (!(bits >> phys & 1u))
                        g.values[o + phys] = 0.0;
                }
            }
            const uint32_t known = dense ? 0xFFFFFFFFu : mask;   // a dense tile's slots are its bits
            auto slot_of = [&](int c) {
                return static_cast<int>(o) +
                       __popc(known & (bit_of(static_cast<unsigned>(c)) - 1u));
            };
            const int n = q - x;
            if (n <= TC && x + TC - e0 <= ns) {
#pragma unroll
                for (int u = 0; u < TC; ++u)
                    if (u < n)
                        s_stage[staged(x + u - e0)] = u > 0 && cb[u] == cb[u - 1] ? kDup : slot_of(cb[u]);
            } else {
                // Runs past the stage, and rows with more entries in the
                // tile than columns (duplicates).
                int y = x;
                while (y < q) {
                    const int c = col(y);
                    const int y0 = y;
                    double s = g.val[y];
                    ++y;
                    while (y < q && col(y) == c) {
                        s += g.val[y];
                        ++y;
                    }
                    const int slot = slot_of(c);
                    g.values[slot] = s;
                    if (g.src_slot) {
                        for (int z = y0; z < y; ++z)
                            g.src_slot[z] = slot;
                        if (y - y0 > 1)
                            g.head->dups = 1u;
                    }
                }
                for (y = x; y < q && y - e0 < ns; ++y)
                    s_stage[staged(y - e0)] = kDone;
            }
            ++t;
            o += dense ? 32 : cnt;
            x = q;
        }
    }
    __syncthreads();
    for (int x0 = tid; x0 < ns; x0 += kLoads * kBuild) {
        int slot[kLoads];
        bool dup[kLoads];
        double v[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int x = x0 + u * kBuild;
            slot[u] = x < ns ? s_stage[staged(x)] : kDone;
            dup[u] = x + 1 < ns && s_stage[staged(x + 1)] == kDup;
            v[u] = slot[u] >= 0 ? g.val[e0 + x] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int x = x0 + u * kBuild;
            if (slot[u] >= 0) {
                if (dup[u]) {
                    g.head->dups = 1u;
                    for (int y = x + 1; y < ns && s_stage[staged(y)] == kDup; ++y) {
                        v[u] += g.val[e0 + y];
                        if (g.src_slot)
                            g.src_slot[e0 + y] = slot[u];
                    }
                }
                g.values[slot[u]] = v[u];
                if (g.src_slot)
                    g.src_slot[e0 + x] = slot[u];
            } else if (slot[u] == kOut && g.src_slot) {
                g.src_slot[e0 + x] = -1;
            }
        }
    }
}

// ---- long tile rows ---------------------------------------------------------
template <int TR>
__device__ __forceinline__ int row_entries(const BuildArgs &g, int64_t tr)
{
    int n = 0;
    for (int r = 0; r < TR; ++r) {
        const int64_t row = tr * TR + r;
        if (row < g.active_rows) {
            const int src = g.row_map ? g.row_map[row] : static_cast<int>(row);
            n += g.rp[src + 1] - g.rp[src];
        }
    }
    return n;
}

template <int TR>
__global__ __launch_bounds__(kThreads) void long_list_kernel(BuildArgs g, int *__restrict__ list)
{
    const int64_t tr = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (tr < g.R && row_entries<TR>(g, tr) > kLongRow * TR)
        list[atomicAdd(&g.head->n_long, 1u)] = static_cast<int>(tr);
}

// A workgroup per listed tile row, in windows of kLongWin tile columns that
// start at the row's next tile: every entry ORs its bit into its tile's mask
// in LDS, the window's nonempty tiles are numbered by a scan, and (FILL)
// every entry then finds its slot from the tile's offset and mask.
template <int TR, int TC, bool B, bool FILL>
__global__ __launch_bounds__(kThreads) void long_rows_kernel(BuildArgs g)
{
    constexpr int kPer = kLongWin / kThreads;
    __shared__ uint32_t s_mask[kLongWin];
    __shared__ int s_off[FILL ? kLongWin : 1];   // first slot of the tile, from the window's
    __shared__ int s_p[TR], s_end[TR], s_hi[TR];
    __shared__ unsigned long long s_w[3][kWaves];
    const int tid = threadIdx.x, w = tid / kWave;
    const int n_long = FILL && !g.head->fits ? 0 : static_cast<int>(g.head->n_long);
    for (int i = blockIdx.x; i < n_long; i += gridDim.x) {
        const int tr = g.long_rows[i];
        if (tid < TR) {
            const int64_t row = static_cast<int64_t>(tr) * TR + tid;
            int p = 0, end = 0;
            if (row < g.active_rows) {
                const int src = g.row_map ? g.row_map[row] : static_cast<int>(row);
                p = g.rp[src];
                end = g.rp[src + 1];
            }
            // First entry at or beyond active_cols.
            int lo = p, hi = end;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (g.ci[mid] < g.active_cols)
                    lo = mid + 1;
                else
                    hi = mid;
            }
            if (FILL && g.src_slot)
                for (int y = lo; y < end; ++y)
                    g.src_slot[y] = -1;
            s_p[tid] = p;
            s_end[tid] = lo;
        }
        long long o0 = 0;
        int t0 = 0;
        int run[kClassesUsed] = {};
        if constexpr (FILL) {
            t0 = g.tile_row_ptr[tr];
            if constexpr (B)
                for (int c = 0; c < kClassesUsed; ++c)
                    run[c] = g.groups[static_cast<int64_t>(kClassSlots) * tr + c];
            o0 = g.long_of[tr].first;
        }
        long long tiles = 0, payload = 0, ndense = 0;
        int cls[kClassesUsed] = {};
        for (int v = tid; v < kLongWin; v += kThreads)
            s_mask[v] = 0u;
        __syncthreads();
        for (;;) {
            int first = INT_MAX;
            for (int r = 0; r < TR; ++r)
                if (s_p[r] < s_end[r])
                    first = min(first, g.ci[s_p[r]] / TC);
            if (first == INT_MAX)
                break;   // the same in every thread
            const int64_t lim = (static_cast<int64_t>(first) + kLongWin) * TC;
            __syncthreads();   // s_p read by all
            if (tid < TR) {
                int lo = s_p[tid], hi = s_end[tid];
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (g.ci[mid] < lim)
                        lo = mid + 1;
                    else
                        hi = mid;
                }
                s_hi[tid] = lo;
            }
            __syncthreads();
            for (int r = 0; r < TR; ++r)
                for (int x = s_p[r] + tid; x < s_hi[r]; x += kThreads) {
                    const int c = g.ci[x];
                    const int lc = c % TC;
                    atomicOr(&s_mask[c / TC - first], 1u << (B ? lc * TR + r : r * TC + lc));
                }
            __syncthreads();
            // Thread v takes kPer consecutive tile columns.
            int nt = 0, pay = 0, nd = 0;
            unsigned long long cl = 0;   // 12 bits a class, at most kPer tiles
            for (int u = 0; u < kPer; ++u) {
                const uint32_t m = s_mask[tid * kPer + u];
                if (!m)
                    continue;
                const int cnt = __popc(m);
                const bool dense = cnt >= g.dense_threshold;
                ++nt;
                nd += dense ? 1 : 0;
                pay += dense ? 32 : cnt;
                if constexpr (B)
                    cl += 1ull << (kClassBits * mask_class(m));
            }
            // Scans of tiles and payload in one word, of the first four class
            // counts (at most kLongWin in a window, 16 bits each) in another,
            // of the last class and the dense tiles in a third.
            const unsigned long long two =
                (static_cast<unsigned long long>(nt) << 32) | static_cast<unsigned int>(pay);
            const unsigned long long it = wave_inclusive_scan(two);
            constexpr unsigned long long kF = (1ull << kClassBits) - 1ull;
            const unsigned long long ca = (cl & kF) | ((cl >> kClassBits & kF) << 16) |
                                          ((cl >> (2 * kClassBits) & kF) << 32) |
                                          ((cl >> (3 * kClassBits) & kF) << 48);
            const unsigned long long cz = (cl >> (4 * kClassBits)) |
                                          (static_cast<unsigned long long>(nd) << 32);
            const unsigned long long ia = wave_inclusive_scan(ca), iz = wave_inclusive_scan(cz);
            if (lane_id() == kWave - 1) {
                s_w[0][w] = it;
                s_w[1][w] = ia;
                s_w[2][w] = iz;
            }
            __syncthreads();
            unsigned long long before[3] = {0, 0, 0}, sum[3] = {0, 0, 0};
            for (int k = 0; k < kWaves; ++k)
                for (int z = 0; z < 3; ++z) {
                    before[z] += k < w ? s_w[z][k] : 0ull;
                    sum[z] += s_w[z][k];
                }
            if constexpr (FILL) {
                const unsigned long long et = before[0] + it - two;
                int t = t0 + static_cast<int>(tiles) + static_cast<int>(et >> 32);
                int off = static_cast<int>(et & 0xFFFFFFFFull);
                const unsigned long long ea = before[1] + ia - ca, ez = before[2] + iz - cz;
                int at[kClassesUsed];
                if constexpr (B) {
                    for (int c = 0; c < 4; ++c)
                        at[c] = run[c] + static_cast<int>(ea >> (16 * c) & 0xFFFFull);
                    at[4] = run[4] + static_cast<int>(ez & 0xFFFFFFFFull);
                }
                for (int u = 0; u < kPer; ++u) {
                    const int v = tid * kPer + u;
                    const uint32_t m = s_mask[v];
                    if (!m)
                        continue;
                    const int cnt = __popc(m);
                    const bool dense = cnt >= g.dense_threshold;
                    const long long o = o0 + payload + off;
                    s_off[v] = off;
                    int tm = t;
                    if constexpr (B) {
                        const int k = mask_class(m);
#pragma unroll
                        for (int c = 0; c < kClassesUsed; ++c)
                            if (c == k)
                                tm = at[c]++;
                    }
                    g.meta[tm] = tile_meta(first + v, m, o, dense);
                    g.tile_col_idx[t] = first + v;
                    g.masks[t] = m;
                    g.value_offsets[t] = static_cast<int>(o);
                    if (dense)
                        for (uint32_t z = ~m; z; z &= z - 1)
                            g.values[o + __builtin_ctz(z)] = 0.0;
                    ++t;
                    off += dense ? 32 : cnt;
                }
                __syncthreads();
                for (int r = 0; r < TR; ++r) {
                    const int p = s_p[r], hi = s_hi[r];
                    for (int x = p + tid; x < hi; x += kThreads) {
                        const int c = g.ci[x];
                        if (x > p && g.ci[x - 1] == c)
                            continue;   // its run's first entry sums it
                        double s = g.val[x];
                        int y = x + 1;
                        for (; y < hi && g.ci[y] == c; ++y)
                            s += g.val[y];
                        const uint32_t m = s_mask[c / TC - first];
                        const int lc = c % TC;
                        const int phys = B ? lc * TR + r : r * TC + lc;
                        const int cnt = __popc(m);
                        const int slot = static_cast<int>(o0 + payload) + s_off[c / TC - first] +
                                         payload_slot(m, cnt >= g.dense_threshold ? 32 : cnt, phys);
                        g.values[slot] = s;
                        if (g.src_slot) {
                            for (int z = x; z < y; ++z)
                                g.src_slot[z] = slot;
                            if (y - x > 1)
                                g.head->dups = 1u;
                        }
                    }
                }
                if constexpr (B) {
                    for (int c = 0; c < 4; ++c)
                        run[c] += static_cast<int>(sum[1] >> (16 * c) & 0xFFFFull);
                    run[4] += static_cast<int>(sum[2] & 0xFFFFFFFFull);
                }
            }
            tiles += static_cast<long long>(sum[0] >> 32);
            payload += static_cast<long long>(sum[0] & 0xFFFFFFFFull);
            ndense += static_cast<long long>(sum[2] >> 32);
            for (int c = 0; c < 4; ++c)
                cls[c] += static_cast<int>(sum[1] >> (16 * c) & 0xFFFFull);
            cls[4] += static_cast<int>(sum[2] & 0xFFFFFFFFull);
            __syncthreads();   // masks and offsets read by all
            for (int v = tid; v < kLongWin; v += kThreads)
                s_mask[v] = 0u;
            if (tid < TR)
                s_p[tid] = s_hi[tid];
            __syncthreads();
        }
        if constexpr (!FILL) {
            if (tid == 0) {
                LongRow lr;
                lr.tiles = static_cast<int>(tiles);
                lr.dense = static_cast<int>(ndense);
                lr.payload = payload;
                for (int c = 0; c < kClassesUsed; ++c)
                    lr.cls[c] = cls[c];
                g.long_of[tr] = lr;
            }
        }
        __syncthreads();   // s_p is reused by the next row
    }
}

__global__ void fill_slots_kernel(int *p, int64_t n, int v)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

// Columns a workgroup stages (a row map disables the staging).
int stage_columns(const DevCsr &src, bool row_map)
{
    if (row_map || src.rows <= 0)
        return 0;
    const double per = 1.1 * kBuild * static_cast<double>(src.nnz) / src.rows;
    const int cap = per >= kStageMax ? kStageMax : (static_cast<int>(per) + 63) / 64 * 64;
    return std::max(kBuild, cap);
}

template <int TR, int TC, bool B>
int run_build(const DevCsr &src, const int *row_map, int active_rows, int active_cols,
              int dense_threshold, DevTiles *out, BuildWork *w, int *src_slot,
              const DevTiles *pairs_of)
{
    hipStream_t s = ctx().stream;
    const int R = out->tile_row_count;
    const int64_t rows = static_cast<int64_t>(R) * TR;
    const int64_t blocks = std::max<int64_t>(1, (rows + kBuild - 1) / kBuild);
    const bool maybe_long = R > 0 && (src.max_row < 0 || src.max_row > kLongRow);
    static_assert(sizeof(BuildHead) % sizeof(unsigned long long) == 0, "head of whole words");
    constexpr int64_t kHeadWords = sizeof(BuildHead) / sizeof(unsigned long long);
    const int64_t words = kHeadWords + 2 * blocks;
    RTT_TRY(w->counters.ensure(static_cast<size_t>(words) * sizeof(unsigned long long)));
    RTT_TRY(w->host_totals.ensure(4 * sizeof(long long)));
    RTT_TRY(out->tile_row_ptr.ensure((static_cast<size_t>(R) + 1) * sizeof(int)));
    if (B)
        RTT_TRY(out->row_groups.ensure((static_cast<size_t>(R) * kClassSlots + 1) * sizeof(int)));
    BuildArgs g;
    g.R = R;
    g.active_rows = active_rows;
    g.active_cols = active_cols;
    g.rp = src.row_ptr.as<int>();
    g.ci = src.col_idx.as<int>();
    g.val = src.values.as<double>();
    g.row_map = row_map;
    g.dense_threshold = dense_threshold;
    g.stage = stage_columns(src, row_map != nullptr);
    g.head = w->counters.as<BuildHead>();
    g.look = w->counters.as<unsigned long long>() + kHeadWords;
    g.tile_row_ptr = out->tile_row_ptr.as<int>();
    g.groups = B ? out->row_groups.as<int>() : nullptr;
    g.src_slot = src_slot;
    long long *totals = w->host_totals.as<long long>();
    g.totals = totals;
    const size_t stage_bytes = static_cast<size_t>(staged(g.stage)) * sizeof(int);
    const unsigned long_blocks = static_cast<unsigned>(8 * (ctx().num_cus > 0 ? ctx().num_cus : 256));
    if (maybe_long) {
        RTT_TRY(w->long_rows.ensure(static_cast<size_t>(R) * sizeof(int)));
        RTT_TRY(w->long_of.ensure(static_cast<size_t>(R) * sizeof(LongRow)));
        g.long_rows = w->long_rows.as<int>();
        g.long_of = w->long_of.as<LongRow>();
    }
    if (B)
        RTT_TRY(out->pair_total.ensure(sizeof(unsigned long long)));
    for (int attempt = 0;; ++attempt) {
        DevBuf &meta = B ? out->records : out->meta;   // B: plane 0 of the records
        const size_t meta_size = B ? sizeof(BRecord) : sizeof(int4);
        g.cap_tiles = std::min({entries_held(out->tile_col_idx.bytes, sizeof(int), 0),
                                entries_held(out->masks.bytes, sizeof(uint32_t), 0),
                                entries_held(meta.bytes, meta_size, 0),
                                entries_held(out->value_offsets.bytes, sizeof(int), 1)});
        // One slot more than the payload: a zero (see DevTiles::values).
        g.cap_payload = entries_held(out->values.bytes, sizeof(double), 1);
        g.tile_col_idx = out->tile_col_idx.as<int>();
        g.masks = out->masks.as<uint32_t>();
        g.value_offsets = out->value_offsets.as<int>();
        g.values = out->values.as<double>();
        g.meta = meta.as<int4>();
        hipLaunchKernelGGL(build_init_kernel, dim3(blocks_for(words, kThreads)), dim3(kThreads), 0,
                           s, w->counters.as<unsigned long long>(), words,
                           B ? out->pair_total.as<unsigned long long>() : nullptr);
        if (maybe_long) {
            hipLaunchKernelGGL(long_list_kernel<TR>, dim3(blocks_for(R, kThreads)), dim3(kThreads),
                               0, s, g, w->long_rows.as<int>());
            hipLaunchKernelGGL((long_rows_kernel<TR, TC, B, false>), dim3(long_blocks),
                               dim3(kThreads), 0, s, g);
        }
        hipLaunchKernelGGL((tile_build_kernel<TR, TC, B>), dim3(static_cast<unsigned>(blocks)),
                           dim3(kBuild), stage_bytes, s, g);
        if (maybe_long)
            hipLaunchKernelGGL((long_rows_kernel<TR, TC, B, true>), dim3(long_blocks),
                               dim3(kThreads), 0, s, g);
        RTT_HIP(hipGetLastError());
        // Queued behind the build, before its totals are read: the extents
        // need B's row structure alone, which is complete either way.
        if (pairs_of)
            RTT_TRY(build_pair_extents(*pairs_of, out, &g.head->dups, totals + 3));
        RTT_HIP(hipStreamSynchronize(s));
        if (totals[0] > INT_MAX || totals[1] > INT_MAX)
            return fail(RTT_ERR_OVERFLOW,
                        "tile count %lld or payload %lld exceeds the int32 tile ABI", totals[0],
                        totals[1]);
        if (totals[0] <= g.cap_tiles && totals[1] <= g.cap_payload)
            break;
        if (attempt > 0)
            return fail(RTT_ERR_DEVICE, "tile build: the sizes changed between two launches");
        const size_t n = static_cast<size_t>(totals[0]);
        RTT_TRY(out->tile_col_idx.ensure(n * sizeof(int)));
        RTT_TRY(out->masks.ensure(n * sizeof(uint32_t)));
        RTT_TRY(out->value_offsets.ensure((n + 1) * sizeof(int)));
        RTT_TRY(out->values.ensure((static_cast<size_t>(totals[1]) + 1) * sizeof(double)));
        RTT_TRY(meta.ensure(std::max<size_t>(n, 1) * meta_size));
    }
    out->num_tiles = totals[0];
    out->payload = totals[1];
    out->dense = totals[2];
    out->sparse = totals[0] - totals[2];
    return RTT_OK;
}

} // namespace

int build_tiles(const DevCsr &src, const int *row_map, int active_rows, int active_cols,
                int logical_rows, int logical_cols, bool b_layout, int dense_threshold,
                DevTiles *out, BuildWork *w, const DevTiles *pairs_of, bool want_source_map)
{
    RTT_TRY(require_ctx());
    const int TR = b_layout ? kTileK : kTileM;
    const int TC = b_layout ? kTileN : kTileK;
    out->rows = logical_rows;
    out->cols = logical_cols;
    out->tile_rows = TR;
    out->tile_cols = TC;
    out->tile_row_count = (active_rows + TR - 1) / TR;
    out->tile_col_count = (active_cols + TC - 1) / TC;
    out->has_csc = false;
    out->arrays_ready = true;
    out->cols_ready = false;
    out->transpose_of = nullptr;
    out->rec_values_ready = !b_layout;
    hipStream_t s = ctx().stream;
    int *src_slot = nullptr;
    out->map_source_id = 0;
    out->map_nnz = 0;
    out->map_dups = false;
    if (want_source_map) {
        RTT_TRY(out->src_slot.ensure(static_cast<size_t>(src.nnz > 0 ? src.nnz : 1) * sizeof(int)));
        src_slot = out->src_slot.as<int>();
        // The build reaches every entry of the rows below active_rows.
        if (src.nnz > 0 && active_rows < src.rows)
            hipLaunchKernelGGL(fill_slots_kernel, dim3(blocks_for(src.nnz, kThreads)),
                               dim3(kThreads), 0, s, src_slot, src.nnz, -1);
        RTT_HIP(hipGetLastError());
    }
    if (b_layout)
        RTT_TRY((run_build<kTileK, kTileN, true>(src, row_map, active_rows, active_cols,
                                                 dense_threshold, out, w, src_slot, pairs_of)));
    else
        RTT_TRY((run_build<kTileM, kTileK, false>(src, row_map, active_rows, active_cols,
                                                  dense_threshold, out, w, src_slot, pairs_of)));
    if (want_source_map) {
        out->map_source_id = src.structure_id;
        out->map_nnz = src.nnz;
        out->map_dups = w->host_totals.as<long long>()[3] != 0;
    }
    return RTT_OK;
}

} // namespace rtt
