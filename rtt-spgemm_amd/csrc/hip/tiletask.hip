// Tile-pair numeric path: C's values computed per 8x8 C tile with matrix
// cores, after the symbolic pass has written C's whole structure.
//
// A C tile (I, J) is the sum over the K where A's tile row I and B's tile
// column J both hold a tile of A(I,K) * B(K,J), an 8x4 by 4x8 product.  This
// is the reference's C8 task (a K-merge of A row I with B column J, then one
// tensor-core product per matched K: src/dmma_spgemm.h:4164-4300,
// 4307-4410); here one gfx950 v_mfma_f64_4x4x4f64 computes a whole pair --
// its four 4x4x4 blocks are the four 4x4 quarters of the 8x8 C tile -- with
// every lane holding one A entry, one B entry and one C entry.  Each C tile
// keeps its running sum in one register per lane and takes its pairs in
// increasing K, so C's values do not depend on scheduling: two calls give the
// same bits.
//
// Work unit: one wave per C tile row, or per part of its C tiles when there
// are too few rows for the chip, in the launch's own order (chunks of
// consecutive rows dealt to the XCDs, so that they work through one window of
// the rows together).  Persistent waves that took rows from eight queue heads
// in one cache line spent 10 ns an atomic on them, 40000 in a launch of any
// size: 0.2 ms of a 2000-row product's 0.23 ms.
//
// Pairs are found from A's side, up to 64 A tiles at a time: every tile (K,
// J) of the B rows those A tiles select is one lane's, which finds J among
// up to 64 C tiles of the row and sets the A tile's bit in that C tile's
// 64-bit word.  The words give every pair its place: C tiles in order, within
// one the number of lower bits (its smaller K).  The pairs are written there
// into an LDS list and run by P::run, which keeps a batch of operand loads in
// flight behind the products and puts each C tile out when its pairs end.
// Every B tile enumerated belongs to a pair (or to no C tile at all), and B
// needs no column structure; the search of A's keys for every entry of every
// B column that this replaces, with the radix sort that made the columns,
// took the block-FEM 500k step 1.5 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <vector>

#include "core.hpp"

namespace rtt {

namespace {

constexpr int kTThreads = 128;
constexpr int kTWaves = kTThreads / kWave;
constexpr int kAVals = 384;     // A payload values of a row staged in LDS
constexpr int kPairCap = 128;   // pairs a wave buffers before running them
constexpr int kBatch = 8;       // pairs whose operand loads are issued together
constexpr int kOutVals = 128;   // C values a wave stages before it stores them
static_assert(kOutVals >= 64, "a C tile fits the stage");
constexpr int kEnumRounds = 2;  // rounds of 64 B tiles whose metas are loaded together (and
                                // kept, when they are all there is)
constexpr int kXcdChunk = 4;    // workgroups of consecutive units dealt to an XCD at a time
constexpr int kPairShards = 256;   // counters of the pairs multiplied, a 128-byte line each (one
constexpr int kShardStride = 16;   // counter would take an atomic from every wave)
constexpr int kWideLeast = 32, kWideMost = 512;   // C tiles of a wide row's unit
constexpr int kMaxParts = 4;    // most units a tile row is cut into
constexpr int kPairWords = kPairCap / 64;
constexpr int kPad = 2 * kBatch;   // pairs of zeros past a list: the batch that its last pairs
                                   // share, and the batch loaded ahead of that one
static_assert(kPairCap % 64 == 0 && kPairWords == 2, "words of the end bits");
static_assert(kPairCap >= kWave, "a C tile has at most 64 pairs per group of A tiles");

struct TileTask {
    int rows;                            // tile rows of A and C
    const int *__restrict__ a_trp;       // A tile row pointer
    const int4 *__restrict__ a_meta;     // {K, mask, per-k bytes, offset | dense}
    const double *__restrict__ a_vals;   // A payload, each tile row-major
    const int4 *__restrict__ a_brange;   // per A tile: {first B tile of row K, -, tiles}
    const int4 *__restrict__ b_meta;     // B tiles row by row: {J, mask, bytes, offset | dense}
    const int *__restrict__ b_groups;    // start of each (row, class) run of B
    const double *__restrict__ b_vals;   // B payload, each tile column-major
    uint32_t a_zero, b_zero;             // slots past the payloads that hold 0.0
    const int *__restrict__ b_cptr;      // tail only: B tile column pointer
    const int4 *__restrict__ b_cent;     // tail only: {K, mask, per-k bytes, offset | dense}
    const int64_t *__restrict__ c_ptr;   // C tile row pointer
    const int *__restrict__ c_col;
    const unsigned long long *__restrict__ c_mask;
    const int64_t *__restrict__ c_off;   // value offset of each C tile
    double *__restrict__ c_val;
    const int *__restrict__ a_row_off;   // A payload offset of each tile row
    float fill;                          // rows taken: A tiles' mean stored values >= fill
    int parts;                           // units per tile row
    unsigned long long *__restrict__ mfma_pairs;   // pairs multiplied (one MFMA each), kPairShards
                                                   // counters; null: not counted
    // Heavy C tiles split into chunks (bit t of heavy: C tile t), used when
    // tail->enabled; null when no admission ran.
    const uint32_t *__restrict__ heavy;
    const struct TailState *__restrict__ tail;
};

// Tail queue (the reference's heavy-task split, src/dmma_spgemm.h:2534-2776,
// 4902-5254, 6003-6049): C tiles whose K-merge costs more than the admission
// threshold are split into chunks of their B-column range; each chunk's
// partial tile goes to a workspace slot, and a reduction sums the chunks of a
// tile in chunk order, so the split tiles are as reproducible as the rest.
struct TailRecord {          // DmmaTailRecord {id, scans, matches, chunks} + the tile row
    long long task;
    int row;
    int scans;
    int matches;
    int chunks;
};
struct TailState {
    unsigned int count;              // records admitted (may exceed capacity)
    int overflow;                    // an admission found the record list full
    unsigned long long chunks;       // chunks of the admitted records
    int reason;                      // gate decision (rtt_stats.tail_reason)
    int enabled;                     // 1: heavy tiles take the chunk kernels
    int chunk_head;                  // work queue of the chunk kernel
    int reduce_head;                 // work queue of the reduction
};

constexpr uint32_t kDense = 0x80000000u;
constexpr int kTailNone = 4;   // gate reason: no heavy tile

// A tile in the pair list is {mask, offset} with a full mask for a dense tile
// (which holds all 32 slots, absent entries as zeros): entry `phys` then lies
// at offset + popc(mask & below), below = (1 << phys) - 1, whatever the kind.
__device__ __forceinline__ uint32_t list_mask(int mask, int offw)
{
    return offw < 0 ? 0xFFFFFFFFu : static_cast<uint32_t>(mask);
}

// Slot of an entry, `zero` (a slot that holds 0.0) when the mask lacks it, so
// that the load is unconditional and its value needs no select.
__device__ __forceinline__ uint32_t entry_slot(uint32_t mask, uint32_t off, int phys,
                                               uint32_t below, uint32_t zero)
{
    const uint32_t at = off + __popc(mask & below);
    return (mask >> phys) & 1u ? at : zero;
}

__device__ __forceinline__ int read_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// Value of lane ^ 8 (a rotation by 8 within rows of 16 lanes).
__device__ __forceinline__ double from_lane_xor8(double v)
{
    const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(v));
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), 0x128, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), 0x128, 0xf, 0xf, false);
    return __longlong_as_double(static_cast<long long>(
        (static_cast<unsigned long long>(static_cast<uint32_t>(hi)) << 32) |
        static_cast<uint32_t>(lo)));
}

// Lane roles of v_mfma_f64_4x4x4f64 (four independent 4x4x4 blocks; block b,
// measured on gfx950): A[b][i][k] in lane i + 4b + 16k, B[b][k][j] in lane
// j + 4b + 16k, D[b][i][j] in lane j + 4b + 16i.  Block b = 2h + v multiplies
// rows 4h..4h+3 of the A tile by columns 4v..4v+3 of the B tile, so D's four
// blocks are the quarters of the 8x8 C tile.
struct LaneRoles {
    int a_phys;   // A tile bit r*4+k this lane supplies
    int b_phys;   // B tile bit c*4+k
    int c_bit;    // C tile bit r*8+c this lane accumulates
    bool lower;   // rows 4..7 of the A tile (h = 1)
    uint32_t a_below, b_below;   // (1 << phys) - 1
    __device__ LaneRoles(int lane)
    {
        const int blk = (lane >> 2) & 3, lo = lane & 3, hi = lane >> 4;
        lower = (blk >> 1) != 0;
        a_phys = ((blk >> 1) * 4 + lo) * 4 + hi;
        b_phys = ((blk & 1) * 4 + lo) * 4 + hi;
        c_bit = ((blk >> 1) * 4 + hi) * 8 + (blk & 1) * 4 + lo;
        a_below = (1u << a_phys) - 1u;
        b_below = (1u << b_phys) - 1u;
    }
};

// 64-bit value held by lane `l` (l uniform across the wave).
__device__ __forceinline__ unsigned long long read_lane64(unsigned long long v, int l)
{
    return (static_cast<unsigned long long>(static_cast<uint32_t>(
                read_lane(static_cast<int>(v >> 32), l))) << 32) |
           static_cast<uint32_t>(read_lane(static_cast<int>(v), l));
}

// ---------------------------------------------------------------------------
// Plain FP64: one v_mfma_f64_4x4x4f64 per pair into a running sum of one
// register per lane.  A batch of kBatch pairs (which may span C tiles) has its
// operand loads issued together.
// ---------------------------------------------------------------------------
struct Fp64Product {
    struct Lane {
        LaneRoles roles;
        __device__ Lane(int lane) : roles(lane) {}
    };
    struct Acc {
        double v = 0.0;
    };
    // Waves per SIMD the tile kernel is compiled for (94 VGPRs); its LDS, 17 KB a
    // workgroup of two waves, lets nine workgroups on a CU, 4.5 waves per SIMD.
    // The waves wait for loads more than half of their time.  Block-FEM
    // 500k, 2.16e7 pairs: 1.69 ms (6.5 TFLOP/s on the matrix cores); 1.80 at
    // four waves with 512 A values staged and four enumeration rounds kept,
    // 1.90 with twice the output stage, 1.89 at six waves, batches of four and
    // spills; 2.17 before the output was staged, 2.95 with the search of B's
    // columns.  B tiles loaded whole and spread by lane permutes, a third of
    // the cache accesses, were slower (2.01 against 1.90).
    static constexpr int kOccupancy = 5;
    static constexpr int kWideOccupancy = 4;

    // C values on their way out: `count` values from `base` on wait in `vals`.
    // The C tiles of a row lie one behind the other, so they leave together,
    // in whole lines.  Stored tile by tile, every batch waited for the stores
    // of the one before: loads and stores come back in one order, and a wait
    // for operands cannot tell how many stores are behind them (8000 cycles a
    // batch of eight pairs): block-FEM 500k 2.17 -> 1.80 ms.
    struct Out {
        double *vals;
        long long base;
        int count;
    };
    static __device__ __forceinline__ void flush(const TileTask &g, Out &out)
    {
        wave_sync();
        for (int i = lane_id(); i < out.count; i += kWave)
            g.c_val[out.base + i] = out.vals[i];
        wave_sync();
        out.count = 0;
    }

    static __device__ __forceinline__ void put(const TileTask &g, const Lane &ln, int c_local,
                                               unsigned long long cm, long long co, const Acc &acc,
                                               Out &out)
    {
        const unsigned long long m = read_lane64(cm, c_local);
        const long long off = static_cast<long long>(read_lane64(static_cast<unsigned long long>(co), c_local));
        const int n = __popcll(m);
        if (off != out.base + out.count || out.count + n > kOutVals) {
            flush(g, out);
            out.base = off;
        }
        const int bit = ln.roles.c_bit;
        if ((m >> bit) & 1ull)
            out.vals[out.count + __popcll(m & ((1ull << bit) - 1ull))] = acc.v;
        out.count += n;
    }

    // Lane's entry of a C tile stored earlier.
    __device__ static double load(const TileTask &g, const Lane &ln, int c_local,
                                  unsigned long long cm, long long co)
    {
        const unsigned long long m = read_lane64(cm, c_local);
        const long long off = static_cast<long long>(read_lane64(static_cast<unsigned long long>(co), c_local));
        const int bit = ln.roles.c_bit;
        return (m >> bit) & 1ull ? g.c_val[off + __popcll(m & ((1ull << bit) - 1ull))] : 0.0;
    }

    // Lane's entry of a finished tile into a 64-slot partial (bit order).
    __device__ static void dump(const Lane &ln, const Acc &acc, double *slot64)
    {
        slot64[ln.roles.c_bit] = acc.v;
    }

    // B entries of listed pairs [p0, p0 + kBatch).  A B entry is needed by two
    // lanes, l and l ^ 8 (the two halves of the A tile's rows), so of every
    // two pairs one half's lanes load the first and the other's the second,
    // and the products take the partner's by a DPP move: half the loads, and
    // twice the pairs in flight per register.
    static __device__ __forceinline__ void load_b(const TileTask &g, const Lane &ln, const int4 *pm,
                                                  int p0, double (&bv)[kBatch / 2])
    {
        const int4 *p = pm + p0 + (ln.roles.lower ? 1 : 0);
#pragma unroll
        for (int i = 0; i < kBatch / 2; ++i) {
            const int2 m = reinterpret_cast<const int2 *>(p + 2 * i)[1];
            bv[i] = g.b_vals[entry_slot(static_cast<uint32_t>(m.x), static_cast<uint32_t>(m.y),
                                        ln.roles.b_phys, ln.roles.b_below, g.b_zero)];
        }
    }

    // Products of listed pairs [0, n), padded to kBatch past the end (see
    // kPad).  The B loads of the next batch are issued before the products
    // of the current one.  after(p0, i) runs after the product of pair p0 + i.
    template <class After>
    static __device__ __forceinline__ void products(const TileTask &g, const Lane &ln,
                                                    const double *a_vals, uint32_t a_zero,
                                                    const int4 *pm, int n, Acc &acc, After &&after)
    {
        double bv[kBatch / 2];
        load_b(g, ln, pm, 0, bv);
        for (int p0 = 0; p0 < n; p0 += kBatch) {
            double bn[kBatch / 2];
            load_b(g, ln, pm, p0 + kBatch, bn);
            double av[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int2 m = reinterpret_cast<const int2 *>(pm + p0 + i)[0];
                av[i] = a_vals[entry_slot(static_cast<uint32_t>(m.x), static_cast<uint32_t>(m.y),
                                          ln.roles.a_phys, ln.roles.a_below, a_zero)];
            }
#pragma unroll
            for (int i = 0; i < kBatch; i += 2) {
                const double own = bv[i / 2], other = from_lane_xor8(own);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const double b = ln.roles.lower == (u == 1) ? own : other;
                    acc.v = __builtin_amdgcn_mfma_f64_4x4x4f64(av[i + u], b, acc.v, 0, 0, 0);
                    after(p0, i + u);
                }
            }
#pragma unroll
            for (int i = 0; i < kBatch / 2; ++i)
                bv[i] = bn[i];
        }
    }

    // Runs a list of whole C tiles in order, putting each out after its last pair.
    // cnt: pairs of the lane's C tile; ends: bit p set when a tile ends with
    // pair p (all of them in scalar registers, off the vector units); live:
    // the listed tiles.  A C tile in `started` has its sum over earlier A
    // tiles in C already.  (Products of the padding follow the last store.)
    static __device__ __forceinline__ void run(const TileTask &g, const Lane &ln, const double *a_vals,
                               uint32_t a_zero, const int4 *pm, int n, int,
                               const unsigned long long (&ends)[kPairWords],
                               unsigned long long live, unsigned long long started,
                               unsigned long long cm, long long co, double *out_vals)
    {
        Acc acc;
        Out out = {out_vals, 0, 0};
        auto begin = [&]() {
            const int t = __builtin_ctzll(live);
            acc.v = (started >> t) & 1ull ? load(g, ln, t, cm, co) : 0.0;
        };
        if (started)
            begin();
        unsigned long long word = 0;
        products(g, ln, a_vals, a_zero, pm, n, acc, [&](int p0, int i) {
            if (i == 0)
                word = (p0 < 64 ? ends[0] : ends[1]) >> (p0 & 63);
            if ((word >> i) & 1ull) {
                put(g, ln, __builtin_ctzll(live), cm, co, acc, out);
                live &= live - 1;
                acc.v = 0.0;
                if (started && live)
                    begin();
            }
        });
        flush(g, out);
    }

    // Adds listed pairs [0, n) to acc.
    static __device__ __forceinline__ void add(const TileTask &g, const Lane &ln, const double *a_vals,
                               uint32_t a_zero, const int4 *pm, int n, Acc &acc)
    {
        products(g, ln, a_vals, a_zero, pm, n, acc, [](int, int) {});
    }
};

// ---------------------------------------------------------------------------
// Split precision (Ozaki scheme, error-free slicing): for a batch of at most
// eight pairs of one C tile, every A entry is written relative to the largest
// exponent E_r of its tile row r over the batch as a 64-bit fixed-point
// fraction, sign * sum_e q_e 2^(E_r - 8(e+1)) with eight integer slices
// q_e in [0, 255] (the bytes of the fraction), and every B entry likewise
// relative to its tile column's largest exponent.  Slices are exact in
// BF16, and a product of two slices is exact in FP32.  All 64 slice pairs
// are kept; grouped by d = e + f (0..14), the sums
//   P_d[r][c] = sum_{k, e+f=d} qa_e[r][k] qb_f[k][c]
// have at most 8 x 4 terms of at most 255^2 per pair, so eight pairs' sums
// stay below 2^24 and the FP32 accumulation of v_mfma_f32_16x16x32_bf16 is
// exact.  The reduction dimension of one instruction is 32 = (k, slot x):
// lane group k holds eight slots of a(r, k), and B has in slot x of output
// column c + 8h the slice qb_{D-x} (zero outside 0..7), D = 3 + 2t + h.  Row r
// of the A operand has qa_x in slot x, which gives P_D; row r + 8 has
// qa_{x-4} for t = 0, 1, which gives P_{D-4}, and qa_{x+4} for t = 2, 3, which
// gives P_{D+4} (the slices those shifts push out meet no slice of B).  So
// four instructions give every P_d, -1..14, once, P_{-1} = 0.  With the
// slices unshifted and rows 8..15 empty it took eight, with twice the
// registers (two waves per SIMD) and FP64 work for the sums, four outputs in
// a quarter of the lanes instead of one in each, and fractions by 64-bit
// shifts: 772 vector instructions a C tile of 3.2 pairs.  Block-FEM 50k, 2.15e6
// pairs: 1.31 -> 0.70 ms.
// Each batch is recombined in FP64 on the GPU,
//   C[r][c] += 2^(E_r + E_c) sum_d P_d 2^(-8(d+2)),
// and batches and C tiles accumulate in FP64.  The only approximation is the
// truncation of every operand 64 bits below its row (column) maximum, a
// relative error of at most 2^-63 of that maximum per entry.  A batch whose
// A rows or B columns span more than kSpreadBits binades (where the smallest
// entries would keep fewer than 43 bits) runs on the FP64 matrix cores
// instead, so every product keeps a relative error below 2^-42 and the
// forward error of C stays below about 2^-41 sum |a||b| whatever the data.
// Lane roles of v_mfma_f32_16x16x32_bf16 (measured on gfx950): A[i][k'] in
// lane i + 16(k' >> 3), element k' & 7; B[k'][j] in lane j + 16(k' >> 3),
// element k' & 7; D[i][j] in lane j + 16(i >> 2), element i & 3.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSplitBatch = 8;   // pairs whose slice sums stay exact in FP32

// A batch whose A row (B column) exponents span more than this many binades
// is multiplied on the FP64 matrix cores instead: its smallest entries would
// keep fewer than 64 - 1 - kSpreadBits = 43 bits of the slices.
constexpr int kSpreadBits = 20;

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Biased exponent of x in the low half (subnormals count as 1), and 0x7FF
// minus it in the high half, zeros for a zero: the larger of each gives both
// extremes.
__device__ __forceinline__ u16x2 extremes(double x)
{
    const uint32_t hi = static_cast<uint32_t>(__double2hiint(x));
    const int e = max(static_cast<int>((hi >> 20) & 0x7FFu), 1);
    const uint32_t w = x != 0.0 ? static_cast<uint32_t>((0x7FF << 16) - __mul24(e, 0xFFFF)) : 0u;
    return __builtin_bit_cast(u16x2, w);
}

// 64-bit fixed-point fraction of |x| / 2^(emax - 1022), floor(|x| 2^(64 -
// (emax - 1022))), high word in y.  emax is at least x's exponent and, unless
// x is zero, at most kSpreadBits above it.
__device__ __forceinline__ uint2 fixed_fraction(double x, int emax)
{
    const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(x));
    const uint32_t hi = static_cast<uint32_t>(b >> 32), lo = static_cast<uint32_t>(b);
    const uint32_t ex = (hi >> 20) & 0x7FFu;
    const uint32_t mh = (hi & 0xFFFFFu) | (min(ex, 1u) << 20);   // |x| = {mh, lo} 2^(ex - 1075)
    const uint32_t d = static_cast<uint32_t>(emax) - max(ex, 1u);
    const uint32_t h1 = __builtin_amdgcn_alignbit(mh, lo, 32 - 11);
    return make_uint2(__builtin_amdgcn_alignbit(h1, lo << 11, d), h1 >> (d & 31u));
}

// Slices (bytes) i of x and j of y, the first in the low half.
__device__ __forceinline__ uint32_t slices(uint32_t x, int i, uint32_t y, int j)
{
    const uint32_t fx = __float_as_uint(static_cast<float>((x >> (8 * i)) & 0xFFu));
    const uint32_t fy = __float_as_uint(static_cast<float>((y >> (8 * j)) & 0xFFu));
    return __builtin_amdgcn_perm(fy, fx, 0x07060302u);
}


struct SplitProduct {
    struct Lane {
        int a_phys;      // A tile bit this lane supplies
        bool high;       // its A operand row is 8..15: shifted slices
        int b_phys;      // B tile bit
        int h;           // output column half: D = 3 + 2t + h
        uint32_t b_low, b_mid, b_top;   // byte selectors: B's slices, one byte up for h = 1
        int c_bit;       // C tile bit of this lane's output
        int d0;          // d of its sums at t = 0, 1 (2 apart); d2: at t = 2, 3
        int d2;
        LaneRoles f64;   // roles in the FP64 fallback (v_mfma_f64_4x4x4f64)
        int f64_lane;    // lane whose FP64 entry is this lane's output
        __device__ Lane(int lane) : f64(lane)
        {
            const int i = lane & 15, k = lane >> 4;
            high = i >= 8;
            a_phys = (i & 7) * 4 + k;
            b_phys = (lane & 7) * 4 + k;
            h = (lane >> 3) & 1;
            b_low = h ? 0x0201000Cu : 0x03020100u;
            b_mid = h ? 0x06050403u : 0x07060504u;
            b_top = h ? 0x0C0C0C07u : 0x0C0C0C0Cu;
            // Outputs before the lanes' sums are shared out: rows 4 (k & 1) +
            // 0..3, those of the A operand's rows 8..15 for k >= 2.
            d0 = (k < 2 ? 3 : -1) + h;
            d2 = (k < 2 ? 7 : 11) + h;
            const int r = 4 * (k & 1) + (k & 2) + h, c = lane & 7;
            c_bit = r * 8 + c;
            f64_lane = (c & 3) + 4 * (((r >> 2) << 1) | (c >> 2)) + 16 * (r & 3);
        }
    };
    struct Acc {
        double v = 0.0;
        double f64 = 0.0;   // FP64-fallback partial, v_mfma_f64_4x4x4f64 layout
    };
    // 144 VGPRs, three waves per SIMD; held to four it spills 30 of them for 5 %.
    // Loading the next batch's B entries before the current one is worked on
    // was no faster: vector instructions take 80 % of its cycles.
    static constexpr int kOccupancy = 3;
    static constexpr int kWideOccupancy = 3;

    // Lane's output with the FP64-fallback partial added (every lane takes part
    // in the shuffle).
    __device__ static double finish(const Lane &ln, const Acc &acc)
    {
        return acc.v + __shfl(acc.f64, ln.f64_lane, kWave);
    }

    __device__ static void store(const TileTask &g, const Lane &ln, int c_local,
                                 unsigned long long cm, long long co, const Acc &acc)
    {
        const unsigned long long m = read_lane64(cm, c_local);
        const long long off = static_cast<long long>(read_lane64(static_cast<unsigned long long>(co), c_local));
        const double out = finish(ln, acc);
        if ((m >> ln.c_bit) & 1ull)
            g.c_val[off + __popcll(m & ((1ull << ln.c_bit) - 1ull))] = out;
    }

    __device__ static void dump(const Lane &ln, const Acc &acc, double *slot64)
    {
        slot64[ln.c_bit] = finish(ln, acc);
    }

    // The larger of each half over the four k of a row (column): lanes x, x +
    // 16, x + 32, x + 48.
    __device__ static u16x2 over_k(u16x2 v)
    {
        const uint32_t w = __builtin_bit_cast(uint32_t, v);
        const auto r = __builtin_amdgcn_permlane32_swap(w, w, false, false);
        const u16x2 m = __builtin_elementwise_max(__builtin_bit_cast(u16x2, static_cast<uint32_t>(r[0])),
                                                  __builtin_bit_cast(u16x2, static_cast<uint32_t>(r[1])));
        const uint32_t x = __builtin_bit_cast(uint32_t, m);
        const auto q = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return __builtin_elementwise_max(__builtin_bit_cast(u16x2, static_cast<uint32_t>(q[0])),
                                         __builtin_bit_cast(u16x2, static_cast<uint32_t>(q[1])));
    }

    __device__ static bool wide_spread(u16x2 e)
    {
        return e.y != 0 && e.x - (0x7FF - e.y) > kSpreadBits;
    }

    // Lanes below 32: a + a of lane + 32; the others: b + b of lane - 32.
    __device__ static double halves_sum(double a, double b)
    {
        const unsigned long long ua = static_cast<unsigned long long>(__double_as_longlong(a)),
                                 ub = static_cast<unsigned long long>(__double_as_longlong(b));
        const auto lo = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(ua),
                                                         static_cast<uint32_t>(ub), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(
            static_cast<uint32_t>(ua >> 32), static_cast<uint32_t>(ub >> 32), false, false);
        auto word = [](uint32_t h, uint32_t l) {
            return __longlong_as_double(
                static_cast<long long>((static_cast<unsigned long long>(h) << 32) | l));
        };
        return word(hi[0], lo[0]) + word(hi[1], lo[1]);
    }

    // 2^(-8 (d + 2))
    __device__ static double slice_weight(int d)
    {
        return __longlong_as_double(static_cast<long long>(1023 - 8 * (d + 2)) << 52);
    }

    __device__ static double entry(const double *vals, int mask, int off, int phys, uint32_t zero)
    {
        return vals[entry_slot(static_cast<uint32_t>(mask), static_cast<uint32_t>(off), phys,
                               (1u << phys) - 1u, zero)];
    }

    // Pairs [p0, p0 + n) of one C tile, n <= kSplitBatch, added into acc.
    __device__ static void batch(const TileTask &g, const Lane &ln, const double *a_vals,
                                 uint32_t a_zero, const int4 *pm, int p0, int n, Acc &acc)
    {
        double av[kSplitBatch], bv[kSplitBatch];
#pragma unroll
        for (int i = 0; i < kSplitBatch; ++i) {
            if (i >= n)
                break;
            const int4 m = pm[p0 + i];
            av[i] = entry(a_vals, m.x, m.y, ln.a_phys, a_zero);
            bv[i] = entry(g.b_vals, m.z, m.w, ln.b_phys, g.b_zero);
        }
        u16x2 xa = {0, 0}, xb = {0, 0};
#pragma unroll
        for (int i = 0; i < kSplitBatch; ++i) {
            if (i >= n)
                break;
            xa = __builtin_elementwise_max(xa, extremes(av[i]));
            xb = __builtin_elementwise_max(xb, extremes(bv[i]));
        }
        xa = over_k(xa);
        xb = over_k(xb);
        if (__ballot(wide_spread(xa) || wide_spread(xb))) {
            // Too wide a spread for the slices: these pairs on the FP64 cores.
#pragma unroll
            for (int i = 0; i < kSplitBatch; ++i) {
                if (i >= n)
                    break;
                const int4 m = pm[p0 + i];
                const double a = entry(a_vals, m.x, m.y, ln.f64.a_phys, a_zero);
                const double b = entry(g.b_vals, m.z, m.w, ln.f64.b_phys, g.b_zero);
                acc.f64 = __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, acc.f64, 0, 0, 0);
            }
            return;
        }
        const int ea = max(static_cast<int>(xa.x), 1), eb = max(static_cast<int>(xb.x), 1);
        f32x4 acc_t[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            acc_t[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kSplitBatch; ++i) {
            if (i >= n)
                break;
            // A's slices, most significant first, two a word.
            const uint2 fa = fixed_fraction(av[i], ea);
            const uint32_t asg = av[i] < 0.0 ? 0x80008000u : 0u;
            const uint32_t a0 = slices(fa.y, 3, fa.y, 2) | asg, a1 = slices(fa.y, 1, fa.y, 0) | asg,
                           a2 = slices(fa.x, 3, fa.x, 2) | asg, a3 = slices(fa.x, 1, fa.x, 0) | asg;
            const u32x4 up = ln.high ? u32x4{0u, 0u, a0, a1} : u32x4{a0, a1, a2, a3};
            const u32x4 down = ln.high ? u32x4{a2, a3, 0u, 0u} : u32x4{a0, a1, a2, a3};
            // B's slices, least significant first (one slot later for h = 1),
            // two a word: instruction t reads four words from word 3 - t.
            const uint2 fb = fixed_fraction(bv[i], eb);
            const uint32_t blo = __builtin_amdgcn_perm(fb.y, fb.x, ln.b_low);
            const uint32_t bhi = __builtin_amdgcn_perm(fb.y, fb.x, ln.b_mid);
            const uint32_t last = __builtin_amdgcn_perm(fb.y, fb.x, ln.b_top);
            const uint32_t bsg = bv[i] < 0.0 ? 0x80008000u : 0u;
            const uint32_t w[7] = {0u,
                                   slices(blo, 0, blo, 1) | bsg,
                                   slices(blo, 2, blo, 3) | bsg,
                                   slices(bhi, 0, bhi, 1) | bsg,
                                   slices(bhi, 2, bhi, 3) | bsg,
                                   (__float_as_uint(static_cast<float>(last & 0xFFu)) >> 16) | bsg,
                                   0u};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const u32x4 bw = {w[3 - t], w[4 - t], w[5 - t], w[6 - t]};
                acc_t[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, t < 2 ? up : down), __builtin_bit_cast(bf16x8, bw),
                    acc_t[t], 0, 0, 0);
            }
        }
        // Recombination in FP64.  A lane has, for four rows, the P_d of d0, d0
        // + 2, d2 and d2 + 2 of one column; the others' lie in the lanes 8 and
        // 32 away, so each lane ends with one of the four rows.
        const double w0 = slice_weight(ln.d0), w1 = slice_weight(ln.d0 + 2),
                     w2 = slice_weight(ln.d2), w3 = slice_weight(ln.d2 + 2);
        double sum[4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
            sum[v] = fma(static_cast<double>(acc_t[0][v]), w0,
                         fma(static_cast<double>(acc_t[1][v]), w1,
                             fma(static_cast<double>(acc_t[2][v]), w2,
                                 static_cast<double>(acc_t[3][v]) * w3)));
        const double s0 = halves_sum(sum[0], sum[2]), s1 = halves_sum(sum[1], sum[3]);
        const double out = (ln.h ? s1 : s0) + from_lane_xor8(ln.h ? s0 : s1);
        const int erow = __shfl(ea, ln.c_bit >> 3, kWave);
        acc.v += ldexp(out, erow + eb - 2 * 1022);
    }

    // Lane's output of a C tile as store() left it.
    __device__ static void load(const TileTask &g, const Lane &ln, int c_local,
                                unsigned long long cm, long long co, Acc &acc)
    {
        const unsigned long long m = read_lane64(cm, c_local);
        const long long off = static_cast<long long>(read_lane64(static_cast<unsigned long long>(co), c_local));
        if ((m >> ln.c_bit) & 1ull)
            acc.v = g.c_val[off + __popcll(m & ((1ull << ln.c_bit) - 1ull))];
    }

    static __device__ __forceinline__ void run(const TileTask &g, const Lane &ln, const double *a_vals,
                               uint32_t a_zero, const int4 *pm, int, int cnt,
                               const unsigned long long (&)[kPairWords], unsigned long long live,
                               unsigned long long started, unsigned long long cm, long long co,
                               double *)
    {
        for (int p = 0; live; live &= live - 1) {
            const int t = __builtin_ctzll(live);
            const int end = p + read_lane(cnt, t);
            Acc acc;
            if ((started >> t) & 1ull)
                load(g, ln, t, cm, co, acc);
            for (; p < end; p += kSplitBatch)
                batch(g, ln, a_vals, a_zero, pm, p, min(kSplitBatch, end - p), acc);
            p = end;
            store(g, ln, t, cm, co, acc);
        }
    }

    static __device__ __forceinline__ void add(const TileTask &g, const Lane &ln, const double *a_vals,
                               uint32_t a_zero, const int4 *pm, int n, Acc &acc)
    {
        for (int p = 0; p < n; p += kSplitBatch)
            batch(g, ln, a_vals, a_zero, pm, p, min(kSplitBatch, n - p), acc);
    }
};

// A wave's LDS.
struct WaveStage {
    double av[kAVals + 2];            // A row's payload, when it fits; then 0.0
    int4 pm[kPairCap + kPad];         // {A mask, A offset, B mask, B offset}
    double out[kOutVals];             // C values on their way out
    unsigned long long word[kWave];   // per C tile: its A tiles
    unsigned long long ends[kPairWords + 1];   // bit p: a C tile ends with pair p
    int2 am[kWave];                   // per A tile: {mask, offset}
    int start[kWave];                 // per A tile: its first B tile in the enumeration
    int b0[kWave];                    // per A tile: first B tile minus start
    int cj[kWave];                    // columns of the C tiles
    int base[kWave];                  // per C tile: its first pair
};

// C tiles [c0, c1) of tile row `row`, up to 64 at a time, over A's tiles, up
// to 64 at a time.  a_vals and a_sub: A's payload staged in LDS and the row's
// first value, or A's array and 0.
template <class P>
__device__ __forceinline__ unsigned long long tile_row(const TileTask &g,
                                                       const typename P::Lane &ln, int64_t c0,
                                                       int64_t c1, int a0, int na,
                                                       const double *a_vals, uint32_t a_sub,
                                                       uint32_t a_zero, WaveStage &s, bool heavy_on)
{
    const int lane = lane_id();
    unsigned long long done = 0;
    for (int64_t cc = c0; cc < c1; cc += kWave) {
        const int nc = static_cast<int>(min<int64_t>(kWave, c1 - cc));
        // Lane c of the chunk holds C tile cc + c: column, mask, offset.
        unsigned long long cm = 0;
        long long co = 0;
        int cj = INT_MAX;
        bool whole = false;   // not a heavy tile (the chunk kernels compute those)
        if (lane < nc) {
            const int64_t t = cc + lane;
            cj = g.c_col[t];
            cm = g.c_mask[t];
            co = g.c_off[t];
            whole = !(heavy_on && ((g.heavy[t >> 5] >> (t & 31)) & 1u));
        }
        s.cj[lane] = cj;
        unsigned long long started = 0;
        for (int ag = 0; ag < na; ag += kWave) {
            const int n = min(kWave, na - ag);
            int nb = 0, b0 = 0;
            if (lane < n) {
                const int4 m = g.a_meta[a0 + ag + lane];
                const int4 br = g.a_brange[a0 + ag + lane];
                s.am[lane] = make_int2(static_cast<int>(list_mask(m.y, m.w)),
                                       static_cast<int>((static_cast<uint32_t>(m.w) & ~kDense) - a_sub));
                b0 = br.x;
                nb = br.z;
            }
            const int incl = wave_inclusive_scan(nb);
            const int total = last_lane(incl);
            s.start[lane] = incl - nb;
            s.b0[lane] = b0 - (incl - nb);
            s.word[lane] = 0ull;
            wave_sync();
            // kEnumRounds rounds of B tiles from e0: each lane's A tile (with
            // the C tile above it, -1 when there is none), mask and offset.
            int key[kEnumRounds], bm[kEnumRounds], bo[kEnumRounds];
            auto enumerate = [&](int e0) {
                int col[kEnumRounds];
#pragma unroll
                for (int i = 0; i < kEnumRounds; ++i) {
                    const int p = e0 + i * kWave + lane;
                    key[i] = -1;
                    if (p < total) {
                        const int k = upper_index(s.start, n, p);
                        const int4 m = g.b_meta[s.b0[k] + p];
                        key[i] = k;
                        col[i] = m.x;
                        bm[i] = static_cast<int>(list_mask(m.y, m.w));
                        bo[i] = static_cast<int>(static_cast<uint32_t>(m.w) & ~kDense);
                    }
                }
#pragma unroll
                for (int i = 0; i < kEnumRounds; ++i) {
                    if (key[i] < 0)
                        continue;
                    int at = 0;   // the C tiles with smaller columns
#pragma unroll
                    for (int step = kWave / 2; step > 0; step >>= 1)
                        at += s.cj[at + step - 1] < col[i] ? step : 0;
                    key[i] = s.cj[at] == col[i] ? key[i] | (at << 8) : -1;
                }
            };
            for (int e0 = 0; e0 < total; e0 += kEnumRounds * kWave) {
                enumerate(e0);
#pragma unroll
                for (int i = 0; i < kEnumRounds; ++i)
                    if (key[i] >= 0)
                        atomicOr(&s.word[key[i] >> 8], 1ull << (key[i] & 63));
            }
            wave_sync();
            const unsigned long long word = whole ? s.word[lane] : 0ull;
            const int cnt = __popcll(word);
            const int pi = wave_inclusive_scan(cnt);
            const int pairs = last_lane(pi);
            s.word[lane] = word;
            s.base[lane] = pi - cnt;
            wave_sync();
            for (int lo = 0; lo < pairs;) {
                // As many whole C tiles as the buffer holds.
                const unsigned long long fit = __ballot(pi <= lo + kPairCap);
                const int hi = __shfl(pi, __popcll(fit) - 1, kWave);
                const bool listed = cnt > 0 && pi > lo && pi <= hi;
                const unsigned long long live = __ballot(listed);
                if (lane < kPairWords)
                    s.ends[lane] = 0ull;
                if (lane < kPad)
                    s.pm[hi - lo + lane] = make_int4(0, 0, 0, 0);
                wave_sync();
                if (listed)
                    atomicOr(&s.ends[(pi - 1 - lo) >> 6], 1ull << ((pi - 1 - lo) & 63));
                for (int e0 = 0; e0 < total; e0 += kEnumRounds * kWave) {
                    if (total > kEnumRounds * kWave)
                        enumerate(e0);   // otherwise as the first pass left it
#pragma unroll
                    for (int i = 0; i < kEnumRounds; ++i) {
                        if (key[i] < 0)
                            continue;
                        const int c = key[i] >> 8, k = key[i] & 63;
                        const unsigned long long w = s.word[c];
                        const int slot =
                            s.base[c] + __popcll(w & ((1ull << k) - 1ull)) - lo;
                        if (((w >> k) & 1ull) && slot >= 0 && slot < hi - lo) {
                            const int2 m = s.am[k];
                            s.pm[slot] = make_int4(m.x, m.y, bm[i], bo[i]);
                        }
                    }
                }
                wave_sync();
                unsigned long long ends[kPairWords];
#pragma unroll
                for (int i = 0; i < kPairWords; ++i)
                    ends[i] = read_lane64(s.ends[i], 0);
                P::run(g, ln, a_vals, a_zero, s.pm, hi - lo, cnt, ends, live, started, cm, co, s.out);
                lo = hi;
                wave_sync();
            }
            done += static_cast<unsigned long long>(pairs);
            started |= __ballot(cnt > 0);
            if (ag + kWave < na) {
                // Other lanes than those that stored them may load the sums.
                __threadfence_block();
            }
            wave_sync();
        }
        wave_sync();
    }
    return done;
}

template <class P>
__global__ __launch_bounds__(kTThreads) __attribute__((amdgpu_waves_per_eu(P::kOccupancy)))
void tile_numeric_kernel(TileTask g)
{
    __shared__ WaveStage s_wave[kTWaves];
    const int w = threadIdx.x / kWave;
    const int lane = lane_id();
    WaveStage &s = s_wave[w];
    const int64_t u =
        static_cast<int64_t>(xcd_chunk_row<kXcdChunk>(static_cast<int>(blockIdx.x),
                                                      static_cast<int>(gridDim.x))) * kTWaves + w;
    const int row = static_cast<int>(u / g.parts), part = static_cast<int>(u % g.parts);
    if (row >= g.rows)
        return;
    const int64_t r0 = g.c_ptr[row], nt = g.c_ptr[row + 1] - r0;
    if (nt > kWideTiles)
        return;   // tile_wide_kernel's
    const int64_t c0 = r0 + nt * part / g.parts, c1 = r0 + nt * (part + 1) / g.parts;
    const int a0 = g.a_trp[row];
    const int na = g.a_trp[row + 1] - a0;
    const int v0 = g.a_row_off[row];
    const int nv = g.a_row_off[row + 1] - v0;
    // Rows below the fill threshold belong to the LDS-accumulator kernels.
    if (c0 == c1 || static_cast<float>(nv) < g.fill * static_cast<float>(na))
        return;
    const bool heavy_on = g.heavy && g.tail->enabled;
    const typename P::Lane ln(lane);
    unsigned long long done = 0;   // pairs this wave multiplied
    if (nv <= kAVals) {
        for (int i = lane; i < nv; i += kWave)
            s.av[i] = g.a_vals[v0 + i];
        if (lane == 0)
            s.av[nv] = 0.0;
        wave_sync();
        done = tile_row<P>(g, ln, c0, c1, a0, na, s.av, static_cast<uint32_t>(v0),
                           static_cast<uint32_t>(nv), s, heavy_on);
    } else {
        done = tile_row<P>(g, ln, c0, c1, a0, na, g.a_vals, 0u, g.a_zero, s, heavy_on);
    }
    if (lane == 0 && done && g.mfma_pairs)
        atomicAdd(&g.mfma_pairs[blockIdx.x % kPairShards * kShardStride], done);
}

// ---------------------------------------------------------------------------
// Rows of more than kWideTiles C tiles.  tile_row above enumerates all of the
// row's B tiles again for every 64 C tiles and every kPairCap pairs of those:
// for rows of hundreds of C tiles that is most of its time.  Here a lane keeps,
// for its A tile, where it is in each class run of its B row (whose columns
// ascend), and takes only the tiles between the first and last column of the
// next few C tiles, as many of those as make one list: every pair is met once.
// The A tiles go 64 at a time around that, so a C tile's sum waits in C between
// them; a tile sums the same pairs in the same order as in tile_row.
// A unit is a stretch of a row's C tiles, of a length that fills the chip.
// R-MAT 2^17 (edge factor 8) on this path: 5434 -> 62 ms; dense 4096^2: 537 -> 19;
// band of 200 either side, 100000 rows (101 C tiles a row): 12.3 -> 8.1.
// Rows of few C tiles stay with tile_row, which starts sooner: with no limit the
// 200k-node FEM square took 1.48 ms against 1.22, dense 256^2 0.42 against 0.35;
// with one of 256 the band 12.4 and dense 2048^2 65 ms against 3.2.
// ---------------------------------------------------------------------------
constexpr int kRuns = 5;   // classes of a row of B: heavy, light k = 0..3
constexpr int kWideList = 2 * kWave;   // B tiles taken at a time
static_assert(kWideList <= kPairCap, "their pairs are one list");

struct WideStage {
    int4 pm[kPairCap + kPad];         // as in WaveStage
    double out[kOutVals];
    unsigned long long word[kWave];
    unsigned long long ends[kPairWords + 1];
    int2 am[kWave];
    int start[kWave];                 // per A tile: its first B tile in the enumeration
    int lo[kRuns][kWave];             // per A tile: first B tile taken of each run,
    int cum[kRuns - 1][kWave];        // and the tiles taken of the runs up to each
    int cj[kWave];
    int base[kWave];
};

// First tile of [lo, hi), columns ascending, in column j or beyond: doubling
// steps, then a binary search in the last one.
__device__ __forceinline__ int tile_at(const int4 *__restrict__ meta, int lo, int hi, int j)
{
    int64_t step = 1;
    while (lo + step <= hi && meta[lo + step - 1].x < j) {
        lo += static_cast<int>(step);
        step <<= 1;
    }
    int end = static_cast<int>(min<int64_t>(lo + step - 1, hi));
    while (lo < end) {
        const int mid = (lo + end) >> 1;
        if (meta[mid].x < j)
            lo = mid + 1;
        else
            end = mid;
    }
    return lo;
}

template <class P>
__global__ __launch_bounds__(kTThreads) __attribute__((amdgpu_waves_per_eu(P::kWideOccupancy)))
void tile_wide_kernel(TileTask g, const int4 *__restrict__ units,
                      const unsigned long long *__restrict__ n_units)
{
    __shared__ WideStage s_wave[kTWaves];
    const int w = threadIdx.x / kWave;
    const int lane = lane_id();
    WideStage &s = s_wave[w];
    const int64_t u =
        static_cast<int64_t>(xcd_chunk_row<kXcdChunk>(static_cast<int>(blockIdx.x),
                                                      static_cast<int>(gridDim.x))) * kTWaves + w;
    if (u >= static_cast<int64_t>(*n_units))
        return;
    const int4 unit = units[u];
    const int row = __builtin_amdgcn_readfirstlane(unit.x),
              part = __builtin_amdgcn_readfirstlane(unit.y),
              parts = __builtin_amdgcn_readfirstlane(unit.z);
    const int64_t r0 = g.c_ptr[row], nt = g.c_ptr[row + 1] - r0;
    const int64_t c0 = r0 + nt * part / parts, c1 = r0 + nt * (part + 1) / parts;
    const int a0 = g.a_trp[row];
    const int na = g.a_trp[row + 1] - a0;
    const bool heavy_on = g.heavy && g.tail->enabled;
    const typename P::Lane ln(lane);
    // Sums of C tiles that wait for later A tiles.
    if (na > kWave) {
        for (int64_t i = g.c_off[c0] + lane; i < g.c_off[c1]; i += kWave)
            g.c_val[i] = 0.0;
        __threadfence_block();
    }
    unsigned long long done = 0;
    for (int ag = 0; ag < na; ag += kWave) {
        const int n = min(kWave, na - ag);
        // The lane's A tile: where it is in the runs of its B row, the column
        // there, and the runs' ends.
        int cur[kRuns], end[kRuns], head[kRuns];
#pragma unroll
        for (int c = 0; c < kRuns; ++c) {
            cur[c] = end[c] = 0;
            head[c] = INT_MAX;
        }
        if (lane < n) {
            const int4 m = g.a_meta[a0 + ag + lane];
            s.am[lane] = make_int2(static_cast<int>(list_mask(m.y, m.w)),
                                   static_cast<int>(static_cast<uint32_t>(m.w) & ~kDense));
            const int *gp = g.b_groups + static_cast<int64_t>(kClassSlots) * m.x;
#pragma unroll
            for (int c = 0; c < kRuns; ++c) {
                cur[c] = gp[c];
                end[c] = gp[c + 1];
                head[c] = cur[c] < end[c] ? g.b_meta[cur[c]].x : INT_MAX;
            }
        }
        int width = kWave;
        for (int64_t cc = c0; cc < c1;) {
            width = static_cast<int>(min<int64_t>(width, c1 - cc));
            unsigned long long cm = 0;
            long long co = 0;
            int cj = INT_MAX;
            bool whole = false;   // not a heavy tile (the chunk kernels compute those)
            if (lane < width) {
                const int64_t t = cc + lane;
                cj = g.c_col[t];
                cm = g.c_mask[t];
                co = g.c_off[t];
                whole = !(heavy_on && ((g.heavy[t >> 5] >> (t & 31)) & 1u));
            }
            const int first = read_lane(cj, 0);
            int to[kRuns], nb = 0;
#pragma unroll
            for (int c = 0; c < kRuns; ++c) {
                if (head[c] < first) {
                    cur[c] = tile_at(g.b_meta, cur[c], end[c], first);
                    head[c] = cur[c] < end[c] ? g.b_meta[cur[c]].x : INT_MAX;
                }
                to[c] = end[c];
            }
            int incl = 0, total = 0;
            for (;;) {
                const int last = read_lane(cj, width - 1);
                nb = 0;
#pragma unroll
                for (int c = 0; c < kRuns; ++c) {
                    to[c] = head[c] <= last ? tile_at(g.b_meta, cur[c] + 1, to[c], last + 1) : cur[c];
                    nb += to[c] - cur[c];
                }
                incl = wave_inclusive_scan(nb);
                total = last_lane(incl);
                // (One C tile meets at most one B tile per A tile.)
                if (total <= kWideList || width == 1)
                    break;
                width >>= 1;
            }
            const bool in = lane < width;
            const int step = width;
            if (total > 0) {
                s.cj[lane] = in ? cj : INT_MAX;
                s.start[lane] = incl - nb;
                s.word[lane] = 0ull;
                int sum = 0;
#pragma unroll
                for (int c = 0; c < kRuns; ++c) {
                    s.lo[c][lane] = cur[c] - sum;
                    sum += to[c] - cur[c];
                    if (c < kRuns - 1)
                        s.cum[c][lane] = sum;
                }
                if (lane < kPairWords)
                    s.ends[lane] = 0ull;
                wave_sync();
                int key[2], bm[2], bo[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int p = i * kWave + lane;
                    key[i] = -1;
                    if (p < total) {
                        const int k = upper_index(s.start, n, p);
                        const int q = p - s.start[k];
                        int c = 0;
#pragma unroll
                        for (int x = 0; x < kRuns - 1; ++x)
                            c += q >= s.cum[x][k] ? 1 : 0;
                        const int4 m = g.b_meta[s.lo[c][k] + q];
                        int at = 0;   // the C tiles with smaller columns
#pragma unroll
                        for (int d = kWave / 2; d > 0; d >>= 1)
                            at += s.cj[at + d - 1] < m.x ? d : 0;
                        if (s.cj[at] == m.x) {
                            key[i] = k | (at << 8);
                            bm[i] = static_cast<int>(list_mask(m.y, m.w));
                            bo[i] = static_cast<int>(static_cast<uint32_t>(m.w) & ~kDense);
                            atomicOr(&s.word[at], 1ull << k);
                        }
                    }
                }
                wave_sync();
                const unsigned long long word = whole && in ? s.word[lane] : 0ull;
                const int cnt = __popcll(word);
                const int pi = wave_inclusive_scan(cnt);
                const int pairs = last_lane(pi);
                s.word[lane] = word;
                s.base[lane] = pi - cnt;
                if (lane < kPad)
                    s.pm[pairs + lane] = make_int4(0, 0, 0, 0);
                if (cnt > 0)
                    atomicOr(&s.ends[(pi - 1) >> 6], 1ull << ((pi - 1) & 63));
                wave_sync();
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (key[i] < 0)
                        continue;
                    const int c = key[i] >> 8, k = key[i] & 63;
                    const unsigned long long wd = s.word[c];
                    if ((wd >> k) & 1ull) {
                        const int2 m = s.am[k];
                        s.pm[s.base[c] + __popcll(wd & ((1ull << k) - 1ull))] =
                            make_int4(m.x, m.y, bm[i], bo[i]);
                    }
                }
                wave_sync();
                if (pairs > 0) {
                    unsigned long long ends[kPairWords];
#pragma unroll
                    for (int i = 0; i < kPairWords; ++i)
                        ends[i] = read_lane64(s.ends[i], 0);
                    P::run(g, ln, g.a_vals, g.a_zero, s.pm, pairs, cnt, ends, __ballot(cnt > 0),
                           ag > 0 ? ~0ull : 0ull, cm, co, s.out);
                    done += static_cast<unsigned long long>(pairs);
                }
                wave_sync();
            }
#pragma unroll
            for (int c = 0; c < kRuns; ++c)
                if (to[c] > cur[c]) {
                    cur[c] = to[c];
                    head[c] = cur[c] < end[c] ? g.b_meta[cur[c]].x : INT_MAX;
                }
            cc += step;
            if (total <= kWideList / 3)
                width = min(2 * width, kWave);
        }
        if (ag + kWave < na)
            __threadfence_block();   // other lanes than those that stored them may load the sums
    }
    if (lane == 0 && done && g.mfma_pairs)
        atomicAdd(&g.mfma_pairs[blockIdx.x % kPairShards * kShardStride], done);
}

// The units of the wide rows: parts of about `target` C tiles.
__global__ __launch_bounds__(256) void wide_units_kernel(
    int rows, const int64_t *__restrict__ c_ptr, const int *__restrict__ a_trp,
    const int *__restrict__ a_row_off, float fill, int target, unsigned long long *n_units,
    int4 *__restrict__ units)
{
    __shared__ int s_tmp[256 / kWave];
    __shared__ unsigned long long s_base;
    const int row = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    int parts = 0;
    if (row < rows) {
        const int64_t nt = c_ptr[row + 1] - c_ptr[row];
        if (nt > kWideTiles && static_cast<float>(a_row_off[row + 1] - a_row_off[row]) >=
                                   fill * static_cast<float>(a_trp[row + 1] - a_trp[row]))
            parts = static_cast<int>((nt + target - 1) / target);
    }
    int all = 0;
    const int before = block_exclusive_scan<256 / kWave>(parts, s_tmp, &all);
    if (threadIdx.x == 0)
        s_base = all ? atomicAdd(n_units, static_cast<unsigned long long>(all)) : 0ull;
    __syncthreads();
    for (int i = 0; i < parts; ++i)
        units[s_base + before + i] = make_int4(row, i, parts, 0);
}

// Chunks of a task whose merge takes `scans` steps with `matches` matched
// pairs: the reference's FP32 admission (cost = scans + 8 matches, strictly
// above the threshold) and chunk count (ceil(cost / target), clamped to
// [2, max_chunks] and to at most one chunk per scan step); 0 = not admitted
// (dmma_tail_chunk_count_from_counts, src/dmma_spgemm.h:2628-2647).
__device__ __forceinline__ int tail_chunks(int scans, int matches, float threshold, float target,
                                           int max_chunks)
{
    const float work = 1.0f * static_cast<float>(scans) + 8.0f * static_cast<float>(matches);
    if (!(work > threshold) || !(target > 0.0f) || scans <= 1 || max_chunks <= 1)
        return 0;
    const float want = ceilf(work / target);
    int c = want >= static_cast<float>(max_chunks) ? max_chunks : static_cast<int>(want);
    c = max(c, 2);
    c = min(c, scans);
    return c >= 2 ? c : 0;
}

struct TailArgs {
    float threshold, target;
    int max_chunks;
    double max_heavy_fraction;
    int force;
    unsigned int capacity;
    unsigned long long workspace_limit;   // bytes
    long long tiles;                      // C tiles of the call
    TailRecord *__restrict__ records;
    TailState *__restrict__ state;
    uint32_t *__restrict__ heavy;
    int *__restrict__ chunk_base;         // capacity + 1
    double *__restrict__ workspace;       // 64 doubles per chunk
};

__global__ void tail_reset_kernel(TailState *st)
{
    if (threadIdx.x == 0) {
        st->count = 0u;
        st->overflow = 0;
        st->chunks = 0ull;
        st->reason = 0;
        st->enabled = 0;
        st->chunk_head = 0;
        st->reduce_head = 0;
    }
}

// One wave per tile row of the tile-pair kernel: the exact merge counts of
// every C tile whose upper bound (all of both lists scanned, every pair of
// the shorter list matched) clears the threshold, and a record for each
// admitted tile.
__global__ __launch_bounds__(kTThreads) void tail_admit_kernel(TileTask g, TailArgs t)
{
    const int row = blockIdx.x * kTWaves + static_cast<int>(threadIdx.x) / kWave;
    const int lane = lane_id();
    if (row >= g.rows)
        return;
    const int64_t c0 = g.c_ptr[row], c1 = g.c_ptr[row + 1];
    const int a0 = g.a_trp[row];
    const int na = g.a_trp[row + 1] - a0;
    if (c0 == c1 || static_cast<float>(g.a_row_off[row + 1] - g.a_row_off[row]) <
                        g.fill * static_cast<float>(na))
        return;
    for (int64_t cc = c0; cc < c1; cc += kWave) {
        const int64_t tile = cc + lane;
        int cb = 0, nb = 0;
        bool cand = false;
        if (tile < c1) {
            const int j = g.c_col[tile];
            cb = g.b_cptr[j];
            nb = g.b_cptr[j + 1] - cb;
            const float ub = 1.0f * static_cast<float>(na + nb) +
                             8.0f * static_cast<float>(min(na, nb));
            cand = ub > t.threshold;
        }
        unsigned long long todo = __ballot(cand);
        while (todo) {
            const int l = __ffsll(static_cast<long long>(todo)) - 1;
            todo &= todo - 1;
            const int tcb = read_lane(cb, l), tnb = read_lane(nb, l);
            // Intersection of A row's K list with B column's K list: lanes
            // take the shorter list, binary search in the longer.
            const bool a_short = na <= tnb;
            const int ns = a_short ? na : tnb, nl = a_short ? tnb : na;
            int matches = 0;
            for (int x0 = 0; x0 < ns; x0 += kWave) {
                const int x = x0 + lane;
                bool hit = false;
                if (x < ns) {
                    const int key = a_short ? g.a_meta[a0 + x].x : g.b_cent[tcb + x].x;
                    int lo = 0, hi = nl;
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        const int k = a_short ? g.b_cent[tcb + mid].x : g.a_meta[a0 + mid].x;
                        if (k < key)
                            lo = mid + 1;
                        else
                            hi = mid;
                    }
                    hit = lo < nl &&
                          (a_short ? g.b_cent[tcb + lo].x : g.a_meta[a0 + lo].x) == key;
                }
                matches += __popcll(__ballot(hit));
            }
            const int scans = na + tnb - matches;
            const int chunks = tail_chunks(scans, matches, t.threshold, t.target, t.max_chunks);
            if (lane == 0 && chunks > 0) {
                const unsigned int slot = atomicAdd(&t.state->count, 1u);
                if (slot < t.capacity) {
                    TailRecord r;
                    r.task = cc + l;
                    r.row = row;
                    r.scans = scans;
                    r.matches = matches;
                    r.chunks = chunks;
                    t.records[slot] = r;
                    atomicAdd(&t.state->chunks, static_cast<unsigned long long>(chunks));
                } else {
                    atomicExch(&t.state->overflow, 1);
                }
            }
        }
    }
}

// The gate (one thread): split only when some tile was admitted, the
// records fit, the heavy fraction is at most max_heavy_fraction (unless
// forced) and the chunk workspace fits its limit.  Reason codes: 1 split,
// 4 no heavy tile, 5 record capacity exceeded, 6 heavy fraction exceeded,
// 7 workspace limit exceeded.
__global__ void tail_gate_kernel(TailArgs t)
{
    if (threadIdx.x != 0)
        return;
    TailState *st = t.state;
    int reason;
    if (st->overflow || st->count > t.capacity)
        reason = 5;
    else if (st->count == 0u)
        reason = kTailNone;
    else if (!t.force && static_cast<double>(st->count) / static_cast<double>(t.tiles) >
                             t.max_heavy_fraction)
        reason = 6;
    else if (st->chunks * 64ull * sizeof(double) > t.workspace_limit)
        reason = 7;
    else
        reason = 1;
    st->reason = reason;
    st->enabled = reason == 1 ? 1 : 0;
}

__global__ void tail_mark_kernel(TailArgs t)
{
    const unsigned int i = blockIdx.x * blockDim.x + threadIdx.x;
    const TailState *st = t.state;
    const unsigned int n = min(st->count, t.capacity);
    if (i == 0)
        t.chunk_base[0] = 0;
    if (i >= n)
        return;
    const TailRecord r = t.records[i];
    if (st->enabled)
        atomicOr(&t.heavy[r.task >> 5], 1u << (r.task & 31));
}

// Exclusive prefix of the records' chunk counts (records in slot order; a
// tile's chunks are contiguous).  Single workgroup, sequential over the
// workgroup's partial sums: the record list is short.
__global__ __launch_bounds__(kTThreads) void tail_chunk_base_kernel(TailArgs t)
{
    __shared__ int s_sum[kTThreads];
    const TailState *st = t.state;
    const int n = static_cast<int>(min(st->count, t.capacity));
    const int per = (n + kTThreads - 1) / kTThreads;
    const int b = threadIdx.x * per, e = min(n, b + per);
    int sum = 0;
    for (int i = b; i < e; ++i)
        sum += t.records[i].chunks;
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int i = 0; i < kTThreads; ++i) {
            const int v = s_sum[i];
            s_sum[i] = run;
            run += v;
        }
    }
    __syncthreads();
    int run = s_sum[threadIdx.x];
    for (int i = b; i < e; ++i) {
        t.chunk_base[i] = run;
        run += t.records[i].chunks;
    }
    if (e == n && b < e)
        t.chunk_base[n] = run;
    if (n == 0 && threadIdx.x == 0)
        t.chunk_base[0] = 0;
}

// Persistent waves over the chunks: chunk j of record r covers B column
// entries [cb + nb j / chunks, cb + nb (j+1) / chunks) of its tile; the
// pairs found there are multiplied like the tile kernel's and the lane's
// partial entries go to the chunk's 64-slot workspace.
template <class P>
__global__ __launch_bounds__(kTThreads) void tail_chunk_kernel(TileTask g, TailArgs t)
{
    __shared__ int4 s_pm[kTWaves][kPairCap + kPad];
    const int w = threadIdx.x / kWave;
    const int lane = lane_id();
    int4 *pm = s_pm[w];
    const typename P::Lane ln(lane);
    const TailState *st = t.state;
    if (!st->enabled)
        return;
    const int n = static_cast<int>(min(st->count, t.capacity));
    const int total = t.chunk_base[n];
    for (;;) {
        int q = 0;
        if (lane == 0)
            q = atomicAdd(&t.state->chunk_head, 1);
        q = read_lane(q, 0);
        if (q >= total)
            break;
        const int r = upper_index(t.chunk_base, n, q);
        const TailRecord rec = t.records[r];
        const int j = q - t.chunk_base[r];
        const int row = rec.row;
        const int a0 = g.a_trp[row];
        const int na = g.a_trp[row + 1] - a0;
        const int jj = g.c_col[rec.task];
        const int cb = g.b_cptr[jj];
        const int nb = g.b_cptr[jj + 1] - cb;
        const int e0 = cb + static_cast<int>(static_cast<long long>(nb) * j / rec.chunks);
        const int e1 = cb + static_cast<int>(static_cast<long long>(nb) * (j + 1) / rec.chunks);
        int npairs = 0;
        typename P::Acc acc;
        for (int p0 = e0; p0 < e1; p0 += kWave) {
            const int p = p0 + lane;
            int ai = -1;
            int4 be = make_int4(0, 0, 0, 0);
            if (p < e1) {
                be = g.b_cent[p];
                int lo = 0, hi = na;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (g.a_meta[a0 + mid].x < be.x)
                        lo = mid + 1;
                    else
                        hi = mid;
                }
                if (lo < na && g.a_meta[a0 + lo].x == be.x)
                    ai = a0 + lo;
            }
            const unsigned long long match = __ballot(ai >= 0);
            if (ai >= 0) {
                const int4 am = g.a_meta[ai];
                const int slot = npairs + __popcll(match & ((1ull << lane) - 1ull));
                pm[slot] = make_int4(static_cast<int>(list_mask(am.y, am.w)),
                                     static_cast<int>(static_cast<uint32_t>(am.w) & ~kDense),
                                     static_cast<int>(list_mask(be.y, be.w)),
                                     static_cast<int>(static_cast<uint32_t>(be.w) & ~kDense));
            }
            npairs += __popcll(match);
            if (npairs + kWave > kPairCap || p0 + kWave >= e1) {
                if (lane < kPad)
                    pm[npairs + lane] = make_int4(0, 0, 0, 0);
                wave_sync();
                P::add(g, ln, g.a_vals, g.a_zero, pm, npairs, acc);
                npairs = 0;
                wave_sync();
            }
        }
        P::dump(ln, acc, t.workspace + static_cast<size_t>(q) * 64);
    }
}

// One wave per admitted tile: its chunks' partials summed in chunk order,
// stored at the tile's entries.
__global__ __launch_bounds__(kTThreads) void tail_reduce_kernel(TileTask g, TailArgs t)
{
    const TailState *st = t.state;
    if (!st->enabled)
        return;
    const int n = static_cast<int>(min(st->count, t.capacity));
    const int lane = lane_id();
    for (;;) {
        int r = 0;
        if (lane == 0)
            r = atomicAdd(&t.state->reduce_head, 1);
        r = read_lane(r, 0);
        if (r >= n)
            break;
        const TailRecord rec = t.records[r];
        const double *ws = t.workspace + static_cast<size_t>(t.chunk_base[r]) * 64;
        double sum = 0.0;
        for (int j = 0; j < rec.chunks; ++j)
            sum += ws[static_cast<size_t>(j) * 64 + lane];
        const unsigned long long m = g.c_mask[rec.task];
        if ((m >> lane) & 1ull)
            g.c_val[g.c_off[rec.task] + __popcll(m & ((1ull << lane) - 1ull))] = sum;
    }
}

__global__ void zero_u32_kernel(uint32_t *p, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0u;
}

__global__ void zero_queue_kernel(int *q, int n, unsigned long long *pairs)
{
    if (static_cast<int>(threadIdx.x) < n)
        q[threadIdx.x] = 0;
    if (threadIdx.x == 0)
        *pairs = 0ull;
}

// The call's tile statistics to the host's buffer: pairs, tail gate reason,
// admitted records, chunks of the split tiles.
__global__ __launch_bounds__(kPairShards) void tile_stats_kernel(const unsigned long long *pairs,
                                                                 const TailState *st, int reason,
                                                                 unsigned long long *host)
{
    __shared__ unsigned long long s_sum[kPairShards / kWave];
    const unsigned long long mine = wave_sum(pairs[threadIdx.x * kShardStride]);
    if (lane_id() == 0)
        s_sum[threadIdx.x / kWave] = mine;
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    unsigned long long all = 0;
    for (int i = 0; i < kPairShards / kWave; ++i)
        all += s_sum[i];
    host[0] = all;
    host[1] = static_cast<unsigned long long>(st ? st->reason : reason);
    host[2] = st ? st->count : 0ull;
    host[3] = st && st->enabled ? st->chunks : 0ull;
}

// The operands, C's structure, the units of a launch and its workgroups.  A
// product of fewer rows than the chip holds waves is cut into parts of a row.
TileTask make_task(const DevTiles &a, const DevTiles &b, const DevC &c, float fill,
                   double *c_values, unsigned long long *pairs, unsigned *blocks)
{
    TileTask g{};
    g.rows = static_cast<int>(c.tilem);
    g.a_trp = a.tile_row_ptr.as<int>();
    g.a_meta = a.meta.as<int4>();
    g.a_vals = a.values.as<double>();
    g.a_brange = b.a_brange.as<int4>();
    g.b_meta = b.records.as<int4>();
    g.b_groups = b.row_groups.as<int>();
    g.b_vals = b.payload_values();
    g.a_zero = static_cast<uint32_t>(a.payload);
    g.b_zero = static_cast<uint32_t>(b.payload);   // of B = A^T: A's, whose payload it is
    g.c_ptr = c.tile_ptr.as<int64_t>();
    g.c_col = c.tile_col.as<int>();
    g.c_mask = c.tile_mask.as<unsigned long long>();
    g.c_off = c.tile_nnz.as<int64_t>();
    g.c_val = c_values;
    g.a_row_off = a.row_payload_off.as<int>();
    g.fill = fill;
    g.mfma_pairs = pairs;
    const int64_t cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    const int64_t waves = cus * 16;
    g.parts = static_cast<int>(std::min<int64_t>(kMaxParts, (waves + g.rows - 1) / g.rows));
    *blocks = blocks_for(static_cast<int64_t>(g.rows) * g.parts, kTWaves);
    return g;
}

// The rows of the tile-pair kernel, then the wide ones by their units.
int launch_tiles(const TileTask &g, int precision, unsigned blocks, const SpgemmWork &w,
                 hipStream_t s)
{
    if (precision == 0)
        hipLaunchKernelGGL(tile_numeric_kernel<Fp64Product>, dim3(blocks), dim3(kTThreads), 0, s, g);
    else
        hipLaunchKernelGGL(tile_numeric_kernel<SplitProduct>, dim3(blocks), dim3(kTThreads), 0, s,
                           g);
    if (w.wide_units_most > 0) {
        const dim3 grid(blocks_for(w.wide_units_most, kTWaves));
        const unsigned long long *n = w.wide_units.as<unsigned long long>();
        const int4 *units = w.wide_units.as<int4>() + 1;
        if (precision == 0)
            hipLaunchKernelGGL(tile_wide_kernel<Fp64Product>, grid, dim3(kTThreads), 0, s, g, units,
                               n);
        else
            hipLaunchKernelGGL(tile_wide_kernel<SplitProduct>, grid, dim3(kTThreads), 0, s, g,
                               units, n);
    }
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

} // namespace

int plan_wide_rows(const DevTiles &a, const DevC &c, float fill, int64_t wide_rows,
                   int64_t wide_tiles, SpgemmWork *w, hipStream_t s)
{
    w->wide_units_most = 0;
    if (wide_rows == 0)
        return RTT_OK;
    const int64_t cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    // Twice the waves the chip holds, and no unit so short that finding its
    // place in every B row shows.
    const int64_t target = std::min<int64_t>(
        kWideMost, std::max<int64_t>(kWideLeast, wide_tiles / (2 * cus * 16)));
    const int64_t most = wide_tiles / target + wide_rows;
    // One int4 in front: the count.
    RTT_TRY(w->wide_units.ensure((static_cast<size_t>(most) + 1) * sizeof(int4)));
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(4), 0, s, w->wide_units.as<uint32_t>(),
                       int64_t(4));
    const int rows = static_cast<int>(c.tilem);
    hipLaunchKernelGGL(wide_units_kernel, dim3(blocks_for(rows, 256)), dim3(256), 0, s, rows,
                       c.tile_ptr.as<int64_t>(), a.tile_row_ptr.as<int>(),
                       a.row_payload_off.as<int>(), fill, static_cast<int>(target),
                       w->wide_units.as<unsigned long long>(), w->wide_units.as<int4>() + 1);
    RTT_HIP(hipGetLastError());
    w->wide_units_most = most;
    return RTT_OK;
}

TileColumns b_columns(const DevTiles &b)
{
    TileColumns v;
    if (b.transpose_of) {
        // B tile (K,J) column-major is A tile (J,K) row-major, bit for bit:
        // B's column J is A's tile row J.
        v.ptr = b.transpose_of->tile_row_ptr.as<int>();
        v.ent = b.transpose_of->meta.as<int4>();
    } else {
        v.ptr = b.col_ptr.as<int>();
        v.ent = b.col_ent.as<int4>();
    }
    return v;
}

// count[0]: tile rows routed to the tile-pair kernel at `fill`; count[1]:
// tile rows holding any tile; count[2]: most tiles in a row.  A grid-stride pass of at most kCountBlocks
// workgroups with one atomic pair per workgroup: an atomic pair per wave on
// the same two counters serialised at the L2 (0.3 ms for 2.6 M rows).
constexpr int kCountThreads = 256;
constexpr int kCountBlocks = 1024;
__global__ __launch_bounds__(kCountThreads) void count_tile_rows_kernel(
    int rows, const int *__restrict__ trp, const int *__restrict__ row_off, float fill,
    unsigned long long *__restrict__ count)
{
    __shared__ unsigned int s_m[kCountThreads / kWave], s_n[kCountThreads / kWave];
    __shared__ int s_l[kCountThreads / kWave];
    unsigned int m = 0, n = 0;
    int longest = 0;
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += gridDim.x * blockDim.x) {
        const int t = trp[r + 1] - trp[r];
        longest = max(longest, t);
        n += t > 0 ? 1u : 0u;
        m += t > 0 && static_cast<float>(row_off[r + 1] - row_off[r]) >= fill * static_cast<float>(t)
                 ? 1u
                 : 0u;
    }
    m = wave_sum(m);
    n = wave_sum(n);
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1)
        longest = max(longest, __shfl_xor(longest, o, kWave));
    if (lane_id() == 0) {
        s_l[threadIdx.x / kWave] = longest;
        s_m[threadIdx.x / kWave] = m;
        s_n[threadIdx.x / kWave] = n;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long bm = 0, bn = 0;
#pragma unroll
        for (int w = 0; w < kCountThreads / kWave; ++w) {
            bm += s_m[w];
            bn += s_n[w];
            longest = max(longest, s_l[w]);
        }
        if (bm)
            atomicAdd(count, bm);
        if (static_cast<unsigned long long>(longest) >
            __hip_atomic_load(count + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(count + 2, static_cast<unsigned long long>(longest));
        if (bn)
            atomicAdd(count + 1, bn);
    }
}

int count_tile_rows(const DevTiles &a, float fill, DevBuf *scratch, RowRouting *out)
{
    if (out->fill == fill)
        return RTT_OK;
    hipStream_t s = ctx().stream;
    RTT_TRY(scratch->ensure(3 * sizeof(unsigned long long)));
    unsigned long long *d = scratch->as<unsigned long long>();
    hipLaunchKernelGGL(zero_queue_kernel, dim3(1), dim3(4), 0, s, reinterpret_cast<int *>(d), 4,
                       d + 2);
    const int R = a.tile_row_count;
    if (R > 0)
        hipLaunchKernelGGL(count_tile_rows_kernel,
                           dim3(std::min<unsigned int>(kCountBlocks, blocks_for(R, kCountThreads))),
                           dim3(kCountThreads), 0, s, R, a.tile_row_ptr.as<int>(),
                           a.row_payload_off.as<int>(), fill, d);
    RTT_HIP(hipGetLastError());
    unsigned long long h[3] = {0, 0, 0};
    RTT_HIP(hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s));
    RTT_HIP(hipStreamSynchronize(s));
    out->longest = static_cast<int>(h[2]);
    out->tile_rows = static_cast<int64_t>(h[0]);
    out->nonempty = static_cast<int64_t>(h[1]);
    out->fill = fill;
    return RTT_OK;
}

int tile_numeric(const DevTiles &a, const DevTiles &b, const DevC &c, const TileOpts &opt,
                 const TileColumns *tail_columns, SpgemmWork *w, hipStream_t s)
{
    if (c.tilem == 0 || c.num_tiles == 0)
        return RTT_OK;
    const int precision = opt.precision;
    if (precision != 0 && precision != 1)
        return fail(RTT_ERR_INVALID, "unknown tile numeric precision %d", precision);
    constexpr int kShardWords = kPairShards * kShardStride;
    RTT_TRY(w->tile_pairs.ensure(kShardWords * sizeof(unsigned long long)));
    RTT_TRY(w->host_tile_stats.ensure(4 * sizeof(unsigned long long)));
    unsigned blocks = 0;
    TileTask g = make_task(a, b, c, opt.fill, c.tile_csr_val.as<double>(),
                           w->tile_pairs.as<unsigned long long>(), &blocks);
    w->tail_ran = tail_columns != nullptr;
    if (tail_columns) {
        g.b_cptr = tail_columns->ptr;
        g.b_cent = tail_columns->ent;
    }
    hipLaunchKernelGGL(zero_u32_kernel, dim3(blocks_for(2 * kShardWords, 256)), dim3(256), 0, s,
                       w->tile_pairs.as<uint32_t>(), static_cast<int64_t>(2 * kShardWords));
    const int cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    TailArgs t{};
    if (tail_columns) {
        // Record capacity as the reference sizes it: one past the admissible
        // heavy count (floor(tiles * max_fraction)), or every tile when the
        // split is forced, and never more than tail_record_capacity
        // (src/dmma_spgemm.h:7000-7016).
        const int64_t T = c.num_tiles;
        const int64_t admissible = static_cast<int64_t>(
            std::floor(static_cast<double>(T) * opt.max_heavy_fraction));
        const int64_t cap = std::max<int64_t>(
            1, std::min<int64_t>(opt.force ? T : admissible + 1, opt.record_capacity));
        const unsigned long long limit = 1ull << 30;   // src/main.cu:89
        const unsigned long long ws_bytes = std::min<unsigned long long>(
            limit, static_cast<unsigned long long>(cap) * opt.max_chunks * 64 * sizeof(double));
        RTT_TRY(w->tail_records.ensure(static_cast<size_t>(cap) * sizeof(TailRecord)));
        RTT_TRY(w->tail_state.ensure(sizeof(TailState)));
        RTT_TRY(w->tail_chunk_base.ensure((static_cast<size_t>(cap) + 1) * sizeof(int)));
        RTT_TRY(w->tail_heavy.ensure(static_cast<size_t>((T + 31) / 32) * sizeof(uint32_t)));
        RTT_TRY(w->tail_workspace.ensure(ws_bytes));
        t.threshold = opt.threshold;
        t.target = opt.target;
        t.max_chunks = opt.max_chunks;
        t.max_heavy_fraction = opt.max_heavy_fraction;
        t.force = opt.force;
        t.capacity = static_cast<unsigned int>(cap);
        t.workspace_limit = ws_bytes;
        t.tiles = T;
        t.records = w->tail_records.as<TailRecord>();
        t.state = w->tail_state.as<TailState>();
        t.heavy = w->tail_heavy.as<uint32_t>();
        t.chunk_base = w->tail_chunk_base.as<int>();
        t.workspace = w->tail_workspace.as<double>();
        hipLaunchKernelGGL(tail_reset_kernel, dim3(1), dim3(1), 0, s, t.state);
        hipLaunchKernelGGL(zero_u32_kernel, dim3(blocks_for((T + 31) / 32, 256)), dim3(256), 0, s,
                           t.heavy, (T + 31) / 32);
        hipLaunchKernelGGL(tail_admit_kernel, dim3(blocks_for(g.rows, kTWaves)), dim3(kTThreads),
                           0, s, g, t);
        hipLaunchKernelGGL(tail_gate_kernel, dim3(1), dim3(1), 0, s, t);
        hipLaunchKernelGGL(tail_mark_kernel, dim3(blocks_for(cap, 256)), dim3(256), 0, s, t);
        hipLaunchKernelGGL(tail_chunk_base_kernel, dim3(1), dim3(kTThreads), 0, s, t);
        RTT_HIP(hipGetLastError());
        g.heavy = t.heavy;
        g.tail = t.state;
    }
    RTT_TRY(launch_tiles(g, precision, blocks, *w, s));
    if (tail_columns) {
        if (precision == 0)
            hipLaunchKernelGGL(tail_chunk_kernel<Fp64Product>, dim3(cus * 4), dim3(kTThreads), 0,
                               s, g, t);
        else
            hipLaunchKernelGGL(tail_chunk_kernel<SplitProduct>, dim3(cus * 4), dim3(kTThreads), 0,
                               s, g, t);
        hipLaunchKernelGGL(tail_reduce_kernel, dim3(cus * 2), dim3(kTThreads), 0, s, g, t);
        RTT_HIP(hipGetLastError());
    }
    // With the queue on and no tile to admit, the gate's answer is known.
    hipLaunchKernelGGL(tile_stats_kernel, dim3(1), dim3(kPairShards), 0, s, g.mfma_pairs, g.tail,
                       opt.tail ? kTailNone : 0, w->host_tile_stats.as<unsigned long long>());
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int tile_values_noalloc(const DevTiles &a, const DevTiles &b, const DevC &c, const SpgemmWork &w,
                        int precision, double *c_values, hipStream_t s)
{
    if (c.tilem > INT_MAX)
        return fail(RTT_ERR_INVALID, "C has %lld tile rows: beyond the kernel's range",
                    (long long)c.tilem);
    if (precision != 0 && precision != 1)
        return fail(RTT_ERR_INVALID, "unknown tile numeric precision %d", precision);
    if (c.tilem == 0 || c.num_tiles == 0)
        return RTT_OK;
    unsigned blocks = 0;
    const TileTask g = make_task(a, b, c, 0.f, c_values, nullptr, &blocks);
    return launch_tiles(g, precision, blocks, w, s);
}

bool tail_possible(int a_tiles, int64_t b_tiles, float threshold)
{
    // The admission kernel's own bound, at the longest lists.
    const float ub = 1.0f * static_cast<float>(a_tiles + b_tiles) +
                     8.0f * static_cast<float>(std::min<int64_t>(a_tiles, b_tiles));
    return ub > threshold;
}

int tail_records(SpgemmWork *w, int max_records, long long *task, int *scans, int *matches,
                 int *chunks, int *count)
{
    *count = 0;
    if (!w->tail_ran)
        return RTT_OK;
    TailState st{};
    RTT_HIP(hipMemcpy(&st, w->tail_state.ptr, sizeof(st), hipMemcpyDeviceToHost));
    const int n = static_cast<int>(std::min<unsigned long long>(
        std::min<unsigned long long>(st.count, w->tail_records.bytes / sizeof(TailRecord)),
        static_cast<unsigned long long>(max_records)));
    std::vector<TailRecord> recs(static_cast<size_t>(n));
    if (n > 0)
        RTT_HIP(hipMemcpy(recs.data(), w->tail_records.ptr, n * sizeof(TailRecord),
                          hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i) {
        task[i] = recs[i].task;
        scans[i] = recs[i].scans;
        matches[i] = recs[i].matches;
        chunks[i] = recs[i].chunks;
    }
    *count = n;
    return RTT_OK;
}

} // namespace rtt
