// CSR upload/validation, B = A^T from A's tiles, and what the SpGEMM core
// reads beside the tiles (records, pair extents, tile columns).  The CSR ->
// tile builder is in tilebuild.hip.
#include <atomic>
#include <hipcub/hipcub.hpp>

#include <climits>

#include "device.hpp"
#include "internal.hpp"

namespace rtt {

namespace {

constexpr int kThreads = 256;

__global__ void set_i64_kernel(int64_t *p, int64_t n, int64_t v)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

__global__ void fill_int_kernel(int *p, int64_t n, int v)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

__global__ void iota_kernel(int *p, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = static_cast<int>(i);
}

__global__ void fill_f64_kernel(double *p, int64_t n, double v)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

// out[x] = in[idx[x]]
__global__ void gather_f64_kernel(int64_t n, const int *__restrict__ idx,
                                  const double *__restrict__ in, double *__restrict__ out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        out[i] = in[idx[i]];
}

// flags: 1 row_ptr not monotone / wrong ends, 2 column out of range,
//        4 some row not column-sorted (duplicates allowed).
__global__ void validate_csr_kernel(int rows, int cols, int64_t nnz,
                                    const int *__restrict__ rp,
                                    const int *__restrict__ ci, int *flags, int *max_row)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i == 0 && (rp[0] != 0 || rp[rows] != nnz))
        atomicOr(flags, 1);
    if (i < rows) {
        const int b = rp[i], e = rp[i + 1];
        // Bounds first: a row outside [0, nnz] is flagged, never walked.
        if (b < 0 || e < b || static_cast<int64_t>(e) > nnz) {
            atomicOr(flags, 1);
        } else {
            if (e - b > __hip_atomic_load(max_row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax(max_row, e - b);
            for (int x = b + 1; x < e; ++x)
                if (ci[x] < ci[x - 1]) {
                    atomicOr(flags, 4);
                    break;
                }
        }
    }
    if (i < nnz) {
        const int c = ci[i];
        if (c < 0 || c >= cols)
            atomicOr(flags, 2);
    }
}

__global__ void narrow_i64_kernel(const int64_t *in, int *out, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        out[i] = static_cast<int>(in[i]);
}

__global__ void tile_row_of_kernel(int rows, const int *__restrict__ trp,
                                   int *__restrict__ out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < rows)
        for (int t = trp[i]; t < trp[i + 1]; ++t)
            out[t] = static_cast<int>(i);
}

__global__ void histogram_kernel(const int *__restrict__ keys, int64_t n,
                                 int64_t *__restrict__ counts)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        atomicAdd(reinterpret_cast<unsigned long long *>(counts + keys[i]), 1ull);
}

// CSC of a tile matrix from its stably sorted tile ids.
__global__ void csc_fill_kernel(int64_t n, const int *__restrict__ sorted_ids,
                                const int *__restrict__ tile_row_of,
                                int *__restrict__ tile_row_idx,
                                int *__restrict__ csc_tile_ids)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) {
        const int t = sorted_ids[i];
        csc_tile_ids[i] = t;
        tile_row_idx[i] = tile_row_of[t];
    }
}

// B tile b (sorted by K) comes from A tile ids[b]; gather its metadata.
__global__ void transpose_meta_kernel(int64_t n, const int *__restrict__ ids,
                                      const int *__restrict__ a_row_of,
                                      const uint32_t *__restrict__ a_masks,
                                      const int *__restrict__ a_off,
                                      int *__restrict__ b_col,
                                      uint32_t *__restrict__ b_masks,
                                      int64_t *__restrict__ spans,
                                      int *__restrict__ b_csc_ids)
{
    const int64_t b = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (b < n) {
        const int a = ids[b];
        b_col[b] = a_row_of[a];
        b_masks[b] = a_masks[a];
        spans[b] = a_off[a + 1] - a_off[a];
        b_csc_ids[a] = static_cast<int>(b);   // A order == B's CSC order
    }
}

// Payload copy, one wave per 2 tiles (32 lanes per tile).
__global__ void transpose_payload_kernel(int64_t n, const int *__restrict__ ids,
                                         const int *__restrict__ a_off,
                                         const double *__restrict__ a_vals,
                                         const int64_t *__restrict__ b_off64,
                                         int *__restrict__ b_off,
                                         double *__restrict__ b_vals)
{
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t b = gid / 32;
    const int s = static_cast<int>(gid % 32);
    if (b >= n)
        return;
    const int a = ids[b];
    const int src = a_off[a];
    const int span = a_off[a + 1] - src;
    const int64_t dst = b_off64[b];
    if (s == 0)
        b_off[b] = static_cast<int>(dst);
    if (s < span)
        b_vals[dst + s] = a_vals[src + s];
}

// Row pointer of a sorted key array: ptr[k] = first index with key >= k.
__global__ void row_ptr_from_sorted_kernel(const int *__restrict__ keys, int64_t n, int rows,
                                           int *__restrict__ ptr)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i > n)
        return;
    const int prev = i == 0 ? -1 : keys[i - 1];
    const int cur = i == n ? rows : keys[i];
    for (int k = prev + 1; k <= cur; ++k)
        ptr[k] = static_cast<int>(i);
}

// Position of the n-th set bit of m (n below its count).
__device__ __forceinline__ int nth_bit(uint32_t m, int n)
{
    int pos = 0;
#pragma unroll
    for (int w = 16; w >= 1; w >>= 1) {
        const int c = __popc((m >> pos) & ((1u << w) - 1u));
        if (n >= c) {
            n -= c;
            pos += w;
        }
    }
    return pos;
}

// Value planes (1 .. kRecParts-1) of B's records and the k-major copy of what
// they do not hold, from the payload.  A record holds its tile's first
// kRecVals values in k-major order (row k's entries contiguous, columns
// ascending); the values past them go to the same places of the k-major copy,
// whose first kRecVals slots per tile nothing reads.  The planes past a
// tile's values are never read.
// Four lanes per tile, lane q the values 2q, 2q + 1 of every eight: a wave
// reads its 16 tiles' values a line at a time and writes 256 contiguous bytes
// of every plane.  (One lane per tile where tiles hold two values or fewer on
// average, which the first lane has anyway: four took 1 % more of a step there,
// scattered columns with 2, 6 and 16 entries a row; above, no difference was seen
// at two to four values, and the batches below gained.)  With a tile per thread every load met 64 lines, and they
// were gone from the L1 before a tile's next value was asked for: banded batch
// 257 -> 168 us, AMG batch 233 -> 222 us (its tiles hold few values).
template <int L>
__global__ void record_values_kernel(int64_t n, const double *__restrict__ vals,
                                     int4 *__restrict__ planes, double *__restrict__ kmajor)
{
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t step = static_cast<int64_t>(gridDim.x) * blockDim.x / L;
    const int q = static_cast<int>(gid % L);
    for (int64_t t = gid / L; t < n; t += step) {
        const int4 m = planes[t];
        const uint32_t mask = static_cast<uint32_t>(m.y);
        const bool dense = m.w < 0;
        const uint32_t off = static_cast<uint32_t>(m.w) & 0x7FFFFFFFu;
        const int nv = __popc(mask);
        const uint32_t mz = static_cast<uint32_t>(m.z);   // bit k * 8 + c
        // Value of the entry at bit pos: bit c * 4 + k of the payload's order.
        auto at = [&](int pos) {
            const int phys = (pos & 7) * 4 + (pos >> 3);
            return vals[off + (dense ? phys : __popc(mask & ((1u << phys) - 1u)))];
        };
        for (int j = 2 * q; j < nv; j += 2 * L) {
            const int p0 = nth_bit(mz, j);
            const uint32_t rest = p0 < 31 ? mz >> (p0 + 1) : 0u;
            double2 v;
            v.x = at(p0);
            v.y = j + 1 < nv ? at(p0 + 1 + __builtin_ctz(rest | 0x80000000u)) : 0.0;
            if (j < kRecVals) {
                planes[(1 + j / 2) * n + t] = *reinterpret_cast<const int4 *>(&v);
            } else {
                kmajor[off + j] = v.x;
                if (j + 1 < nv)
                    kmajor[off + j + 1] = v.y;
            }
        }
    }
}

// Values-only update: the first source entry of each slot's run sums the
// run in entry order (the order the tile build sums duplicates in).  Runs
// are adjacent because duplicates of a coordinate are adjacent in a
// row-sorted CSR.
__global__ void scatter_runs_kernel(int64_t nnz, const int *__restrict__ slot,
                                    const double *__restrict__ v, double *__restrict__ values)
{
    const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= nnz)
        return;
    const int s = slot[e];
    if (s < 0 || (e > 0 && slot[e - 1] == s))
        return;
    double sum = v[e];
    for (int64_t f = e + 1; f < nnz && slot[f] == s; ++f)
        sum += v[f];
    values[s] = sum;
}

// Part `part` of the record of a tile with meta m and k-major payload.
__device__ __forceinline__ int4 record_part(int part, const int4 &m, const double *kmajor)
{
    if (part == 0)
        return m;
    const uint32_t off = static_cast<uint32_t>(m.w) & 0x7FFFFFFFu;
    const int nv = min(kRecVals, __popc(static_cast<uint32_t>(m.y)));
    const int j = 2 * (part - 1);
    double2 v;
    v.x = j < nv ? kmajor[off + j] : 0.0;
    v.y = j + 1 < nv ? kmajor[off + j + 1] : 0.0;
    return *reinterpret_cast<const int4 *>(&v);
}

// Offline, per A tile: the record a B tile built as A^T takes over, its meta
// with the tile column replaced by the tile row.
// The B tile's k-major order is the A tile's column-major order.
__global__ void transpose_source_kernel(int64_t n, const int *__restrict__ a_row_of,
                                        const int4 *__restrict__ a_meta,
                                        const double *__restrict__ a_vals_cm,
                                        BRecord *__restrict__ out)
{
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t t = gid / kRecParts;
    if (t >= n)
        return;
    int4 m = a_meta[t];
    m.x = a_row_of[t];
    const int part = static_cast<int>(gid % kRecParts);
    reinterpret_cast<int4 *>(out + t)[part] = record_part(part, m, a_vals_cm);
}

// B = A^T: B tile b is A tile ids[b], so its record is a copy of that A
// tile's transpose record, one tile per thread: a thread reads its record
// (80 contiguous bytes) and consecutive threads write consecutive entries
// of every plane (3 % faster than a thread per 16-byte part).
__global__ void transposed_records_kernel(int64_t n, const int *__restrict__ ids,
                                          const BRecord *__restrict__ src,
                                          int4 *__restrict__ planes)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n)
        return;
    const int4 *r = reinterpret_cast<const int4 *>(src + ids[t]);
    int4 v[kRecParts];
#pragma unroll
    for (int part = 0; part < kRecParts; ++part)
        v[part] = r[part];
#pragma unroll
    for (int part = 0; part < kRecParts; ++part)
        planes[part * n + t] = v[part];
}

// Class of a B tile within its row: 0 for heavy tiles (kHeavyMin entries or
// more, or entries in more than one row k), else 1 + k for a light tile whose
// entries all lie in row k.  bytes holds the per-k column bytes of the tile
// (for B = A^T, the per-k row bytes of the A tile).
__device__ __forceinline__ int b_tile_class(uint32_t mask, uint32_t bytes)
{
    uint32_t rows = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        rows |= ((bytes >> (8 * k)) & 0xFFu) ? (1u << k) : 0u;
    if (__popc(mask) >= kHeavyMin || __popc(rows) != 1)
        return 0;
    return 1 + __builtin_ctz(rows);
}

// Counting transpose of A's tiles into B = A^T rows, for operands whose tile
// columns hold at most kShortCol tiles: a count per B row, a scan, a scatter
// in arbitrary order within each row, then one workgroup per kOrderRows rows
// ranks every entry within its row by (class, A tile id).  The result is the
// stable sort by (row, class) that the radix path produces, entry for entry.
constexpr int kShortCol = 64;     // most tiles in an A tile column it takes
constexpr int kOrderRows = 64;    // B rows per ordering workgroup
constexpr int kOrderIdBits = 28;  // A tile ids below 2^28; the class above them

// B class of the A^T tile made from each A tile, and its arrival rank in its
// B row (the tile's column of A).
__global__ void column_rank_kernel(int64_t n, const int *__restrict__ col,
                                   const uint32_t *__restrict__ masks, int *__restrict__ counts,
                                   int *__restrict__ rank_cls)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n)
        return;
    const uint32_t mask = masks[t];
    uint32_t bytes = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        bytes |= stride4_bits(mask, k) << (8 * k);
    const int r = atomicAdd(&counts[col[t]], 1);
    rank_cls[t] = (r << 3) | b_tile_class(mask, bytes);
}

__global__ void column_scatter_kernel(int64_t n, const int *__restrict__ col,
                                      const int *__restrict__ rank_cls,
                                      const int *__restrict__ rp, uint32_t *__restrict__ ent)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n)
        return;
    const int rc = rank_cls[t];
    ent[rp[col[t]] + (rc >> 3)] = (static_cast<uint32_t>(rc & 7) << kOrderIdBits) |
                                  static_cast<uint32_t>(t);
}

// Rows r0 .. r0 + kOrderRows - 1 of B: each entry's place is its row's start
// plus the number of the row's entries below it by (class, id); each
// (row, class) run starts after the row's entries of lower classes.
__global__ void __launch_bounds__(kThreads)
    order_rows_kernel(int R, int64_t n, const int *__restrict__ rp,
                      const uint32_t *__restrict__ ent, int *__restrict__ sorted_ids,
                      int *__restrict__ groups)
{
    __shared__ int s_rp[kOrderRows + 1];
    __shared__ uint32_t s_ent[kOrderRows * kShortCol];
    const int r0 = blockIdx.x * kOrderRows;
    const int nr = min(kOrderRows, R - r0);
    for (int i = threadIdx.x; i <= nr; i += blockDim.x)
        s_rp[i] = rp[r0 + i];
    __syncthreads();
    const int base = s_rp[0];
    const int total = s_rp[nr] - base;
    // At most nr * kShortCol when every column holds at most kShortCol
    // tiles, which the host checks before taking this path; the bound keeps
    // the stage in its LDS whatever the input.
    if (total > kOrderRows * kShortCol)
        return;
    for (int e = threadIdx.x; e < total; e += blockDim.x)
        s_ent[e] = ent[base + e];
    __syncthreads();
    for (int e = threadIdx.x; e < total; e += blockDim.x) {
        int lo = 0, hi = nr - 1;   // last row starting at or before e
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_rp[mid] - base <= e)
                lo = mid;
            else
                hi = mid - 1;
        }
        const int b = s_rp[lo] - base, end = s_rp[lo + 1] - base;
        const uint32_t v = s_ent[e];
        int rank = 0;
        for (int x = b; x < end; ++x)
            rank += s_ent[x] < v ? 1 : 0;
        sorted_ids[base + b + rank] = static_cast<int>(v & ((1u << kOrderIdBits) - 1u));
    }
    for (int i = threadIdx.x; i < nr * kClassSlots; i += blockDim.x) {
        const int r = i / kClassSlots;
        const uint32_t c = static_cast<uint32_t>(i % kClassSlots);
        const int b = s_rp[r] - base, end = s_rp[r + 1] - base;
        int below = 0;
        for (int x = b; x < end; ++x)
            below += (s_ent[x] >> kOrderIdBits) < c ? 1 : 0;
        groups[static_cast<int64_t>(r0 + r) * kClassSlots + c] = base + b + below;
    }
    if (r0 + nr == R && threadIdx.x == 0)
        groups[static_cast<int64_t>(R) * kClassSlots] = static_cast<int>(n);
}

// Tiles per tile column; column_max_kernel then puts the largest count in
// counts[cols].
__global__ void column_count_kernel(int64_t n, const int *__restrict__ col, int *__restrict__ counts)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < n)
        atomicAdd(&counts[col[t]], 1);
}

// At most one atomic per workgroup, and none once the largest count so far
// is as large: an atomic per wave on the one address serialises (0.1 ms on
// 2^19 columns).
__global__ void __launch_bounds__(kThreads) column_max_kernel(int cols, int *__restrict__ counts)
{
    __shared__ int s_max[kThreads / kWave];
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    int m = j < cols ? counts[j] : 0;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1)
        m = max(m, __shfl_xor(m, o, kWave));
    if (lane_id() == 0)
        s_max[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / kWave; ++w)
            m = max(m, s_max[w]);
        if (m > __hip_atomic_load(&counts[cols], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&counts[cols], m);
    }
}

// Per A tile t in column K: {first B tile of row K, heavy tiles, all tiles}
// and the light run its pairs need: for an A tile whose entries all lie in
// one column k, only the light tiles of row k can meet it.
__global__ __launch_bounds__(kThreads) void pair_extent_kernel(
    int64_t n, const int4 *__restrict__ a_meta, const int *__restrict__ groups,
    int4 *__restrict__ out, int2 *__restrict__ light, unsigned long long *__restrict__ pairs,
    const unsigned int *__restrict__ flag, long long *__restrict__ flag_out)
{
    // Passes the tile build's duplicate flag on to the host's buffer.
    if (flag && blockIdx.x == 0 && threadIdx.x == 0)
        *flag_out = *flag;
    // Grid-stride, so that the pair total takes one atomic per workgroup.
    __shared__ unsigned long long s_sum[kThreads / kWave];
    unsigned long long sum = 0;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < n;
         t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int4 m = a_meta[t];
        const int *gp = groups + static_cast<int64_t>(kClassSlots) * m.x;
        const int b0 = gp[0];
        const int total = gp[kClassSlots] - b0;
        out[t] = make_int4(b0, gp[1] - b0, total, 0);
        sum += static_cast<unsigned long long>(total);
        const uint32_t bytes = static_cast<uint32_t>(m.z);
        uint32_t cols = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            cols |= ((bytes >> (8 * k)) & 0xFFu) ? (1u << k) : 0u;
        if (__popc(cols) == 1) {
            const int k0 = __builtin_ctz(cols);
            light[t] = make_int2(gp[1 + k0], gp[2 + k0] - gp[1 + k0]);
        } else {
            light[t] = make_int2(gp[1], gp[5] - gp[1]);
        }
    }
    sum = wave_sum(sum);
    if (lane_id() == 0)
        s_sum[threadIdx.x / kWave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long all = 0;
        for (int w = 0; w < kThreads / kWave; ++w)
            all += s_sum[w];
        if (all)
            atomicAdd(pairs, all);
    }
}

// Sort key of a B tile: its row times kClassSlots plus its class.
__global__ void class_keys_kernel(int64_t n, const int *__restrict__ row,
                                  const int4 *__restrict__ meta, int *__restrict__ keys)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < n) {
        const int4 m = meta[t];
        keys[t] = kClassSlots * row[t] +
                  b_tile_class(static_cast<uint32_t>(m.y), static_cast<uint32_t>(m.z));
    }
}

// B's row pointer from the row pointer over (row, class) keys.
__global__ void group_row_ptr_kernel(int rows, const int *__restrict__ groups,
                                     int *__restrict__ trp)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r <= rows)
        trp[r] = groups[static_cast<int64_t>(kClassSlots) * r];
}

__global__ void entry_rows_kernel(int rows, const int *__restrict__ rp,
                                  int *__restrict__ out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < rows)
        for (int e = rp[i]; e < rp[i + 1]; ++e)
            out[e] = static_cast<int>(i);
}

__global__ void gather_transposed_kernel(int64_t nnz, const int *__restrict__ order,
                                         const int *__restrict__ entry_row,
                                         const double *__restrict__ val,
                                         int *__restrict__ t_col,
                                         double *__restrict__ t_val)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < nnz) {
        const int e = order[i];
        t_col[i] = entry_row[e];
        t_val[i] = val[e];
    }
}

__global__ void nnz_cub_kernel(int64_t nnz, const int *__restrict__ ci,
                               const int *__restrict__ rp,
                               const int64_t *__restrict__ coldeg,
                               unsigned long long *__restrict__ out)
{
    __shared__ unsigned long long part[kThreads / kWave];
    unsigned long long v = 0;
    // Grid-stride, so that only a few hundred workgroups add into *out.
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < nnz;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int c = ci[i];
        v += coldeg ? static_cast<unsigned long long>(coldeg[c])
                    : static_cast<unsigned long long>(rp[c + 1] - rp[c]);
    }
    v = wave_sum(v);
    if (lane_id() == 0)
        part[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long s = 0;
        for (int w = 0; w < kThreads / kWave; ++w)
            s += part[w];
        atomicAdd(out, s);
    }
}

int bits_for(int64_t max_value)
{
    int bits = 1;
    while (bits < 62 && (int64_t(1) << bits) <= max_value)
        ++bits;
    return bits;
}

// Stable sort of int keys with int payload (hipcub LSD radix sort).
int sort_pairs(const int *k_in, int *k_out, const int *v_in, int *v_out, int64_t n,
               int bits, DevBuf *tmp, hipStream_t s)
{
    size_t bytes = 0;
    RTT_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k_in, k_out, v_in, v_out,
                                               static_cast<int>(n), 0, bits, s));
    RTT_TRY(tmp->ensure(bytes));
    RTT_HIP(hipcub::DeviceRadixSort::SortPairs(tmp->ptr, bytes, k_in, k_out, v_in, v_out,
                                               static_cast<int>(n), 0, bits, s));
    return RTT_OK;
}

int read_i64(const int64_t *d, int64_t *h, hipStream_t s)
{
    RTT_HIP(hipMemcpyAsync(h, d, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    RTT_HIP(hipStreamSynchronize(s));
    return RTT_OK;
}

// Builds B's tile CSC (tile_col_ptr, tile_row_idx, csc_tile_ids) from its
// tile CSR: tiles of each tile column in increasing tile-row order
// (src/gpu_dmma_tiles.h:1003-1088 semantics).
int build_csc(DevTiles *t, BuildWork *w)
{
    hipStream_t s = ctx().stream;
    const int64_t n = t->num_tiles;
    const int ncols = t->tile_col_count;
    RTT_TRY(t->tile_col_ptr.ensure((ncols + 1) * sizeof(int)));
    RTT_TRY(t->tile_row_idx.ensure(n * sizeof(int)));
    RTT_TRY(t->csc_tile_ids.ensure(n * sizeof(int)));
    RTT_TRY(fill_tile_row_of(t));
    RTT_TRY(w->spans.ensure((ncols + 1) * sizeof(int64_t)));
    RTT_TRY(w->counters.ensure((ncols + 1) * sizeof(int64_t)));
    int64_t *cnt = w->spans.as<int64_t>();
    hipLaunchKernelGGL(set_i64_kernel, dim3(blocks_for(ncols + 1, kThreads)), dim3(kThreads),
                       0, s, cnt, static_cast<int64_t>(ncols) + 1, int64_t(0));
    if (n > 0) {
        hipLaunchKernelGGL(histogram_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0,
                           s, t->tile_col_idx.as<int>(), n, cnt);
        RTT_TRY(w->ids_in.ensure(n * sizeof(int)));
        RTT_TRY(w->ids_out.ensure(n * sizeof(int)));
        RTT_TRY(w->keys_out.ensure(n * sizeof(int)));
        hipLaunchKernelGGL(iota_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s,
                           w->ids_in.as<int>(), n);
        RTT_TRY(sort_pairs(t->tile_col_idx.as<int>(), w->keys_out.as<int>(),
                           w->ids_in.as<int>(), w->ids_out.as<int>(), n, bits_for(ncols),
                           &w->scan_tmp, s));
        hipLaunchKernelGGL(csc_fill_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0,
                           s, n, w->ids_out.as<int>(), t->tile_row_of.as<int>(),
                           t->tile_row_idx.as<int>(), t->csc_tile_ids.as<int>());
    }
    int64_t *ptr64 = w->counters.as<int64_t>();
    RTT_TRY(exclusive_scan_i64(cnt, ptr64, ncols, &w->scan_tmp, s));
    hipLaunchKernelGGL(narrow_i64_kernel, dim3(blocks_for(ncols + 1, kThreads)),
                       dim3(kThreads), 0, s, ptr64, t->tile_col_ptr.as<int>(),
                       static_cast<int64_t>(ncols) + 1);
    RTT_HIP(hipGetLastError());
    t->has_csc = true;
    return RTT_OK;
}

} // namespace

void DevTiles::view(rtt_device_tiles *v) const
{
    v->rows = rows;
    v->cols = cols;
    v->tile_rows = tile_rows;
    v->tile_cols = tile_cols;
    v->tile_row_count = tile_row_count;
    v->tile_col_count = tile_col_count;
    v->num_tiles = static_cast<int>(num_tiles);
    v->payload_size = static_cast<int>(payload);
    v->dense_tiles = static_cast<int>(dense);
    v->sparse_tiles = static_cast<int>(sparse);
    v->tile_row_ptr = tile_row_ptr.as<int>();
    v->tile_col_idx = tile_col_idx.as<int>();
    v->value_offsets = value_offsets.as<int>();
    v->masks = masks.as<uint32_t>();
    v->values = values.as<double>();
    v->tile_col_ptr = has_csc ? tile_col_ptr.as<int>() : nullptr;
    v->tile_row_idx = has_csc ? tile_row_idx.as<int>() : nullptr;
    v->csc_tile_ids = has_csc ? csc_tile_ids.as<int>() : nullptr;
}

static int write_record_values(DevTiles *b)
{
    RTT_TRY(b->values_cm.ensure(static_cast<size_t>(b->payload > 0 ? b->payload : 1) *
                                sizeof(double)));
    auto launch = [&](auto kernel, int lanes) {
        hipLaunchKernelGGL(kernel, dim3(std::min(blocks_for(b->num_tiles * lanes, kThreads), 1u << 22)),
                           dim3(kThreads), 0, ctx().stream, b->num_tiles, b->values.as<double>(),
                           b->records.as<int4>(), b->values_cm.as<double>());
    };
    if (b->num_tiles > 0 && b->payload <= 2 * b->num_tiles)
        launch(record_values_kernel<1>, 1);
    else if (b->num_tiles > 0)
        launch(record_values_kernel<4>, 4);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int ensure_record_values(DevTiles *b)
{
    if (b->transpose_of || b->rec_values_ready)
        return RTT_OK;
    RTT_TRY(write_record_values(b));
    b->rec_values_ready = true;
    return RTT_OK;
}

int build_pair_extents(const DevTiles &a, DevTiles *b, const unsigned int *flag,
                       long long *flag_out)
{
    RTT_TRY(b->a_brange.ensure(a.num_tiles * sizeof(int4)));
    RTT_TRY(b->a_blight.ensure(a.num_tiles * sizeof(int2)));
    hipStream_t s = ctx().stream;
    const int cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(
        4 * cus, std::max<int64_t>(1, blocks_for(a.num_tiles, kThreads))));
    hipLaunchKernelGGL(pair_extent_kernel, dim3(blocks), dim3(kThreads), 0, s, a.num_tiles,
                       a.meta.as<int4>(), b->row_groups.as<int>(), b->a_brange.as<int4>(),
                       b->a_blight.as<int2>(), b->pair_total.as<unsigned long long>(), flag,
                       flag_out);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

// Tile columns of B for the tile-pair numeric path: the tiles of each tile
// column J in increasing tile-row order, each as {tile row K, mask, per-k
// byte sets, payload offset | dense bit}.  A stable sort of the (class
// ordered) tiles by column keeps rows ascending within a column.
__global__ void column_keys_kernel(int64_t n, const int4 *__restrict__ meta, int *__restrict__ keys)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < n)
        keys[t] = meta[t].x;
}

__global__ void column_entries_kernel(int64_t n, const int *__restrict__ ids,
                                      const int *__restrict__ row_of,
                                      const int4 *__restrict__ meta, int4 *__restrict__ out)
{
    const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= n)
        return;
    const int t = ids[p];
    const int4 m = meta[t];
    out[p] = make_int4(row_of[t], m.y, m.z, m.w);
}

__global__ void column_longest_kernel(const int *counts, int cols, unsigned long long *host)
{
    *host = static_cast<unsigned long long>(counts[cols]);
}

int longest_b_column(const DevTiles &b, DevBuf *scratch, unsigned long long *host)
{
    hipStream_t s = ctx().stream;
    const int C = b.tile_col_count;
    RTT_TRY(scratch->ensure((static_cast<size_t>(C) + 1) * sizeof(int)));
    int *counts = scratch->as<int>();
    hipLaunchKernelGGL(fill_int_kernel, dim3(blocks_for(C + 1, kThreads)), dim3(kThreads), 0, s,
                       counts, static_cast<int64_t>(C) + 1, 0);
    if (b.num_tiles > 0) {
        hipLaunchKernelGGL(column_count_kernel, dim3(blocks_for(b.num_tiles, kThreads)),
                           dim3(kThreads), 0, s, b.num_tiles, b.tile_col_idx.as<int>(), counts);
        hipLaunchKernelGGL(column_max_kernel, dim3(blocks_for(C, kThreads)), dim3(kThreads), 0, s,
                           C, counts);
    }
    hipLaunchKernelGGL(column_longest_kernel, dim3(1), dim3(1), 0, s, counts, C, host);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int build_b_columns(DevTiles *b, BuildWork *w)
{
    if (b->transpose_of || b->cols_ready)
        return RTT_OK;   // B = A^T reads A's tile rows as its columns
    hipStream_t s = ctx().stream;
    const int64_t n = b->num_tiles;
    const int BC = b->tile_col_count;
    RTT_TRY(b->col_ptr.ensure((static_cast<size_t>(BC) + 1) * sizeof(int)));
    RTT_TRY(b->col_ent.ensure((n > 0 ? n : 1) * sizeof(int4)));
    if (n > 0) {
        RTT_TRY(fill_tile_row_of(b));
        RTT_TRY(w->keys_in.ensure(n * sizeof(int)));
        RTT_TRY(w->keys_out.ensure(n * sizeof(int)));
        RTT_TRY(w->ids_in.ensure(n * sizeof(int)));
        RTT_TRY(w->ids_out.ensure(n * sizeof(int)));
        hipLaunchKernelGGL(column_keys_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s,
                           n, b->records.as<int4>(), w->keys_in.as<int>());
        hipLaunchKernelGGL(iota_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s,
                           w->ids_in.as<int>(), n);
        RTT_TRY(sort_pairs(w->keys_in.as<int>(), w->keys_out.as<int>(), w->ids_in.as<int>(),
                           w->ids_out.as<int>(), n, bits_for(BC), &w->scan_tmp, s));
        hipLaunchKernelGGL(column_entries_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0,
                           s, n, w->ids_out.as<int>(), b->tile_row_of.as<int>(),
                           b->records.as<int4>(), b->col_ent.as<int4>());
    }
    hipLaunchKernelGGL(row_ptr_from_sorted_kernel, dim3(blocks_for(n + 1, kThreads)),
                       dim3(kThreads), 0, s, w->keys_out.as<int>(), n, BC, b->col_ptr.as<int>());
    RTT_HIP(hipGetLastError());
    b->cols_ready = true;
    return RTT_OK;
}

// An 8x4 A tile's payload re-packed column-major: entry (r, k) goes to off +
// (rows of columns < k) + (rows < r in column k).  LANES = 8: lane r takes
// tile row r (physical slots r * 4 .. r * 4 + 3), so the lanes of a
// well-filled tile read its payload as one stretch.  LANES = 1: one lane
// walks the mask of a tile of a few entries, leaving no lanes idle.
template <int LANES>
__global__ void colmajor_values_kernel(int64_t n, const int4 *__restrict__ meta,
                                       const double *__restrict__ vals, double *__restrict__ out)
{
    static_assert(LANES == 1 || LANES == 8, "a lane per tile or per tile row");
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t t = gid / LANES;
    if (t >= n)
        return;
    const int4 m = meta[t];
    const uint32_t mask = static_cast<uint32_t>(m.y);
    const uint32_t rb = static_cast<uint32_t>(m.z);
    const uint32_t w = static_cast<uint32_t>(m.w);
    const bool dense = (w & 0x80000000u) != 0;
    const uint32_t off = w & 0x7FFFFFFFu;
    if constexpr (LANES == 1) {
        int start[4];
        int acc = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            start[k] = acc;
            acc += __popc((rb >> (8 * k)) & 0xFFu);
        }
        uint32_t mm = mask;
        int j = 0;
        while (mm) {
            const int phys = __builtin_ctz(mm);
            mm &= mm - 1;
            const int r = phys >> 2, k = phys & 3;
            const uint32_t col_rows = (rb >> (8 * k)) & 0xFFu;
            out[off + start[k] + __popc(col_rows & ((1u << r) - 1u))] =
                vals[off + (dense ? phys : j)];
            ++j;
        }
    } else {
        const int r = static_cast<int>(gid & 7);
        uint32_t bits = (mask >> (4 * r)) & 0xFu;
        int rank = __popc(mask & ((1u << (4 * r)) - 1u));   // entries of rows < r (r < 8)
        while (bits) {
            const int k = __builtin_ctz(bits);
            bits &= bits - 1;
            const int before = __popc(rb & ((1u << (8 * k)) - 1u));   // rows of columns < k
            const uint32_t col_rows = (rb >> (8 * k)) & 0xFFu;
            out[off + before + __popc(col_rows & ((1u << r) - 1u))] =
                vals[off + (dense ? 4 * r + k : rank)];
            ++rank;
        }
    }
}

__global__ void row_payload_off_kernel(int rows, const int *__restrict__ trp,
                                       const int *__restrict__ off, int *__restrict__ out)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r <= rows)
        out[r] = off[trp[r]];
}

int build_transpose_source(DevTiles *t, BuildWork *w)
{
    // The longest tile column decides how the B = A^T update orders B's rows.
    const int C = t->tile_col_count;
    RTT_TRY(w->counters.ensure((static_cast<size_t>(C) + 1) * sizeof(int)));
    int *counts = w->counters.as<int>();
    hipLaunchKernelGGL(fill_int_kernel, dim3(blocks_for(C + 1, kThreads)), dim3(kThreads), 0,
                       ctx().stream, counts, static_cast<int64_t>(C) + 1, 0);
    if (t->num_tiles > 0) {
        hipLaunchKernelGGL(column_count_kernel, dim3(blocks_for(t->num_tiles, kThreads)),
                           dim3(kThreads), 0, ctx().stream, t->num_tiles,
                           t->tile_col_idx.as<int>(), counts);
        hipLaunchKernelGGL(column_max_kernel, dim3(blocks_for(C, kThreads)), dim3(kThreads), 0,
                           ctx().stream, C, counts);
    }
    int longest = 0;
    RTT_HIP(hipMemcpyAsync(&longest, counts + C, sizeof(int), hipMemcpyDeviceToHost,
                           ctx().stream));
    RTT_HIP(hipStreamSynchronize(ctx().stream));
    t->max_col_tiles = longest;
    RTT_TRY(t->row_payload_off.ensure((static_cast<size_t>(t->tile_row_count) + 1) * sizeof(int)));
    hipLaunchKernelGGL(row_payload_off_kernel, dim3(blocks_for(t->tile_row_count + 1, kThreads)),
                       dim3(kThreads), 0, ctx().stream, t->tile_row_count,
                       t->tile_row_ptr.as<int>(), t->value_offsets.as<int>(),
                       t->row_payload_off.as<int>());
    RTT_TRY(t->transpose_src.ensure(static_cast<size_t>(t->num_tiles > 0 ? t->num_tiles : 1) *
                                    sizeof(BRecord)));
    if (t->num_tiles > 0)
        hipLaunchKernelGGL(transpose_source_kernel, dim3(blocks_for(t->num_tiles * kRecParts, kThreads)),
                           dim3(kThreads), 0, ctx().stream, t->num_tiles,
                           t->tile_row_of.as<int>(), t->meta.as<int4>(), t->values_cm.as<double>(),
                           t->transpose_src.as<BRecord>());
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int build_colmajor_values(DevTiles *t)
{
    RTT_TRY(t->values_cm.ensure(static_cast<size_t>(t->payload > 0 ? t->payload : 1) *
                                sizeof(double)));
    // Tiles of a few entries on average (prolongators, Galerkin products)
    // take one lane each, fuller tiles eight.
    if (t->num_tiles > 0 && t->payload < 6 * t->num_tiles)
        hipLaunchKernelGGL((colmajor_values_kernel<1>), dim3(blocks_for(t->num_tiles, kThreads)),
                           dim3(kThreads), 0, ctx().stream, t->num_tiles, t->meta.as<int4>(),
                           t->values.as<double>(), t->values_cm.as<double>());
    else if (t->num_tiles > 0)
        hipLaunchKernelGGL((colmajor_values_kernel<8>),
                           dim3(blocks_for(t->num_tiles * 8, kThreads)), dim3(kThreads), 0,
                           ctx().stream, t->num_tiles, t->meta.as<int4>(),
                           t->values.as<double>(), t->values_cm.as<double>());
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int fill_tile_row_of(DevTiles *t)
{
    RTT_TRY(t->tile_row_of.ensure(t->num_tiles * sizeof(int)));
    if (t->tile_row_count > 0)
        hipLaunchKernelGGL(tile_row_of_kernel, dim3(blocks_for(t->tile_row_count, kThreads)),
                           dim3(kThreads), 0, ctx().stream, t->tile_row_count,
                           t->tile_row_ptr.as<int>(), t->tile_row_of.as<int>());
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int upload_csr(const rtt_smatrix &host, DevCsr *out, BuildWork *w, double *h2d_ms,
               double *validate_ms, double *sort_ms, int *rows_were_sorted)
{
    RTT_TRY(require_ctx());
    hipStream_t s = ctx().stream;
    if (host.m < 0 || host.n < 0 || host.nnz < 0 || (host.m > 0 && !host.rowpointer) ||
        (host.nnz > 0 && (!host.columnindex || !host.value)))
        return fail(RTT_ERR_INVALID, "malformed host CSR");
    auto t0 = Clock::now();
    out->rows = host.m;
    out->cols = host.n;
    out->nnz = host.nnz;
    RTT_TRY(out->row_ptr.ensure((static_cast<size_t>(host.m) + 1) * sizeof(int)));
    RTT_TRY(out->col_idx.ensure(static_cast<size_t>(host.nnz) * sizeof(int)));
    RTT_TRY(out->values.ensure(static_cast<size_t>(host.nnz) * sizeof(double)));
    if (host.m > 0)
        RTT_HIP(hipMemcpyAsync(out->row_ptr.ptr, host.rowpointer,
                               (static_cast<size_t>(host.m) + 1) * sizeof(int),
                               hipMemcpyHostToDevice, s));
    else {
        int zero = 0;
        RTT_HIP(hipMemcpyAsync(out->row_ptr.ptr, &zero, sizeof(int), hipMemcpyHostToDevice, s));
    }
    if (host.nnz > 0) {
        RTT_HIP(hipMemcpyAsync(out->col_idx.ptr, host.columnindex,
                               static_cast<size_t>(host.nnz) * sizeof(int),
                               hipMemcpyHostToDevice, s));
        RTT_HIP(hipMemcpyAsync(out->values.ptr, host.value,
                               static_cast<size_t>(host.nnz) * sizeof(double),
                               hipMemcpyHostToDevice, s));
    }
    RTT_HIP(hipStreamSynchronize(s));
    *h2d_ms = ms_since(t0);

    t0 = Clock::now();
    RTT_TRY(w->counters.ensure(sizeof(int64_t)));
    int *flags = w->counters.as<int>();   // the flags, then the longest row
    RTT_HIP(hipMemsetAsync(flags, 0, 2 * sizeof(int), s));
    const int64_t work = std::max<int64_t>(host.m, host.nnz) + 1;
    hipLaunchKernelGGL(validate_csr_kernel, dim3(blocks_for(work, kThreads)), dim3(kThreads), 0,
                       s, host.m, host.n, static_cast<int64_t>(host.nnz),
                       out->row_ptr.as<int>(), out->col_idx.as<int>(), flags, flags + 1);
    RTT_HIP(hipGetLastError());
    int got[2] = {0, 0};
    RTT_HIP(hipMemcpyAsync(got, flags, sizeof(got), hipMemcpyDeviceToHost, s));
    RTT_HIP(hipStreamSynchronize(s));
    const int hflags = got[0];
    out->max_row = got[1];
    *validate_ms = ms_since(t0);
    if (hflags & 3)
        return fail(RTT_ERR_INVALID, "CSR validation failed (flags %d)", hflags);
    *rows_were_sorted = (hflags & 4) ? 0 : 1;

    t0 = Clock::now();
    out->reordered = false;
    if (hflags & 4) {
        // Stable per-row sort by column; duplicates keep their input order.
        // input_of[x] = input position of sorted entry x, kept for value updates.
        DevBuf keys, ids_in, vals;
        RTT_TRY(keys.ensure(static_cast<size_t>(host.nnz) * sizeof(int)));
        RTT_TRY(ids_in.ensure(static_cast<size_t>(host.nnz) * sizeof(int)));
        RTT_TRY(vals.ensure(static_cast<size_t>(host.nnz) * sizeof(double)));
        RTT_TRY(out->input_of.ensure(static_cast<size_t>(host.nnz) * sizeof(int)));
        hipLaunchKernelGGL(iota_kernel, dim3(blocks_for(host.nnz, kThreads)), dim3(kThreads), 0,
                           s, ids_in.as<int>(), static_cast<int64_t>(host.nnz));
        size_t bytes = 0;
        const int *rp = out->row_ptr.as<int>();
        RTT_HIP(hipcub::DeviceSegmentedRadixSort::SortPairs(
            nullptr, bytes, out->col_idx.as<int>(), keys.as<int>(), ids_in.as<int>(),
            out->input_of.as<int>(), host.nnz, host.m, rp, rp + 1, 0, bits_for(host.n), s));
        RTT_TRY(w->scan_tmp.ensure(bytes));
        RTT_HIP(hipcub::DeviceSegmentedRadixSort::SortPairs(
            w->scan_tmp.ptr, bytes, out->col_idx.as<int>(), keys.as<int>(), ids_in.as<int>(),
            out->input_of.as<int>(), host.nnz, host.m, rp, rp + 1, 0, bits_for(host.n), s));
        hipLaunchKernelGGL(gather_f64_kernel, dim3(blocks_for(host.nnz, kThreads)),
                           dim3(kThreads), 0, s, static_cast<int64_t>(host.nnz),
                           out->input_of.as<int>(), out->values.as<double>(), vals.as<double>());
        RTT_HIP(hipGetLastError());
        RTT_HIP(hipMemcpyAsync(out->col_idx.ptr, keys.ptr,
                               static_cast<size_t>(host.nnz) * sizeof(int),
                               hipMemcpyDeviceToDevice, s));
        RTT_HIP(hipMemcpyAsync(out->values.ptr, vals.ptr,
                               static_cast<size_t>(host.nnz) * sizeof(double),
                               hipMemcpyDeviceToDevice, s));
        RTT_HIP(hipStreamSynchronize(s));
        out->reordered = true;
    }
    static std::atomic<uint64_t> next_structure_id{1};
    out->structure_id = next_structure_id.fetch_add(1);
    *sort_ms = ms_since(t0);
    return RTT_OK;
}

int transpose_tiles(const DevTiles &a, int b_cols, DevTiles *b, BuildWork *w)
{
    RTT_TRY(require_ctx());
    hipStream_t s = ctx().stream;
    const int64_t n = a.num_tiles;
    b->rows = a.cols;
    b->cols = b_cols;
    b->tile_rows = kTileK;
    b->tile_cols = kTileN;
    b->tile_row_count = a.tile_col_count;
    b->tile_col_count = (b_cols + kTileN - 1) / kTileN;
    b->num_tiles = n;
    b->payload = a.payload;
    b->dense = a.dense;
    b->sparse = a.sparse;
    b->transpose_of = &a;
    b->arrays_ready = false;
    b->has_csc = false;
    b->cols_ready = false;
    const int R = b->tile_row_count;
    const int64_t slots = static_cast<int64_t>(kClassSlots) * R;
    RTT_TRY(b->tile_row_ptr.ensure((R + 1) * sizeof(int)));
    RTT_TRY(b->row_groups.ensure((slots + 1) * sizeof(int)));
    RTT_TRY(b->sorted_ids.ensure(n * sizeof(int)));
    RTT_TRY(w->ids_in.ensure(n * sizeof(int)));
    RTT_TRY(w->keys_in.ensure(n * sizeof(int)));
    RTT_TRY(w->keys_out.ensure(n * sizeof(int)));
    RTT_TRY(b->pair_total.ensure(sizeof(unsigned long long)));
    hipLaunchKernelGGL(set_i64_kernel, dim3(1), dim3(1), 0, s, b->pair_total.as<int64_t>(),
                       int64_t(1), int64_t(0));
    if (n > 0 && a.max_col_tiles >= 0 && a.max_col_tiles <= kShortCol &&
        n < (int64_t(1) << kOrderIdBits)) {
        // The same order by counting: B's rows are short.
        RTT_TRY(w->keys_out.ensure((std::max<int64_t>(n, R + 1)) * sizeof(int)));
        int *counts = w->keys_out.as<int>();
        int *rp = b->tile_row_ptr.as<int>();
        hipLaunchKernelGGL(fill_int_kernel, dim3(blocks_for(R + 1, kThreads)), dim3(kThreads), 0,
                           s, counts, static_cast<int64_t>(R) + 1, 0);
        hipLaunchKernelGGL(column_rank_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0,
                           s, n, a.tile_col_idx.as<int>(), a.masks.as<uint32_t>(), counts,
                           w->keys_in.as<int>());
        size_t bytes = 0;
        RTT_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, counts, rp, R + 1, s));
        RTT_TRY(w->scan_tmp.ensure(bytes));
        RTT_HIP(hipcub::DeviceScan::ExclusiveSum(w->scan_tmp.ptr, bytes, counts, rp, R + 1, s));
        hipLaunchKernelGGL(column_scatter_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads),
                           0, s, n, a.tile_col_idx.as<int>(), w->keys_in.as<int>(), rp,
                           w->ids_in.as<uint32_t>());
        hipLaunchKernelGGL(order_rows_kernel, dim3(blocks_for(R, kOrderRows)), dim3(kThreads), 0,
                           s, R, n, rp, w->ids_in.as<uint32_t>(), b->sorted_ids.as<int>(),
                           b->row_groups.as<int>());
        RTT_TRY(b->records.ensure(n * sizeof(BRecord)));
        hipLaunchKernelGGL(transposed_records_kernel, dim3(blocks_for(n, kThreads)),
                           dim3(kThreads), 0, s, n, b->sorted_ids.as<int>(),
                           a.transpose_src.as<BRecord>(), b->records.as<int4>());
        RTT_HIP(hipGetLastError());
        return RTT_OK;
    }
    if (n > 0) {
        // Stable radix sort of A's tiles by (tile column, class): B's row
        // order with every row's heavy tiles first, then its light tiles by
        // the row k they occupy.
        hipLaunchKernelGGL(iota_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s,
                           w->ids_in.as<int>(), n);
        hipLaunchKernelGGL(class_keys_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s,
                           n, a.tile_col_idx.as<int>(), a.meta.as<int4>(), w->keys_in.as<int>());
        RTT_TRY(sort_pairs(w->keys_in.as<int>(), w->keys_out.as<int>(), w->ids_in.as<int>(),
                           b->sorted_ids.as<int>(), n, bits_for(slots), &w->scan_tmp, s));
        RTT_TRY(b->records.ensure(n * sizeof(BRecord)));
        hipLaunchKernelGGL(transposed_records_kernel, dim3(blocks_for(n, kThreads)),
                           dim3(kThreads), 0, s, n, b->sorted_ids.as<int>(),
                           a.transpose_src.as<BRecord>(), b->records.as<int4>());
    }
    hipLaunchKernelGGL(row_ptr_from_sorted_kernel, dim3(blocks_for(n + 1, kThreads)),
                       dim3(kThreads), 0, s, w->keys_out.as<int>(), n, static_cast<int>(slots),
                       b->row_groups.as<int>());
    hipLaunchKernelGGL(group_row_ptr_kernel, dim3(blocks_for(R + 1, kThreads)), dim3(kThreads), 0,
                       s, R, b->row_groups.as<int>(), b->tile_row_ptr.as<int>());
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int materialize_tiles(DevTiles *b, BuildWork *w)
{
    RTT_TRY(require_ctx());
    hipStream_t s = ctx().stream;
    const int64_t n = b->num_tiles;
    if (!b->arrays_ready) {
        const DevTiles &a = *b->transpose_of;
        const int R = b->tile_row_count;
        const int C = b->tile_col_count;
        RTT_TRY(b->tile_col_idx.ensure(n * sizeof(int)));
        RTT_TRY(b->masks.ensure(n * sizeof(uint32_t)));
        RTT_TRY(b->value_offsets.ensure((n + 1) * sizeof(int)));
        RTT_TRY(b->values.ensure(b->payload * sizeof(double)));
        RTT_TRY(b->tile_col_ptr.ensure((C + 1) * sizeof(int)));
        RTT_TRY(b->tile_row_idx.ensure(n * sizeof(int)));
        RTT_TRY(b->csc_tile_ids.ensure(n * sizeof(int)));
        RTT_TRY(w->spans.ensure((n + 1) * sizeof(int64_t)));
        RTT_TRY(w->counters.ensure((n + 1) * sizeof(int64_t)));
        if (n > 0) {
            // The timed update orders each B row heavy tiles first; the
            // standard arrays keep the tiles of a row in column order, which
            // a sort of A's tiles by column alone gives.
            RTT_TRY(w->ids_in.ensure(n * sizeof(int)));
            RTT_TRY(w->keys_out.ensure(n * sizeof(int)));
            RTT_TRY(w->ids_out.ensure(n * sizeof(int)));
            hipLaunchKernelGGL(iota_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, s,
                               w->ids_in.as<int>(), n);
            RTT_TRY(sort_pairs(a.tile_col_idx.as<int>(), w->keys_out.as<int>(),
                               w->ids_in.as<int>(), w->ids_out.as<int>(), n, bits_for(R),
                               &w->scan_tmp, s));
            const int *col_order = w->ids_out.as<int>();
            int64_t *spans = w->spans.as<int64_t>();
            hipLaunchKernelGGL(set_i64_kernel, dim3(1), dim3(1), 0, s, spans + n, int64_t(1),
                               int64_t(0));
            hipLaunchKernelGGL(transpose_meta_kernel, dim3(blocks_for(n, kThreads)),
                               dim3(kThreads), 0, s, n, col_order,
                               a.tile_row_of.as<int>(), a.masks.as<uint32_t>(),
                               a.value_offsets.as<int>(), b->tile_col_idx.as<int>(),
                               b->masks.as<uint32_t>(), spans, b->csc_tile_ids.as<int>());
            int64_t *off64 = w->counters.as<int64_t>();
            RTT_TRY(exclusive_scan_i64(spans, off64, n, &w->scan_tmp, s));
            hipLaunchKernelGGL(transpose_payload_kernel, dim3(blocks_for(n * 32, kThreads)),
                               dim3(kThreads), 0, s, n, col_order,
                               a.value_offsets.as<int>(), a.values.as<double>(), off64,
                               b->value_offsets.as<int>(), b->values.as<double>());
            hipLaunchKernelGGL(narrow_i64_kernel, dim3(1), dim3(1), 0, s, off64 + n,
                               b->value_offsets.as<int>() + n, int64_t(1));
            // CSC of B = CSR of A: tile_row_idx = A.tile_col_idx and
            // tile_col_ptr = A.tile_row_ptr padded to C + 1 entries.
            RTT_HIP(hipMemcpyAsync(b->tile_row_idx.ptr, a.tile_col_idx.ptr, n * sizeof(int),
                                   hipMemcpyDeviceToDevice, s));
        } else {
            int zero = 0;
            RTT_HIP(hipMemcpyAsync(b->value_offsets.ptr, &zero, sizeof(int),
                                   hipMemcpyHostToDevice, s));
        }
        const int ar = a.tile_row_count;
        RTT_HIP(hipMemcpyAsync(b->tile_col_ptr.ptr, a.tile_row_ptr.ptr, (ar + 1) * sizeof(int),
                               hipMemcpyDeviceToDevice, s));
        if (C > ar) {
            std::vector<int> tail(C - ar, static_cast<int>(n));
            RTT_HIP(hipMemcpyAsync(b->tile_col_ptr.as<int>() + ar + 1, tail.data(),
                                   tail.size() * sizeof(int), hipMemcpyHostToDevice, s));
            RTT_HIP(hipStreamSynchronize(s));
        }
        b->arrays_ready = true;
        b->has_csc = true;
    }
    if (!b->has_csc)
        RTT_TRY(build_csc(b, w));
    RTT_HIP(hipGetLastError());
    RTT_HIP(hipStreamSynchronize(s));
    return RTT_OK;
}

int transpose_csr(const DevCsr &src, DevCsr *out, BuildWork *w)
{
    RTT_TRY(require_ctx());
    hipStream_t s = ctx().stream;
    const int64_t nnz = src.nnz;
    out->rows = src.cols;
    out->cols = src.rows;
    out->nnz = nnz;
    out->max_row = -1;
    RTT_TRY(out->row_ptr.ensure((static_cast<size_t>(src.cols) + 1) * sizeof(int)));
    RTT_TRY(out->col_idx.ensure(nnz * sizeof(int)));
    RTT_TRY(out->values.ensure(nnz * sizeof(double)));
    RTT_TRY(w->row_tiles.ensure((static_cast<size_t>(src.cols) + 1) * sizeof(int64_t)));
    RTT_TRY(w->row_payload.ensure((static_cast<size_t>(src.cols) + 1) * sizeof(int64_t)));
    int64_t *cnt = w->row_tiles.as<int64_t>();
    hipLaunchKernelGGL(set_i64_kernel, dim3(blocks_for(src.cols + 1, kThreads)), dim3(kThreads),
                       0, s, cnt, static_cast<int64_t>(src.cols) + 1, int64_t(0));
    if (nnz > 0) {
        RTT_TRY(w->ids_in.ensure(nnz * sizeof(int)));
        RTT_TRY(w->ids_out.ensure(nnz * sizeof(int)));
        RTT_TRY(w->keys_out.ensure(nnz * sizeof(int)));
        RTT_TRY(w->spans.ensure(nnz * sizeof(int)));
        hipLaunchKernelGGL(histogram_kernel, dim3(blocks_for(nnz, kThreads)), dim3(kThreads), 0,
                           s, src.col_idx.as<int>(), nnz, cnt);
        hipLaunchKernelGGL(iota_kernel, dim3(blocks_for(nnz, kThreads)), dim3(kThreads), 0, s,
                           w->ids_in.as<int>(), nnz);
        RTT_TRY(sort_pairs(src.col_idx.as<int>(), w->keys_out.as<int>(), w->ids_in.as<int>(),
                           w->ids_out.as<int>(), nnz, bits_for(src.cols), &w->scan_tmp, s));
        int *entry_row = w->spans.as<int>();
        hipLaunchKernelGGL(entry_rows_kernel, dim3(blocks_for(src.rows, kThreads)),
                           dim3(kThreads), 0, s, src.rows, src.row_ptr.as<int>(), entry_row);
        hipLaunchKernelGGL(gather_transposed_kernel, dim3(blocks_for(nnz, kThreads)),
                           dim3(kThreads), 0, s, nnz, w->ids_out.as<int>(), entry_row,
                           src.values.as<double>(), out->col_idx.as<int>(),
                           out->values.as<double>());
    }
    int64_t *ptr64 = w->row_payload.as<int64_t>();
    RTT_TRY(exclusive_scan_i64(cnt, ptr64, src.cols, &w->scan_tmp, s));
    hipLaunchKernelGGL(narrow_i64_kernel, dim3(blocks_for(src.cols + 1, kThreads)),
                       dim3(kThreads), 0, s, ptr64, out->row_ptr.as<int>(),
                       static_cast<int64_t>(src.cols) + 1);
    RTT_HIP(hipGetLastError());
    return RTT_OK;
}

int nnz_cub(const DevCsr &csr, bool aat, unsigned long long *result, BuildWork *w)
{
    RTT_TRY(require_ctx());
    hipStream_t s = ctx().stream;
    RTT_TRY(w->counters.ensure(sizeof(unsigned long long)));
    unsigned long long *acc = w->counters.as<unsigned long long>();
    RTT_HIP(hipMemsetAsync(acc, 0, sizeof(unsigned long long), s));
    const int64_t *deg = nullptr;
    if (aat) {
        RTT_TRY(w->row_tiles.ensure((static_cast<size_t>(csr.cols) + 1) * sizeof(int64_t)));
        int64_t *d = w->row_tiles.as<int64_t>();
        hipLaunchKernelGGL(set_i64_kernel, dim3(blocks_for(csr.cols + 1, kThreads)),
                           dim3(kThreads), 0, s, d, static_cast<int64_t>(csr.cols) + 1,
                           int64_t(0));
        if (csr.nnz > 0)
            hipLaunchKernelGGL(histogram_kernel, dim3(blocks_for(csr.nnz, kThreads)),
                               dim3(kThreads), 0, s, csr.col_idx.as<int>(), csr.nnz, d);
        deg = d;
    }
    if (csr.nnz > 0)
        hipLaunchKernelGGL(nnz_cub_kernel,
                           dim3(static_cast<unsigned>(std::min<int64_t>(1024, blocks_for(csr.nnz, kThreads)))),
                           dim3(kThreads),
                           0, s, csr.nnz, csr.col_idx.as<int>(), csr.row_ptr.as<int>(), deg,
                           acc);
    RTT_HIP(hipGetLastError());
    RTT_HIP(hipMemcpyAsync(result, acc, sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    RTT_HIP(hipStreamSynchronize(s));
    return RTT_OK;
}

int set_csr_values(DevCsr *csr, const double *host_values, BuildWork *w)
{
    RTT_TRY(require_ctx());
    hipStream_t s = ctx().stream;
    if (csr->nnz == 0)
        return RTT_OK;
    if (!host_values)
        return fail(RTT_ERR_INVALID, "NULL values for a CSR with %lld entries",
                    (long long)csr->nnz);
    const size_t bytes = static_cast<size_t>(csr->nnz) * sizeof(double);
    if (!csr->reordered) {
        RTT_HIP(hipMemcpyAsync(csr->values.ptr, host_values, bytes, hipMemcpyHostToDevice, s));
    } else {
        RTT_TRY(w->staging.ensure(bytes));
        RTT_HIP(hipMemcpyAsync(w->staging.ptr, host_values, bytes, hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(gather_f64_kernel, dim3(blocks_for(csr->nnz, kThreads)),
                           dim3(kThreads), 0, s, csr->nnz, csr->input_of.as<int>(),
                           w->staging.as<double>(), csr->values.as<double>());
        RTT_HIP(hipGetLastError());
    }
    RTT_HIP(hipStreamSynchronize(s));
    return RTT_OK;
}

int update_b_values(const DevCsr &src, bool clear, DevTiles *b)
{
    RTT_TRY(require_ctx());
    hipStream_t s = ctx().stream;
    if (b->map_source_id == 0 || b->map_source_id != src.structure_id ||
        b->map_nnz != src.nnz || b->transpose_of)
        return fail(RTT_ERR_INVALID, "B has no source map for this CSR");
    if (clear && b->payload > 0)
        hipLaunchKernelGGL(fill_f64_kernel, dim3(blocks_for(b->payload, kThreads)),
                           dim3(kThreads), 0, s, b->values.as<double>(), b->payload, 0.0);
    if (src.nnz > 0)
        hipLaunchKernelGGL(scatter_runs_kernel, dim3(blocks_for(src.nnz, kThreads)),
                           dim3(kThreads), 0, s, src.nnz, b->src_slot.as<int>(),
                           src.values.as<double>(), b->values.as<double>());
    RTT_HIP(hipGetLastError());
    // The records are kept current only once a kernel has asked for them
    // (ensure_record_values); otherwise they are written when next needed.
    if (b->rec_values_ready)
        RTT_TRY(write_record_values(b));
    return RTT_OK;
}

int nnz_cub_ab(const DevCsr &a, const DevCsr &b, unsigned long long *result, BuildWork *w)
{
    RTT_TRY(require_ctx());
    if (a.cols != b.rows)
        return fail(RTT_ERR_INVALID, "A has %d columns but B has %d rows", a.cols, b.rows);
    hipStream_t s = ctx().stream;
    RTT_TRY(w->counters.ensure(sizeof(unsigned long long)));
    unsigned long long *acc = w->counters.as<unsigned long long>();
    RTT_HIP(hipMemsetAsync(acc, 0, sizeof(unsigned long long), s));
    if (a.nnz > 0)
        hipLaunchKernelGGL(nnz_cub_kernel,
                           dim3(static_cast<unsigned>(std::min<int64_t>(1024, blocks_for(a.nnz, kThreads)))),
                           dim3(kThreads), 0, s, a.nnz, a.col_idx.as<int>(), b.row_ptr.as<int>(),
                           static_cast<const int64_t *>(nullptr), acc);
    RTT_HIP(hipGetLastError());
    RTT_HIP(hipMemcpyAsync(result, acc, sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    RTT_HIP(hipStreamSynchronize(s));
    return RTT_OK;
}

} // namespace rtt
