// ESC SpGEMM (Z_ik = sum_j A_ij B_jk, CSR x CSR -> CSR) for gfx950 with 64-bit product and
// result offsets.
//
// Reference path replaced: the spgemm kernel (compiler.cpp:145-148), lowered as a scatter
// reduction (compile.cpp:40-72): an expand phase partitioned over the intermediate-product
// count (compile.cpp:122-221, partition.cpp:1039-1193), then CUB DeviceSegmentedSort by column
// within each row, mark_heads / InclusiveSum / extract_offsets and a warp-32 segmented scan
// with atomicAdd (stitch_and_generate_gpu.cpp:14-138, 257-366).  The reference keeps every
// count in int32, which the R-MAT scale-20 square (6.0e9 products, 3.6e9 results) overflows.
//
// Pipeline (every count and offset is int64):
//   1. sizes: a row's products are the lengths of its A entries' B rows; exclusive scan ->
//      row_off, P: row i's products are [row_off[i], row_off[i+1]) in natural (j, k) order.
//      (Small products are bound by launches and waits for counts: the scans of one step run
//      together, counts reach the host through pinned words, and steps of long rows are
//      skipped where there are none; 2^8 vertices 251 -> 129 us, 2^13 412 -> 316 us.)
//   2. segments: a row with at most kShort products is one segment.  A longer row is split by
//      column into nb buckets of 2^shift columns (one device-wide radix digit, k >> shift);
//      each bucket is a segment.  Segments are numbered row-major, bucket-minor, so their
//      concatenation in order is every row's products grouped by column range.
//   3. expand to runs: a product (k, a_ij * b_jk) is never written to memory.  B's rows are
//      cut into runs of equal column bucket; a segment's products are the concatenation of
//      its runs, each run one A entry times a contiguous range of one B row, described by
//      {first B entry, length, a_ij} (a short row's runs are its A entries' whole B rows, in
//      natural order; a long row's runs of bucket b come from B's run table).  A histogram
//      over B's runs gives each long-row segment's products and runs without visiting a
//      product; scans give segment product offsets and run offsets; the run descriptors are
//      then written per segment (4.4e8 of 16 bytes at C4, against 6.0e9 products of 8).
//   4. units: a segment with more than kShort products is a dense unit; smaller segments
//      whose first product falls in the same kShort-aligned window share one sort unit
//      (fewer than 2*kShort products), or one bitmap unit when they are at most
//      kMaxBitmapBuckets narrow column buckets of long rows.  Each kind gets a compacted list.
//   5. reduce: a unit expands its runs, gathering (k, a_ij * b_jk) from B.  A sort unit sorts
//      (segment ordinal, k) in LDS and sums each run of equal keys in float64; a bitmap unit
//      ranks each bucket's columns in an LDS bitmap and sums by rank; a dense unit accumulates
//      its 2^shift-column range in an LDS float64 array (windows of kDenseCols columns) and
//      compacts the touched columns in order.  All write the distinct (k, sum rounded once to
//      float32) at the unit's product offset in an output staging buffer and record the
//      unit's count and the local offset of every row starting in it.
//   6. output, sized one of two ways (output_mode).  Staged: the units write at their product
//      offsets in a staging buffer; a scan of unit counts gives result offsets, each unit's
//      entries are copied, row offsets come from the unit offsets.  Symbolic (columns below
//      2^20): before the runs, a symbolic pass counts every segment's distinct columns from
//      A and B (long rows in an LDS bitmap of the row's columns, short rows in a per-wave LDS
//      hash table); their scan gives segment and row offsets, the result is allocated at its
//      exact size and the units write straight into it.  Every distinct column is kept
//      (structural result, as the reference).
// Summation order inside a segment follows the runs' order and LDS atomics, so values are
// reproducible to within one float32 rounding of the float64 sum (the reference's own order
// is not deterministic either).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#include "device_utils.hpp"
#include "runtime.hpp"
#include "scan.hpp"

namespace nacho {
namespace spgemm {

constexpr int kBlock = 256;
constexpr int kTile = 4096;             // LDS capacity of a sort unit
constexpr int kPer = kTile / kBlock;    // 16 positions per lane
constexpr int kShort = kTile / 2;       // segments with at most this many products are sorted
constexpr int kOrdBits = 12;            // a sort unit holds fewer than 2^12 segments
constexpr int kDenseBits = 13;          // dense accumulation window: 8192 columns
constexpr int kDenseCols = 1 << kDenseBits;
constexpr int kMaxBucketBits = 10;      // at most 1024 column buckets per long row
constexpr int kMaxBuckets = 1 << kMaxBucketBits;
// A long row's bucket with more products than this is accumulated densely (its 8192-column
// window in LDS) rather than by a bitmap or sort unit.  At C4, 1536 / 2048 (one box, two
// rounds): 95.46 / 95.45 against 96.66 / 95.98 ms; 1024 and 1280 lose.
constexpr int kDenseMin = 1536;
constexpr int kMaxBitmapSegs = 256;     // segments (empty ones included) of a bitmap unit
constexpr int kMaxBitmapBuckets = 32;   // nonempty buckets of a bitmap unit (larger buckets)
constexpr int kBitmapWords = 8192 / 32; // one bit per column of an 8192-column bucket
constexpr int kBitmapBlock = 512;       // threads of a bitmap unit's workgroup
constexpr int kHistGrid = 8192;         // workgroups of the long-row histogram
// Units in list order on one XCD at a time, kXcdGroup consecutive ones per XCD: a long row's
// neighbouring buckets gather adjacent ranges of the same B rows, which then share one L2.
// At C4 the unit kernels fetched 124 -> 105 GB per call (96.97 -> 95.58 ms) with groups of
// 64; one contiguous range per XCD fetched as little but took 102.2 ms (the XCDs' loads no
// longer matched).  Groups of 128 / 256 against 64, one box, two rounds each: 96.10 / 95.88,
// 95.67 / 95.54 against 96.66 / 95.98 ms.
constexpr unsigned kXcdGroup = 256;

static_assert(kTile == 1 << kOrdBits, "segment ordinals must fit kOrdBits");
static_assert(kTile == kBlock * kPer, "a unit's products are kPer per lane");

// ---- small device helpers --------------------------------------------------------------

// LDS index with one pad word per kPer words: a lane's kPer consecutive (blocked) positions
// then start kPer + 1 words after its neighbour's, so blocked accesses are free of bank
// conflicts.
constexpr int kPadded = kTile + kTile / 16;
__device__ __forceinline__ int pad(int i) { return i + (i >> 4); }

using dev::last_le;

// ---- 1-2: sizes and segments -----------------------------------------------------------

// Per row of A: its products, the A entries whose B row is not empty, its segments (1, or nb
// for a long row) and, for a long row, its work blocks of kBlock A entries.
struct RowCounts {
    int64_t *products;
    int *entries;
    int64_t *segments;
    int64_t *blocks;
    int nb;
    // One entry of A, in column j.
    static __device__ __forceinline__ void add(const int *__restrict__ pos_b, int j, int64_t &sum,
                                               int &some) {
        const int n = pos_b[j + 1] - pos_b[j];
        sum += n;
        some += n > 0 ? 1 : 0;
    }
    __device__ __forceinline__ void store(int64_t row, int len, int64_t sum, int some) const {
        products[row] = sum;
        entries[row] = some;
        finish(row, len, sum);
    }
    __device__ __forceinline__ void finish(int64_t row, int len, int64_t sum) const {
        segments[row] = sum > kShort ? nb : 1;
        blocks[row] = sum > kShort ? (len + kBlock - 1) / kBlock : 0;
    }
};

// LANES lanes per row.  A row of more than kWave entries is taken by its whole wavefront or, with
// `split`, only zeroed: long_products_kernel adds it up.
constexpr int kRowLanes = 8;
constexpr int kOneLaneEntries = 4;  // per row on average, below which a row takes one lane
// A's entries from which long rows are split: R-MAT graphs hold their longest rows side by side,
// and one wavefront for each took 364 us at scale 20 (both kernels now: 176).  The launch costs
// 3 us, a wavefront 80 us for all of fewer entries at worst.
constexpr int64_t kSplitEntries = int64_t{1} << 15;

template <int LANES>
__global__ __launch_bounds__(kBlock) void row_products_kernel(
    const int *__restrict__ pos_a, const int *__restrict__ crd_a, int rows,
    const int *__restrict__ pos_b, bool split, RowCounts out) {
    const int l = dev::lane();
    const int64_t i = (blockIdx.x * static_cast<int64_t>(kBlock) + threadIdx.x) / LANES;
    const bool lead = l % LANES == 0;
    int s = 0, e = 0;
    if (i < rows) {
        s = pos_a[i];
        e = pos_a[i + 1];
    }
    const bool is_long = e - s > dev::kWave;
    int64_t sum = 0;
    int some = 0;
    if (!is_long) {
#pragma unroll 4
        for (int p = s + l % LANES; p < e; p += LANES) out.add(pos_b, crd_a[p], sum, some);
    }
#pragma unroll
    for (int d = LANES / 2; d > 0; d >>= 1) {
        sum += __shfl_xor(sum, d, dev::kWave);
        some += __shfl_xor(some, d, dev::kWave);
    }
    if (lead && i < rows && !is_long) out.store(i, e - s, sum, some);
    if (split) {  // uniform
        if (lead && is_long) {
            out.products[i] = out.segments[i] = 0;
            out.entries[i] = 0;
        }
        return;
    }
    unsigned long long rest = __ballot(is_long && lead);
    while (rest) {  // uniform
        const int src = __ffsll(static_cast<long long>(rest)) - 1;
        rest &= rest - 1;
        const int hs = __shfl(s, src, dev::kWave), he = __shfl(e, src, dev::kWave);
        sum = 0;
        some = 0;
#pragma unroll 4
        for (int p = hs + l; p < he; p += dev::kWave) out.add(pos_b, crd_a[p], sum, some);
        sum = dev::wave_sum(sum);
        some = dev::wave_sum(some);
        if (l == src) out.store(i, e - s, sum, some);
    }
}

// The rows of more than kWave entries: workgroup b takes A's entries [b * kLongSpan,
// (b + 1) * kLongSpan), its wavefronts kLongPart entries of one such row among them at a time.
// The parts of a row that reaches into several spans are added where they are counted, its
// segments' word counts the parts, and the workgroup that adds the last one stores what follows
// from the sum.
constexpr int kLongSpan = 4096;
constexpr int kLongPart = 4 * dev::kWave;

__global__ __launch_bounds__(kBlock) void long_products_kernel(
    const int *__restrict__ pos_a, const int *__restrict__ crd_a, int rows, int64_t nnz_a,
    const int *__restrict__ pos_b, RowCounts out) {
    constexpr int kWaves = kBlock / dev::kWave;
    __shared__ int s_ends[2];
    constexpr int kRows = kLongSpan / dev::kWave + 2;  // (the first and last may reach outside)
    __shared__ int s_row[kRows];
    __shared__ int s_rows;
    __shared__ unsigned long long s_sum[kRows];
    __shared__ int s_some[kRows];
    const int lo = static_cast<int>(blockIdx.x) * kLongSpan;
    const int hi = static_cast<int>(min(static_cast<int64_t>(lo) + kLongSpan, nnz_a));
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / dev::kWave), l = dev::lane();
    if (w < 2) {  // the row of the first and of the last entry
        const int at = w == 0 ? lo : hi - 1;
        const int r = dev::group_last_true<dev::kWave>(0, rows - 1,
                                                       [&](int x) { return pos_a[x] <= at; });
        if (l == 0) s_ends[w] = r;
    }
    if (threadIdx.x == 0) s_rows = 0;
    if (threadIdx.x < kRows) {
        s_sum[threadIdx.x] = 0;
        s_some[threadIdx.x] = 0;
    }
    __syncthreads();
    for (int r = s_ends[0] + static_cast<int>(threadIdx.x); r <= s_ends[1]; r += kBlock) {
        const int e = pos_a[r + 1];
        if (e - pos_a[r] > dev::kWave && e > lo) s_row[atomicAdd(&s_rows, 1)] = r;
    }
    __syncthreads();
    for (int k = 0; k < s_rows; ++k) {
        const int row = s_row[k];
        const int s = max(pos_a[row], lo), e = min(pos_a[row + 1], hi);
        // (row k's first part is wavefront k's: most rows have one)
        for (int at = s + ((w - k) & (kWaves - 1)) * kLongPart; at < e; at += kWaves * kLongPart) {
            int64_t sum = 0;
            int some = 0;
#pragma unroll
            for (int u = 0; u < kLongPart; u += dev::kWave) {
                if (at + u + l < e) out.add(pos_b, crd_a[at + u + l], sum, some);
            }
            sum = dev::wave_sum(sum);
            some = dev::wave_sum(some);
            if (l == 0) {
                atomicAdd(&s_sum[k], static_cast<unsigned long long>(sum));
                atomicAdd(&s_some[k], some);
            }
        }
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) >= s_rows) return;
    const int row = s_row[threadIdx.x], some = s_some[threadIdx.x];
    const unsigned long long sum = s_sum[threadIdx.x];
    const int s = pos_a[row], e = pos_a[row + 1];
    if (s >= lo && e <= hi) {
        out.store(row, e - s, static_cast<int64_t>(sum), some);
        return;
    }
    auto *products = reinterpret_cast<unsigned long long *>(&out.products[row]);
    auto *parts = reinterpret_cast<unsigned long long *>(&out.segments[row]);
    atomicAdd(products, sum);
    atomicAdd(&out.entries[row], some);
    const unsigned long long before =
        __hip_atomic_fetch_add(parts, 1ull, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (before == static_cast<unsigned long long>((e - 1) / kLongSpan - s / kLongSpan)) {
        out.finish(row, e - s,
                   static_cast<int64_t>(__hip_atomic_load(products, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT)));
    }
}

// Segment table: row of each segment, product and run counts (short rows known now: one run
// per A entry whose B row is not empty; long rows counted by the histogram pass) and the
// zeroed fill counters of the long rows' run emission.  blk_row[b] = the row of work block b
// (kBlock consecutive A entries of one long row; blocks numbered by the scan blk_off).
__global__ void segments_kernel(const int64_t *__restrict__ row_off,
                                const int64_t *__restrict__ seg_prefix, int rows,
                                const int *__restrict__ entries,
                                const int64_t *__restrict__ blk_off, int *__restrict__ blk_row,
                                int *__restrict__ seg_row, int64_t *__restrict__ seg_len,
                                int64_t *__restrict__ seg_runs, int64_t *__restrict__ seg_fill) {
    // One row per lane; a long row's segments (one per column bucket) are then written by
    // the whole wavefront, 64 consecutive segments per store, instead of by its own lane.
    const int l = dev::lane();
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i0 = static_cast<int64_t>(blockIdx.x) * blockDim.x + (threadIdx.x - l);
         i0 < rows; i0 += stride) {  // uniform per wavefront
        const int i = static_cast<int>(i0) + l;
        int64_t s0 = 0, s1 = 0, runs = 0, prod = 0;
        if (i < rows) {
            s0 = seg_prefix[i];
            s1 = seg_prefix[i + 1];
            prod = row_off[i + 1] - row_off[i];
            if (prod <= kShort) runs = entries[i];
            for (int64_t b = blk_off[i]; b < blk_off[i + 1]; ++b) blk_row[b] = i;
            if (s1 - s0 == 1) {  // a short row's single segment
                seg_row[s0] = i;
                seg_len[s0] = prod > kShort ? 0 : prod;
                seg_runs[s0] = runs;
                seg_fill[s0] = 0;
            }
        }
        unsigned long long many = __ballot(i < rows && s1 - s0 > 1);
        while (many) {  // uniform
            const int src = __ffsll(static_cast<long long>(many)) - 1;
            many &= many - 1;
            const int64_t a0 = __shfl(s0, src, dev::kWave), a1 = __shfl(s1, src, dev::kWave);
            const int row = __shfl(i, src, dev::kWave);
            const int64_t plen = __shfl(prod, src, dev::kWave);
            const int64_t prun = __shfl(runs, src, dev::kWave);
            for (int64_t sg = a0 + l; sg < a1; sg += dev::kWave) {
                seg_row[sg] = row;
                seg_len[sg] = plen > kShort ? 0 : plen;
                seg_runs[sg] = prun;
                seg_fill[sg] = 0;
            }
        }
    }
}

// ---- 3a: long-row histogram from B's column-bucket runs --------------------------------
//
// Long rows need their products counted per column bucket before the scatter.  B's rows
// have sorted columns, so each B row is a short list of runs of equal bucket (at most nb,
// however long the row); a long row's bucket counts are the sums of its B rows' run
// lengths.  At C4 (R-MAT 2^20, 128 buckets) this is 4.3e8 run visits instead of 5.9e9
// products.

// B's columns and value bits as one array of pairs, read by the reduce units' gathers, and
// (flag not null) flag[p] = 1 where B entry p starts a run: its bucket differs from entry
// p - 1's.  Row starts are flagged by run_row_starts_kernel, launched after this one.
__global__ void pairs_flags_kernel(const int *__restrict__ crd_b, const float *__restrict__ val_b,
                                   int64_t nnz_b, int shift, int2 *__restrict__ cv_b,
                                   int64_t *__restrict__ flag) {
    for (int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; p < nnz_b;
         p += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int c = crd_b[p];
        cv_b[p] = make_int2(c, __float_as_int(val_b[p]));
        if (flag) flag[p] = (p == 0 || (c >> shift) != (crd_b[p - 1] >> shift)) ? 1 : 0;
    }
}

__global__ void run_row_starts_kernel(const int *__restrict__ pos_b, int rows_b,
                                      int64_t *__restrict__ flag) {
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rows_b; r += gridDim.x * blockDim.x) {
        if (pos_b[r] < pos_b[r + 1]) flag[pos_b[r]] = 1;
    }
}

// Run q (numbered by the exclusive scan run_idx of the flags): its bucket (run[q].x) and
// its first B entry; run_start[total runs] = nnz_b closes the last run.  B row k's runs are
// [run_idx[pos_b[k]], run_idx[pos_b[k + 1]]).
__global__ void runs_kernel(const int *__restrict__ crd_b, int64_t nnz_b, int shift,
                            const int64_t *__restrict__ flag, const int64_t *__restrict__ run_idx,
                            int2 *__restrict__ run, int *__restrict__ run_start) {
    for (int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; p < nnz_b;
         p += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        if (flag[p]) {
            const int64_t q = run_idx[p];
            run[q].x = crd_b[p] >> shift;
            run_start[q] = static_cast<int>(p);
        }
        if (p == 0) run_start[run_idx[nnz_b]] = static_cast<int>(nnz_b);
    }
}

// run[q].y = the length of run q (runs numbered below run_idx[nnz_b]).
__global__ void run_lengths_kernel(const int64_t *__restrict__ run_idx, int64_t nnz_b,
                                   const int *__restrict__ run_start, int2 *__restrict__ run) {
    const int64_t n_runs = run_idx[nnz_b];
    for (int64_t q = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; q < n_runs;
         q += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        run[q].y = run_start[q + 1] - run_start[q];
    }
}

// B row k's runs, packed (bucket, length) in run[] and first entries in run_start[].
struct BRuns {
    const int64_t *run_idx;  // B row k's runs are [run_idx[pos_b[k]], run_idx[pos_b[k + 1]])
    const int2 *run;
    const int *run_start;
};

// The runs of a work block's A entries, dealt evenly over the workgroup: an A entry's B row
// may hold one run or a hundred (a hub), so one lane per entry leaves most lanes of a
// wavefront waiting for its longest.  Every lane publishes its entry's run count, first run
// and A value; the block's T runs (entry by entry) are then taken kRunsPer per lane per
// round, run j by lane j mod kBlock, which finds the entry owning j with a fixed eight-step
// search of the entries' run offsets in LDS (the kRunsPer searches interleaved).
constexpr int kRunsPer = 4;

struct BlockRuns {
    int off[kBlock];      // exclusive scan of the entries' run counts
    int64_t q0[kBlock];   // first run of the entry's B row in br.run
    float a[kBlock];      // the entry's A value
    int wave[kBlock / dev::kWave];
};

// Publishes this lane's entry (n_runs runs from q0, A value a); returns T.  Ends synchronised.
__device__ __forceinline__ int publish_runs(BlockRuns &sh, int n_runs, int64_t q0, float a) {
    int total = 0;
    const int off = dev::block_exclusive_sum<kBlock>(n_runs, sh.wave, total);
    sh.off[threadIdx.x] = off;
    sh.q0[threadIdx.x] = q0;
    sh.a[threadIdx.x] = a;
    __syncthreads();
    return total;
}

// Run j of the block (j < T): its index in br.run and its entry's A value.
__device__ __forceinline__ void block_run(const BlockRuns &sh, int j, int64_t &q, float &a) {
    int lo = 0;  // last entry whose first run is at or before j (off[0] = 0)
#pragma unroll
    for (int step = kBlock / 2; step > 0; step >>= 1) {
        lo += sh.off[lo + step] <= j ? step : 0;
    }
    q = sh.q0[lo] + (j - sh.off[lo]);
    a = sh.a[lo];
}

// Work blocks strided over the grid (a heavy row's blocks land on different workgroups):
// every thread takes one A entry of the block and adds, per run of its B row, the run's
// length and one run to LDS histograms of the row's buckets; nonzero bins are then added to
// the row's seg_len and seg_runs (zeroed by segments_kernel), stored directly when the row
// has a single block.
__global__ __launch_bounds__(kBlock) void long_hist_kernel(
    const int *__restrict__ pos_a, const int *__restrict__ crd_a,
    const int64_t *__restrict__ blk_off, const int *__restrict__ blk_row, int rows,
    const int *__restrict__ pos_b, BRuns br, int nb, const int64_t *__restrict__ seg_prefix,
    int64_t *__restrict__ seg_len, int64_t *__restrict__ seg_runs) {
    __shared__ int s_hist[kMaxBuckets];
    __shared__ int s_runs[kMaxBuckets];
    __shared__ BlockRuns sh;
    const int64_t n_blk = blk_off[rows];
    for (int64_t blk = blockIdx.x; blk < n_blk; blk += gridDim.x) {
        const int i = blk_row[blk];
        const int64_t first = blk_off[i];
        for (int b = threadIdx.x; b < nb; b += kBlock) {
            s_hist[b] = 0;
            s_runs[b] = 0;
        }
        const int p = pos_a[i] + static_cast<int>(blk - first) * kBlock + threadIdx.x;
        int64_t q0 = 0;
        int n_runs = 0;
        if (p < pos_a[i + 1]) {
            const int k = crd_a[p];
            q0 = br.run_idx[pos_b[k]];
            n_runs = static_cast<int>(br.run_idx[pos_b[k + 1]] - q0);
        }
        // (its barriers also order the clears above before the adds below)
        const int T = publish_runs(sh, n_runs, q0, 0.0f);
        for (int j0 = 0; j0 < T; j0 += kRunsPer * kBlock) {  // uniform
            int2 x[kRunsPer];
#pragma unroll
            for (int u = 0; u < kRunsPer; ++u) {
                int64_t q;
                float a;
                block_run(sh, min(j0 + u * kBlock + static_cast<int>(threadIdx.x), T - 1), q, a);
                x[u] = br.run[q];
            }
#pragma unroll
            for (int u = 0; u < kRunsPer; ++u) {
                if (j0 + u * kBlock + static_cast<int>(threadIdx.x) < T && x[u].x < nb) {
                    atomicAdd(&s_hist[x[u].x], x[u].y);
                    atomicAdd(&s_runs[x[u].x], 1);
                }
            }
        }
        __syncthreads();
        const int64_t s0 = seg_prefix[i];
        const bool alone = blk_off[i + 1] - first == 1;
        for (int b = threadIdx.x; b < nb; b += kBlock) {
            const int c = s_hist[b], n = s_runs[b];
            if (alone) {
                seg_len[s0 + b] = c;
                seg_runs[s0 + b] = n;
            } else if (c > 0) {
                atomicAdd(reinterpret_cast<unsigned long long *>(&seg_len[s0 + b]),
                          static_cast<unsigned long long>(c));
                atomicAdd(reinterpret_cast<unsigned long long *>(&seg_runs[s0 + b]),
                          static_cast<unsigned long long>(n));
            }
        }
        __syncthreads();  // the histograms are read before the next block clears them
    }
}

// ---- 3b: run descriptors -----------------------------------------------------------------

// A run of products: B entries [x, x + y) times the A value with bits z (w unused).
__device__ __forceinline__ int4 make_run(int first, int length, float a) {
    return make_int4(first, length, __float_as_int(a), 0);
}

// Long rows: the same work blocks as the histogram.  Each bucket's runs from the block are
// counted in LDS, a range of the segment's run slots is reserved with one atomic per
// nonempty bucket (none when the row has a single block), and every run is written at the
// next slot of its bucket's range.  The order of runs inside a segment is free: the reduce
// is order-independent (up to float64 rounding).  (Staging a block's runs in LDS to store
// each bucket's range coalesced cost more in occupancy than it saved: 8.4 -> 12.6 ms at C4.)
__global__ __launch_bounds__(kBlock) void long_runs_kernel(
    const int *__restrict__ pos_a, const int *__restrict__ crd_a, const float *__restrict__ val_a,
    const int64_t *__restrict__ blk_off, const int *__restrict__ blk_row, int rows,
    const int *__restrict__ pos_b, BRuns br, int nb, const int64_t *__restrict__ seg_prefix,
    const int64_t *__restrict__ seg_roff, int64_t *__restrict__ seg_fill,
    int4 *__restrict__ desc) {
    __shared__ int s_cnt[kMaxBuckets];
    __shared__ int64_t s_base[kMaxBuckets];
    __shared__ BlockRuns sh;
    const int64_t n_blk = blk_off[rows];
    for (int64_t blk = blockIdx.x; blk < n_blk; blk += gridDim.x) {
        const int i = blk_row[blk];
        const int64_t first = blk_off[i];
        for (int b = threadIdx.x; b < nb; b += kBlock) s_cnt[b] = 0;
        const int p = pos_a[i] + static_cast<int>(blk - first) * kBlock + threadIdx.x;
        int64_t q0 = 0;
        int n_runs = 0;
        float a_mine = 0.0f;
        if (p < pos_a[i + 1]) {
            const int k = crd_a[p];
            a_mine = val_a[p];
            q0 = br.run_idx[pos_b[k]];
            n_runs = static_cast<int>(br.run_idx[pos_b[k + 1]] - q0);
        }
        // (its barriers also order the clears above before the counts below)
        const int T = publish_runs(sh, n_runs, q0, a_mine);
        for (int j0 = 0; j0 < T; j0 += kRunsPer * kBlock) {  // uniform
            int2 x[kRunsPer];
#pragma unroll
            for (int u = 0; u < kRunsPer; ++u) {
                int64_t q;
                float a;
                block_run(sh, min(j0 + u * kBlock + static_cast<int>(threadIdx.x), T - 1), q, a);
                x[u] = br.run[q];
            }
#pragma unroll
            for (int u = 0; u < kRunsPer; ++u) {
                if (j0 + u * kBlock + static_cast<int>(threadIdx.x) < T && x[u].x < nb) {
                    atomicAdd(&s_cnt[x[u].x], 1);
                }
            }
        }
        __syncthreads();
        const int64_t s0 = seg_prefix[i];
        const bool alone = blk_off[i + 1] - first == 1;
        for (int b = threadIdx.x; b < nb; b += kBlock) {
            const int c = s_cnt[b];
            int64_t at = 0;
            if (c > 0 && !alone) {
                at = static_cast<int64_t>(atomicAdd(
                    reinterpret_cast<unsigned long long *>(&seg_fill[s0 + b]),
                    static_cast<unsigned long long>(c)));
            }
            s_base[b] = seg_roff[s0 + b] + at;
            s_cnt[b] = 0;
        }
        __syncthreads();
        for (int j0 = 0; j0 < T; j0 += kRunsPer * kBlock) {  // uniform
            int2 x[kRunsPer];
            int first_b[kRunsPer];
            float av[kRunsPer];
#pragma unroll
            for (int u = 0; u < kRunsPer; ++u) {
                int64_t q;
                block_run(sh, min(j0 + u * kBlock + static_cast<int>(threadIdx.x), T - 1), q,
                          av[u]);
                x[u] = br.run[q];
                first_b[u] = br.run_start[q];
            }
#pragma unroll
            for (int u = 0; u < kRunsPer; ++u) {
                if (j0 + u * kBlock + static_cast<int>(threadIdx.x) < T && x[u].x < nb) {
                    const int64_t slot = s_base[x[u].x] + atomicAdd(&s_cnt[x[u].x], 1);
                    desc[slot] = make_run(first_b[u], x[u].y, av[u]);
                }
            }
        }
        __syncthreads();  // s_cnt, s_base and sh are read before the next block resets them
    }
}

// Short rows: one run per A entry whose B row is not empty, in natural order (the row's
// products in their natural order).  One thread per row.
__global__ void short_runs_kernel(const int *__restrict__ pos_a, const int *__restrict__ crd_a,
                                  const float *__restrict__ val_a, int rows,
                                  const int64_t *__restrict__ row_off,
                                  const int64_t *__restrict__ seg_prefix,
                                  const int64_t *__restrict__ seg_roff,
                                  const int *__restrict__ pos_b, int4 *__restrict__ desc) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows; i += gridDim.x * blockDim.x) {
        const int64_t prod = row_off[i + 1] - row_off[i];
        if (prod == 0 || prod > kShort) continue;
        int64_t slot = seg_roff[seg_prefix[i]];
        for (int p = pos_a[i]; p < pos_a[i + 1]; ++p) {
            const int k = crd_a[p];
            const int b0 = pos_b[k], b1 = pos_b[k + 1];
            if (b1 > b0) desc[slot++] = make_run(b0, b1 - b0, val_a[p]);
        }
    }
}

// Products by windows: the runs of up to kTile products laid end to end, each window of 64
// consecutive products a wavefront's, lane x on product x, so that a window's gathers are
// consecutive entries of a few runs (R-MAT scale 20: 14 products per run) and a product's run
// costs two bit counts.  Eight consecutive products per lane instead (a search or a running
// maximum for the first, then a walk; every gather instruction on 64 cache lines) took 35.4 ms
// in the bitmap units, 17.3 ms in the dense units and 13.4 ms in the sort units at scale 20;
// windows 31.4, 15.3 and 12.7.  s_mask has a bit per product that starts a run (every
// run has at least one product); lane l of a wavefront keeps word l and the number of bits
// before it, and a product's run is a count of bits.
struct RunWindows {
    unsigned long long word;
    int before;
    // Run of lane l's product in window i (uniform), counted from `before`'s first run.
    __device__ __forceinline__ int run(int i) const {
        const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readlane(
            static_cast<int>(static_cast<unsigned>(word)), i));
        const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readlane(
            static_cast<int>(static_cast<unsigned>(word >> 32)), i));
        const unsigned long long m = (static_cast<unsigned long long>(hi) << 32) | lo;
        // the bits up to lane l's own: those below it, and its own
        const int own = __builtin_amdgcn_inverse_ballot_w64(m) ? 1 : 0;
        return __builtin_amdgcn_readlane(before, i) +
               static_cast<int>(__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u))) +
               own - 1;
    }
};

__device__ __forceinline__ RunWindows load_windows(const unsigned *s_mask, int first) {
    const unsigned long long word = reinterpret_cast<const unsigned long long *>(s_mask)[dev::lane()];
    const int bits = __popcll(word);
    return RunWindows{word, first + dev::wave_inclusive_sum(bits) - bits};
}

// ---- 4: units --------------------------------------------------------------------------

// A segment is accumulated densely when it has more than kShort products, or more than
// dense_min products and is a column bucket of a long row (dense_min is kShort when buckets
// are wider than one kDenseCols window).  Dense accumulation costs a fixed LDS clear and
// scan of the window plus one atomic per product; sorting costs several passes per product.
__device__ __forceinline__ bool dense_segment(int64_t len, int64_t s,
                                              const int *__restrict__ seg_row,
                                              const int64_t *__restrict__ row_off,
                                              int dense_min) {
    if (len > kShort) return true;
    if (len <= dense_min) return false;
    const int r = seg_row[s];
    return row_off[r + 1] - row_off[r] > kShort;
}

// Units owned by segment s: 1 for a dense segment and for the first nonempty sorted segment
// whose products start in a kShort window (the previous nonempty segment is dense or starts
// in an earlier window); 0 otherwise.
__global__ void unit_count_kernel(const int64_t *__restrict__ seg_len,
                                  const int64_t *__restrict__ seg_off, int64_t n_seg,
                                  const int *__restrict__ seg_row,
                                  const int64_t *__restrict__ row_off, int dense_min,
                                  int64_t *__restrict__ seg_units) {
    for (int64_t s = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; s < n_seg;
         s += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t len = seg_len[s], start = seg_off[s];
        int64_t u;
        if (len == 0) {
            u = 0;
        } else if (start == 0 || dense_segment(len, s, seg_row, row_off, dense_min)) {
            u = 1;
        } else {
            // previous nonempty segment: last x < s with seg_off[x] < start
            int64_t lo = 0, hi = s - 1;
            while (lo < hi) {
                const int64_t mid = (lo + hi + 1) >> 1;
                if (seg_off[mid] < start) {
                    lo = mid;
                } else {
                    hi = mid - 1;
                }
            }
            const int64_t ps = seg_off[lo];
            u = (dense_segment(start - ps, lo, seg_row, row_off, dense_min) ||
                 ps / kShort != start / kShort)
                    ? 1
                    : 0;
        }
        seg_units[s] = u;
    }
}

// Unit table: first segment and product offset of each unit, and whether it is dense.
__global__ void unit_map_kernel(const int64_t *__restrict__ seg_units,
                                const int64_t *__restrict__ unit_prefix,
                                const int64_t *__restrict__ seg_off,
                                const int64_t *__restrict__ seg_len,
                                const int *__restrict__ seg_row,
                                const int64_t *__restrict__ row_off, int dense_min,
                                int64_t n_seg, int64_t P, int *__restrict__ unit_seg,
                                int64_t *__restrict__ unit_start,
                                int64_t *__restrict__ unit_dense) {
    for (int64_t s = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; s <= n_seg;
         s += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        if (s == n_seg) {
            unit_start[unit_prefix[n_seg]] = P;
        } else if (seg_units[s]) {
            const int64_t u = unit_prefix[s];
            unit_seg[u] = static_cast<int>(s);
            unit_start[u] = seg_off[s];
            unit_dense[u] = dense_segment(seg_len[s], s, seg_row, row_off, dense_min) ? 1 : 0;
        }
    }
}

// A unit that is not dense is a bitmap unit when its buckets span at most 8192 columns and
// every one of its (at most kMaxBitmapSegs) segments is a column bucket of a long row: each
// bucket's distinct columns then fit one 8192-bit LDS bitmap.  A bitmap bucket has a fixed
// cost (clearing and scanning its bitmap), so units of many small buckets are sorted
// instead: at most kMaxBitmapBuckets nonempty buckets.  At C4 (units of about 2000
// products) the limits 16 / 32 / 64 / 256 gave a call of 99.6 / 96.6 / 96.9 / 98.0 ms.
// *units of the `bound` entries are units; the others' flags are cleared.
__global__ void unit_bitmap_kernel(const int *__restrict__ unit_seg,
                                   int64_t *__restrict__ unit_dense,
                                   const int64_t *__restrict__ units, int64_t bound,
                                   int64_t n_seg, const int64_t *__restrict__ seg_len,
                                   const int *__restrict__ seg_row,
                                   const int64_t *__restrict__ row_off, bool narrow_buckets,
                                   int64_t *__restrict__ unit_bitmap) {
    const int64_t n_units = *units;
    for (int64_t u = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; u < bound;
         u += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        if (u >= n_units) {
            unit_dense[u] = unit_bitmap[u] = 0;
            continue;
        }
        const int64_t s0 = unit_seg[u];
        const int64_t s1 = u + 1 < n_units ? unit_seg[u + 1] : n_seg;
        bool ok = narrow_buckets && !unit_dense[u] && s1 - s0 <= kMaxBitmapSegs;
        int buckets = 0;
        for (int64_t s = s0; ok && s < s1; ++s) {
            if (seg_len[s] == 0) continue;
            const int r = seg_row[s];
            ok = row_off[r + 1] - row_off[r] > kShort && ++buckets <= kMaxBitmapBuckets;
        }
        unit_bitmap[u] = ok ? 1 : 0;
    }
}

// The three work lists, in unit order: each unit at its rank among units of its kind
// (dense_rank and bitmap_rank are exclusive scans of the kind flags).
__global__ void unit_lists_kernel(const int64_t *__restrict__ unit_dense,
                                  const int64_t *__restrict__ dense_rank,
                                  const int64_t *__restrict__ unit_bitmap,
                                  const int64_t *__restrict__ bitmap_rank, int64_t n_units,
                                  int *__restrict__ dense_list, int *__restrict__ bitmap_list,
                                  int *__restrict__ sort_list) {
    for (int64_t u = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; u < n_units;
         u += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t rd = dense_rank[u], rb = bitmap_rank[u];
        if (unit_dense[u]) {
            dense_list[rd] = static_cast<int>(u);
        } else if (unit_bitmap[u]) {
            bitmap_list[rb] = static_cast<int>(u);
        } else {
            sort_list[u - rd - rb] = static_cast<int>(u);
        }
    }
}

// ---- 5a: sort units --------------------------------------------------------------------

// Ascending sort of one lane's kPer (key, value) pairs in registers (bitonic network with
// compile-time indices).
template <typename K>
__device__ __forceinline__ void sort_registers(K (&k)[kPer], float (&v)[kPer]) {
#pragma unroll
    for (int size = 2; size <= kPer; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool ascending = (i & size) == 0;
                    const bool swap = (k[i] > k[j]) == ascending;
                    const K ki = k[i], kj = k[j];
                    const float vi = v[i], vj = v[j];
                    k[i] = swap ? kj : ki;
                    k[j] = swap ? ki : kj;
                    v[i] = swap ? vj : vi;
                    v[j] = swap ? vi : vj;
                }
            }
        }
    }
}

// Merge-path split of output diagonal d over A[0, na) and B[0, nb), equal keys from A first:
// the number of A items among the first d outputs.
// A and B are offsets of the two runs in the padded LDS array.
template <typename K>
__device__ __forceinline__ int merge_split(const K *s_key, int A, int B, int na, int nb, int d) {
    int lo = max(0, d - nb), hi = min(d, na);
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s_key[pad(A + mid)] <= s_key[pad(B + d - 1 - mid)]) {
            lo = mid + 1;
        } else {
            hi = mid;
        }
    }
    return lo;
}

// Ascending sort of n2 (a power of two, kPer <= n2 <= kTile) pairs: lane t holds positions
// [t*kPer, (t+1)*kPer) in k/v (registers), sorts them, then sorted runs of kPer << l are
// merged pairwise through LDS, each lane producing its kPer outputs from a merge-path split.
// On return s_key/s_val hold the sorted sequence and k/v the lane's part of it.
template <typename K>
__device__ __forceinline__ void merge_sort(K (&k)[kPer], float (&v)[kPer], K *s_key,
                                           float *s_val, int n2) {
    const int base = threadIdx.x * kPer;
    const bool active = base < n2;
    sort_registers(k, v);
    if (active) {
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            s_key[pad(base + u)] = k[u];
            s_val[pad(base + u)] = v[u];
        }
    }
    for (int len = kPer; len < n2; len <<= 1) {
        __syncthreads();
        const int A = base & ~(2 * len - 1);
        const int B = A + len;
        // runs already in order (typically two different segments) merge to themselves: the
        // lane's registers and LDS positions already hold its outputs
        const bool merge = active && s_key[pad(B - 1)] > s_key[pad(B)];
        if (merge) {
            int a = merge_split(s_key, A, B, len, len, base - A);
            int b = (base - A) - a;
            K ka = s_key[pad(A + min(a, len - 1))];
            K kb = s_key[pad(B + min(b, len - 1))];
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const bool take_a = a < len && (b >= len || ka <= kb);
                const int src = take_a ? A + a : B + min(b, len - 1);
                k[u] = take_a ? ka : kb;
                v[u] = s_val[pad(src)];
                a += take_a;
                b += !take_a;
                // the head that advanced, read at an index inside its run, then selected:
                // no branch whose sides wait for their own reads
                const K kn = s_key[pad(take_a ? A + min(a, len - 1) : B + min(b, len - 1))];
                ka = take_a ? kn : ka;
                kb = take_a ? kb : kn;
            }
        }
        __syncthreads();
        if (merge) {
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                s_key[pad(base + u)] = k[u];
                s_val[pad(base + u)] = v[u];
            }
        }
    }
    __syncthreads();
}

// Exclusive segmented sum across the workgroup's lanes.  Lane input: f = the lane holds a run
// start, s = the sum of its positions after its last start (all of them if none).  Output:
// the sum of the run open where the lane begins (from earlier lanes; 0 if none).
__device__ __forceinline__ double block_segmented_carry(bool f, double s, double *s_sum,
                                                        int *s_flag) {
    const int l = dev::lane();
    const int w = threadIdx.x / dev::kWave;
    int fi = f ? 1 : 0;
    double si = s;
#pragma unroll
    for (int o = 1; o < dev::kWave; o <<= 1) {
        const int fu = __shfl_up(fi, o, dev::kWave);
        const double su = __shfl_up(si, o, dev::kWave);
        if (l >= o) {
            if (!fi) si += su;
            fi |= fu;
        }
    }
    int fe = __shfl_up(fi, 1, dev::kWave);
    double se = __shfl_up(si, 1, dev::kWave);
    if (l == 0) {
        fe = 0;
        se = 0.0;
    }
    if (l == dev::kWave - 1) {
        s_flag[w] = fi;
        s_sum[w] = si;
    }
    __syncthreads();
    double cs = 0.0;
    for (int i = 0; i < w; ++i) cs = s_flag[i] ? s_sum[i] : cs + s_sum[i];
    __syncthreads();
    return fe ? se : cs + se;
}

// One workgroup per sort unit (from the sort list).  Sorts the unit's products by
// (segment ordinal, k), sums each run in float64, writes the distinct entries at the unit's
// start in ukey/uval, the unit's count, and (row_unit, row_local) for rows starting here.
// K is uint32_t when kOrdBits + col_shift <= 32, else uint64_t (col_shift = 32).
template <typename K>
__global__ __launch_bounds__(kBlock) void sort_unit_kernel(
    const int *__restrict__ sort_list, const int *__restrict__ unit_seg,
    const int64_t *__restrict__ unit_start, int64_t n_units,
    int64_t n_seg, const int64_t *__restrict__ seg_len, const int64_t *__restrict__ seg_off,
    const int *__restrict__ seg_row, const int64_t *__restrict__ row_off, int col_shift,
    const int4 *__restrict__ desc, const int64_t *__restrict__ seg_roff,
    const int2 *__restrict__ cv_b, int *__restrict__ ukey,
    float *__restrict__ uval, int64_t *__restrict__ unit_nnz, int *__restrict__ row_unit,
    int *__restrict__ row_local, const int64_t *__restrict__ seg_out) {
    static_assert(sizeof(K) >= sizeof(int), "run starts are staged in s_key");
    __shared__ K s_key[kPadded];
    __shared__ float s_val[kPadded];
    __shared__ int s_mark[kPadded];
    __shared__ __align__(8) unsigned s_mask[kTile / 32];  // products that start a run
    __shared__ int s_wave[kBlock / dev::kWave];
    __shared__ double s_sum[kBlock / dev::kWave];
    __shared__ int s_flag[kBlock / dev::kWave];
    const int64_t u = sort_list[dev::xcd_block<kXcdGroup>()];
    const int s0 = unit_seg[u];
    const int64_t start = unit_start[u];
    const int n = static_cast<int>(unit_start[u + 1] - start);
    const int64_t s_end = u + 1 < n_units ? unit_seg[u + 1] : n_seg;
    const int64_t r0 = seg_roff[s0];
    const int R = static_cast<int>(seg_roff[s_end] - r0);
    int4 d = desc[r0 + min(static_cast<int>(threadIdx.x), R - 1)];
    if (threadIdx.x < kTile / 32) s_mask[threadIdx.x] = 0u;
    __syncthreads();
    {
        // the unit's products from its runs, by windows, held in registers until every lane is
        // done with the runs' tables, then staged in LDS
        constexpr int kWaves = kBlock / dev::kWave;
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / dev::kWave), l = dev::lane();
        int *s_bs = reinterpret_cast<int *>(s_key);  // product 0's B entry
        float *s_a = s_val;                          // A value
        int products = 0;
        for (int rb = 0; rb < R; rb += kBlock) {  // uniform
            const int r = rb + static_cast<int>(threadIdx.x);
            if (rb > 0) d = desc[r0 + min(r, R - 1)];
            int total = 0;
            const int off =
                products + dev::block_exclusive_sum<kBlock>(r < R ? d.y : 0, s_wave, total);
            if (r < R) {
                s_bs[r] = d.x - off;
                s_a[r] = __int_as_float(d.z);
                if (d.y > 0) atomicOr(&s_mask[off >> 5], 1u << (off & 31));
            }
            products += total;
        }
        __syncthreads();
        const RunWindows runs = load_windows(s_mask, 0);
        int2 e[kPer];
        float av[kPer];
#pragma unroll
        for (int g = 0; g < kPer; g += 4) {
            if ((g * kWaves + w) * dev::kWave >= n) break;  // uniform
#pragma unroll
            for (int j = g; j < g + 4; ++j) {
                const int i = j * kWaves + w;
                const int r = runs.run(i);
                e[j] = cv_b[s_bs[r] + min(i * dev::kWave + l, n - 1)];
                av[j] = s_a[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int q = (j * kWaves + w) * dev::kWave + l;
            s_mark[pad(q)] = 0;
            if (q < n) {
                s_key[pad(q)] = static_cast<K>(static_cast<uint32_t>(e[j].x));
                s_val[pad(q)] = av[j] * __int_as_float(e[j].y);
            }
        }
    }
    __syncthreads();
    for (int64_t s = s0 + threadIdx.x; s < s_end; s += kBlock) {
        if (seg_len[s] > 0) s_mark[pad(static_cast<int>(seg_off[s] - start))] = static_cast<int>(s) + 1;
    }
    __syncthreads();
    const int base = threadIdx.x * kPer;  // blocked positions of this lane
    int c = 0;
#pragma unroll
    for (int v = 0; v < kPer; ++v) c += s_mark[pad(base + v)] != 0;
    int total = 0;
    int ord = dev::block_exclusive_sum<kBlock>(c, s_wave, total) - 1;
    int n2 = kPer;
    while (n2 < n) n2 <<= 1;
    K rk0[kPer];
    float rv0[kPer];
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        const int q = base + v;
        ord += s_mark[pad(q)] != 0;
        rk0[v] = q < n ? (static_cast<K>(ord) << col_shift) | s_key[pad(q)] : ~static_cast<K>(0);
        rv0[v] = q < n ? s_val[pad(q)] : 0.0f;
    }
    __syncthreads();
    merge_sort(rk0, rv0, s_key, s_val, n2);
    // Segments keep their positions (sorted by ordinal first), so s_mark still marks them.
    // rk0/rv0 hold this lane's sorted positions; neighbours come from LDS.
    const K prev = base > 0 && base < n ? s_key[pad(base - 1)] : ~static_cast<K>(0);
    unsigned st = 0;
    double acc = 0.0;
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        const int q = base + v;
        const bool start_run = q < n && (q == 0 || rk0[v] != (v > 0 ? rk0[v - 1] : prev));
        if (start_run) st |= 1u << v;
        const double x = q < n ? static_cast<double>(rv0[v]) : 0.0;
        acc = start_run ? x : acc + x;
    }
    int runs = 0;
    const int rank0 =
        dev::block_exclusive_sum<kBlock>(static_cast<int>(__popc(st)), s_wave, runs);
    const double carry = block_segmented_carry(st != 0, acc, s_sum, s_flag);
    const K next = base + kPer < n ? s_key[pad(base + kPer)] : ~static_cast<K>(0);
    const K mask = (static_cast<K>(1) << col_shift) - 1;
    // second pass: each run's sum is complete at its last position; it goes to the index of
    // the run's start (one entry per run, in order)
    acc = carry;
    int idx = rank0 - 1;
    int ok[kPer];
    float ov[kPer];
    unsigned ends = 0;
    int first_end = 0;  // run index of the lane's first run end (its later ends follow)
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        const int q = base + v;
        ok[v] = 0;
        ov[v] = 0.0f;
        if (q < n) {
            const bool start_run = (st >> v) & 1u;
            if (start_run) ++idx;
            acc = start_run ? static_cast<double>(rv0[v]) : acc + static_cast<double>(rv0[v]);
            const K after = v + 1 < kPer ? rk0[v + 1] : next;
            if (q + 1 == n || after != rk0[v]) {
                if (ends == 0) first_end = idx;
                ends |= 1u << v;
                ok[v] = static_cast<int>(rk0[v] & mask);
                ov[v] = static_cast<float>(acc);
            }
            // rows starting here: the first position of their first nonempty segment
            if (s_mark[pad(q)]) {
                const int sg = s_mark[pad(q)] - 1;
                const int r = seg_row[sg];
                if (row_off[r] == seg_off[sg]) {
                    row_unit[r] = static_cast<int>(u);
                    row_local[r] = idx;
                }
            }
        }
    }
    // stage the unit's distinct entries in LDS (run j at slot j), then store them coalesced
    __syncthreads();
    int *s_ok = s_mark;
    idx = first_end;
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        if ((ends >> v) & 1u) {
            s_ok[pad(idx)] = ok[v];
            s_val[pad(idx)] = ov[v];
            ++idx;
        }
    }
    __syncthreads();
    const int64_t out = seg_out ? seg_out[s0] : start;
    for (int j = threadIdx.x; j < runs; j += kBlock) {
        ukey[out + j] = s_ok[pad(j)];
        uval[out + j] = s_val[pad(j)];
    }
    if (threadIdx.x == 0) unit_nnz[u] = runs;
}

// ---- 5b: bitmap units ------------------------------------------------------------------

using dev::wave_sync;

// Marks the columns of a bucket (window offsets s_col[x0, x1)) in bm.
__device__ __forceinline__ void mark_bucket(unsigned *bm, const unsigned short *s_col, int x0,
                                            int x1) {
    const int l = dev::lane();
#pragma unroll
    for (int i = 0; i < kBitmapWords / dev::kWave; ++i) bm[l + i * dev::kWave] = 0u;
    wave_sync();
    for (int xb = x0 + l; xb < x1; xb += 4 * dev::kWave) {  // four reads in flight
        int c[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) c[j] = s_col[min(xb + j * dev::kWave, x1 - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (xb + j * dev::kWave < x1) atomicOr(&bm[c[j] >> 5], 1u << (c[j] & 31));
        }
    }
    wave_sync();
}

// One workgroup per bitmap unit; one wavefront per bucket at a time.  A bucket's distinct
// columns are the set bits of its 8192-bit window bitmap; the rank of a column (prefix
// popcount) indexes its float64 accumulator, and each product then writes its column at
// its rank, which lists the distinct columns sorted (a loop over each word's set bits
// instead cost 7.7 of the units' 40 ms at C4: a wavefront waits for its lane with the most
// bits; the products are spread evenly).  Accumulators and the listed columns of a bucket
// live in its own product range of the unit; once every bucket is done, a scan of their
// counts gives the output offsets and the workgroup stores the unit's entries with
// consecutive lanes on consecutive outputs.
// At R-MAT scale 20 (1.5 million units) 30.1 ms, LDS about half busy.  A bucket of up to 512
// products keeps its columns, values and ranks in registers, which leaves out a quarter of the
// LDS instructions (31.4 -> 30.4 ms); tables loaded up front 30.4 -> 30.1.
__global__ __launch_bounds__(kBitmapBlock) void bitmap_unit_kernel(
    const int *__restrict__ bitmap_list, const int *__restrict__ unit_seg,
    const int64_t *__restrict__ unit_start, int64_t n_units, int64_t n_seg,
    const int64_t *__restrict__ seg_len, const int64_t *__restrict__ seg_off,
    const int64_t *__restrict__ seg_prefix, const int *__restrict__ seg_row,
    const int64_t *__restrict__ row_off, int shift, const int4 *__restrict__ desc,
    const int64_t *__restrict__ seg_roff, const int2 *__restrict__ cv_b,
    int *__restrict__ ukey, float *__restrict__ uval,
    int64_t *__restrict__ unit_nnz, int *__restrict__ row_unit, int *__restrict__ row_local,
    const int64_t *__restrict__ seg_out) {
    constexpr int kWaves = kBitmapBlock / dev::kWave;
    constexpr int kPerB = kTile / kBitmapBlock;
    constexpr int kHeld = 8;  // products per lane of a bucket held in registers
    __shared__ double s_acc[kTile];
    __shared__ unsigned short s_col[kTile];  // column offset inside its bucket's window
    __shared__ float s_pv[kTile];            // product values
    __shared__ __align__(16) unsigned s_bits[kWaves][kBitmapWords];
    __shared__ __align__(16) int s_pre[kWaves][kBitmapWords];
    __shared__ int s_x0[kMaxBitmapSegs + 1];
    __shared__ int s_base[kMaxBitmapSegs];
    __shared__ int s_row[kMaxBitmapSegs];
    __shared__ int s_out[kMaxBitmapSegs];
    __shared__ int s_wave[kWaves];
    __shared__ int s_next;  // the next bucket to claim
    const int64_t u = bitmap_list[dev::xcd_block<kXcdGroup>()];
    const int64_t s0 = unit_seg[u];
    const int64_t s1 = u + 1 < n_units ? unit_seg[u + 1] : n_seg;
    const int64_t start = unit_start[u];
    const int n = static_cast<int>(unit_start[u + 1] - start);
    // Everything the unit reads of the tables is loaded up front, four dependent steps (list,
    // unit, segment, row and runs) before the gathers: with two workgroups per CU each step
    // costs its latency.
    const int64_t s = min(s0 + static_cast<int64_t>(threadIdx.x), s1 - 1);
    const int64_t r0 = seg_roff[s0];
    const int R = static_cast<int>(seg_roff[s1] - r0);
    const int64_t out = seg_out ? seg_out[s0] : start;
    const bool here = s0 + threadIdx.x < s1 && seg_len[s] > 0;
    const int64_t first = seg_off[s];
    const int row = seg_row[s];
    int4 d = desc[r0 + min(static_cast<int>(threadIdx.x), R - 1)];
    const int64_t row_seg = seg_prefix[row], row_first = row_off[row];
    // the unit's nonempty buckets in order (at most kMaxBitmapSegs segments: one per lane)
    int n_buckets = 0;
    const int ord = dev::block_exclusive_sum<kBitmapBlock>(here ? 1 : 0, s_wave, n_buckets);
    if (here) {
        s_x0[ord] = static_cast<int>(first - start);
        s_base[ord] = static_cast<int>((s - row_seg) << shift);
        s_row[ord] = first == row_first ? row : -1;  // the row that starts with the bucket
    }
    if (threadIdx.x == 0) {
        s_x0[n_buckets] = n;
        s_next = kWaves;  // wavefront w starts with bucket w
    }
    // the unit's products from its runs: window offsets (bucket = column >> shift, so the
    // offset is the column's low bits) and values, staged once
    const int low = (1 << shift) - 1;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / dev::kWave), l = dev::lane();
    {
        int *s_bs = reinterpret_cast<int *>(s_acc);                 // product 0's B entry
        float *s_a = reinterpret_cast<float *>(s_acc) + kTile;      // A value
        unsigned *s_mask = s_bits[0];
        if (threadIdx.x < kTile / 32) s_mask[threadIdx.x] = 0u;
        __syncthreads();
        int products = 0;
        for (int rb = 0; rb < R; rb += kBitmapBlock) {  // uniform
            const int r = rb + static_cast<int>(threadIdx.x);
            if (rb > 0) d = desc[r0 + min(r, R - 1)];
            int total = 0;
            const int off = products + dev::block_exclusive_sum<kBitmapBlock>(
                                           r < R ? d.y : 0, s_wave, total);
            if (r < R) {
                s_bs[r] = d.x - off;
                s_a[r] = __int_as_float(d.z);
                if (d.y > 0) atomicOr(&s_mask[off >> 5], 1u << (off & 31));
            }
            products += total;
        }
        __syncthreads();
        const RunWindows runs = load_windows(s_mask, 0);
        constexpr int kGroup = 4;  // windows whose gathers are issued together
#pragma unroll
        for (int g = 0; g < kPerB; g += kGroup) {
            if ((g * kWaves + w) * dev::kWave >= n) break;  // uniform
            int2 e[kGroup];
            float av[kGroup];
#pragma unroll
            for (int j = 0; j < kGroup; ++j) {
                const int i = (g + j) * kWaves + w;
                const int r = runs.run(i);
                e[j] = cv_b[s_bs[r] + min(i * dev::kWave + l, n - 1)];
                av[j] = s_a[r];
            }
#pragma unroll
            for (int j = 0; j < kGroup; ++j) {
                const int q = ((g + j) * kWaves + w) * dev::kWave + l;
                if (q < n) {
                    s_col[q] = static_cast<unsigned short>(e[j].x & low);
                    s_pv[q] = av[j] * __int_as_float(e[j].y);
                }
            }
        }
    }
    __syncthreads();
    unsigned *bm = s_bits[w];
    int *pre = s_pre[w];
    // accumulate each bucket by rank; its distinct columns (window offsets, in order) and
    // their sums are left in its own product range, s_col / s_acc[x0 + rank]
    constexpr int kWordsPerLane = kBitmapWords / dev::kWave;
    static_assert(kWordsPerLane == 4, "a lane's words are one 16-byte access");
    // exclusive popcount prefix per word (lane l owns words [4 l, 4 l + 4)); the bucket's count
    auto ranks = [&]() {
        const uint4 m = reinterpret_cast<const uint4 *>(bm)[l];
        const int c0 = __popc(m.x), c1 = c0 + __popc(m.y), c2 = c1 + __popc(m.z);
        const int mine = c2 + __popc(m.w);
        const int incl = dev::wave_inclusive_sum_dpp(mine);
        const int run = incl - mine;
        reinterpret_cast<int4 *>(pre)[l] = make_int4(run, run + c0, run + c1, run + c2);
        wave_sync();
        return incl;
    };
    auto rank_of = [&](int c) {
        return pre[c >> 5] + __popc(bm[c >> 5] & ((1u << (c & 31)) - 1u));
    };
    int *s_ocol = reinterpret_cast<int *>(s_pv);
    // Buckets differ widely in size: a wavefront that finishes one claims the next.
    for (int o = w; o < n_buckets;) {  // uniform per wavefront
        const int x0 = __builtin_amdgcn_readfirstlane(s_x0[o]);
        const int x1 = __builtin_amdgcn_readfirstlane(s_x0[o + 1]);
        for (int x = x0 + l; x < x1; x += dev::kWave) s_acc[x] = 0.0;
        int distinct = 0;
        if (x1 - x0 <= kHeld * dev::kWave) {
            // columns, values and ranks stay in registers
            int c[kHeld];
            float v[kHeld];
            reinterpret_cast<uint4 *>(bm)[l] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
            for (int g = 0; g < kHeld; g += 4) {
                if (x0 + g * dev::kWave >= x1) break;  // uniform
#pragma unroll
                for (int j = g; j < g + 4; ++j) {
                    const int x = min(x0 + j * dev::kWave + l, x1 - 1);
                    c[j] = s_col[x];
                    v[j] = s_pv[x];
                }
            }
            wave_sync();
#pragma unroll
            for (int j = 0; j < kHeld; ++j) {
                if (x0 + j * dev::kWave + l < x1) atomicOr(&bm[c[j] >> 5], 1u << (c[j] & 31));
            }
            wave_sync();
            distinct = ranks();
#pragma unroll
            for (int g = 0; g < kHeld; g += 4) {
                if (x0 + g * dev::kWave >= x1) break;  // uniform
                int r[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) r[j] = rank_of(c[g + j]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (x0 + (g + j) * dev::kWave + l < x1) {
                        atomicAdd(&s_acc[x0 + r[j]], static_cast<double>(v[g + j]));
                        s_ocol[x0 + r[j]] = c[g + j];
                    }
                }
            }
        } else {
            mark_bucket(bm, s_col, x0, x1);
            distinct = ranks();
            for (int xb = x0 + l; xb < x1; xb += 4 * dev::kWave) {
                // every read of four products first (clamped to the bucket), then the adds
                float vv[4];
                int r[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int x = min(xb + j * dev::kWave, x1 - 1);
                    vv[j] = s_pv[x];
                    r[j] = rank_of(s_col[x]);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (xb + j * dev::kWave < x1) {
                        atomicAdd(&s_acc[x0 + r[j]], static_cast<double>(vv[j]));
                    }
                }
            }
            wave_sync();  // every product value of the bucket is read: its slots take the columns
            // Each product writes its column at its rank into the bucket's own product-value
            // slots (s_pv), so the distinct columns land there in order; products of one
            // column write the same word.  Four products per lane per round, as above.
            for (int xb = x0 + l; xb < x1; xb += 4 * dev::kWave) {
                int c[4], r[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    c[j] = s_col[min(xb + j * dev::kWave, x1 - 1)];
                    r[j] = rank_of(c[j]);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (xb + j * dev::kWave < x1) s_ocol[x0 + r[j]] = c[j];
                }
            }
        }
        if (l == dev::kWave - 1) s_out[o] = distinct;  // the bucket's distinct columns
        wave_sync();
        int claim = 0;
        if (l == 0) claim = atomicAdd(&s_next, 1);
        o = __builtin_amdgcn_readfirstlane(claim);
    }
    __syncthreads();
    // output offset of each bucket inside the unit
    int total = 0;
    const int cnt = static_cast<int>(threadIdx.x) < n_buckets ? s_out[threadIdx.x] : 0;
    const int off = dev::block_exclusive_sum<kBitmapBlock>(cnt, s_wave, total);
    if (static_cast<int>(threadIdx.x) < n_buckets) s_out[threadIdx.x] = off;
    __syncthreads();
    // the unit's entries, consecutive lanes on consecutive outputs: output i belongs to the
    // last bucket whose offset is at most i (a lane's outputs only move forward)
    int o = 0;
    for (int i = threadIdx.x; i < total; i += kBitmapBlock) {
        while (o + 1 < n_buckets && s_out[o + 1] <= i) ++o;
        const int x = s_x0[o] + (i - s_out[o]);
        ukey[out + i] = s_base[o] + reinterpret_cast<const int *>(s_pv)[x];
        uval[out + i] = static_cast<float>(s_acc[x]);
    }
    // rows starting in this unit, and the unit's count
    if (static_cast<int>(threadIdx.x) < n_buckets) {
        const int r = s_row[threadIdx.x];
        if (r >= 0) {
            row_unit[r] = static_cast<int>(u);
            row_local[r] = s_out[threadIdx.x];
        }
    }
    if (threadIdx.x == 0) unit_nnz[u] = total;
}

// ---- 5c: dense units -------------------------------------------------------------------

// One workgroup of kDenseBlock threads per dense unit (from the dense list): the 64 KB
// accumulator allows two resident workgroups per CU, so the workgroup is wide.  The
// segment's column range [bucket << shift, (bucket + 1) << shift) is accumulated kDenseCols
// columns at a time in an LDS float64 array (plus a bitmap of touched columns), then
// compacted in column order, 16 columns per lane.  At R-MAT scale 20 (577,000 units) 14.9 ms.
// Twice the wavefronts (1024 threads) took 1.0 ms more, and outputs compacted in LDS and stored
// with consecutive lanes on consecutive outputs 0.4 ms more: neither bounds it.
constexpr int kDenseBlock = 512;
constexpr int kDenseWaves = kDenseBlock / dev::kWave;
constexpr int kDenseGroup = 4;  // windows whose gathers are issued together

__global__ __launch_bounds__(kDenseBlock) void dense_unit_kernel(
    const int *__restrict__ dense_list, const int *__restrict__ unit_seg,
    const int64_t *__restrict__ unit_start,
    const int64_t *__restrict__ seg_len, const int64_t *__restrict__ seg_prefix,
    const int *__restrict__ seg_row, const int64_t *__restrict__ row_off, int shift, int cols,
    const int4 *__restrict__ desc, const int64_t *__restrict__ seg_roff,
    const int2 *__restrict__ cv_b, int *__restrict__ ukey,
    float *__restrict__ uval, int64_t *__restrict__ unit_nnz, int *__restrict__ row_unit,
    int *__restrict__ row_local, const int64_t *__restrict__ seg_out) {
    __shared__ double s_acc[kDenseCols];
    __shared__ unsigned s_bits[kDenseCols / 32];
    __shared__ int s_wave[kDenseBlock / dev::kWave];
    // a batch of up to kDenseBlock runs: B entry of the batch's product 0, A value
    __shared__ int s_bs[kDenseBlock];
    __shared__ float s_a[kDenseBlock];
    __shared__ __align__(8) unsigned s_mask[kTile / 32];  // a round's run starts
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / dev::kWave), l = dev::lane();
    static_assert(kDenseCols / 16 == kDenseBlock, "16 bitmap bits per lane");
    const int64_t u = dense_list[dev::xcd_block<kXcdGroup>()];
    const int s = unit_seg[u];
    const int64_t start = unit_start[u];
    const int row = seg_row[s];
    // (the unit's tables and first runs up front, as in a bitmap unit)
    const int64_t r0 = seg_roff[s], r1 = seg_roff[s + 1];
    const int64_t seg_first = seg_out ? seg_out[s] : start;
    const int64_t lane_run = r0 + threadIdx.x;
    const int4 d0 = desc[min(lane_run, r1 - 1)];
    const int64_t bucket = s - seg_prefix[row];
    const int64_t c_lo = bucket << shift;
    const int64_t c_hi = min(static_cast<int64_t>(cols), (bucket + 1) << shift);
    if (threadIdx.x == 0 && row_off[row] == start) {
        row_unit[row] = static_cast<int>(u);
        row_local[row] = 0;
    }
    int64_t written = seg_first;
    const int64_t out0 = written;
    for (int64_t w0 = c_lo; w0 < c_hi; w0 += kDenseCols) {
        for (int i = threadIdx.x; i < kDenseCols; i += kDenseBlock) s_acc[i] = 0.0;
        if (threadIdx.x < kDenseCols / 32) s_bits[threadIdx.x] = 0u;
        __syncthreads();
        // runs in batches of kDenseBlock (one per lane); the batch's products in rounds of
        // kTile, by windows
        for (int64_t rb = r0; rb < r1; rb += kDenseBlock) {
            const bool mine = rb + threadIdx.x < r1;
            const int4 d = rb == r0 ? d0 : desc[min(rb + threadIdx.x, r1 - 1)];
            int total = 0;
            const int off = dev::block_exclusive_sum<kDenseBlock>(mine ? d.y : 0, s_wave, total);
            s_bs[threadIdx.x] = d.x - off;
            s_a[threadIdx.x] = __int_as_float(d.z);
            for (int x0 = 0; x0 < total; x0 += kTile) {
                if (threadIdx.x < kTile / 32) s_mask[threadIdx.x] = 0u;
                __syncthreads();
                const int at = off - x0;
                if (mine && at >= 0 && at < kTile) atomicOr(&s_mask[at >> 5], 1u << (at & 31));
                const int before = __syncthreads_count(mine && at < 0);
                const RunWindows runs = load_windows(s_mask, before);
                const int left = min(total - x0, kTile);
#pragma unroll
                for (int g = 0; g < kTile / kDenseBlock; g += kDenseGroup) {
                    if ((g * kDenseWaves + w) * dev::kWave >= left) break;  // uniform
                    int2 e[kDenseGroup];
                    float av[kDenseGroup];
#pragma unroll
                    for (int j = 0; j < kDenseGroup; ++j) {
                        const int i = (g + j) * kDenseWaves + w;
                        const int r = runs.run(i);
                        e[j] = cv_b[s_bs[r] + x0 + min(i * dev::kWave + l, left - 1)];
                        av[j] = s_a[r];
                    }
#pragma unroll
                    for (int j = 0; j < kDenseGroup; ++j) {
                        const int64_t c = e[j].x - w0;
                        if (((g + j) * kDenseWaves + w) * dev::kWave + l < left && c >= 0 &&
                            c < kDenseCols) {
                            atomicAdd(&s_acc[c],
                                      static_cast<double>(av[j] * __int_as_float(e[j].y)));
                            atomicOr(&s_bits[c >> 5], 1u << (c & 31));
                        }
                    }
                }
                __syncthreads();  // the round's tables are read before the next one's
            }
        }
        const unsigned half = (s_bits[threadIdx.x >> 1] >> ((threadIdx.x & 1) * 16)) & 0xffffu;
        int total = 0;
        int rank = dev::block_exclusive_sum<kDenseBlock>(static_cast<int>(__popc(half)), s_wave,
                                                         total);
        unsigned m = half;
        while (m) {
            const int bit = __ffs(m) - 1;
            m &= m - 1;
            const int c = threadIdx.x * 16 + bit;
            ukey[written + rank] = static_cast<int>(w0 + c);
            uval[written + rank] = static_cast<float>(s_acc[c]);
            ++rank;
        }
        written += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) unit_nnz[u] = written - out0;
}

// ---- symbolic pass: the result's size before the reduce ----------------------------------
//
// When every column index fits kSymColBits bits, the distinct columns of every segment are
// counted before any unit reduces, from A and B directly (no run descriptors): seg_nnz[s].
// Their exclusive scan gives every segment's result offset, the result is allocated at its
// exact size, and the reduce units write straight into it (a unit's entries are its
// segments' distinct entries in segment order, so the unit starts at its first segment's
// offset).  A row starts at its first segment's offset.  The reference sizes its result the
// same way before reducing into it, from the head flags of its sorted products
// (stitch_and_generate_gpu.cpp:96-126).
//
// Long rows: one workgroup per row (rows claimed from a list, the heaviest first) ORs each
// product's column into a bitmap of the row's columns in LDS (2^20 bits, 128 KB), then counts
// each bucket's bits (a bucket is 8192 columns, 256 words, or the whole row when nb = 1) and
// clears the words it read.  The row's A entries are staged kSymChunk at a time (their B
// rows' starts and product offsets; empty B rows dropped); each wavefront takes an equal
// share of the chunk's products in windows of 64 consecutive products, lane x on product x
// of the window, so that a window's loads are consecutive entries of a few B rows.  The
// entry of lane x's product is the window's first entry plus the number of entries starting
// inside the window at or before x, counted in a 64-bit mask of those starts (an OR over the
// wavefront).  The first entries of kSymBatch windows are searched at once, one lane each,
// and the windows' loads are all issued before their ORs.
// Short rows (at most kShort products): one wavefront per row inserts the columns into an
// open-addressing table of its own in LDS (kSymSlots 32-bit slots, at most half full) and
// counts the keys it added; then it refills the table with the empty key.
constexpr int kSymColBits = 20;
constexpr int kSymBlock = 1024;
constexpr int kSymWords = 1 << (kSymColBits - 5);
constexpr int kSymChunk = kSymBlock;
constexpr int kSymBatch = 16;
constexpr int64_t kSymHeavy = int64_t{1} << 18;  // long rows with more products go first
constexpr int kSymShortBlock = 512;
constexpr int kSymSlots = 4096;
constexpr unsigned kSymEmpty = 0xffffffffu;  // above every column index (< 2^kSymColBits)
static_assert(kSymWords == 32 * kSymBlock, "a thread counts 32 words of the bitmap");
static_assert(kDenseCols / 32 == 8 * 32, "a bucket of 8192 columns is 8 threads' words");
static_assert(kSymSlots >= 2 * kShort, "a short row's table stays at most half full");

// OR of v over the 64 lanes, returned to every lane (DPP inclusive OR scan, then lane 63).
// Every lane must be active.
__device__ __forceinline__ unsigned wave_or(unsigned v) {
    int x = static_cast<int>(v);
    x |= __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x |= __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x |= __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x |= __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x |= __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x |= __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return static_cast<unsigned>(__builtin_amdgcn_readlane(x, dev::kWave - 1));
}

// Entry of lane l's product in a window of 64 products starting at wb, given e0, the entry
// holding product wb: entries e0 + 1 + l (l < 63) may start inside the window (off: their
// first products, ne entries in all, nonempty, so their starts are distinct and > wb).
// Uniform control flow.
__device__ __forceinline__ int window_entry(const int *off, int ne, int e0, int wb, int l) {
    const int e = e0 + 1 + l;
    const int d = e < ne ? off[e] - wb : dev::kWave;
    const bool in = d < dev::kWave;
    const unsigned mlo = wave_or(in && d < 32 ? 1u << d : 0u);
    const unsigned mhi = wave_or(in && d >= 32 ? 1u << (d - 32) : 0u);
    const int cnt = l < 32 ? __popc(mlo & ((2u << l) - 1u))
                           : __popc(mlo) + __popc(mhi & ((2u << (l - 32)) - 1u));
    return e0 + cnt;
}

// Work lists of the symbolic pass.  key1[i] = 2^32 for a long row with more than kSymHeavy
// products, 1 for another long row; key2[i] = 1 for a short row with products.  An empty
// row's segment count is 0.  Zeroes the long-row work counter.
__global__ void sym_flags_kernel(const int64_t *__restrict__ row_off, int rows,
                                 const int64_t *__restrict__ seg_prefix,
                                 int64_t *__restrict__ key1, int64_t *__restrict__ key2,
                                 int64_t *__restrict__ seg_nnz, int *__restrict__ work) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows; i += gridDim.x * blockDim.x) {
        const int64_t prod = row_off[i + 1] - row_off[i];
        key1[i] = prod > kShort ? (prod > kSymHeavy ? (int64_t{1} << 32) : 1) : 0;
        key2[i] = prod > 0 && prod <= kShort ? 1 : 0;
        if (prod == 0) seg_nnz[seg_prefix[i]] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *work = 0;
}

// long_list: the heavy long rows, then the others (each group in row order); short_list:
// the short rows with products.  counts[0] / counts[1]: their lengths.  rank1 / rank2 are
// the exclusive scans of key1 / key2 (rank1 packs both groups' ranks, heavy in the high half).
__global__ void sym_lists_kernel(const int64_t *__restrict__ row_off, int rows,
                                 const int64_t *__restrict__ rank1,
                                 const int64_t *__restrict__ rank2, int *__restrict__ long_list,
                                 int *__restrict__ short_list, int64_t *__restrict__ counts) {
    const int64_t t1 = rank1[rows];
    const int64_t n_heavy = t1 >> 32;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows; i += gridDim.x * blockDim.x) {
        const int64_t prod = row_off[i + 1] - row_off[i];
        if (prod > kShort) {
            const int64_t r = rank1[i];
            long_list[prod > kSymHeavy ? (r >> 32) : n_heavy + (r & 0xffffffffll)] = i;
        } else if (prod > 0) {
            short_list[rank2[i]] = i;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        counts[0] = n_heavy + (t1 & 0xffffffffll);
        counts[1] = rank2[rows];
    }
}

// Distinct columns of every bucket of the long rows (see above).  One resident workgroup
// per CU; workgroup g starts with long-list item g and claims its next item from `work`
// (zeroed) when it starts a row, so the next chunk of A entries (the rest of this row's, or
// the claimed item's first) is known in advance: its column loads are issued before this
// chunk's batches and its B row starts after them, off the chunk-to-chunk path.
__global__ __launch_bounds__(kSymBlock) void sym_long_kernel(
    const int *__restrict__ pos_a, const int *__restrict__ crd_a,
    const int *__restrict__ pos_b, const int *__restrict__ crd_b,
    const int *__restrict__ long_list, const int64_t *__restrict__ counts,
    int *__restrict__ work, const int64_t *__restrict__ seg_prefix, int nb, int cols,
    int64_t *__restrict__ seg_nnz) {
    constexpr int kWaves = kSymBlock / dev::kWave;
    __shared__ uint4 s_bm4[kSymWords / 4];
    __shared__ int s_off[kSymChunk + 1];
    __shared__ int s_bs[kSymChunk];
    __shared__ int64_t s_wave[kWaves];
    __shared__ int s_sum[kWaves];
    __shared__ int64_t s_next;  // the item claimed for after the current row
    unsigned *s_bm = reinterpret_cast<unsigned *>(s_bm4);
    const int tid = threadIdx.x, w = tid / dev::kWave, l = dev::lane();
    const int64_t n_long = counts[0];
    int64_t item = blockIdx.x;
    if (item >= n_long) return;  // uniform
    const int words = (cols + 31) >> 5;  // <= kSymWords
    for (int i = tid; i < kSymWords / 4; i += kSymBlock) s_bm4[i] = make_uint4(0u, 0u, 0u, 0u);
    int row = long_list[item];
    int p0 = pos_a[row], p_end = pos_a[row + 1];
    bool row_start = true;
    int bs = 0, len = 0;  // this thread's A entry of the current chunk: its B row
    if (p0 + tid < p_end) {
        const int k = crd_a[p0 + tid];
        bs = pos_b[k];
        len = pos_b[k + 1] - bs;
    }
    for (;;) {
        // (every thread read the previous claim before the last chunk's final barrier; this
        // one is read after this chunk's barriers)
        if (row_start && tid == 0) s_next = static_cast<int64_t>(gridDim.x) + atomicAdd(work, 1);
        // the next chunk, and its column loads (in flight during this chunk)
        int64_t n_item = item;
        int n_row = row, n_p0 = p0 + kSymChunk, n_end = p_end;
        const bool row_done = n_p0 >= p_end;
        if (row_done) {
            __syncthreads();  // the claim
            n_item = s_next;
            if (n_item < n_long) {
                n_row = long_list[n_item];
                n_p0 = pos_a[n_row];
                n_end = pos_a[n_row + 1];
            }
        }
        const bool more = n_item < n_long;
        const int n_k = more && n_p0 + tid < n_end ? crd_a[n_p0 + tid] : -1;
        // one scan for both the nonempty entries' ranks (high half) and product offsets
        // (low half: a chunk's products are at most nnz(B), its B rows being distinct)
        int64_t tot = 0;
        const int64_t ex = dev::block_exclusive_sum<kSymBlock, int64_t>(
            (static_cast<int64_t>(len > 0) << 32) | static_cast<int64_t>(len), s_wave, tot);
        const int ne = static_cast<int>(tot >> 32);
        const int T = static_cast<int>(tot & 0xffffffffll);
        if (len > 0) {
            const int e = static_cast<int>(ex >> 32);
            const int off = static_cast<int>(ex & 0xffffffffll);
            s_off[e] = off;
            s_bs[e] = bs - off;  // product x of entry e is B entry s_bs[e] + x
        }
        if (tid == 0) s_off[ne] = T;
        __syncthreads();
        const int share = (T + kWaves - 1) / kWaves;
        const int lo = min(T, w * share), hi = min(T, lo + share);
        for (int x0 = lo; x0 < hi; x0 += dev::kWave * kSymBatch) {  // uniform per wave
            int first = 0;  // lane j < kSymBatch: the entry of window j's first product
            {
                const int q = x0 + l * dev::kWave;
                if (l < kSymBatch && q < hi) {
                    first = static_cast<int>(dev::last_le(s_off, 0, ne - 1, q));
                }
            }
            int c[kSymBatch];
#pragma unroll
            for (int j = 0; j < kSymBatch; ++j) {
                const int wb = x0 + j * dev::kWave;
                c[j] = -1;
                if (wb < hi) {  // uniform
                    const int e0 = __builtin_amdgcn_readlane(first, j);
                    const int e = window_entry(s_off, ne, e0, wb, l);
                    if (wb + l < hi) c[j] = crd_b[s_bs[e] + wb + l];
                }
            }
#pragma unroll
            for (int j = 0; j < kSymBatch; ++j) {
                if (c[j] >= 0) atomicOr(&s_bm[c[j] >> 5], 1u << (c[j] & 31));
            }
        }
        // the next chunk's B rows (in flight during the barrier and the bucket counts)
        int n_bs = 0, n_len = 0;
        if (n_k >= 0) {
            n_bs = pos_b[n_k];
            n_len = pos_b[n_k + 1] - n_bs;
        }
        __syncthreads();  // the chunk's tables are read; the ORs are done
        if (row_done) {
            // count and clear: thread t holds words [32t, 32t + 32).  The next chunk's scan
            // barrier orders the clears before its ORs.
            int bits = 0;
            if (32 * tid < words) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint4 v = s_bm4[8 * tid + i];
                    bits += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
                    s_bm4[8 * tid + i] = make_uint4(0u, 0u, 0u, 0u);
                }
            }
            const int64_t s0 = seg_prefix[row];
            if (nb == 1) {
                int total = 0;
                (void)dev::block_exclusive_sum<kSymBlock>(bits, s_sum, total);
                if (tid == 0) seg_nnz[s0] = total;
            } else {  // buckets of 8192 columns: 8 consecutive threads each
                bits += __shfl_xor(bits, 1, dev::kWave);
                bits += __shfl_xor(bits, 2, dev::kWave);
                bits += __shfl_xor(bits, 4, dev::kWave);
                if ((tid & 7) == 0 && (tid >> 3) < nb) seg_nnz[s0 + (tid >> 3)] = bits;
            }
        }
        if (!more) break;  // uniform
        row_start = row_done;
        item = n_item;
        row = n_row;
        p0 = n_p0;
        p_end = n_end;
        bs = n_bs;
        len = n_len;
    }
}

// Distinct columns of every short row (see above): one wavefront per row; wave v of the
// grid takes short-list items v, v + V, v + 2V, ... (V waves), and loads the next item's
// row and offsets while it counts the current one.
__global__ __launch_bounds__(kSymShortBlock) void sym_short_kernel(
    const int *__restrict__ pos_a, const int *__restrict__ crd_a,
    const int *__restrict__ pos_b, const int *__restrict__ crd_b,
    const int *__restrict__ short_list, const int64_t *__restrict__ counts,
    const int64_t *__restrict__ seg_prefix, int64_t *__restrict__ seg_nnz) {
    constexpr int kWaves = kSymShortBlock / dev::kWave;
    __shared__ uint4 s_tab4[kWaves][kSymSlots / 4];
    __shared__ int s_off[kWaves][dev::kWave + 1];
    __shared__ int s_bs[kWaves][dev::kWave];
    const int w = threadIdx.x / dev::kWave, l = dev::lane();
    unsigned *tab = reinterpret_cast<unsigned *>(s_tab4[w]);
    int *off = s_off[w];
    int *bsw = s_bs[w];
    const uint4 empty4 = make_uint4(kSymEmpty, kSymEmpty, kSymEmpty, kSymEmpty);
    const int64_t n_short = counts[1];
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kWaves;
    int64_t item = static_cast<int64_t>(blockIdx.x) * kWaves + w;
    for (int i = l; i < kSymSlots / 4; i += dev::kWave) s_tab4[w][i] = empty4;
    if (item >= n_short) return;  // uniform per wave (no barriers below)
    int row = short_list[item];
    int p_lo = pos_a[row], p_end = pos_a[row + 1];
    for (;;) {
        const int64_t n_item = item + stride;
        const bool more = n_item < n_short;
        int n_row = 0, n_lo = 0, n_end = 0;
        if (more) {  // next item's row and offsets, in flight during this row
            n_row = short_list[n_item];
            n_lo = pos_a[n_row];
            n_end = pos_a[n_row + 1];
        }
        int fresh = 0;
        for (int p0 = p_lo; p0 < p_end; p0 += dev::kWave) {  // 64 A entries at a time
            const int p = p0 + l;
            int bs = 0, len = 0;
            if (p < p_end) {
                const int k = crd_a[p];
                bs = pos_b[k];
                len = pos_b[k + 1] - bs;
            }
            const unsigned long long nz = __ballot(len > 0);
            const int e = static_cast<int>(__popcll(nz & ((1ull << l) - 1ull)));
            const int ne = static_cast<int>(__popcll(nz));
            const int incl = dev::wave_inclusive_sum_dpp(len);
            const int T = __builtin_amdgcn_readlane(incl, dev::kWave - 1);
            if (len > 0) {
                off[e] = incl - len;
                bsw[e] = bs - (incl - len);
            }
            if (l == 0) off[ne] = T;
            wave_sync();
            for (int x0 = 0; x0 < T; x0 += dev::kWave * kSymBatch) {  // uniform
                int first = 0;
                {
                    const int q = x0 + l * dev::kWave;
                    if (l < kSymBatch && q < T) {
                        first = static_cast<int>(dev::last_le(off, 0, ne - 1, q));
                    }
                }
                int c[kSymBatch];
#pragma unroll
                for (int j = 0; j < kSymBatch; ++j) {
                    const int wb = x0 + j * dev::kWave;
                    c[j] = -1;
                    if (wb < T) {  // uniform
                        const int e0 = __builtin_amdgcn_readlane(first, j);
                        const int ee = window_entry(off, ne, e0, wb, l);
                        if (wb + l < T) c[j] = crd_b[bsw[ee] + wb + l];
                    }
                }
#pragma unroll
                for (int j = 0; j < kSymBatch; ++j) {
                    if (c[j] >= 0) {
                        const unsigned key = static_cast<unsigned>(c[j]);
                        unsigned h = (key * 0x9e3779b1u) >> (32 - 12);
                        for (;;) {
                            const unsigned old = atomicCAS(&tab[h], kSymEmpty, key);
                            if (old == kSymEmpty) {
                                ++fresh;
                                break;
                            }
                            if (old == key) break;
                            h = (h + 1u) & (kSymSlots - 1);
                        }
                    }
                }
            }
            wave_sync();  // off / bsw are read before the next 64 entries replace them
        }
        const int total = dev::wave_sum(fresh);
        if (l == 0) seg_nnz[seg_prefix[row]] = total;
        for (int i = l; i < kSymSlots / 4; i += dev::kWave) s_tab4[w][i] = empty4;
        wave_sync();
        if (!more) break;
        item = n_item;
        row = n_row;
        p_lo = n_lo;
        p_end = n_end;
    }
}

// Row offsets from the segment offsets: row i starts at its first segment's offset
// (seg_prefix[rows] = n_seg, whose offset is nnz).
template <typename PosT>
__global__ void seg_pos_kernel(const int64_t *__restrict__ seg_prefix, int rows,
                               const int64_t *__restrict__ seg_out, PosT *__restrict__ pos) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i <= rows; i += gridDim.x * blockDim.x) {
        pos[i] = static_cast<PosT>(seg_out[seg_prefix[i]]);
    }
}

// ---- 6: output -------------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void copy_units_kernel(
    const int64_t *__restrict__ unit_start, const int64_t *__restrict__ unit_nnz,
    const int64_t *__restrict__ unit_out, const int *__restrict__ ukey,
    const float *__restrict__ uval, int *__restrict__ out_crd, float *__restrict__ out_val) {
    const int64_t u = blockIdx.x;
    const int64_t src = unit_start[u], dst = unit_out[u], n = unit_nnz[u];
    for (int64_t x = threadIdx.x; x < n; x += kBlock) {
        out_crd[dst + x] = ukey[src + x];
        out_val[dst + x] = uval[src + x];
    }
}

// Row offsets: a row with products starts at its unit's offset plus its local offset; the
// empty rows just before it share that offset; rows starting at P (and pos[rows]) get nnz.
template <typename PosT>
__global__ void row_pos_kernel(const int64_t *__restrict__ row_off, int rows, int64_t P,
                               int64_t nnz, const int *__restrict__ row_unit,
                               const int *__restrict__ row_local,
                               const int64_t *__restrict__ unit_out, PosT *__restrict__ pos) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i <= rows; i += gridDim.x * blockDim.x) {
        const int64_t rs = row_off[i];
        if (rs == P) {
            pos[i] = static_cast<PosT>(nnz);
        } else if (row_off[i + 1] > rs) {
            const PosT v = static_cast<PosT>(unit_out[row_unit[i]] + row_local[i]);
            pos[i] = v;
            for (int x = i - 1; x >= 0 && row_off[x] == rs; --x) pos[x] = v;
        }
    }
}

// ---- host ------------------------------------------------------------------------------

bool bad_csr(const nacho_csr *t) {
    if (!t || t->dim_i_size < 0 || t->dim_j_size < 0 || t->dim_j_length < 0) return true;
    if (!t->dim_j_offsets) return true;
    if (t->dim_j_length > 0 && (!t->dim_j_indices || !t->values)) return true;
    return false;
}

unsigned grid_for(int64_t n, int per_block) {
    const int64_t g = (n + per_block - 1) / per_block;
    return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(g, 1 << 20)));
}

// Bits that hold every column index of a matrix with `cols` columns.
int col_bits(int cols) {
    int b = 1;
    while (b < 31 && (static_cast<int64_t>(1) << b) < cols) ++b;
    return b;
}

// Workgroups of the long rows' kernels, which stride over their work blocks.
unsigned long_grid(int64_t blocks) {
    return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(blocks, kHistGrid)));
}

// At most this many products (64 MB of run descriptors) or segments are taken as the bound of
// the runs or units; more are counted, which costs a wait of the host for the device.
constexpr int64_t kBoundRuns = int64_t{1} << 22;
constexpr int64_t kBoundUnits = int64_t{1} << 18;

// How the result is sized.  Staged: the reduce units write their distinct entries at their
// units' product offsets in a staging buffer of 8 bytes per product, and a copy moves them
// into the result once every unit's count is known.  Symbolic: the symbolic pass counts
// every segment's distinct columns first, and the units write straight into the result
// (no staging buffer; possible when every column fits the pass's 2^kSymColBits-bit row
// bitmap).  At C4 the copy costs 11.0 ms and the symbolic pass 20.6 ms (its long-row kernel
// is bound by the per-row chain of one workgroup per CU), so the staged path is taken
// while its buffer fits in half of the device memory that is free or cached by the
// library, the symbolic one otherwise.  NACHO_SPGEMM_OUTPUT=staged or =symbolic chooses
// one (symbolic only where it applies).
enum class Output { Staged, Symbolic };

Output output_mode(int64_t products, bool symbolic_fits) {
    const char *v = std::getenv("NACHO_SPGEMM_OUTPUT");
    if (v != nullptr && std::strcmp(v, "staged") == 0) return Output::Staged;
    if (!symbolic_fits) return Output::Staged;
    if (v != nullptr && std::strcmp(v, "symbolic") == 0) return Output::Symbolic;
    if (products <= kBoundRuns) return Output::Staged;  // 32 MB: not worth asking
    size_t free_bytes = 0, total_bytes = 0;
    if (hipMemGetInfo(&free_bytes, &total_bytes) != hipSuccess) return Output::Symbolic;
    const double room = (static_cast<double>(free_bytes) + static_cast<double>(nacho_cached_bytes())) / 2;
    return 8.0 * static_cast<double>(products) <= room ? Output::Staged : Output::Symbolic;
}

struct Product {
    int rows = 0, cols = 0;
    int64_t nnz = 0;
    void *pos = nullptr;
    int *crd = nullptr;
    float *val = nullptr;
};

// Runs the pipeline; result offsets are PosT.  With int32 offsets the call fails with
// NACHO_ERR_INDEX_OVERFLOW (before allocating the result) when nnz(Z) exceeds INT_MAX.
template <typename PosT>
int multiply(Call &call, const nacho_csr *a, const nacho_csr *b, Product *z) {
    const hipStream_t st = call.stream();
    const int rows = a->dim_i_size;
    const int cols = b->dim_j_size;
    const int cb = col_bits(cols);
    // one radix digit over the columns: buckets of 2^shift columns, at most kMaxBuckets
    const int shift = std::max(std::min(kDenseBits, cb), cb - kMaxBucketBits);
    const int nb = cols > 0 ? ((cols - 1) >> shift) + 1 : 1;
    const int dense_min = shift <= kDenseBits ? kDenseMin : kShort;
    const char *name = "spgemm: runs+reduce+output";
    NACHO_TRY(call.timer_start(name));

    // 1-2. products, segments and long-row work blocks per row
    int64_t *per_row = nullptr, *row_off = nullptr, *seg_prefix = nullptr, *blk_off = nullptr;
    int *entries = nullptr;
    NACHO_TRY(call.scratch_n(3 * (static_cast<size_t>(rows) + 1), &per_row));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &entries));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &row_off));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &seg_prefix));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &blk_off));
    int64_t *products = per_row, *seg_count = per_row + (rows + 1),
            *nblk = per_row + 2 * (static_cast<size_t>(rows) + 1);
    if (rows > 0) {
        const int64_t nnz_a = a->dim_j_length;
        const bool split = nnz_a > kSplitEntries;
        const RowCounts counts{products, entries, seg_count, nblk, nb};
        // (short rows: lanes of a row idle, and its counts are stored eight rows at a time)
        const bool one = nnz_a < kOneLaneEntries * static_cast<int64_t>(rows);
        const int64_t lanes = static_cast<int64_t>(rows) * (one ? 1 : kRowLanes);
        auto kernel = one ? row_products_kernel<1> : row_products_kernel<kRowLanes>;
        kernel<<<static_cast<unsigned>((lanes + kBlock - 1) / kBlock), kBlock, 0, st>>>(
            a->dim_j_offsets, a->dim_j_indices, rows, b->dim_j_offsets, split, counts);
        NACHO_TRY_HIP(hipGetLastError());
        if (split) {
            const int64_t spans = (nnz_a + kLongSpan - 1) / kLongSpan;
            long_products_kernel<<<static_cast<unsigned>(spans), kBlock, 0, st>>>(
                a->dim_j_offsets, a->dim_j_indices, rows, nnz_a, b->dim_j_offsets, counts);
            NACHO_TRY_HIP(hipGetLastError());
        }
    }
    int64_t *word[3] = {nullptr, nullptr, nullptr};  // counts read back on the way
    auto words = [&](int n) {
        for (int i = 0; i < n; ++i) NACHO_TRY(call.value_word(i, &word[i]));
        return static_cast<int>(NACHO_OK);
    };
    // The n words' values, once the kernels queued so far have stored them.
    auto values = [&](int n, int64_t *v) {
        NACHO_TRY(call.timer_stop());
        for (int i = 0; i < n; ++i) NACHO_TRY(call.value(i, v + i));
        NACHO_TRY(call.collect_timer());
        return call.timer_start(name);
    };
    NACHO_TRY(words(3));
    const scan::Job row_jobs[3] = {{products, rows, row_off, word[0]},
                                   {seg_count, rows, seg_prefix, word[1]},
                                   {nblk, rows, blk_off, word[2]}};
    NACHO_TRY(scan::exclusive_scans(call, row_jobs, 3));
    int64_t counts3[3] = {0, 0, 0};
    NACHO_TRY(values(3, counts3));
    const int64_t P = counts3[0], n_seg = counts3[1], n_blk = counts3[2];
    if (n_seg >= INT_MAX) return NACHO_ERR_INDEX_OVERFLOW;  // segment ids are int32
    const bool symbolic =
        P > 0 && output_mode(P, cb <= kSymColBits &&
                                    b->dim_j_length <= static_cast<int64_t>(INT_MAX) -
                                                           4 * kSymChunk) == Output::Symbolic;

    int64_t n_units = 0;
    int64_t *seg_out = nullptr;  // symbolic pass: result offset of every segment
    int64_t *unit_start = nullptr, *unit_nnz = nullptr, *unit_out = nullptr;
    int *row_unit = nullptr, *row_local = nullptr;
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &row_unit));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &row_local));
    if (P > 0) {
        // segment table
        int *seg_row = nullptr;
        int64_t *seg_len = nullptr, *seg_off = nullptr, *seg_fill = nullptr;
        int64_t *seg_runs = nullptr, *seg_roff = nullptr;
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg), &seg_row));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg) + 1, &seg_len));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg) + 1, &seg_off));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg), &seg_fill));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg) + 1, &seg_runs));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg) + 1, &seg_roff));
        int *blk_row = nullptr;
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_blk) + 1, &blk_row));
        segments_kernel<<<grid_for(rows, 256), 256, 0, st>>>(row_off, seg_prefix, rows, entries,
                                                            blk_off, blk_row, seg_row, seg_len,
                                                            seg_runs, seg_fill);
        NACHO_TRY_HIP(hipGetLastError());

        // symbolic pass: distinct columns per segment, scanned into result offsets
        if (symbolic) {
            int64_t *seg_nnz = nullptr, *keys = nullptr, *ranks = nullptr, *counts = nullptr;
            int *lists = nullptr, *work = nullptr;
            NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg) + 1, &seg_nnz));
            NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg) + 1, &seg_out));
            NACHO_TRY(call.scratch_n(2 * (static_cast<size_t>(rows) + 1), &keys));
            NACHO_TRY(call.scratch_n(2 * (static_cast<size_t>(rows) + 1), &ranks));
            NACHO_TRY(call.scratch_n(2 * static_cast<size_t>(rows) + 2, &lists));
            NACHO_TRY(call.scratch_n(2, &counts));
            NACHO_TRY(call.scratch_n(1, &work));
            int64_t *key2 = keys + (rows + 1), *rank2 = ranks + (rows + 1);
            int *long_list = lists, *short_list = lists + (rows + 1);
            sym_flags_kernel<<<grid_for(rows, 256), 256, 0, st>>>(row_off, rows, seg_prefix,
                                                                 keys, key2, seg_nnz, work);
            NACHO_TRY_HIP(hipGetLastError());
            NACHO_TRY(scan::exclusive_scan_i64(call, keys, rows, ranks));
            NACHO_TRY(scan::exclusive_scan_i64(call, key2, rows, rank2));
            sym_lists_kernel<<<grid_for(rows, 256), 256, 0, st>>>(row_off, rows, ranks, rank2,
                                                                 long_list, short_list, counts);
            NACHO_TRY_HIP(hipGetLastError());
            int g_long = 0, g_short = 0;
            NACHO_TRY(resident_grid(reinterpret_cast<const void *>(sym_long_kernel), kSymBlock,
                                    &g_long));
            NACHO_TRY(resident_grid(reinterpret_cast<const void *>(sym_short_kernel),
                                    kSymShortBlock, &g_short));
            sym_long_kernel<<<static_cast<unsigned>(g_long), kSymBlock, 0, st>>>(
                a->dim_j_offsets, a->dim_j_indices, b->dim_j_offsets, b->dim_j_indices,
                long_list, counts, work, seg_prefix, nb, cols, seg_nnz);
            NACHO_TRY_HIP(hipGetLastError());
            sym_short_kernel<<<static_cast<unsigned>(g_short), kSymShortBlock, 0, st>>>(
                a->dim_j_offsets, a->dim_j_indices, b->dim_j_offsets, b->dim_j_indices,
                short_list, counts, seg_prefix, seg_nnz);
            NACHO_TRY_HIP(hipGetLastError());
            NACHO_TRY(scan::exclusive_scan_i64(call, seg_nnz, n_seg, seg_out));
        }

        // 3. histogram, segment offsets, runs
        int *ukey = nullptr;  // the units' output: staged at product offsets, or the result
        float *uval = nullptr;
        if (!symbolic) {
            NACHO_TRY(call.scratch_n(static_cast<size_t>(P), &ukey));
            NACHO_TRY(call.scratch_n(static_cast<size_t>(P), &uval));
        }
        // long rows' bucket counts from B's runs (P > 0, so B has entries)
        const int64_t nnz_b = b->dim_j_length;
        const int rows_b = b->dim_i_size;
        int2 *cv_b = nullptr;
        NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_b), &cv_b));
        int64_t *flag = nullptr, *run_idx = nullptr;
        int2 *run = nullptr;
        int *run_start = nullptr;
        if (n_blk > 0) {
            NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_b) + 1, &flag));
            NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_b) + 1, &run_idx));
            NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_b), &run));
            NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_b) + 1, &run_start));
        }
        pairs_flags_kernel<<<grid_for(nnz_b, 256), 256, 0, st>>>(b->dim_j_indices, b->values,
                                                                 nnz_b, shift, cv_b, flag);
        NACHO_TRY_HIP(hipGetLastError());
        const BRuns br{run_idx, run, run_start};
        if (n_blk > 0) {
            run_row_starts_kernel<<<grid_for(rows_b, 256), 256, 0, st>>>(b->dim_j_offsets,
                                                                          rows_b, flag);
            NACHO_TRY_HIP(hipGetLastError());
            NACHO_TRY(scan::exclusive_scan_i64(call, flag, nnz_b, run_idx));
            runs_kernel<<<grid_for(nnz_b, 256), 256, 0, st>>>(b->dim_j_indices, nnz_b, shift,
                                                              flag, run_idx, run, run_start);
            NACHO_TRY_HIP(hipGetLastError());
            run_lengths_kernel<<<grid_for(nnz_b, 256), 256, 0, st>>>(run_idx, nnz_b, run_start,
                                                                     run);
            NACHO_TRY_HIP(hipGetLastError());
            long_hist_kernel<<<long_grid(n_blk), kBlock, 0, st>>>(
                a->dim_j_offsets, a->dim_j_indices, blk_off, blk_row, rows, b->dim_j_offsets, br,
                nb, seg_prefix, seg_len, seg_runs);
            NACHO_TRY_HIP(hipGetLastError());
        }
        // A product lies in one run: few products bound the runs without waiting for their
        // count.
        int64_t n_runs = P, nnz_sym = 0;
        const bool count_runs = P > kBoundRuns;
        if (count_runs) NACHO_TRY(words(1));
        const scan::Job seg_jobs[2] = {{seg_len, n_seg, seg_off},
                                       {seg_runs, n_seg, seg_roff, count_runs ? word[0] : nullptr}};
        NACHO_TRY(scan::exclusive_scans(call, seg_jobs, 2));
        if (count_runs) NACHO_TRY(values(1, &n_runs));
        if (symbolic) {
            NACHO_TRY(call.timer_stop());
            NACHO_TRY(call.read_back(&nnz_sym, seg_out + n_seg, sizeof(nnz_sym)));
            NACHO_TRY(call.timer_start(name));
            if (sizeof(PosT) == sizeof(int32_t) && nnz_sym > INT_MAX) {
                return NACHO_ERR_INDEX_OVERFLOW;
            }
            NACHO_TRY(call.result_n(static_cast<size_t>(nnz_sym), &z->crd));
            NACHO_TRY(call.result_n(static_cast<size_t>(nnz_sym), &z->val));
            ukey = z->crd;
            uval = z->val;
        }
        int4 *desc = nullptr;
        NACHO_TRY(call.scratch_n(static_cast<size_t>(std::max<int64_t>(n_runs, 1)), &desc));
        if (n_blk > 0) {
            long_runs_kernel<<<long_grid(n_blk), kBlock, 0, st>>>(
                a->dim_j_offsets, a->dim_j_indices, a->values, blk_off, blk_row, rows,
                b->dim_j_offsets, br, nb, seg_prefix, seg_roff, seg_fill, desc);
            NACHO_TRY_HIP(hipGetLastError());
        }
        short_runs_kernel<<<grid_for(rows, 256), 256, 0, st>>>(
            a->dim_j_offsets, a->dim_j_indices, a->values, rows, row_off, seg_prefix, seg_roff,
            b->dim_j_offsets, desc);
        NACHO_TRY_HIP(hipGetLastError());

        // 4. units
        int64_t *seg_units = seg_fill;  // the run fill counters are spent
        int64_t *unit_prefix = nullptr;
        NACHO_TRY(call.scratch_n(static_cast<size_t>(n_seg) + 1, &unit_prefix));
        unit_count_kernel<<<grid_for(n_seg, 256), 256, 0, st>>>(
            seg_len, seg_off, n_seg, seg_row, row_off, dense_min, seg_units);
        NACHO_TRY_HIP(hipGetLastError());
        NACHO_TRY(words(3));
        NACHO_TRY(scan::exclusive_scan_i64(call, seg_units, n_seg, unit_prefix, word[0]));
        // (a unit starts at a segment: few segments bound the units without waiting)
        int64_t bound = n_seg;
        const bool count_units = n_seg > kBoundUnits;
        if (count_units) {
            NACHO_TRY(values(1, &bound));
            if (bound > INT_MAX) return NACHO_ERR_INDEX_OVERFLOW;
        }
        int *unit_seg = nullptr;
        NACHO_TRY(call.scratch_n(static_cast<size_t>(bound), &unit_seg));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(bound) + 1, &unit_start));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(bound) + 1, &unit_nnz));
        NACHO_TRY(call.scratch_n(static_cast<size_t>(bound) + 1, &unit_out));
        int *lists = nullptr;  // dense list, bitmap list, sort list
        int64_t *kinds = nullptr;  // dense flags, their ranks, bitmap flags, their ranks
        NACHO_TRY(call.scratch_n(3 * static_cast<size_t>(bound), &lists));
        NACHO_TRY(call.scratch_n(4 * (static_cast<size_t>(bound) + 1), &kinds));
        int64_t *unit_dense = kinds, *dense_rank = kinds + (bound + 1);
        int64_t *unit_bitmap = kinds + 2 * (bound + 1), *bitmap_rank = kinds + 3 * (bound + 1);
        int *dense_list = lists, *bitmap_list = lists + bound, *sort_list = lists + 2 * bound;
        unit_map_kernel<<<grid_for(n_seg + 1, 256), 256, 0, st>>>(
            seg_units, unit_prefix, seg_off, seg_len, seg_row, row_off, dense_min, n_seg, P,
            unit_seg, unit_start, unit_dense);
        NACHO_TRY_HIP(hipGetLastError());
        unit_bitmap_kernel<<<grid_for(bound, 256), 256, 0, st>>>(
            unit_seg, unit_dense, unit_prefix + n_seg, bound, n_seg, seg_len, seg_row, row_off,
            shift <= kDenseBits, unit_bitmap);
        NACHO_TRY_HIP(hipGetLastError());
        const scan::Job kind_jobs[2] = {{unit_dense, bound, dense_rank, word[1]},
                                        {unit_bitmap, bound, bitmap_rank, word[2]}};
        NACHO_TRY(scan::exclusive_scans(call, kind_jobs, 2));
        int64_t kinds3[3] = {0, 0, 0};
        NACHO_TRY(values(3, kinds3));
        n_units = kinds3[0];
        const int64_t n_dense = kinds3[1], n_bitmap = kinds3[2];
        unit_lists_kernel<<<grid_for(n_units, 256), 256, 0, st>>>(
            unit_dense, dense_rank, unit_bitmap, bitmap_rank, n_units, dense_list, bitmap_list,
            sort_list);
        NACHO_TRY_HIP(hipGetLastError());
        const int n_kind[3] = {static_cast<int>(n_dense),
                               static_cast<int>(n_units - n_dense - n_bitmap),
                               static_cast<int>(n_bitmap)};

        // 5. reduce
        const unsigned ug = static_cast<unsigned>(n_units);
        if (n_kind[1] > 0 && cb + kOrdBits <= 32) {
            sort_unit_kernel<uint32_t><<<static_cast<unsigned>(n_kind[1]), kBlock, 0, st>>>(
                sort_list, unit_seg, unit_start, n_units, n_seg, seg_len, seg_off, seg_row,
                row_off, cb, desc, seg_roff, cv_b, ukey, uval, unit_nnz, row_unit, row_local,
                seg_out);
        } else if (n_kind[1] > 0) {
            sort_unit_kernel<uint64_t><<<static_cast<unsigned>(n_kind[1]), kBlock, 0, st>>>(
                sort_list, unit_seg, unit_start, n_units, n_seg, seg_len, seg_off, seg_row,
                row_off, 32, desc, seg_roff, cv_b, ukey, uval, unit_nnz, row_unit, row_local,
                seg_out);
        }
        NACHO_TRY_HIP(hipGetLastError());
        if (n_kind[2] > 0) {
            bitmap_unit_kernel<<<static_cast<unsigned>(n_kind[2]), kBitmapBlock, 0, st>>>(
                bitmap_list, unit_seg, unit_start, n_units, n_seg, seg_len, seg_off, seg_prefix,
                seg_row, row_off, shift, desc, seg_roff, cv_b, ukey, uval, unit_nnz, row_unit,
                row_local, seg_out);
            NACHO_TRY_HIP(hipGetLastError());
        }
        if (n_kind[0] > 0) {
            dense_unit_kernel<<<static_cast<unsigned>(n_kind[0]), kDenseBlock, 0, st>>>(
                dense_list, unit_seg, unit_start, seg_len, seg_prefix, seg_row, row_off, shift,
                cols, desc, seg_roff, cv_b, ukey, uval, unit_nnz, row_unit, row_local, seg_out);
            NACHO_TRY_HIP(hipGetLastError());
        }
        if (symbolic) {
            z->nnz = nnz_sym;  // the units wrote straight into the result
        } else {
            NACHO_TRY(words(1));
            NACHO_TRY(scan::exclusive_scan_i64(call, unit_nnz, n_units, unit_out, word[0]));
            int64_t nnz = 0;
            NACHO_TRY(values(1, &nnz));
            if (sizeof(PosT) == sizeof(int32_t) && nnz > INT_MAX) return NACHO_ERR_INDEX_OVERFLOW;

            // 6. output
            NACHO_TRY(call.result_n(static_cast<size_t>(nnz), &z->crd));
            NACHO_TRY(call.result_n(static_cast<size_t>(nnz), &z->val));
            if (nnz > 0) {
                copy_units_kernel<<<ug, kBlock, 0, st>>>(unit_start, unit_nnz, unit_out, ukey,
                                                         uval, z->crd, z->val);
                NACHO_TRY_HIP(hipGetLastError());
            }
            z->nnz = nnz;
        }
    }
    PosT *pos = nullptr;
    NACHO_TRY(call.result_n(static_cast<size_t>(rows) + 1, &pos));
    if (seg_out) {
        seg_pos_kernel<PosT><<<grid_for(static_cast<int64_t>(rows) + 1, 256), 256, 0, st>>>(
            seg_prefix, rows, seg_out, pos);
    } else {
        row_pos_kernel<PosT><<<grid_for(static_cast<int64_t>(rows) + 1, 256), 256, 0, st>>>(
            row_off, rows, P, z->nnz, row_unit, row_local, unit_out, pos);
    }
    NACHO_TRY_HIP(hipGetLastError());
    NACHO_TRY(call.timer_stop());
    NACHO_TRY(call.collect_timer());

    z->rows = rows;
    z->cols = cols;
    z->pos = pos;
    return NACHO_OK;
}

int check_operands(const nacho_csr *a, const nacho_csr *b, int32_t num_blocks,
                   int32_t threads_per_block) {
    NACHO_TRY(check_launch_hints(num_blocks, threads_per_block));
    if (bad_csr(a) || bad_csr(b)) return NACHO_ERR_INVALID_ARGUMENT;
    if (a->dim_j_size != b->dim_i_size) return NACHO_ERR_INVALID_ARGUMENT;
    return NACHO_OK;
}

}  // namespace spgemm
}  // namespace nacho

extern "C" {

int nacho_gpu_spgemm64_f32(const nacho_csr *a, const nacho_csr *b, nacho_csr64 *z,
                           int32_t num_blocks, int32_t threads_per_block, void *stream,
                           const nacho_allocator *alloc) {
    using namespace nacho;
    if (!z) return NACHO_ERR_INVALID_ARGUMENT;
    *z = nacho_csr64{};
    NACHO_TRY(spgemm::check_operands(a, b, num_blocks, threads_per_block));
    Call call(stream, alloc);
    spgemm::Product p;
    NACHO_TRY(spgemm::multiply<int64_t>(call, a, b, &p));
    z->dim_i_size = p.rows;
    z->dim_j_size = p.cols;
    z->dim_j_offsets = static_cast<int64_t *>(p.pos);
    z->dim_j_length = p.nnz;
    z->dim_j_indices = p.crd;
    z->values = p.val;
    z->nnz = p.nnz;
    call.commit();
    return NACHO_OK;
}

int nacho_gpu_spgemm_f32(const nacho_csr *a, const nacho_csr *b, nacho_csr *z,
                         int32_t num_blocks, int32_t threads_per_block, void *stream,
                         const nacho_allocator *alloc) {
    using namespace nacho;
    if (!z) return NACHO_ERR_INVALID_ARGUMENT;
    *z = nacho_csr{};
    NACHO_TRY(spgemm::check_operands(a, b, num_blocks, threads_per_block));
    Call call(stream, alloc);
    spgemm::Product p;
    NACHO_TRY(spgemm::multiply<int32_t>(call, a, b, &p));
    z->dim_i_size = p.rows;
    z->dim_j_size = p.cols;
    z->dim_j_offsets = static_cast<int32_t *>(p.pos);
    z->dim_j_length = static_cast<int32_t>(p.nnz);
    z->dim_j_indices = p.crd;
    z->values = p.val;
    z->nnz = static_cast<int32_t>(p.nnz);
    call.commit();
    return NACHO_OK;
}

}  // extern "C"
