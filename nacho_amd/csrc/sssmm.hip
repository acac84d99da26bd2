// Masked SpGEMM (sssmm): Z_ik = sum_j a_ij * b_jk * c_ik over the (i, k) stored in C that
// at least one product reaches, for gfx950.
//
// Reference path replaced: sssmm (compiler.cpp:150-153, GPU-only), whose generated kernel
// expands the products of A B restricted to C's pattern through the scatter-reduction path
// (stitch_and_generate_gpu.cpp:14-138).  Its benchmark checks the structure against
// cuSPARSE A*B followed by csr_mul with C (benchmarks/sssmm.py:46-51): the result is C's
// pattern intersected with the product's pattern, and no entry of A B outside C is formed.
//
// Here every mask entry (i, k) is an inner product of row i of A with column k of B.  Both
// operands are indexed by j through per-row / per-column hash tables, so the entry costs
// min(|A_i|, |B_k|) probes: the shorter list is walked and each j is looked up in the other
// operand's table.  On power-law inputs that is far less than expanding every product of
// A B (R-MAT scale 20 squared and masked by itself: 1.1e9 probes against 6.0e9 products).
//
//   count_cols_kernel, scan          column counts of B, column offsets
//   table_sizes_kernel, scans        hash table sizes (power of two >= 2 * length) and bases
//   fill_kernel                      empty tables, zeroed filter
//   transpose_kernel                 B's entries into columns (row ids + values), and into
//                                    the per-column tables keyed by row id
//   rows_table_kernel                A's entries into the per-row tables keyed by column id
//   work_kernel, scan                per mask entry: row, probes = min(|A_i|, |B_k|), which
//                                    side is walked, which table is probed
//   chunk_bounds_kernel              first / last mask entry of every 4096-probe chunk
//   probe_kernel                     one chunk per workgroup: load-balanced decode of probes
//                                    to mask entries (max-scan of entry start marks in LDS),
//                                    walk, filter, probe, (a * b) * c per hit in float32 as
//                                    written, summed per entry in float64 in LDS, one atomic
//                                    add per entry and chunk (of few mask entries) or per
//                                    entry and wavefront
//   keep_kernel, scan, output_kernel the entries that some product reached, in C's order
//
// Values: each term is rounded as the reference writes it, ((a * b) * c) in float32, and the
// terms of an entry are summed in float64 and rounded once.  The order of the float64 sums
// follows atomic arrival, so values are reproducible within one float32 rounding; the structure
// is exact.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>

#include "device_utils.hpp"
#include "runtime.hpp"
#include "scan.hpp"

namespace nacho {
namespace sssmm {

constexpr int kBlock = 256;
constexpr int kChunk = 4096;       // probes per workgroup
constexpr int kPer = kChunk / kBlock;
constexpr int kBatch = 4;  // probe rounds whose loads are issued together
constexpr uint32_t kEmptyKey = 0xffffffffu;
constexpr uint64_t kEmptySlot = 0x00000000ffffffffull;  // value bits 0, key empty
constexpr uint32_t kWalkB = 0x80000000u;  // entry flag: walk B's column, probe A's row table

using dev::block_exclusive_max;
using dev::last_le;

__device__ __forceinline__ int pad(int i) { return i + (i >> 4); }
constexpr int kPadded = kChunk + kChunk / 16;

__device__ __forceinline__ uint32_t mix(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// The filter's bit of a key in its home slot's byte.
__device__ __forceinline__ uint32_t filter_bit(uint32_t hash) { return hash >> 29; }

// Inserts the key into its table; the caller has set its bit in the filter (hash: mix(key)).
__device__ __forceinline__ void table_insert(uint64_t *table, int64_t base, uint32_t mask,
                                             uint32_t key, uint32_t hash, float value) {
    const uint64_t word = (static_cast<uint64_t>(__float_as_uint(value)) << 32) | key;
    uint32_t h = hash & mask;
    for (;;) {
        auto *slot = reinterpret_cast<unsigned long long *>(table + base + h);
        if (atomicCAS(slot, static_cast<unsigned long long>(kEmptySlot),
                      static_cast<unsigned long long>(word)) == kEmptySlot) {
            return;
        }
        h = (h + 1) & mask;
    }
}

// A key's bit in the filter's word (of four slots) of its home slot.
__device__ __forceinline__ unsigned filter_word_bit(int64_t home, uint32_t hash) {
    return 1u << (8u * static_cast<uint32_t>(home & 3) + filter_bit(hash));
}

__global__ void fill_kernel(uint64_t *__restrict__ p, int64_t n, uint64_t v) {
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        p[i] = v;
    }
}

// The mask entries' sums and hit flags, zeroed.
__global__ void zero_sums_kernel(double *__restrict__ acc, int *__restrict__ hit, int64_t n) {
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        acc[i] = 0.0;
        hit[i] = 0;
    }
}

// Workgroup b counts the columns of entries [b*kSpan, (b+1)*kSpan): columns below kHotCols in
// an LDS histogram flushed with one global atomic per nonzero bin (power-law operands put
// most entries in a few low-numbered hub columns, whose global counters would serialise
// every entry's atomic), the others with a global atomic each.
constexpr int kHotCols = 8192;
constexpr int kSpan = 16 * kBlock;  // entries per workgroup of the two kernels below

__global__ __launch_bounds__(kBlock) void count_cols_kernel(const int *__restrict__ crd,
                                                            int64_t n, int cols,
                                                            unsigned long long *__restrict__ count) {
    __shared__ unsigned hist[kHotCols];
    const int hot = min(cols, kHotCols);
    for (int i = threadIdx.x; i < hot; i += kBlock) hist[i] = 0u;
    __syncthreads();
    const int64_t lo = static_cast<int64_t>(blockIdx.x) * kSpan;
    const int64_t hi = min(n, lo + kSpan);
    for (int64_t e = lo + threadIdx.x; e < hi; e += kBlock) {
        const int k = crd[e];
        if (k < hot) {
            atomicAdd(&hist[k], 1u);
        } else {
            atomicAdd(&count[k], 1ull);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < hot; i += kBlock) {
        if (hist[i]) atomicAdd(&count[i], static_cast<unsigned long long>(hist[i]));
    }
}

// Table of a list of `len` entries: the smallest power of two >= 2 * len (0 when empty).
__device__ __forceinline__ int64_t table_size(int64_t len) {
    if (len == 0) return 0;
    int64_t s = 2;
    while (s < 2 * len) s <<= 1;
    return s;
}

// Table sizes of B's columns (lengths `count`) and of A's rows (offsets `pos`).
__global__ void table_sizes_kernel(const int64_t *__restrict__ count, int cols,
                                   int64_t *__restrict__ size_b, const int *__restrict__ pos,
                                   int rows, int64_t *__restrict__ size_a) {
    const int stride = gridDim.x * blockDim.x;
    const int first = blockIdx.x * blockDim.x + threadIdx.x;
    for (int x = first; x < cols; x += stride) size_b[x] = table_size(count[x]);
    for (int x = first; x < rows; x += stride) size_a[x] = table_size(pos[x + 1] - pos[x]);
}

// Entries per workgroup of the two table builders: kSpan, less where that would leave most of
// the chip idle (40,000 entries in 10 workgroups took 88 and 72 us).
inline int table_span(int64_t nnz) {
    const int64_t rounds = (nnz + 2048 * kBlock - 1) / (2048 * kBlock);
    return static_cast<int>(std::min<int64_t>(kSpan, std::max<int64_t>(rounds, 1) * kBlock));
}

// Workgroup b takes entries [lo, hi) = [b*span, (b+1)*span) of a list split by the offsets
// p (n + 1 entries); [r_lo, r_hi] holds the rows of its first and last entry and so bounds
// every entry's row search.  False (for the whole workgroup) when the span is empty.
__device__ __forceinline__ bool span_rows(const int *__restrict__ p, int n, int64_t nnz, int span,
                                          int64_t &lo, int64_t &hi, int &r_lo, int &r_hi) {
    __shared__ int s_rows[2];
    lo = static_cast<int64_t>(blockIdx.x) * span;
    hi = min(nnz, lo + span);
    if (lo >= hi) return false;
    if (threadIdx.x == 0) {
        const int first = static_cast<int>(last_le(p, 0, n - 1, lo));
        s_rows[0] = first;
        s_rows[1] = static_cast<int>(last_le(p, first, n - 1, hi - 1));
    }
    __syncthreads();
    r_lo = s_rows[0];
    r_hi = s_rows[1];
    return true;
}

// B's entries into columns (CSC) and into the per-column tables keyed by row id.
__global__ __launch_bounds__(kBlock) void transpose_kernel(
    const int *__restrict__ pb, int inner, const int *__restrict__ cb,
    const float *__restrict__ vb, int64_t nnz_b, int span, const int64_t *__restrict__ col_off,
    unsigned long long *__restrict__ col_fill, const int64_t *__restrict__ tab_off,
    int *__restrict__ csc_row, float *__restrict__ csc_val, uint64_t *__restrict__ tab_b,
    unsigned *__restrict__ filter) {
    int64_t lo, hi;
    int r_lo, r_hi;
    if (!span_rows(pb, inner, nnz_b, span, lo, hi, r_lo, r_hi)) return;
    for (int64_t e = lo + threadIdx.x; e < hi; e += kBlock) {
        const int j = static_cast<int>(last_le(pb, r_lo, r_hi, e));
        const int k = cb[e];
        const float v = vb[e];
        const int64_t slot = col_off[k] + static_cast<int64_t>(atomicAdd(&col_fill[k], 1ull));
        csc_row[slot] = j;
        csc_val[slot] = v;
        const int64_t base = tab_off[k];
        const uint32_t mask = static_cast<uint32_t>(tab_off[k + 1] - base - 1);
        const uint32_t hash = mix(static_cast<uint32_t>(j));
        const int64_t home = base + (hash & mask);
        atomicOr(&filter[home >> 2], filter_word_bit(home, hash));
        table_insert(tab_b, base, mask, static_cast<uint32_t>(j), hash, v);
    }
}

// A's entries into the per-row tables keyed by column id, which start at slot `first`.  The filter
// of the rows that lie inside the workgroup's span, whose tables are neighbours, is built in LDS
// and stored; that of a row which reaches out of it by global atomics.  (All by global atomics,
// where the entries of a short row meet in a few words: 310 us for the 3.9M entries of a band of
// 15 a row, 182 so, 195 without a filter.)
__global__ __launch_bounds__(kBlock) void rows_table_kernel(
    const int *__restrict__ pa, int rows, const int *__restrict__ ca,
    const float *__restrict__ va, int64_t nnz_a, int span, const int64_t *__restrict__ tab_off,
    uint64_t *__restrict__ tab, unsigned *__restrict__ filter, int64_t first) {
    // (a list's table is smaller than four times its length, and starts anywhere in a word)
    constexpr int kWords = kSpan + 1;
    __shared__ unsigned s_filter[kWords];
    int64_t lo, hi;
    int r_lo, r_hi;
    if (!span_rows(pa, rows, nnz_a, span, lo, hi, r_lo, r_hi)) return;
    const int i0 = pa[r_lo] >= lo ? r_lo : r_lo + 1;       // rows [i0, i1) lie inside
    const int i1 = pa[r_hi + 1] <= hi ? r_hi + 1 : r_hi;
    const int64_t s0 = i0 < i1 ? first + tab_off[i0] : 0;  // their slots
    const int64_t s1 = i0 < i1 ? first + tab_off[i1] : 0;
    const int64_t w0 = s0 >> 2;
    const int words = static_cast<int>((s1 + 3) / 4 - w0);
    for (int x = threadIdx.x; x < words; x += kBlock) s_filter[x] = 0u;
    __syncthreads();
    for (int64_t e = lo + threadIdx.x; e < hi; e += kBlock) {
        const int i = static_cast<int>(last_le(pa, r_lo, r_hi, e));
        const int64_t base = first + tab_off[i];
        const uint32_t mask = static_cast<uint32_t>(first + tab_off[i + 1] - base - 1);
        const uint32_t key = static_cast<uint32_t>(ca[e]);
        const uint32_t hash = mix(key);
        const int64_t home = base + (hash & mask);
        const unsigned bit = filter_word_bit(home, hash);
        if (i >= i0 && i < i1) {
            atomicOr(&s_filter[static_cast<int>((home >> 2) - w0)], bit);
        } else {
            atomicOr(&filter[home >> 2], bit);
        }
        table_insert(tab, base, mask, key, hash, va[e]);
    }
    __syncthreads();
    for (int x = threadIdx.x; x < words; x += kBlock) {
        const unsigned v = s_filter[x];
        if (v == 0) continue;
        const int64_t at = 4 * (w0 + x);
        if (at >= s0 && at + 4 <= s1) {
            filter[w0 + x] = v;  // (zeroed before)
        } else {
            atomicOr(&filter[w0 + x], v);  // shared with a neighbour's table
        }
    }
}

// Per mask entry e = (i, k): probes = min(|A_i|, |B_k|) (0 when either is empty), the walked
// list's base, and the probed table's base and mask (kWalkB set when B's column is walked).
__global__ void work_kernel(const int *__restrict__ pc, int rows, const int *__restrict__ cc,
                            int64_t nnz_c, const int *__restrict__ pa,
                            const unsigned long long *__restrict__ col_count,
                            const int64_t *__restrict__ col_off,
                            const int64_t *__restrict__ tab_a_off, int64_t first_a,
                            const int64_t *__restrict__ tab_b_off, int64_t *__restrict__ work,
                            int64_t *__restrict__ walk_base, int64_t *__restrict__ probe_base,
                            uint32_t *__restrict__ probe_mask) {
    for (int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; e < nnz_c;
         e += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int i = static_cast<int>(last_le(pc, 0, rows - 1, e));
        const int k = cc[e];
        const int64_t la = pa[i + 1] - pa[i];
        const int64_t lb = static_cast<int64_t>(col_count[k]);
        const bool walk_b = lb < la;
        work[e] = (la == 0 || lb == 0) ? 0 : (walk_b ? lb : la);
        walk_base[e] = walk_b ? col_off[k] : static_cast<int64_t>(pa[i]);
        const int64_t t0 = walk_b ? tab_a_off[i] : tab_b_off[k];
        const int64_t t1 = walk_b ? tab_a_off[i + 1] : tab_b_off[k + 1];
        probe_base[e] = walk_b ? first_a + t0 : t0;
        probe_mask[e] = static_cast<uint32_t>(t1 - t0 - 1) | (walk_b ? kWalkB : 0u);
    }
}

// First and last mask entry of every chunk of kChunk probes.
__global__ void chunk_bounds_kernel(const int64_t *__restrict__ woff, int64_t nnz_c,
                                    int64_t total, int64_t chunks, int64_t *__restrict__ bounds) {
    for (int64_t x = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
         x < 2 * chunks; x += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t c = x >> 1;
        const int64_t q = (x & 1) ? min((c + 1) * kChunk, total) - 1 : c * kChunk;
        bounds[x] = last_le(woff, 0, nnz_c - 1, q);
    }
}

// A chunk of at most this many mask entries (a few dozen where lists are long) keeps their
// fields in LDS and sums them there (binary64 LDS atomics, then one global atomic per entry); a
// chunk of more, short ones reads the fields from memory, and each wavefront sums an entry's hits
// in LDS before one global atomic for its 64 probes.  (With a global atomic for every hit, the
// probes of a band of 15 entries a row, where most hit, took 2088 us instead of 439.  A band of 17,
// 241 mask entries a chunk: 1368 us a call in LDS, 1505 the other way.)
constexpr int kAccEntries = 256;
static_assert(kAccEntries == kBlock, "or one slot per lane");

// What a probe needs of its mask entry: the walked list's position of probe 0 of the chunk (as
// if the list went on to it), the probed table's slots and mask | kWalkB.
struct EntryFields {
    int walk;
    uint32_t mask;
    int64_t table;
};

// Bound by the lines that its random reads fetch: R-MAT 2^20 masked by itself, 1.14e9 probes into
// 134 MB of slots each side, 23 GB in 5.7 ms.  Without the filter, whose bytes mostly stay in L2
// and which tells most misses, one line per probe: 58 GB in 10.5 ms.  On the way: sums in LDS
// instead of a segmented sum by shuffles per 64 probes 10.5 -> 9.7 ms; the filter 6.9; the entries'
// fields in LDS and the values read after the filter, four rounds at a time, 5.7 (two rounds 6.0,
// eight 7.0).
__global__ __launch_bounds__(kBlock) void probe_kernel(
    const int64_t *__restrict__ woff, const int64_t *__restrict__ bounds, int64_t total,
    const int64_t *__restrict__ walk_base, const int64_t *__restrict__ probe_base,
    const uint32_t *__restrict__ probe_mask, const int *__restrict__ ca,
    const float *__restrict__ va, const int *__restrict__ csc_row,
    const float *__restrict__ csc_val, const uint64_t *__restrict__ tab,
    const unsigned char *__restrict__ filter, const float *__restrict__ vc,
    double *__restrict__ acc, int *__restrict__ hit) {
    __shared__ EntryFields s_field[kAccEntries];
    __shared__ double s_acc[kAccEntries];
    __shared__ unsigned char s_hit[kAccEntries];
    __shared__ int s_e[kPadded];
    __shared__ int s_wave[kBlock / dev::kWave];
    // neighbouring chunks (a mask row's probes into one table) on one XCD, 64 at a time:
    // probe_kernel fetched 11% less at C4
    const int64_t chunk = dev::xcd_block<64>();
    const int64_t c0 = chunk * kChunk;
    const int n = static_cast<int>(min(static_cast<int64_t>(kChunk), total - c0));
    const int64_t e_lo = bounds[2 * chunk], e_hi = bounds[2 * chunk + 1];
    const int l = dev::lane();
    // a chunk of at most kAccEntries mask entries sums them here
    const bool local = e_hi - e_lo < kAccEntries;
    const int entries = static_cast<int>(min(e_hi - e_lo + 1, static_cast<int64_t>(kAccEntries)));
    auto fields = [&](int64_t e) {
        // (positions stay below 2^31: a list's own do, and the chunk's probes inside it too)
        return EntryFields{static_cast<int>(walk_base[e] - (woff[e] - c0)), probe_mask[e],
                           probe_base[e]};
    };
    for (int x = threadIdx.x; x < entries; x += kBlock) {
        s_acc[x] = 0.0;
        s_hit[x] = 0;
        if (local) s_field[x] = fields(e_lo + x);
    }
    // decode: s_e[x] = (mask entry of probe c0 + x) - e_lo
    for (int x = threadIdx.x; x < kChunk; x += kBlock) s_e[pad(x)] = 0;
    __syncthreads();
    for (int64_t e = e_lo + 1 + threadIdx.x; e <= e_hi; e += kBlock) {
        const int64_t x = woff[e] - c0;
        if (x >= 0 && x < n) atomicMax(&s_e[pad(static_cast<int>(x))], static_cast<int>(e - e_lo));
    }
    __syncthreads();
    const int base = threadIdx.x * kPer;
    int m = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) m = max(m, s_e[pad(base + u)]);
    int run = block_exclusive_max(m, s_wave);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        run = max(run, s_e[pad(base + u)]);
        s_e[pad(base + u)] = run;
    }
    __syncthreads();
    // probes, kBlock consecutive ones per round so a wavefront holds 64 consecutive probes.
    // kBatch rounds at a time: each step of a probe's chain of dependent loads (the entry's
    // fields, the walked entry, the table slot) is issued for all of them before the next,
    // so that kBatch chains are in flight per lane.
    static_assert(kPer % kBatch == 0, "rounds come in whole batches");
    for (int r0 = 0; r0 < kPer; r0 += kBatch) {
        bool live[kBatch];
        int ent[kBatch], wb[kBatch];  // mask entry (from e_lo), position in the walked list
        int64_t tb[kBatch];
        uint32_t pm[kBatch];
#pragma unroll
        for (int g = 0; g < kBatch; ++g) {
            const int x = threadIdx.x + (r0 + g) * kBlock;
            live[g] = x < n;
            ent[g] = live[g] ? s_e[pad(x)] : 0;
            const EntryFields f = local ? s_field[ent[g]] : fields(e_lo + ent[g]);
            pm[g] = f.mask;
            wb[g] = f.walk + x;
            tb[g] = f.table;
        }
        uint32_t key[kBatch];
#pragma unroll
        for (int g = 0; g < kBatch; ++g) {
            key[g] = 0;
            if (live[g]) {
                key[g] = static_cast<uint32_t>(((pm[g] & kWalkB) ? csc_row : ca)[wb[g]]);
            }
        }
        // The filter first: one byte of a home slot's keys, a sixteenth of the table's
        // footprint, tells most misses.
        uint32_t hash[kBatch], bits[kBatch];
#pragma unroll
        for (int g = 0; g < kBatch; ++g) {
            hash[g] = mix(key[g]);
            bits[g] = live[g] ? filter[tb[g] + (hash[g] & (pm[g] & ~kWalkB))] : 0u;
        }
        bool maybe[kBatch];
        uint64_t w[kBatch];
        float cv[kBatch], own[kBatch];  // the mask's and the walked entry's values
#pragma unroll
        for (int g = 0; g < kBatch; ++g) {
            maybe[g] = ((bits[g] >> filter_bit(hash[g])) & 1u) != 0;
            w[g] = kEmptySlot;
            cv[g] = own[g] = 0.0f;
            if (maybe[g]) {
                w[g] = tab[tb[g] + (hash[g] & (pm[g] & ~kWalkB))];
                own[g] = ((pm[g] & kWalkB) ? csc_val : va)[wb[g]];
                cv[g] = vc[e_lo + ent[g]];
            }
        }
#pragma unroll
        for (int g = 0; g < kBatch; ++g) {
            double v = 0.0;
            bool found = false;
            if (maybe[g]) {
                const uint32_t mask = pm[g] & ~kWalkB;
                uint64_t ww = w[g];
                uint32_t hh = hash[g] & mask;
                // collisions: the next two slots per step, both loads issued together (a
                // wavefront waits for its longest chain; the second slot is nearly always in
                // the same line); the first of them that holds the key or is empty ends it
                while (static_cast<uint32_t>(ww) != key[g] &&
                       static_cast<uint32_t>(ww) != kEmptyKey) {
                    const uint32_t h1 = (hh + 1) & mask, h2 = (hh + 2) & mask;
                    const uint64_t w1 = tab[tb[g] + h1], w2 = tab[tb[g] + h2];
                    const bool first = static_cast<uint32_t>(w1) == key[g] ||
                                       static_cast<uint32_t>(w1) == kEmptyKey;
                    ww = first ? w1 : w2;
                    hh = first ? h1 : h2;
                }
                found = static_cast<uint32_t>(ww) == key[g];
                const float other = __uint_as_float(static_cast<uint32_t>(ww >> 32));
                // a * b with a from A and b from B, as the reference writes it
                const float ab = (pm[g] & kWalkB) ? other * own[g] : own[g] * other;
                v = static_cast<double>(ab * cv[g]);
            }
            if (local) {  // uniform
                if (found) {
                    atomicAdd(&s_acc[ent[g]], v);
                    s_hit[ent[g]] = 1;
                }
                continue;
            }
            const unsigned long long hits = __ballot(found);
            if (hits == 0) continue;  // uniform in the wavefront
            // the lanes of one entry are neighbours: its sum forms in its first lane's slot
            const int prev = __shfl_up(ent[g], 1, dev::kWave);  // (every lane takes part)
            const unsigned long long first = __ballot(l == 0 || ent[g] != prev);
            const unsigned long long upto = first & (~0ull >> (63 - l));
            const int lead = 63 - __clzll(static_cast<long long>(upto));
            double *sum = s_acc + (threadIdx.x - l);  // the wavefront's slots
            sum[l] = 0.0;
            dev::wave_sync();
            if (found) atomicAdd(&sum[lead], v);
            dev::wave_sync();
            const unsigned long long after = first & ~(2ull * (1ull << l) - 1ull);
            const unsigned long long mine =
                (after ? (after & -after) - 1ull : ~0ull) & ~((1ull << l) - 1ull);
            if (lead == l && (hits & mine) != 0) {
                atomicAdd(&acc[e_lo + ent[g]], sum[l]);
                hit[e_lo + ent[g]] = 1;
            }
            dev::wave_sync();
        }
    }
    if (local) {
        __syncthreads();
        for (int x = threadIdx.x; x < entries; x += kBlock) {
            if (s_hit[x]) {
                atomicAdd(&acc[e_lo + x], s_acc[x]);
                hit[e_lo + x] = 1;
            }
        }
    }
}

__global__ void keep_kernel(const int *__restrict__ hit, int64_t n, int64_t *__restrict__ keep) {
    for (int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; e < n;
         e += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        keep[e] = hit[e] ? 1 : 0;
    }
}

// Z.pos[r] = kept entries of C before row r; kept entries copied in C's order.
__global__ void output_kernel(const int *__restrict__ pc, int rows, const int *__restrict__ cc,
                              int64_t nnz_c, const int64_t *__restrict__ koff,
                              const int *__restrict__ hit, const double *__restrict__ acc,
                              int *__restrict__ pz, int *__restrict__ cz, float *__restrict__ vz) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    const int64_t first = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    for (int64_t r = first; r <= rows; r += stride) pz[r] = static_cast<int>(koff[pc[r]]);
    for (int64_t e = first; e < nnz_c; e += stride) {
        if (hit[e]) {
            const int64_t o = koff[e];
            cz[o] = cc[e];
            vz[o] = static_cast<float>(acc[e]);
        }
    }
}

__global__ void zero_pos_kernel(int *__restrict__ p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i <= n; i += gridDim.x * blockDim.x) p[i] = 0;
}

unsigned grid_for(int64_t n) {
    const int64_t g = (n + kBlock - 1) / kBlock;
    return static_cast<unsigned>(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}

bool bad_csr(const nacho_csr *t) {
    if (!t || t->dim_i_size < 0 || t->dim_j_size < 0 || t->dim_j_length < 0) return true;
    if (!t->dim_j_offsets) return true;
    if (t->dim_j_length > 0 && (!t->dim_j_indices || !t->values)) return true;
    return false;
}

int multiply(const nacho_csr *a, const nacho_csr *b, const nacho_csr *c, nacho_csr *z,
             int32_t num_blocks, int32_t threads_per_block, void *stream,
             const nacho_allocator *alloc) {
    if (!z) return NACHO_ERR_INVALID_ARGUMENT;
    *z = nacho_csr{};
    NACHO_TRY(check_launch_hints(num_blocks, threads_per_block));
    if (bad_csr(a) || bad_csr(b) || bad_csr(c)) return NACHO_ERR_INVALID_ARGUMENT;
    if (a->dim_j_size != b->dim_i_size || c->dim_i_size != a->dim_i_size ||
        c->dim_j_size != b->dim_j_size) {
        return NACHO_ERR_INVALID_ARGUMENT;
    }
    const int rows = a->dim_i_size, inner = b->dim_i_size, cols = b->dim_j_size;
    const int64_t nnz_a = a->dim_j_length, nnz_b = b->dim_j_length, nnz_c = c->dim_j_length;
    Call call(stream, alloc);
    const hipStream_t st = call.stream();
    const char *name = "sssmm: tables+probe+output";
    int *pz = nullptr;
    NACHO_TRY(call.result_n(static_cast<size_t>(rows) + 1, &pz));
    NACHO_TRY(call.timer_start(name));
    if (nnz_a == 0 || nnz_b == 0 || nnz_c == 0) {
        zero_pos_kernel<<<grid_for(static_cast<int64_t>(rows) + 1), kBlock, 0, st>>>(pz, rows);
        NACHO_TRY_HIP(hipGetLastError());
        NACHO_TRY(call.timer_stop());
        NACHO_TRY(call.collect_timer());
        z->dim_i_size = rows;
        z->dim_j_size = cols;
        z->dim_j_offsets = pz;
        call.commit();
        return NACHO_OK;
    }

    // columns of B and the table sizes
    int64_t *col_count = nullptr, *col_off = nullptr, *col_fill = nullptr;
    int64_t *tsize_b = nullptr, *toff_b = nullptr, *tsize_a = nullptr, *toff_a = nullptr;
    NACHO_TRY(call.scratch_n(2 * (static_cast<size_t>(cols) + 1), &col_count));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(cols) + 1, &col_off));
    col_fill = col_count + cols + 1;
    NACHO_TRY(call.scratch_n(static_cast<size_t>(cols) + 1, &tsize_b));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(cols) + 1, &toff_b));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &tsize_a));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(rows) + 1, &toff_a));
    fill_kernel<<<grid_for(2 * (static_cast<int64_t>(cols) + 1)), kBlock, 0, st>>>(
        reinterpret_cast<uint64_t *>(col_count), 2 * (static_cast<int64_t>(cols) + 1), 0ull);
    const unsigned span_grid =
        static_cast<unsigned>(std::max<int64_t>(1, (nnz_b + kSpan - 1) / kSpan));
    count_cols_kernel<<<span_grid, kBlock, 0, st>>>(
        b->dim_j_indices, nnz_b, cols, reinterpret_cast<unsigned long long *>(col_count));
    NACHO_TRY_HIP(hipGetLastError());
    table_sizes_kernel<<<grid_for(std::max(cols, rows)), kBlock, 0, st>>>(
        col_count, cols, tsize_b, a->dim_j_offsets, rows, tsize_a);
    NACHO_TRY_HIP(hipGetLastError());
    int64_t *word[2] = {nullptr, nullptr};
    NACHO_TRY(call.value_word(0, &word[0]));
    NACHO_TRY(call.value_word(1, &word[1]));
    const scan::Job size_jobs[3] = {{tsize_b, cols, toff_b, word[0]},
                                    {tsize_a, rows, toff_a, word[1]},
                                    {col_count, cols, col_off}};
    NACHO_TRY(scan::exclusive_scans(call, size_jobs, 3));
    NACHO_TRY(call.timer_stop());
    int64_t sizes[2] = {0, 0};
    NACHO_TRY(call.value(0, &sizes[0]));
    NACHO_TRY(call.value(1, &sizes[1]));
    NACHO_TRY(call.collect_timer());
    // A table's mask is kept in 31 bits (bit 31 flags the walked side), so no table may
    // exceed 2^31 slots.  Table sizes are powers of two, so a larger one (2^32 slots or
    // more, for a row or column of more than 2^30 entries) would make its side's total at
    // least 2^32.
    if (sizes[0] >= (int64_t{1} << 32) || sizes[1] >= (int64_t{1} << 32)) {
        return NACHO_ERR_INDEX_OVERFLOW;
    }
    NACHO_TRY(call.timer_start(name));

    // tables and B's columns
    // (one array: B's tables, then A's from slot sizes[0] on; one filter byte per slot)
    uint64_t *tab = nullptr;
    unsigned *filter = nullptr;
    int *csc_row = nullptr;
    float *csc_val = nullptr;
    const int64_t slots = sizes[0] + sizes[1];
    const int64_t filter_words = (slots + 7) / 8;  // 64-bit
    NACHO_TRY(call.scratch_n(static_cast<size_t>(slots), &tab));
    NACHO_TRY(call.scratch_n(2 * static_cast<size_t>(filter_words), &filter));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_b), &csc_row));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_b), &csc_val));
    fill_kernel<<<grid_for(slots), kBlock, 0, st>>>(tab, slots, kEmptySlot);
    fill_kernel<<<grid_for(filter_words), kBlock, 0, st>>>(reinterpret_cast<uint64_t *>(filter),
                                                           filter_words, 0ull);
    const int span_b = table_span(nnz_b), span_a = table_span(nnz_a);
    transpose_kernel<<<static_cast<unsigned>((nnz_b + span_b - 1) / span_b), kBlock, 0, st>>>(
        b->dim_j_offsets, inner, b->dim_j_indices, b->values, nnz_b, span_b, col_off,
        reinterpret_cast<unsigned long long *>(col_fill), toff_b, csc_row, csc_val, tab, filter);
    rows_table_kernel<<<static_cast<unsigned>((nnz_a + span_a - 1) / span_a), kBlock, 0, st>>>(
        a->dim_j_offsets, rows, a->dim_j_indices, a->values, nnz_a, span_a, toff_a, tab, filter,
        sizes[0]);
    NACHO_TRY_HIP(hipGetLastError());

    // probes per mask entry
    int64_t *work = nullptr, *woff = nullptr, *walk_base = nullptr, *probe_base = nullptr;
    uint32_t *probe_mask = nullptr;
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_c) + 1, &work));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_c) + 1, &woff));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_c), &walk_base));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_c), &probe_base));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_c), &probe_mask));
    work_kernel<<<grid_for(nnz_c), kBlock, 0, st>>>(
        c->dim_j_offsets, rows, c->dim_j_indices, nnz_c, a->dim_j_offsets,
        reinterpret_cast<const unsigned long long *>(col_count), col_off, toff_a, sizes[0], toff_b, work,
        walk_base, probe_base, probe_mask);
    NACHO_TRY_HIP(hipGetLastError());
    NACHO_TRY(call.value_word(0, &word[0]));
    NACHO_TRY(scan::exclusive_scan_i64(call, work, nnz_c, woff, word[0]));
    // (queued ahead of the wait for the probes' number)
    double *acc = nullptr;
    int *hit = nullptr;
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_c), &acc));
    NACHO_TRY(call.scratch_n(static_cast<size_t>(nnz_c), &hit));
    zero_sums_kernel<<<grid_for(nnz_c), kBlock, 0, st>>>(acc, hit, nnz_c);
    NACHO_TRY_HIP(hipGetLastError());
    NACHO_TRY(call.timer_stop());
    int64_t total = 0;
    NACHO_TRY(call.value(0, &total));
    NACHO_TRY(call.collect_timer());
    NACHO_TRY(call.timer_start(name));
    const int64_t chunks = (total + kChunk - 1) / kChunk;
    if (chunks > INT_MAX) return NACHO_ERR_INDEX_OVERFLOW;

    // probes
    if (chunks > 0) {
        int64_t *bounds = nullptr;
        NACHO_TRY(call.scratch_n(2 * static_cast<size_t>(chunks), &bounds));
        chunk_bounds_kernel<<<grid_for(2 * chunks), kBlock, 0, st>>>(woff, nnz_c, total, chunks,
                                                                     bounds);
        probe_kernel<<<static_cast<unsigned>(chunks), kBlock, 0, st>>>(
            woff, bounds, total, walk_base, probe_base, probe_mask, a->dim_j_indices, a->values,
            csc_row, csc_val, tab, reinterpret_cast<const unsigned char *>(filter), c->values, acc,
            hit);
        NACHO_TRY_HIP(hipGetLastError());
    }

    // result
    int64_t *keep = work, *koff = woff;  // the work counts are spent
    keep_kernel<<<grid_for(nnz_c), kBlock, 0, st>>>(hit, nnz_c, keep);
    NACHO_TRY_HIP(hipGetLastError());
    NACHO_TRY(call.value_word(0, &word[0]));
    NACHO_TRY(scan::exclusive_scan_i64(call, keep, nnz_c, koff, word[0]));
    NACHO_TRY(call.timer_stop());
    int64_t nnz = 0;
    NACHO_TRY(call.value(0, &nnz));
    NACHO_TRY(call.collect_timer());
    NACHO_TRY(call.timer_start(name));
    int *cz = nullptr;
    float *vz = nullptr;
    NACHO_TRY(call.result_n(static_cast<size_t>(nnz), &cz));
    NACHO_TRY(call.result_n(static_cast<size_t>(nnz), &vz));
    output_kernel<<<grid_for(nnz_c > rows ? nnz_c : static_cast<int64_t>(rows) + 1), kBlock, 0,
                    st>>>(c->dim_j_offsets, rows, c->dim_j_indices, nnz_c, koff, hit, acc, pz,
                          cz, vz);
    NACHO_TRY_HIP(hipGetLastError());
    NACHO_TRY(call.timer_stop());
    NACHO_TRY(call.collect_timer());
    z->dim_i_size = rows;
    z->dim_j_size = cols;
    z->dim_j_offsets = pz;
    z->dim_j_length = static_cast<int32_t>(nnz);
    z->dim_j_indices = cz;
    z->values = vz;
    z->nnz = static_cast<int32_t>(nnz);
    call.commit();
    return NACHO_OK;
}

}  // namespace sssmm
}  // namespace nacho

extern "C" int nacho_gpu_sssmm_f32(const nacho_csr *a, const nacho_csr *b, const nacho_csr *c,
                                   nacho_csr *z, int32_t num_blocks, int32_t threads_per_block,
                                   void *stream, const nacho_allocator *alloc) {
    return nacho::sssmm::multiply(a, b, c, z, num_blocks, threads_per_block, stream, alloc);
}
