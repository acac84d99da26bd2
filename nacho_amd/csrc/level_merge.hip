// The level merge for gfx950: union or intersection of two compressed levels, row by row.
// CSR / COO / DCSR add and multiply, CSF3 add (three chained levels) and the inner products
// all run on it.
//
// Reference path replaced: the generated partition_ij / precompute_ij / compute_ij kernels
// (src/backend/partition.cpp:59-336, 813-993; src/backend/compute.cpp:151-395, 619-1388) and
// their host orchestration (src/backend/stitch_and_generate.cpp:8-112, 438-527;
// stitch_and_generate_gpu.cpp:379-715).  The reference runs one thread per merge-path
// partition with a serial, uncoalesced merge, a count pass, a CUB scan, a blocking length
// readback and a write pass that merges again.  Here the merge is done once and its outcome,
// two bits per entry, is what the write pass reads:
//
//  * csr_partition_kernel cuts the merged sequence (every row's A entries, B entries and one
//    row end) into tiles; no equal A/B pair is split across tiles.
//  * order_kernel merges one tile per workgroup in registers and LDS (a bitonic merging
//    network, no data-dependent control flow) and stores the tile's merge order: for each
//    slot of the merged entries, whether it is a B entry, and whether it is the second of an
//    equal A/B pair.  It also counts the pairs, which gives the result length.
//  * emit_kernel streams the result: a slot's operand index is a population count over the
//    order bits before it, so consecutive lanes read consecutive entries straight from the
//    operands and store consecutive outputs, with no merge, no staging and no barrier.
//
// Measured on MI355X per call, against two merge walks per level (count, then write) that
// this replaces: csr_add of 950K x 1M, 7.8M entries each, evenly spread, 142 -> 106 us; C2
// (2^20 rows, Zipf, 16.7M each) 161 -> 146; csr_mul C3 148 -> 133; csf_add C5 496 -> 416;
// coo3d_add C5 464 -> 420; inner_prod C5 241 -> 228; 200 x 180 with 1800 entries 33.6 -> 29.2.
//
// Emission order and values follow the reference's lattice (compute.cpp:476-491,
// 1169-1198, 1297-1337): coordinates ascending within a row; union emits a+b where both
// exist and a copy otherwise; intersection emits a*b only where both exist.  Explicit zeros
// are kept.  Each value is one IEEE binary32 operation, so results are bit-identical to the
// reference's.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>

#include "csr_merge.hpp"
#include "csr_partition.hpp"
#include "device_utils.hpp"
#include "runtime.hpp"

namespace nacho {
namespace csr {

namespace {

enum class Op { Union, Intersect };

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / dev::kWave;
constexpr int kPer = 16;                // slots per lane of the merging network
constexpr int kSlots = kBlock * kPer;   // merged entries of a tile, padded
// Items per tile: with the entry that the pair rule may add, a wavefront's width of padding
// stays between a tile's A and B slots.
constexpr int kTile = kSlots - dev::kWave - 1;
constexpr int kWords = kSlots / 64;     // 64-slot order words per tile
static_assert(kLevelItemSlack >= kTile, "an item count rounded up to tiles fits 32 bits");
static_assert(kWords == dev::kWave, "one order word per lane");
// Tiles per pair total: a wavefront of the emit kernel sums the chunks before its tile's and
// the tiles before it in its own chunk (at most 2^31 / kTile / kChunk + kChunk loads).
constexpr int kChunk = 256;
// Levels of at most this many tiles take one launch (fused_kernel): one per CU.  Per call, one
// launch against three: 4 tiles 28.7 / 30.6 us, 42 tiles 29.0 / 34.0, 253 tiles 30.8 / 35.3, but
// 421 tiles 34.9 / 34.0 (csr_add, 8 entries per row and operand).
constexpr int kFusedTiles = 256;
// 32-bit words between the totals: atomics are serialised per cache line.
constexpr int kChunkStride = 32;

// Set bits of m below this lane.
__device__ __forceinline__ int bits_below(unsigned long long m) {
    return static_cast<int>(__builtin_amdgcn_mbcnt_hi(
        static_cast<unsigned>(m >> 32),
        __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m), 0u)));
}

// ---- sparse tiles ----------------------------------------------------------------------
//
// Rows where one operand is empty need no merging, and in a row that holds few entries of
// one operand it is cheaper to search those in the other's.  Power-law operands are mostly
// such rows (C2: 0.24M searches for 33M entries), so where rows are long on average the
// partition kernel is replaced by this one, which also writes the order of every tile whose
// rows hold at most kMaxSearches entries on their smaller sides; the order kernel then
// merges the other tiles only.
//
// A tile's B slots are written as toggles: a run of B entries flips the bit where it starts
// and the bit after its end, and a prefix XOR over the tile's bits gives the side of every
// slot.  One wavefront per tile, four tiles per workgroup: the searches are chains of
// dependent loads, so what counts is how many tiles are in flight.  C2: 24 us with the split,
// and 11 us for the order kernel on the tiles left (2%), against 8.5 us for the split and 65
// for ordering every tile.  Where rows hold few entries (or, in tensors, thousands of both
// operands) most tiles are dense and the look is lost.
constexpr int kMaxSearches = 256;  // entries to search
constexpr int kMaxSearchRows = 512;
constexpr int kSearchWays = 8;     // of a lower bound: probes per round + 1
// Entries of both operands per row from which a union looks for sparse tiles.  How even the rows
// are, which decides what the look brings, is not known here.  csr_add of 700,000 rows, looking /
// not: Zipf rows of 5, 6, 8, 10, 16, 32 entries per operand 48.3 / 48.4, 53.5 / 54.5, 59.1 /
// 64.1, 67.7 / 78.2, 103.5 / 117.3, 183.5 / 216.1 us, even rows 51.8 / 47.2, 58.4 / 53.3, 69.2 /
// 62.3, 83.1 / 80.3, 134.7 / 129.3, 240.6 / 231.1.
constexpr int kSparseEntriesPerRow = 8;
constexpr unsigned kDense = UINT_MAX;  // tile_pairs of a tile left to the order kernel

// A row's entries in its tile: A's [a, a + la), B's [b, b + lb).
struct TileRow {
    int a, la, b, lb;
};

struct SparseLds {
    unsigned toggle[kSlots / 32];
    unsigned dup[kSlots / 32];
    uint2 first_of[kMaxSearches];  // the row whose searches start here: {a | la << 16, b | lb << 16}
};

// Lower bound of x in v[p, q): kSearchWays - 1 independent probes per round.
__device__ __forceinline__ int lower_bound(const int *__restrict__ v, int p, int q, int x) {
    while (p < q) {
        const int step = (q - p + kSearchWays - 1) / kSearchWays;
        int below = 0;  // probes p + j * step - 1 inside the range that hold less than x
#pragma unroll
        for (int j = 1; j < kSearchWays; ++j) {
            const int at = p + j * step - 1;
            const int c = v[min(at, q - 1)];
            below += (at < q && c < x) ? 1 : 0;
        }
        const int np = p + below * step;
        q = below == kSearchWays - 1 ? q : min(np + step - 1, q);
        p = np;
    }
    return p;
}

// Boundaries [4 b, 4 b + 4] by 16 lanes each, then tile 4 b + w by wavefront w.
__global__ __launch_bounds__(kBlock) void split_sparse_kernel(
    const int *__restrict__ pa, const int *__restrict__ ca, const int *__restrict__ pb,
    const int *__restrict__ cb, int rows, int total, int num_tiles, int *__restrict__ split_r,
    int *__restrict__ split_a, int *__restrict__ split_b,
    unsigned long long *__restrict__ side_out, unsigned long long *__restrict__ dup_out,
    unsigned *__restrict__ state, unsigned *__restrict__ tile_pairs,
    unsigned long long *__restrict__ done, unsigned *__restrict__ zero_counts, int n_counts) {
    constexpr int kGroup = 16;
    __shared__ int s_split[3 * (kWaves + 1)];
    __shared__ SparseLds s_tiles[kWaves];
    const int tid = threadIdx.x;
    const int l = tid % dev::kWave;
    const int w = __builtin_amdgcn_readfirstlane(tid / dev::kWave);
    const int t0 = blockIdx.x * kWaves;
    SparseLds &sh = s_tiles[w];
    for (int i = l; i < kSlots / 32; i += dev::kWave) sh.toggle[i] = sh.dup[i] = 0u;
    for (int i = l; i < kMaxSearches; i += dev::kWave) sh.first_of[i] = uint2{0, 0};
    {
        const int g = tid / kGroup, t = t0 + g;
        const bool lead = tid % kGroup == 0;
        if (blockIdx.x == 0 && tid == kBlock - 1) dev::zero_total(done);
        for (int i = blockIdx.x * kBlock + tid; i < n_counts; i += gridDim.x * kBlock) {
            zero_counts[i * kChunkStride] = 0u;
        }
        if (g <= kWaves && t <= num_tiles) {
            const long long d64 = static_cast<long long>(t) * kTile;
            int r, a, b;
            find_split<kGroup>(pa, ca, pb, cb, rows,
                               d64 > total ? total : static_cast<int>(d64), r, a, b);
            if (lead) {
                s_split[3 * g] = r;
                s_split[3 * g + 1] = a;
                s_split[3 * g + 2] = b;
                if (g < kWaves || t == num_tiles) {
                    split_r[t] = r;
                    split_a[t] = a;
                    split_b[t] = b;
                }
            }
        }
    }
    __syncthreads();
    const int t = t0 + w;
    if (t >= num_tiles) return;  // (no barrier follows)
    auto u = [&](int i) { return __builtin_amdgcn_readfirstlane(s_split[3 * w + i]); };
    const TileSplit sp{u(0), u(1), u(2), u(3), u(4), u(5)};
    const int na = sp.a1 - sp.a0, nb = sp.b1 - sp.b0, nr = sp.r1 - sp.r0 + 1;
    if (nr > kMaxSearchRows) {
        if (l == 0) state[t] = kDense;
        return;
    }
    // The tile's rows, one per lane and round; every load is issued before the first is used.
    constexpr int kRounds = kMaxSearchRows / dev::kWave;
    int a0[kRounds], a1[kRounds], b0[kRounds], b1[kRounds];
#pragma unroll
    for (int j = 0; j < kRounds; ++j) {
        if (j * dev::kWave >= nr) break;  // uniform
        const int r = sp.r0 + min(j * dev::kWave + l, nr - 1);
        const int next = min(r + 1, rows);
        a0[j] = pa[r];
        a1[j] = pa[next];
        b0[j] = pb[r];
        b1[j] = pb[next];
    }
    auto row = [&](int j) {  // (empty past the tile's last row)
        TileRow x{0, 0, 0, 0};
        const int k = j * dev::kWave + l;
        if (k < nr) {
            x.a = max(a0[j] - sp.a0, 0);
            x.b = max(b0[j] - sp.b0, 0);
            x.la = min(a1[j] - sp.a0, na) - x.a;
            x.lb = min(b1[j] - sp.b0, nb) - x.b;
        }
        return x;
    };
    auto toggle = [&](int s) { atomicXor(&sh.toggle[s >> 5], 1u << (s & 31)); };
    auto searches = [](const TileRow &x) { return x.la > 0 && x.lb > 0 ? min(x.la, x.lb) : 0; };
    int work = 0;
#pragma unroll
    for (int j = 0; j < kRounds; ++j) {
        if (j * dev::kWave >= nr) break;
        work += searches(row(j));
    }
    const int incl = dev::wave_inclusive_sum_dpp(work);
    const int all = __builtin_amdgcn_readlane(incl, dev::kWave - 1);
    if (all > kMaxSearches) {
        if (l == 0) state[t] = kDense;
        return;
    }
    // Whole rows: the B entries of a row with fewer A entries (or none) are one run, cut
    // below by its A entries; a row with fewer B entries starts as all A.
    int at = incl - work;
#pragma unroll
    for (int j = 0; j < kRounds; ++j) {
        if (j * dev::kWave >= nr) break;
        const TileRow x = row(j);
        const int m = searches(x);
        if (x.lb > 0 && x.la <= x.lb) {
            toggle(x.a + x.b);
            toggle(x.a + x.b + x.la + x.lb);
        }
        if (m > 0) {
            sh.first_of[at] = uint2{static_cast<unsigned>(x.a | (x.la << 16)),
                                    static_cast<unsigned>(x.b | (x.lb << 16))};
        }
        at += m;
    }
    dev::wave_sync();
    uint2 carry{0, 0};  // the row in effect before the round
    int carry_at = 0;   // and its first search
    for (int i0 = 0; i0 < all; i0 += dev::kWave) {  // uniform
        const int i = i0 + l;
        const uint2 f = sh.first_of[min(i, kMaxSearches - 1)];
        const unsigned long long starts = __ballot(i < all && f.x != 0);
        const unsigned long long upto = starts & (~0ull >> (63 - l));
        const int from = upto ? 63 - __clzll(static_cast<long long>(upto)) : 0;
        const unsigned fx = __shfl(f.x, from, dev::kWave), fy = __shfl(f.y, from, dev::kWave);
        const uint2 rec = upto ? uint2{fx, fy} : carry;
        const int nth = i - (upto ? i0 + from : carry_at);
        if (starts) {  // uniform
            const int top = 63 - __clzll(static_cast<long long>(starts));
            carry.x = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(f.x), top));
            carry.y = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(f.y), top));
            carry_at = i0 + top;
        }
        if (i < all) {
            const TileRow x{static_cast<int>(rec.x & 0xffffu), static_cast<int>(rec.x >> 16),
                            static_cast<int>(rec.y & 0xffffu), static_cast<int>(rec.y >> 16)};
            const bool a_small = x.la <= x.lb;
            const int own = a_small ? sp.a0 + x.a + nth : sp.b0 + x.b + nth;
            const int c = (a_small ? ca : cb)[own];
            const int *__restrict__ large = a_small ? cb : ca;
            const int p = a_small ? sp.b0 + x.b : sp.a0 + x.a;
            const int q = p + (a_small ? x.lb : x.la);
            const int lb = lower_bound(large, p, q, c);
            const bool pair = lb < q && large[lb] == c;
            // (a pair's A entry comes first)
            const int s = x.a + x.b + nth + (lb - p) + (pair && !a_small ? 1 : 0);
            toggle(s);
            toggle(s + 1);
            if (pair) {
                const int d = a_small ? s + 1 : s;  // its B slot
                atomicOr(&sh.dup[d >> 5], 1u << (d & 31));
            }
        }
    }
    dev::wave_sync();
    unsigned long long bits = (static_cast<unsigned long long>(sh.toggle[2 * l + 1]) << 32) |
                              sh.toggle[2 * l];
    const unsigned long long dup = (static_cast<unsigned long long>(sh.dup[2 * l + 1]) << 32) |
                                   sh.dup[2 * l];
    const unsigned long long odd = __ballot((__popcll(bits) & 1) != 0);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) bits ^= bits << d;
    if (bits_below(odd) & 1) bits = ~bits;  // (the toggles are even in number: 0 past the end)
    side_out[static_cast<size_t>(t) * kWords + l] = bits;
    dup_out[static_cast<size_t>(t) * kWords + l] = dup;
    // Two searches of an unsorted row may land on one slot and their toggles cancel; a tile whose
    // B slots are not nb, or whose pairs end on another slot, is left to the order kernel.
    const bool stray = __any((dup & ~bits) != 0);
    const unsigned sums = static_cast<unsigned>(dev::wave_inclusive_sum_dpp(
        __popcll(bits) << 16 | __popcll(dup)));  // (at most kSlots each)
    if (l == dev::kWave - 1) {
        const bool whole = !stray && sums >> 16 == static_cast<unsigned>(nb);
        tile_pairs[t] = state[t] = whole ? sums & 0xffffu : kDense;
    }
}

// ---- order kernel ----------------------------------------------------------------------
//
// A tile's entries become keys (row in tile, coordinate, side), side 0 for A and 1 for B, so
// that an equal pair sorts A first.  A's keys ascending, then padding, then B's reversed are a
// bitonic sequence of kSlots keys, which log2(kSlots) = 12 compare-exchange stages sort:
// strides 2048 .. 256 between a lane's own registers (slot lane + 256 j), 128 .. 16 after one
// transposition through LDS, 8 .. 1 after a second one inside each wavefront.  Every lane
// does the same 12 minima and maxima per key, all independent within a stage, where a merge
// walk is a serial chain of LDS reads per lane with its wavefront's lanes on both branches.
//
// Keys are 32-bit where row, coordinate and side fit (decided per tile, for coordinates of the
// declared extent), else binary64 numbers whose order is that of the key.  A tile with a
// coordinate that its keys do not hold (past the extent, or negative) is walked afterwards
// instead (walk_tile), so coordinates are ordered as the int32 numbers they are.  (Key widths
// chosen by each tile's largest coordinate made the keys wait for one more reduction: 1 to 2%
// per call; one kernel for both widths took 47 us more at C5's k level, where the 32-bit one's
// 7 wavefronts per SIMD are worth it.)
//
// Bound by LDS and VALU issue together (about 60% and 55% busy at C3: 560 VALU and 73 LDS
// instructions per lane and tile): 61 us for C3's 33M entries, 96 us for the 40M of the C5 k
// level, 7.3 ns per tile in either key width and at 4 or 7 resident workgroups per CU.
//
// Rows: each row marks its first A slot (and, in B's reversed order, the slot of its last B
// entry), and a running maximum over the slots gives every entry its row and side: a mark is
// the tile row k for A, ~k for B, and kPadMark for the padding between them.
//
// Whatever coordinates a tile's rows hold, its order (here and in split_sparse_kernel) has
// exactly nb B slots among its n, so the emit kernel's indices stay inside the tile's ranges of
// the operands.  (The ranges themselves come from searches that take rows for sorted.)

// LDS word of slot p's key: the wavefront's lanes fall on distinct banks in all three layouts,
// and a lane's 16 consecutive slots stay 16-byte aligned.
constexpr int kLdsWords = kSlots + kSlots / 4 + kSlots / 16;
__device__ __forceinline__ int lds_word(int p) { return p + ((p >> 4) << 2) + ((p >> 8) << 4); }
// LDS half word of slot p's mark: 48 bytes per 16 slots, so that 16-byte reads of consecutive
// lanes' slots fall on distinct banks.
constexpr int kMarkHalves = kSlots / 16 * 24;
__device__ __forceinline__ int mark_half(int p) { return (p >> 4) * 24 + (p & 15); }
// Padding's mark: above every A mark, below every B mark; its row has every bit set that a
// key holds, which no row of the tile has.
constexpr unsigned kPadMark = 0xe000u;
typedef unsigned short half2_t __attribute__((ext_vector_type(2)));

struct OrderLds {
    union {
        unsigned word[kLdsWords];
        unsigned short mark[kMarkHalves];
    };
    unsigned wave_max[kWaves];
    unsigned first[2 * kWaves], last[2 * kWaves];
    unsigned pairs[kWaves];
    unsigned sides[kWaves];
};

// One 32-bit word of every key through LDS, from slots tid + 256 j to slots
// (tid / 16) * 256 + 16 r + tid % 16: get(j) is the word of register j, set(r, word) replaces
// it.  No barrier after the reads.
template <typename Get, typename Set>
__device__ __forceinline__ void transpose_block(unsigned *s, int tid, Get get, Set set) {
    const int w = lds_word(tid);
    const int r0 = lds_word((tid >> 4) << 8) + (tid & 15);
#pragma unroll
    for (int j = 0; j < kPer; ++j) s[w + 336 * j] = get(j);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPer; ++r) set(r, s[r0 + 20 * r]);
}

// The same from slots (tid / 16) * 256 + 16 r + tid % 16 to slots 16 tid + r: each wavefront
// reads and writes only its own 1024 slots.
template <typename Get, typename Set>
__device__ __forceinline__ void transpose_wave(unsigned *s, int tid, Get get, Set set) {
    const int r0 = lds_word((tid >> 4) << 8) + (tid & 15);
    const int c0 = lds_word(kPer * tid);
#pragma unroll
    for (int r = 0; r < kPer; ++r) s[r0 + 20 * r] = get(r);
    dev::wave_sync();
#pragma unroll
    for (int q = 0; q < kPer / 4; ++q) {
        const uint4 x = *reinterpret_cast<const uint4 *>(s + c0 + 4 * q);
        set(4 * q, x.x);
        set(4 * q + 1, x.y);
        set(4 * q + 2, x.z);
        set(4 * q + 3, x.w);
    }
    dev::wave_sync();
}

// Keys from a row (before the coordinate's bits) and the low word (crd << 1 | side).
struct NarrowKey {
    using T = unsigned;
    static __device__ __forceinline__ T make(unsigned row, unsigned low, int bits) {
        return (row << (bits + 1)) | low;
    }
    static __device__ __forceinline__ T lower(T a, T b) { return min(a, b); }
    static __device__ __forceinline__ T upper(T a, T b) { return max(a, b); }
    static __device__ __forceinline__ unsigned low(T k) { return k; }
    static __device__ __forceinline__ unsigned high(T) { return 0u; }
    static __device__ __forceinline__ void to_mid(T (&k)[kPer], unsigned *s, int tid) {
        transpose_block(s, tid, [&](int r) { return k[r]; }, [&](int r, T v) { k[r] = v; });
    }
    static __device__ __forceinline__ void to_runs(T (&k)[kPer], unsigned *s, int tid) {
        transpose_wave(s, tid, [&](int r) { return k[r]; }, [&](int r, T v) { k[r] = v; });
    }
};

// The row beside kHigh is the high word: finite binary64 numbers, ordered as the keys.
struct WideKey {
    using T = double;
    static constexpr unsigned kHigh = 0x40000000u;
    static __device__ __forceinline__ T make(unsigned row, unsigned low, int) {
        return __hiloint2double(static_cast<int>(kHigh | row), static_cast<int>(low));
    }
    // (the instructions themselves: the keys are no NaN, so nothing needs canonicalising)
    static __device__ __forceinline__ T lower(T a, T b) {
        T r;
        asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
        return r;
    }
    static __device__ __forceinline__ T upper(T a, T b) {
        T r;
        asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
        return r;
    }
    static __device__ __forceinline__ unsigned low(T k) {
        return static_cast<unsigned>(__double2loint(k));
    }
    static __device__ __forceinline__ unsigned high(T k) {
        return static_cast<unsigned>(__double2hiint(k));
    }
    static __device__ __forceinline__ T join(unsigned hi, unsigned lo) {
        return __hiloint2double(static_cast<int>(hi), static_cast<int>(lo));
    }
    // (one half at a time: a register holds halves of two keys in between)
    static __device__ __forceinline__ void to_mid(T (&k)[kPer], unsigned *s, int tid) {
        transpose_block(s, tid, [&](int r) { return low(k[r]); },
                        [&](int r, unsigned v) { k[r] = join(high(k[r]), v); });
        __syncthreads();
        transpose_block(s, tid, [&](int r) { return high(k[r]); },
                        [&](int r, unsigned v) { k[r] = join(v, low(k[r])); });
    }
    static __device__ __forceinline__ void to_runs(T (&k)[kPer], unsigned *s, int tid) {
        transpose_wave(s, tid, [&](int r) { return low(k[r]); },
                       [&](int r, unsigned v) { k[r] = join(high(k[r]), v); });
        transpose_wave(s, tid, [&](int r) { return high(k[r]); },
                       [&](int r, unsigned v) { k[r] = join(v, low(k[r])); });
    }
};

// Four compare-exchange stages between a lane's registers.
template <typename Key>
__device__ __forceinline__ void exchange(typename Key::T (&k)[kPer]) {
#pragma unroll
    for (int d = kPer / 2; d > 0; d >>= 1) {
#pragma unroll
        for (int r = 0; r < kPer; ++r) {
            if (r & d) continue;
            const typename Key::T lo = Key::lower(k[r], k[r | d]);
            const typename Key::T hi = Key::upper(k[r], k[r | d]);
            k[r] = lo;
            k[r | d] = hi;
        }
    }
}

// Sorts the tile's keys (x: coordinates of slots tid + 256 j; mark: their marks' running
// maxima) and gives slots 16 tid .. 16 tid + 15 of the sorted tile as bit masks: `side` (B
// entries) and `dup` (a B entry equal to the A entry before it).  The first slot of a
// wavefront is compared after the next barrier (sh.first, sh.last).
template <typename Key>
__device__ __forceinline__ void sort_tile(OrderLds &sh, const unsigned (&x)[kPer],
                                          const unsigned (&mark)[kPer], int n, int bits, int tid,
                                          unsigned &side, unsigned &dup) {
    typename Key::T k[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const unsigned row = mark[j] ^ static_cast<unsigned>(static_cast<int>(mark[j]) >> 31);
        k[j] = Key::make(row, __builtin_amdgcn_alignbit(x[j], mark[j], 31), bits);
    }
    exchange<Key>(k);
    Key::to_mid(k, sh.word, tid);
    exchange<Key>(k);
    Key::to_runs(k, sh.word, tid);
    exchange<Key>(k);
    // the slot before this lane's first: the previous lane's last
    const unsigned last_lo = Key::low(k[kPer - 1]), last_hi = Key::high(k[kPer - 1]);
    const int l = tid % dev::kWave, w = tid / dev::kWave;
    if (l == dev::kWave - 1) {
        sh.last[2 * w] = last_lo;
        sh.last[2 * w + 1] = last_hi;
    }
    // (wave_shr:1)
    unsigned plo = __builtin_amdgcn_update_dpp(0, static_cast<int>(last_lo), 0x138, 0xf, 0xf, true);
    unsigned phi = __builtin_amdgcn_update_dpp(0, static_cast<int>(last_hi), 0x138, 0xf, 0xf, true);
    if (l == 0) {
        plo = Key::low(k[0]);
        phi = Key::high(k[0]);
        sh.first[2 * w] = plo;
        sh.first[2 * w + 1] = phi;
    }
    side = 0;
    dup = 0;
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        const unsigned lo = Key::low(k[r]), hi = Key::high(k[r]);
        side = __builtin_amdgcn_alignbit(lo, side, 1);
        dup = dup + dup + static_cast<unsigned>((lo ^ plo) == 1u && hi == phi);
        plo = lo;
        phi = hi;
    }
    const int valid = min(max(n - kPer * tid, 0), kPer);
    side = (side >> (32 - kPer)) & ((1u << valid) - 1u);
    dup = (__builtin_bitreverse32(dup) >> (32 - kPer)) & side;
}

// dev::two_level_total for a launch whose workgroups do not all take part: chunk c's first
// workgroup adds the pairs of its written tiles with kChunkTickets tickets less the chunk's
// dense tiles, each of which adds its own pairs with one ticket, so a group of chunks is
// complete exactly when it holds kChunkTickets tickets per chunk (before a chunk's first
// workgroup has added, its dense tiles give fewer).
constexpr int kChunkTickets = 4 * kChunk;

__device__ __forceinline__ int64_t ticket_total(unsigned pairs, int tickets, int c, int tiles,
                                                unsigned long long *acc) {
    const int chunks = (tiles + kChunk - 1) / kChunk;
    const int groups = min(chunks, dev::kTotalGroups);
    const int g = c % dev::kTotalGroups;
    const int members = (chunks - g + dev::kTotalGroups - 1) / dev::kTotalGroups;
    const unsigned long long mine = (static_cast<unsigned long long>(tickets) << 32) | pairs;
    const unsigned long long now = atomicAdd(&acc[(g + 1) * dev::kTotalStride], mine) + mine;
    if ((now >> 32) != static_cast<unsigned long long>(members) * kChunkTickets) return -1;
    const unsigned long long sum = (1ull << 32) | (now & 0xffffffffull);
    const unsigned long long top = atomicAdd(&acc[0], sum) + sum;
    if ((top >> 32) != static_cast<unsigned long long>(groups)) return -1;
    return static_cast<int64_t>(top & 0xffffffffull);
}

// The word `bytes` (>= 0) after a scalar base: one 32-bit lane offset.
__device__ __forceinline__ unsigned load_at(const int *base, int bytes) {
    return *reinterpret_cast<const unsigned *>(reinterpret_cast<const char *>(base) +
                                               static_cast<unsigned>(bytes));
}

// The merge order of a tile whose keys do not hold its coordinates, as order_tile gives it: a lane
// finds its first slot by searches in the operands and takes 16 entries one by one (ties: A
// first).  Unsorted rows keep the searches and the walk inside the tile's ranges as well.
__device__ __forceinline__ void walk_tile(const TileSplit &sp, const int *__restrict__ pa,
                                          const int *__restrict__ ca, const int *__restrict__ pb,
                                          const int *__restrict__ cb, int tid, unsigned &side,
                                          unsigned &dup) {
    const int na = sp.a1 - sp.a0, nb = sp.b1 - sp.b0, nr = sp.r1 - sp.r0 + 1;
    const int first = kPer * tid, count = min(max(na + nb - first, 0), kPer);
    side = dup = 0;
    if (count == 0) return;
    auto begin_a = [&](int k) {
        return k == 0 ? 0 : k >= nr ? na : min(max(pa[sp.r0 + k] - sp.a0, 0), na);
    };
    auto begin_b = [&](int k) {
        return k == 0 ? 0 : k >= nr ? nb : min(max(pb[sp.r0 + k] - sp.b0, 0), nb);
    };
    int k = 0;  // the last row that begins at or before the slot
    for (int hi = nr - 1; k < hi;) {
        const int mid = (k + hi + 1) >> 1;
        if (begin_a(mid) + begin_b(mid) <= first) {
            k = mid;
        } else {
            hi = mid - 1;
        }
    }
    int a = begin_a(k), b = begin_b(k), ae = begin_a(k + 1), be = begin_b(k + 1);
    const int d = first - a - b;
    int lo = max(0, d - (be - b)), hi = min(d, ae - a);  // A entries among the row's first d
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (ca[sp.a0 + a + mid] <= cb[sp.b0 + b + d - 1 - mid]) {
            lo = mid + 1;
        } else {
            hi = mid;
        }
    }
    int as = a;  // the row's first A entry
    a += lo;
    b += d - lo;
    for (int i = 0; i < count; ++i) {
        while (a >= ae && b >= be && k + 1 < nr) {
            ++k;
            as = a;
            ae = begin_a(k + 1);
            be = begin_b(k + 1);
        }
        if (a < ae && (b >= be || ca[sp.a0 + a] <= cb[sp.b0 + b])) {
            ++a;
        } else if (b < be) {
            side |= 1u << i;
            dup |= a > as && ca[sp.a0 + a - 1] == cb[sp.b0 + b] ? 1u << i : 0u;
            ++b;
        }
    }
}

// The merge order of the tile `sp`: lane tid's 16 slots as bit masks `side` and `dup`, and the
// tile's pairs, the same in every lane.  `some`: any readable word.  Ends without a barrier.
template <bool WIDE>
__device__ __forceinline__ unsigned order_tile(OrderLds &sh, const TileSplit &sp,
                                               const int *__restrict__ pa,
                                               const int *__restrict__ ca,
                                               const int *__restrict__ pb,
                                               const int *__restrict__ cb, const int *some,
                                               int bits, int tid, unsigned &side, unsigned &dup) {
    const int l = tid % dev::kWave;
    const int w = __builtin_amdgcn_readfirstlane(tid / dev::kWave);
    const int na = sp.a1 - sp.a0, nb = sp.b1 - sp.b0, nr = sp.r1 - sp.r0 + 1;

    // Slot tid + 256 j is A's entry of that index, or B's entry kSlots - 1 - slot.  The
    // padding is at least a wavefront wide, so a wavefront's 64 slots hold entries of one
    // side only: a scalar base and one clamped lane offset.  Padding slots load a coordinate of
    // the tile, so that every coordinate loaded counts for whether the keys hold it.
    const int *pad = na > 0 ? ca + sp.a0 : nb > 0 ? cb + sp.b0 : some;
    unsigned x[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int first = kBlock * j + dev::kWave * w;  // the wavefront's slots
        const int base = kSlots - kBlock * (j + 1);     // B's entry of tid == kBlock - 1
        const bool in_a = first < na, in_b = first + dev::kWave > kSlots - nb;
        const int *from = in_a ? ca + sp.a0 + kBlock * j : in_b ? cb + sp.b0 + base : pad;
        const int last = in_a ? na - 1 - kBlock * j : in_b ? nb - 1 - base : 0;
        x[j] = load_at(from, min(in_a ? 4 * tid : 4 * (kBlock - 1 - tid), 4 * last));
    }

    static_assert(kMarkHalves % (8 * kBlock) == 0, "cleared in 16-byte stores");
#pragma unroll
    for (int i = 0; i < kMarkHalves / (8 * kBlock); ++i) {
        reinterpret_cast<uint4 *>(sh.mark)[tid + i * kBlock] = uint4{0, 0, 0, 0};
    }
    __syncthreads();
    if (tid == 0) sh.mark[mark_half(na)] = static_cast<unsigned short>(kPadMark);
    for (int k = tid; k < nr; k += kBlock) {
        const bool end = k == nr - 1;
        const int r = sp.r0 + k;
        const int a0 = max(pa[r] - sp.a0, 0), a1 = end ? na : pa[r + 1] - sp.a0;
        const int b0 = max(pb[r] - sp.b0, 0), b1 = end ? nb : pb[r + 1] - sp.b0;
        if (a1 > a0) sh.mark[mark_half(a0)] = static_cast<unsigned short>(k);
        if (b1 > b0) sh.mark[mark_half(kSlots - b1)] = static_cast<unsigned short>(~k);
    }
    __syncthreads();
    // Running maximum: 16 consecutive slots per lane (two per register), then over the lanes
    // and wavefronts.
    half2_t run[kPer / 2];
    uint4 *runs = reinterpret_cast<uint4 *>(sh.mark + mark_half(kPer * tid));
#pragma unroll
    for (int q = 0; q < kPer / 8; ++q) {
        const uint4 v = runs[q];
        run[4 * q] = __builtin_bit_cast(half2_t, v.x);
        run[4 * q + 1] = __builtin_bit_cast(half2_t, v.y);
        run[4 * q + 2] = __builtin_bit_cast(half2_t, v.z);
        run[4 * q + 3] = __builtin_bit_cast(half2_t, v.w);
    }
#pragma unroll
    for (int r = 0; r < kPer / 2; ++r) {
        if (r > 0) run[r] = __builtin_elementwise_max(run[r], run[r - 1].yy);
        run[r] = __builtin_elementwise_max(run[r], run[r].xx);
    }
    const unsigned incl = dev::wave_inclusive_umax_dpp(run[kPer / 2 - 1].y);
    if (l == dev::kWave - 1) sh.wave_max[w] = incl;
    unsigned before = static_cast<unsigned>(  // (wave_shr:1)
        __builtin_amdgcn_update_dpp(0, static_cast<int>(incl), 0x138, 0xf, 0xf, true));
    __syncthreads();
    for (int i = 0; i < w; ++i) before = max(before, sh.wave_max[i]);
    const half2_t carry = static_cast<unsigned short>(before);
#pragma unroll
    for (int q = 0; q < kPer / 8; ++q) {
        auto word = [&](int i) {
            return __builtin_bit_cast(unsigned,
                                      __builtin_elementwise_max(run[4 * q + i], carry));
        };
        runs[q] = uint4{word(0), word(1), word(2), word(3)};
    }
    __syncthreads();
    unsigned mark[kPer];  // sign-extended: k for A, ~k for B
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        mark[j] = static_cast<unsigned>(static_cast<int>(
            static_cast<short>(sh.mark[mark_half(tid) + (kBlock / 16 * 24) * j])));
    }
    __syncthreads();  // (the keys replace the marks)

    // (bits of nr, not of nr - 1: the padding's row, all ones, is no row of the tile)
    const int row_bits = 32 - __builtin_clz(static_cast<unsigned>(nr));
    const bool wide = WIDE && row_bits + bits + 1 > 32;
    unsigned crds = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) crds |= x[j];
    const bool past = __any(crds >> (wide ? 31 : bits));  // of no key's coordinate
    if (wide) {  // uniform
        sort_tile<WideKey>(sh, x, mark, na + nb, bits, tid, side, dup);
    } else {
        sort_tile<NarrowKey>(sh, x, mark, na + nb, bits, tid, side, dup);
    }
    // The tile's pairs and B slots per wavefront (flag: bit 31 of the pairs).
    auto count = [&](bool flag) {
        const int found = dev::wave_inclusive_sum_dpp(__popc(dup));
        const int in_b = dev::wave_inclusive_sum_dpp(__popc(side));
        if (l == dev::kWave - 1) {
            sh.pairs[w] = static_cast<unsigned>(found) | (flag ? 1u << 31 : 0u);
            sh.sides[w] = static_cast<unsigned>(in_b);
        }
        __syncthreads();
    };
    count(past);
    // pairs across two wavefronts: the last slot of i - 1 and the first of i
    auto across = [&](int i) {
        return kPer * dev::kWave * i < na + nb &&
               (sh.first[2 * i] ^ sh.last[2 * i - 2]) == 1u && (sh.first[2 * i] & 1u) == 1u &&
               (!wide || sh.first[2 * i + 1] == sh.last[2 * i - 1]);
    };
    unsigned pairs = sh.pairs[0], sides = sh.sides[0], flags = pairs;
#pragma unroll
    for (int i = 1; i < kWaves; ++i) {
        const bool p = across(i);
        flags |= sh.pairs[i];
        pairs += sh.pairs[i] + static_cast<unsigned>(p);
        sides += sh.sides[i];
        if (p && tid == dev::kWave * i) dup |= 1u;
    }
    if (flags >> 31) {  // uniform
        __syncthreads();  // (the counts are read)
        walk_tile(sp, pa, ca, pb, cb, tid, side, dup);
        count(false);
        pairs = sides = 0;
        for (int i = 0; i < kWaves; ++i) {
            pairs += sh.pairs[i];
            sides += sh.sides[i];
        }
    }
    if (sides != static_cast<unsigned>(nb)) {  // uniform
        // Only operands that break the contract (unsorted rows): any order with nb B slots
        // keeps the emit kernel inside them.
        const int b_from = min(max(na - kPer * tid, 0), kPer);
        const int b_to = min(max(na + nb - kPer * tid, 0), kPer);
        side = ((1u << b_to) - 1u) & ~((1u << b_from) - 1u);
        dup = 0;
        pairs = 0;
    }
    return pairs;
}

// One tile per workgroup.  side / dup: kBlock 16-bit masks per tile; tile_pairs[t] gets the
// tile's pairs, which are also added into chunk_pairs[t / kChunk] (zeroed by the partition
// kernel).  The last workgroup stores the result length: the pairs (intersection), or the
// entries that the operands' offsets span less the pairs.  WIDE: the level's extent may need 64-bit
// keys.  SPARSE: split_sparse_kernel ran; state[t] holds the pairs of a tile that it
// wrote, or kDense.
template <bool WIDE, bool SPARSE>
__global__ __launch_bounds__(kBlock, WIDE ? 4 : 6) void order_kernel(
    const int *__restrict__ pa, const int *__restrict__ ca, const int *__restrict__ pb,
    const int *__restrict__ cb, const int *__restrict__ split_r, const int *__restrict__ split_a,
    const int *__restrict__ split_b, int bits, unsigned short *__restrict__ side_out,
    unsigned short *__restrict__ dup_out, const unsigned *__restrict__ state,
    unsigned *__restrict__ tile_pairs, unsigned *__restrict__ chunk_pairs,
    unsigned long long *__restrict__ done,
    int64_t *__restrict__ length_out, int intersect) {
    __shared__ __align__(16) OrderLds sh;
    const int tid = threadIdx.x;
    const int l = tid % dev::kWave;
    const int w = __builtin_amdgcn_readfirstlane(tid / dev::kWave);
    const int t = blockIdx.x;
    const int c = t / kChunk;
    // The tile's pairs, or those of a chunk's written tiles, `tickets` of the chunk's (one
    // thread).
    auto total = [&](unsigned pairs, int tickets) {
        if (pairs) atomicAdd(&chunk_pairs[c * kChunkStride], pairs);
        const int64_t all = SPARSE ? ticket_total(pairs, tickets, c, gridDim.x, done)
                                   : dev::two_level_total(pairs, done);
        if (all >= 0) {  // (the last one; an operand's arrays may be longer than its offsets say)
            const int64_t items = static_cast<int64_t>(split_a[gridDim.x]) + split_b[gridDim.x];
            dev::store_system(length_out, intersect ? all : items - all);
        }
    };
    if (SPARSE) {
        if (t % kChunk == 0) {  // uniform: the chunk's tiles whose order is written
            const int at = t + tid;
            const unsigned v = at < static_cast<int>(gridDim.x) ? state[at] : 0u;
            const unsigned long long dense = __ballot(v == kDense);
            const int sum = dev::wave_inclusive_sum_dpp(v == kDense ? 0 : static_cast<int>(v));
            if (l == dev::kWave - 1) {
                sh.pairs[w] = static_cast<unsigned>(sum);
                sh.sides[w] = static_cast<unsigned>(__popcll(dense));
            }
            __syncthreads();
            if (tid == 0) {
                unsigned pairs = 0, left = 0;
#pragma unroll
                for (int i = 0; i < kWaves; ++i) {
                    pairs += sh.pairs[i];
                    left += sh.sides[i];
                }
                total(pairs, kChunkTickets - static_cast<int>(left));
            }
            __syncthreads();
        }
        if (state[t] != kDense) return;  // uniform
    }
    const TileSplit sp = load_split(split_r, split_a, split_b, t);
    unsigned side, dup;
    const unsigned pairs =
        order_tile<WIDE>(sh, sp, pa, ca, pb, cb, split_r, bits, tid, side, dup);
    side_out[static_cast<size_t>(t) * kBlock + tid] = static_cast<unsigned short>(side);
    dup_out[static_cast<size_t>(t) * kBlock + tid] = static_cast<unsigned short>(dup);
    if (tid == 0) {
        tile_pairs[t] = pairs;
        total(pairs, 1);
    }
}

// ---- emit kernel -----------------------------------------------------------------------

__device__ __forceinline__ unsigned long long readlane64(unsigned long long v, int i) {
    const unsigned lo = static_cast<unsigned>(
        __builtin_amdgcn_readlane(static_cast<int>(static_cast<unsigned>(v)), i));
    const unsigned hi = static_cast<unsigned>(
        __builtin_amdgcn_readlane(static_cast<int>(static_cast<unsigned>(v >> 32)), i));
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

struct EmitArgs {
    const int *pa, *ca;
    const float *va;
    const int *pb, *cb;
    const float *vb;
    const int *split_r, *split_a, *split_b;
    const unsigned long long *side, *dup;
    const unsigned *tile_pairs, *chunk_pairs;
    int num_tiles;
    int *pc, *cc;
    float *vc;
    const int *next_a, *next_b;
    int *child_a, *child_b;
    int nnz_a, nnz_b;
    int *rc, *ck;
    int kbits;
    double *partial;
};

// Pairs of the tiles before t, summed by one wavefront.
__device__ __forceinline__ int pairs_before(const EmitArgs &g, int t, int l) {
    const int c = t / kChunk;
    int sum = 0;
    for (int i = l; i < c; i += dev::kWave) sum += static_cast<int>(g.chunk_pairs[i * kChunkStride]);
#pragma unroll
    for (int i = 0; i < kChunk / dev::kWave; ++i) {
        const int at = c * kChunk + i * dev::kWave + l;
        if (at < t) sum += static_cast<int>(g.tile_pairs[at]);
    }
    return __builtin_amdgcn_readlane(dev::wave_inclusive_sum_dpp(sum), dev::kWave - 1);
}

// LDS of a tile's output rows (ROWS).
template <bool ROWS>
struct RowLds {
    alignas(16) unsigned short mark[ROWS ? kSlots : 8];
    int carry[kWaves];
};

// Writes one tile's outputs, a quarter of its slots and of its row ends per wavefront; nothing
// is shared between wavefronts (but for the row marks of ROWS).  Lane l of every wavefront
// holds order word l of the tile (side_w, dup_w) and the running counts of B entries and pairs
// before it; `pairs` is the pairs of the tiles before.  A wavefront's 16 words are loaded kGroup at a time before
// any of them is stored: the loads in flight are what the memory's latency is hidden by.
// C2's 547 MB take 105 us (5.2 TB/s; a copy reaches 5.5); with 4 words at a time and a
// resident grid walking chunks of tiles it took 127 us.
//
// VALUES: crd and val.  CHILD: crd and child pointers: for output o, child_a[o] = next_a[a]
// and child_b[o] = next_b[b] at the A / B positions a, b reached before o, so that
// [child[o], child[o + 1]) is the operand's child range under o, empty when absent (null
// next: the position itself).  ROWS: rc receives each output's row.  ck (optional, with
// ROWS): outputs stored split, c >> kbits to cc and the low kbits to ck.  DOT
// (intersection): the products are added to acc instead.
//
// The operands' arrays are never null (the host passes some valid array for an empty one):
// every load is unconditional, at an entry of the operand.
template <Op OP, bool VALUES, bool CHILD, bool ROWS, bool DOT>
__device__ __forceinline__ void emit_tile(const EmitArgs &g, const TileSplit &sp, int t,
                                          unsigned long long side_w, unsigned long long dup_w,
                                          int pairs, int tid, RowLds<ROWS> &lds, double &acc) {
    static_assert(!(VALUES && CHILD) && (VALUES || !ROWS), "a level carries one kind of payload");
    static_assert(!DOT || (OP == Op::Intersect && VALUES), "the inner product: intersection");
    constexpr int kGroup = OP == Op::Union && VALUES ? 16 : 8;  // words loaded together
    constexpr int kWordsPerWave = kWords / kWaves;
    const int l = tid % dev::kWave;
    const int w = __builtin_amdgcn_readfirstlane(tid / dev::kWave);
    const int n = sp.a1 - sp.a0 + sp.b1 - sp.b0;
    const int ends = sp.r1 - sp.r0;  // rows r0 .. r0 + ends - 1 end in the tile
    const int side_n = __popcll(side_w), dup_n = __popcll(dup_w);
    const int side_before = dev::wave_inclusive_sum_dpp(side_n) - side_n;
    const int dup_incl = dev::wave_inclusive_sum_dpp(dup_n);
    const int dup_before = dup_incl - dup_n;
    const int tile_pairs = __builtin_amdgcn_readlane(dup_incl, dev::kWave - 1);
    const int out0 = OP == Op::Union ? sp.a0 + sp.b0 - pairs : pairs;  // first output

    if (ROWS) {  // row marks by slot, as in the order kernel but in merged order
        uint4 *clear = reinterpret_cast<uint4 *>(lds.mark);
        clear[tid] = uint4{0, 0, 0, 0};
        clear[tid + kBlock] = uint4{0, 0, 0, 0};
        if (tid < kWaves) lds.carry[tid] = 0;
        __syncthreads();
        for (int k = tid; k <= ends; k += kBlock) {
            const int s = k == 0 ? 0 : g.pa[sp.r0 + k] - sp.a0 + g.pb[sp.r0 + k] - sp.b0;
            const int e = k == ends ? n
                                    : g.pa[sp.r0 + k + 1] - sp.a0 + g.pb[sp.r0 + k + 1] - sp.b0;
            if (e > s) {
                lds.mark[s] = static_cast<unsigned short>(k);
                atomicMax(&lds.carry[s / (kSlots / kWaves)], k);
            }
        }
        __syncthreads();
    }
    int row_carry = 0;  // last row started before the wavefront's next word (tile-local)
    if (ROWS) {
        for (int i = 0; i < w; ++i) row_carry = max(row_carry, lds.carry[i]);
        row_carry = __builtin_amdgcn_readfirstlane(row_carry);
    }

    for (int i0 = w * kWordsPerWave; i0 < (w + 1) * kWordsPerWave; i0 += kGroup) {
        if (i0 * 64 >= n) break;  // uniform
        if (OP == Op::Intersect && !ROWS) {  // words without pairs: next (uniform)
            const unsigned long long any = __ballot(dup_w != 0);
            // (a pair's A slot may be the last one before its B slot's word; with ROWS,
            // every word carries its last row to the next)
            if (((any >> i0) & ((2ull << kGroup) - 1ull)) == 0) continue;
        }
        int c[kGroup], ra[CHILD ? kGroup : 1], rb[CHILD ? kGroup : 1];
        float v[kGroup], v2[OP == Op::Intersect ? kGroup : 1];
        // slots of word i that hold an entry
        auto valid_of = [&](int i) {
            const int left = n - i * 64;
            return left >= 64 ? ~0ull : left <= 0 ? 0ull : (1ull << left) - 1ull;
        };
        // A entries of pairs in word i: the slot after them is a pair's B entry
        auto pairs_of = [&](int i, unsigned long long dup) {
            const unsigned long long next =
                i + 1 < kWords ? readlane64(dup_w, min(i + 1, kWords - 1)) : 0ull;
            return (dup >> 1) | (next << 63);
        };
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
            const int i = i0 + u;
            const unsigned long long side = readlane64(side_w, i);
            const int sb = __builtin_amdgcn_readlane(side_before, i);
            const int below = bits_below(side);
            const int ib = sp.b0 + sb + below;                 // B position reached
            const int ia = sp.a0 + i * 64 - sb + (l - below);  // A position reached
            if (OP == Op::Union) {
                const bool is_b = __builtin_amdgcn_inverse_ballot_w64(side);
                const bool in = __builtin_amdgcn_inverse_ballot_w64(valid_of(i));
                const int at = in ? (is_b ? ib : ia) : 0;
                c[u] = (is_b ? g.cb : g.ca)[at];
                if (VALUES) v[u] = (is_b ? g.vb : g.va)[at];
                if (CHILD) {
                    const int xa = in ? ia : 0, xb = in ? ib : 0;
                    ra[u] = g.next_a ? g.next_a[xa] : xa;
                    rb[u] = g.next_b ? g.next_b[xb] : xb;
                }
            } else {
                // Lanes without a pair load too: no branch between the loads.  The
                // result's: the entries reached, whose lines its neighbours need; the
                // inner product's, where pairs are few: entry 0.
                const bool in = !DOT || __builtin_amdgcn_inverse_ballot_w64(
                                            pairs_of(i, readlane64(dup_w, i)));
                const int xa = in ? min(ia, max(g.nnz_a - 1, 0)) : 0;
                const int xb = in ? min(ib, max(g.nnz_b - 1, 0)) : 0;
                if (!DOT) c[u] = g.ca[xa];
                v[u] = g.va[xa];
                v2[u] = g.vb[xb];
            }
        }
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
            const int i = i0 + u;
            const unsigned long long dup = readlane64(dup_w, i);
            const unsigned long long pair_a = pairs_of(i, dup);
            const unsigned long long emit = OP == Op::Union ? valid_of(i) & ~dup : pair_a;
            float val = v[u];
            if (OP == Op::Intersect) {
                val = v[u] * v2[u];
            } else if (VALUES && pair_a != 0) {  // uniform
                // the pair's B value was loaded by the next slot (wave_shl:1)
                float other = __int_as_float(__builtin_amdgcn_update_dpp(
                    0, __float_as_int(v[u]), 0x130, 0xf, 0xf, true));
                if (pair_a >> 63) {  // the next word's first slot
                    float next = 0.0f;
                    if (u + 1 < kGroup) {
                        next = __int_as_float(__builtin_amdgcn_readlane(
                            __float_as_int(v[(u + 1) % kGroup]), 0));
                    } else {
                        const unsigned long long side = readlane64(side_w, i);
                        next = g.vb[sp.b0 + __builtin_amdgcn_readlane(side_before, i) +
                                    __popcll(side)];
                    }
                    if (l == dev::kWave - 1) other = next;
                }
                if (__builtin_amdgcn_inverse_ballot_w64(pair_a)) val = v[u] + other;
            }
            if (DOT) {
                if (__builtin_amdgcn_inverse_ballot_w64(emit)) acc += static_cast<double>(val);
                continue;
            }
            int row = 0;
            if (ROWS) {
                const int m = dev::wave_inclusive_max_dpp(lds.mark[i * 64 + l]);
                row = max(m, row_carry);
                row_carry = max(row_carry, __builtin_amdgcn_readlane(m, dev::kWave - 1));
            }
            const int db = __builtin_amdgcn_readlane(dup_before, i);
            const int first = OP == Op::Union ? out0 + i * 64 - db : out0 + db;
            const int o = first + (OP == Op::Union ? l - bits_below(dup) : bits_below(dup));
            if (__builtin_amdgcn_inverse_ballot_w64(emit)) {
                if (ROWS && g.ck) {
                    g.cc[o] = c[u] >> g.kbits;
                    g.ck[o] = static_cast<int>(static_cast<unsigned>(c[u]) &
                                               ((1u << g.kbits) - 1u));
                } else {
                    g.cc[o] = c[u];
                }
                if (VALUES) g.vc[o] = val;
                if (CHILD) {
                    g.child_a[o] = ra[u];
                    g.child_b[o] = rb[u];
                }
                if (ROWS) g.rc[o] = sp.r0 + row;
            }
        }
    }

    if (!DOT) {  // row ends: row r0 + k ends before slot s of the tile
        for (int k0 = w * dev::kWave; k0 < ends; k0 += kBlock) {  // uniform in the wave
            const int k = min(k0 + l, ends - 1);
            const int s = g.pa[sp.r0 + k + 1] - sp.a0 + g.pb[sp.r0 + k + 1] - sp.b0;
            int d = 0;
            if (tile_pairs != 0) {  // pairs whose B slot lies before s
                const int at = min(s >> 6, kWords - 1);
                const unsigned long long word = __shfl(dup_w, at, dev::kWave);
                const int used = s - (at << 6);  // 0 .. 64
                const unsigned long long low = used >= 64 ? ~0ull : (1ull << used) - 1ull;
                d = __shfl(dup_before, at, dev::kWave) + __popcll(word & low);
            }
            if (k0 + l < ends) g.pc[sp.r0 + k + 1] = out0 + (OP == Op::Union ? s - d : d);
        }
        if (t == 0 && tid == 0) g.pc[0] = 0;
    }
    if (CHILD && t == g.num_tiles - 1 && tid == 0) {
        const int end = out0 + n - tile_pairs;
        g.child_a[end] = g.next_a ? g.next_a[g.nnz_a] : g.nnz_a;
        g.child_b[end] = g.next_b ? g.next_b[g.nnz_b] : g.nnz_b;
    }
}

// One tile per workgroup (DOT: tiles strided over the grid, the workgroup's products summed
// to partial[w]).
template <Op OP, bool VALUES, bool CHILD, bool ROWS, bool DOT>
__global__ __launch_bounds__(kBlock) void emit_kernel(EmitArgs g) {
    __shared__ RowLds<ROWS> lds;
    __shared__ double s_dot[DOT ? kBlock : 1];
    const int tid = threadIdx.x;
    const int l = tid % dev::kWave;
    double acc = 0.0;
    for (int t = blockIdx.x; t < g.num_tiles; t += gridDim.x) {  // (once but for DOT)
        const unsigned long long side_w = g.side[static_cast<size_t>(t) * kWords + l];
        const unsigned long long dup_w = g.dup[static_cast<size_t>(t) * kWords + l];
        const TileSplit sp = load_split(g.split_r, g.split_a, g.split_b, t);
        emit_tile<OP, VALUES, CHILD, ROWS, DOT>(g, sp, t, side_w, dup_w,
                                                DOT ? 0 : pairs_before(g, t, l), tid, lds, acc);
    }
    if (DOT) {
        s_dot[tid] = acc;
#pragma unroll
        for (int h = kBlock / 2; h > 0; h >>= 1) {
            __syncthreads();
            if (tid < h) s_dot[tid] += s_dot[tid + h];
        }
        if (tid == 0) g.partial[blockIdx.x] = s_dot[0];
    }
}

// Binary64 sum of the kBlock values of `sh` into sh[0], in a fixed order; ends synchronised.
__device__ __forceinline__ void block_sum_fixed(double *sh) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        __syncthreads();
        if (tid < w) sh[tid] += sh[tid + w];
    }
    __syncthreads();
}

// ---- small levels ----------------------------------------------------------------------
//
// A level of few tiles in one launch: a workgroup finds its tile's boundaries, orders it,
// publishes its pairs, waits for those of the tiles before it and writes its outputs.  Tiles
// are dealt by a ticket, so a workgroup only waits for workgroups that have started; with few
// tiles they all run at once and the wait is the spread of their starts.  (With thousands, the
// first tile's output would wait for nothing while the memory is idle: three launches are
// better.)
//
// `sync` is a block of words that only these kernels write: two counters that keep counting
// from launch to launch (this launch's counts start at `base` and `done_base`) and, per tile, the
// pairs tagged with the launch's epoch, so that it is never cleared.
//
// Every wait is bounded, for a block whose counts are not what the host believes, and a level
// whose length was stored is whole: the length is the last tile's to store, and it withholds it
// where it gives up itself or sees that another tile did.  A tile that gives up says so first
// and then waits once more, for seconds: had the last tile missed the word, every count would
// have been published by then.
constexpr int kSyncGaveUp = 2;  // word that holds the epoch of a launch in which a tile gave up
constexpr int kSyncTiles = 16;  // word of tile 0
constexpr size_t kSyncBytes = (kSyncTiles + kFusedTiles) * sizeof(unsigned long long);

template <Op OP, bool VALUES, bool CHILD, bool ROWS, bool DOT, bool WIDE>
__global__ __launch_bounds__(kBlock) void fused_kernel(EmitArgs g, int rows, int total, int bits,
                                                       unsigned long long *__restrict__ sync,
                                                       unsigned epoch, unsigned base,
                                                       unsigned done_base, unsigned max_polls,
                                                       int64_t *__restrict__ length_out,
                                                       float *__restrict__ dot) {
    __shared__ double s_dot[DOT ? kBlock : 1];
    __shared__ __align__(16) OrderLds sh;
    __shared__ __align__(8) unsigned short s_side[kBlock], s_dup[kBlock];
    __shared__ RowLds<ROWS> lds;
    __shared__ int s_split[6];
    __shared__ int s_ticket, s_wave[kWaves];
    const int tid = threadIdx.x;
    const int l = tid % dev::kWave;
    const int w = __builtin_amdgcn_readfirstlane(tid / dev::kWave);
    int t = 0;
    if (g.num_tiles > 1) {  // uniform
        if (tid == 0) s_ticket = static_cast<int>(atomicAdd(reinterpret_cast<unsigned *>(sync), 1u) - base);
        __syncthreads();
        t = __builtin_amdgcn_readfirstlane(s_ticket);
        if (t < 0 || t >= g.num_tiles) {  // no tile: the block's counts are others
            if (DOT && tid == 0) *dot = __builtin_nanf("");
            return;
        }
    }
    if (w < 2) {  // boundary t + w
        const int b = t + w;
        int r = 0, x = 0, y = 0;
        if (b == g.num_tiles) {
            r = rows;
            x = g.pa[rows];
            y = g.pb[rows];
        } else if (b > 0) {
            find_split<dev::kWave>(g.pa, g.ca, g.pb, g.cb, rows,
                                   static_cast<int>(min(static_cast<long long>(b) * kTile,
                                                        static_cast<long long>(total))),
                                   r, x, y);
        }
        if (l == 0) {
            s_split[3 * w] = r;
            s_split[3 * w + 1] = x;
            s_split[3 * w + 2] = y;
        }
    }
    __syncthreads();
    auto u = [&](int i) { return __builtin_amdgcn_readfirstlane(s_split[i]); };
    const TileSplit sp{u(0), u(1), u(2), u(3), u(4), u(5)};
    unsigned side, dup;
    const unsigned own = order_tile<WIDE>(sh, sp, g.pa, g.ca, g.pb, g.cb, g.pa, bits, tid, side, dup);
    double acc = 0.0;
    if (DOT) {
        // No offsets to wait for: every tile's sum goes to partial, and the workgroup that
        // finishes last (the second counter) adds them in tile order.
        s_side[tid] = static_cast<unsigned short>(side);
        s_dup[tid] = static_cast<unsigned short>(dup);
        __syncthreads();
        emit_tile<OP, VALUES, CHILD, ROWS, DOT>(
            g, sp, t, reinterpret_cast<const unsigned long long *>(s_side)[l],
            reinterpret_cast<const unsigned long long *>(s_dup)[l], 0, tid, lds, acc);
        s_dot[tid] = acc;
        block_sum_fixed(s_dot);
        if (g.num_tiles > 1) {  // uniform
            if (tid == 0) {
                __hip_atomic_store(&g.partial[t], s_dot[0], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                const unsigned done = __hip_atomic_fetch_add(
                    reinterpret_cast<unsigned *>(sync + 1), 1u, __ATOMIC_ACQ_REL,
                    __HIP_MEMORY_SCOPE_AGENT);
                s_ticket = done - done_base == static_cast<unsigned>(g.num_tiles) - 1u;
            }
            __syncthreads();
            if (!s_ticket) return;  // uniform
            acc = 0.0;
            for (int i = tid; i < g.num_tiles; i += kBlock) {
                acc += __hip_atomic_load(&g.partial[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            s_dot[tid] = acc;
            block_sum_fixed(s_dot);
        }
        if (tid == 0) *dot = static_cast<float>(s_dot[0]);
        return;
    }
    if (tid == 0 && t + 1 < g.num_tiles) {
        __hip_atomic_store(&sync[kSyncTiles + t],
                           (static_cast<unsigned long long>(epoch) << 32) | own,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    s_side[tid] = static_cast<unsigned short>(side);
    s_dup[tid] = static_cast<unsigned short>(dup);
    // (The waits end: the workgroups of the tiles before have started and wait for earlier
    // ones only.)
    static_assert(kFusedTiles <= kBlock, "a lane waits for one tile");
    const bool last = t == g.num_tiles - 1;
    int before = 0;
    bool found = true;
    if (tid < t) {
        unsigned long long v = 0;
        auto published = [&](unsigned polls) {
            for (unsigned i = 0; i < polls; ++i) {
                v = __hip_atomic_load(&sync[kSyncTiles + tid], __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
                const unsigned long long gave_up =  // (issued with the load above)
                    last ? __hip_atomic_load(&sync[kSyncGaveUp], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT)
                         : 0ull;
                if ((v >> 32) == epoch) return gave_up != epoch;
            }
            return false;
        };
        found = published(max_polls);
        if (!found && !last) {
            __hip_atomic_store(&sync[kSyncGaveUp], static_cast<unsigned long long>(epoch),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            found = published(SyncBlock::kMaxPolls);
        }
        before = static_cast<int>(v & 0xffffffffull);
    }
    int pairs = 0;
    (void)dev::block_exclusive_sum<kBlock>(before, s_wave, pairs);
    pairs = __builtin_amdgcn_readfirstlane(pairs);
    if (__syncthreads_or(!found)) return;
    if (tid == 0 && t == g.num_tiles - 1) {
        const int64_t all = static_cast<int64_t>(pairs) + own;
        dev::store_system(length_out,
                          OP == Op::Union ? static_cast<int64_t>(sp.a1) + sp.b1 - all : all);
    }
    const unsigned long long side_w = reinterpret_cast<const unsigned long long *>(s_side)[l];
    const unsigned long long dup_w = reinterpret_cast<const unsigned long long *>(s_dup)[l];
    emit_tile<OP, VALUES, CHILD, ROWS, false>(g, sp, t, side_w, dup_w, pairs, tid, lds, acc);
}

// ---- fixed-order sums ------------------------------------------------------------------

// Workgroups of the two-level sums below: few enough that one workgroup then adds their
// partials in a handful of loads per thread.
constexpr int kDotBlocks = 1024;

// One workgroup: the sum of the n partials in a fixed order, rounded once to *dot.
__global__ __launch_bounds__(kBlock) void dot_final_kernel(const double *__restrict__ partial,
                                                           int n, float *__restrict__ dot) {
    __shared__ double sh[kBlock];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += kBlock) acc += partial[i];
    sh[threadIdx.x] = acc;
    block_sum_fixed(sh);
    if (threadIdx.x == 0) *dot = static_cast<float>(sh[0]);
}

// Workgroup b of G sums v[b*n/G, (b+1)*n/G) in binary64, in a fixed order: partial[b].
__global__ __launch_bounds__(kBlock) void sum_blocks_kernel(const float *__restrict__ v,
                                                            long long n,
                                                            double *__restrict__ partial) {
    __shared__ double sh[kBlock];
    const long long g = gridDim.x;
    const long long lo = n * static_cast<long long>(blockIdx.x) / g;
    const long long hi = n * (static_cast<long long>(blockIdx.x) + 1) / g;
    double acc = 0.0;
    for (long long i = lo + threadIdx.x; i < hi; i += kBlock) acc += static_cast<double>(v[i]);
    sh[threadIdx.x] = acc;
    block_sum_fixed(sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

}  // namespace

// ---- host ------------------------------------------------------------------------------

int sum_values(Call &call, const float *v, long long n, float *out) {
    const int blocks = static_cast<int>(
        std::max<long long>(1, std::min<long long>(kDotBlocks, (n + kBlock - 1) / kBlock)));
    double *partial = nullptr;
    NACHO_TRY(call.scratch_n(static_cast<size_t>(blocks), &partial));
    const hipStream_t s = call.stream();
    sum_blocks_kernel<<<blocks, kBlock, 0, s>>>(v, n, partial);
    NACHO_TRY_HIP(hipGetLastError());
    dot_final_kernel<<<1, kBlock, 0, s>>>(partial, blocks, out);
    NACHO_TRY_HIP(hipGetLastError());
    return NACHO_OK;
}

int merge_level(Call &call, bool intersect, bool values, bool child, int rows, int crd_bits,
                const LevelOperand &A, const LevelOperand &B, const LevelResult &Z,
                long long *out_len, const char *kernel_name, bool *length_pending) {
    if (length_pending) *length_pending = false;
    const long long total = static_cast<long long>(A.len) + B.len + rows;
    if (total > static_cast<long long>(INT_MAX) - kLevelItemSlack) {
        return NACHO_ERR_INDEX_OVERFLOW;
    }
    // the kinds of level this merge knows
    if (values ? child : !child || intersect) return NACHO_ERR_INVALID_ARGUMENT;
    if (Z.crd_low && (!Z.row || intersect)) return NACHO_ERR_INVALID_ARGUMENT;
    if (Z.dot && !intersect) return NACHO_ERR_INVALID_ARGUMENT;
    if (!intersect) {  // unions take int32 arrays at multiples of 4 bytes only
        for (const int *p : {A.pos, A.crd, B.pos, B.crd}) {
            if (reinterpret_cast<uintptr_t>(p) & 3u) return NACHO_ERR_INVALID_ARGUMENT;
        }
    }
    const int num_tiles = total > 0 ? static_cast<int>((total + kTile - 1) / kTile) : 1;

    void (*emit)(EmitArgs) =
        child       ? emit_kernel<Op::Union, false, true, false, false>
        : intersect ? (Z.dot   ? emit_kernel<Op::Intersect, true, false, false, true>
                       : Z.row ? emit_kernel<Op::Intersect, true, false, true, false>
                               : emit_kernel<Op::Intersect, true, false, false, false>)
        : Z.row     ? emit_kernel<Op::Union, true, false, true, false>
                    : emit_kernel<Op::Union, true, false, false, false>;
    // One workgroup per tile; an inner product's partial sums come from a resident grid.
    int grid = num_tiles;
    if (Z.dot) {
        NACHO_TRY(resident_grid(reinterpret_cast<const void *>(emit), kBlock, &grid));
        grid = std::min(grid, num_tiles);
    }
    const int chunks = (num_tiles + kChunk - 1) / kChunk;

    const hipStream_t s = call.stream();
    const long long items = static_cast<long long>(A.len) + B.len;
    // 32-bit keys hold any tile's rows (12 bits) beside coordinates of up to 19 bits.
    const bool wide = crd_bits + 13 > 32;
    // (an empty operand's arrays may be null: A's offsets stand in, never used as values)
    const int *ca = A.len > 0 ? A.crd : A.pos, *cb = B.len > 0 ? B.crd : A.pos;
    const float *va = A.len > 0 && values ? A.val : reinterpret_cast<const float *>(A.pos);
    const float *vb = B.len > 0 && values ? B.val : reinterpret_cast<const float *>(A.pos);
    EmitArgs args{A.pos, ca, va, B.pos, cb, vb, nullptr, nullptr, nullptr, nullptr, nullptr,
                  nullptr, nullptr, num_tiles, Z.pos, Z.crd, Z.val, A.next, B.next, Z.child_a,
                  Z.child_b, A.len, B.len, Z.row, Z.crd_low, Z.low_bits, nullptr};
    SyncBlock sync{};
    if (num_tiles <= kFusedTiles) {
        // (one tile takes no ticket)
        const unsigned tickets = num_tiles > 1 ? num_tiles : 0;
        NACHO_TRY(call.sync_block(kSyncBytes, tickets, Z.dot ? tickets : 0, Z.dot != nullptr, &sync));
    }
    // A small inner product, which the host never waits for, may be recorded: each replay clears
    // the words first.  They come with the partial sums, so that a recorded call allocates what
    // the calls that warmed the cache up did.  (A level whose length the host waits for fails
    // under capture.)
    const bool recorded = Z.dot && sync.recorded;
    if (sync.words || recorded) {
        if (Z.dot) {
            NACHO_TRY(call.scratch(static_cast<size_t>(num_tiles) * sizeof(double) + kSyncBytes,
                                   reinterpret_cast<void **>(&args.partial)));
        }
        if (recorded) {
            sync.words = reinterpret_cast<unsigned long long *>(args.partial + num_tiles);
            sync.epoch = 1;
            NACHO_TRY(clear_words(s, sync.words, kSyncBytes / sizeof(unsigned long long)));
        }
        void (*fused)(EmitArgs, int, int, int, unsigned long long *, unsigned, unsigned,
                      unsigned, unsigned, int64_t *, float *) =
#define NACHO_FUSED(OP, VAL, CHD, ROWS, DOT)             \
    (wide ? fused_kernel<OP, VAL, CHD, ROWS, DOT, true> \
          : fused_kernel<OP, VAL, CHD, ROWS, DOT, false>)
            child       ? NACHO_FUSED(Op::Union, false, true, false, false)
            : intersect ? (Z.dot   ? NACHO_FUSED(Op::Intersect, true, false, false, true)
                           : Z.row ? NACHO_FUSED(Op::Intersect, true, false, true, false)
                                   : NACHO_FUSED(Op::Intersect, true, false, false, false))
            : Z.row     ? NACHO_FUSED(Op::Union, true, false, true, false)
                        : NACHO_FUSED(Op::Union, true, false, false, false);
#undef NACHO_FUSED
        int64_t *length_out = nullptr;
        if (!Z.dot) NACHO_TRY(call.length_word(&length_out));
        NACHO_TRY(call.timer_start(kernel_name));
        fused<<<num_tiles, kBlock, 0, s>>>(args, rows, static_cast<int>(total), crd_bits,
                                           sync.words, sync.epoch, sync.base, sync.done,
                                           sync.polls, length_out, Z.dot);
        NACHO_TRY_HIP(hipGetLastError());
        if (Z.dot) {
            call.sync_launched();
        } else {
            NACHO_TRY(call.mark_length());
        }
        NACHO_TRY(call.timer_stop());
        if (Z.dot) {
            NACHO_TRY(call.collect_timer());  // (kernel timing only: waits for the stream)
            *out_len = 0;
            return NACHO_OK;
        }
        if (length_pending) {
            *length_pending = true;
            return NACHO_OK;
        }
        int64_t len = 0;
        NACHO_TRY(call.wait_length(&len));
        *out_len = len;
        return NACHO_OK;
    }

    int *splits = nullptr;
    unsigned *counts = nullptr;
    unsigned short *order = nullptr;
    double *partial = nullptr;
    NACHO_TRY(call.scratch_n(3 * (static_cast<size_t>(num_tiles) + 1), &splits));
    int *split_r = splits, *split_a = splits + num_tiles + 1,
        *split_b = splits + 2 * (num_tiles + 1);
    const size_t chunk_words = static_cast<size_t>(chunks) * kChunkStride;
    NACHO_TRY(call.scratch_n(chunk_words + 2 * dev::kTotalWords + 2 * static_cast<size_t>(num_tiles),
                             &counts));
    // 64-bit accumulator of the length total
    unsigned long long *done = reinterpret_cast<unsigned long long *>(counts + chunk_words);
    unsigned *tile_pairs = counts + chunk_words + 2 * dev::kTotalWords;
    unsigned *state = tile_pairs + num_tiles;  // (levels that look for sparse tiles)
    NACHO_TRY(call.scratch_n(static_cast<size_t>(num_tiles) * (2 * kBlock), &order));
    unsigned short *side = order, *dup = order + static_cast<size_t>(num_tiles) * kBlock;
    // The result length goes straight to a pinned host word as soon as the kernel that
    // totals it ends; the host waits for that kernel only, not for the writes after it.  An
    // inner product's host waits for nothing: its length goes to scratch.
    int64_t *length_out = nullptr;
    if (Z.dot) {
        NACHO_TRY(call.scratch_n(static_cast<size_t>(grid), &partial));
        NACHO_TRY(call.scratch_n(1, &length_out));
    } else {
        NACHO_TRY(call.length_word(&length_out));
    }

    NACHO_TRY(call.timer_start(kernel_name));  // the whole device pipeline of this level
    unsigned long long *side64 = reinterpret_cast<unsigned long long *>(side);
    unsigned long long *dup64 = reinterpret_cast<unsigned long long *>(dup);
    const bool sparse =
        !intersect && values && !Z.crd_low &&
        static_cast<long long>(rows) * kSparseEntriesPerRow <= items;
    if (sparse) {
        split_sparse_kernel<<<(num_tiles + kWaves - 1) / kWaves, kBlock, 0, s>>>(
            A.pos, A.crd, B.pos, B.crd, rows, static_cast<int>(total), num_tiles, split_r,
            split_a, split_b, side64, dup64, state, tile_pairs, done, counts, chunks);
    } else {
        csr_partition_kernel<kTile><<<partition_blocks(num_tiles), kPartBlock, 0, s>>>(
            A.pos, A.crd, B.pos, B.crd, rows, static_cast<int>(total), num_tiles, split_r,
            split_a, split_b, done, counts, chunks, kChunkStride);
    }
    NACHO_TRY_HIP(hipGetLastError());
    auto order_fn = sparse ? (wide ? order_kernel<true, true> : order_kernel<false, true>)
                           : (wide ? order_kernel<true, false> : order_kernel<false, false>);
    order_fn<<<num_tiles, kBlock, 0, s>>>(A.pos, A.crd, B.pos, B.crd, split_r, split_a, split_b,
                                          crd_bits, side, dup, state, tile_pairs, counts, done,
                                          length_out, intersect ? 1 : 0);
    NACHO_TRY_HIP(hipGetLastError());
    if (!Z.dot) NACHO_TRY(call.mark_length());
    args.split_r = split_r;
    args.split_a = split_a;
    args.split_b = split_b;
    args.side = side64;
    args.dup = dup64;
    args.tile_pairs = tile_pairs;
    args.chunk_pairs = counts;
    args.partial = partial;
    emit<<<grid, kBlock, 0, s>>>(args);
    NACHO_TRY_HIP(hipGetLastError());
    if (Z.dot) {
        dot_final_kernel<<<1, kBlock, 0, s>>>(partial, grid, Z.dot);
        NACHO_TRY_HIP(hipGetLastError());
        NACHO_TRY(call.timer_stop());
        NACHO_TRY(call.collect_timer());  // (kernel timing only: waits for the stream)
        *out_len = 0;
        return NACHO_OK;
    }
    NACHO_TRY(call.timer_stop());
    if (length_pending) {
        *length_pending = true;
        return NACHO_OK;
    }
    int64_t len = 0;
    NACHO_TRY(call.wait_length(&len));
    *out_len = len;
    return NACHO_OK;
}

}  // namespace csr
}  // namespace nacho
