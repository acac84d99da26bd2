// csr_add and csr_mul: argument checks and result buffers around the level merge
// (level_merge.hip), and the allocation-free csr_add, whose scratch is a small static device
// array: the level merge's order bits (two per entry) do not fit there, so it merges twice.
//
// Allocation-free csr_add (reference path as in level_merge.hip):
//
//  * csr_partition_kernel cuts the merged row sequence into tiles of kTile items.
//  * pair_count_kernel and walk_write_kernel: each workgroup owns a fixed, contiguous chunk
//    of tiles.  The count kernel reads only coordinates and row offsets and adds each write
//    chunk's output count (a tile emits na + nb - pairs); the write kernel starts from the
//    sum of the preceding chunks' counts and carries a running offset through its tiles.
//  * Inside a tile (both kernels): the tile's crd/val ranges of A and B and a packed word per
//    row are staged in LDS from registers that were loaded one tile ahead; lane t owns items
//    [t*IPT, (t+1)*IPT) of the tile, found by a merge-path search in LDS, and walks them in a
//    fixed, unrolled number of steps (take A's head with ties to A, take B's head, or consume a
//    row end).  An equal A/B pair is combined when its A entry is taken and its B entry is
//    skipped when reached, so pairs may straddle lanes.  Outputs stay in registers until the
//    workgroup scan gives their offsets, then go through LDS to coalesced stores.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <mutex>

#include "csr_merge.hpp"
#include "csr_partition.hpp"
#include "device_utils.hpp"
#include "runtime.hpp"

namespace nacho {
namespace csr {
namespace {

constexpr int kBlock = 256;
constexpr int kItemsPerLane = 15;  // odd: lanes' LDS walks spread over banks
constexpr int kTile = kBlock * kItemsPerLane;
// A tile whose rows need at least this many searches counts its pairs by walking each
// lane's items instead (about 16 dependent LDS steps per lane against about 14 per search).
constexpr int kWalkMin = 2 * kBlock;
// ---- tile staging ----------------------------------------------------------------------

// The splits of a workgroup's whole chunk, staged in LDS once: reading them from global
// memory per tile would use scalar loads, whose wait counter is shared with LDS and would
// stall the next LDS access on a memory round trip.
constexpr int kMaxChunk = 64;

__device__ __forceinline__ void stage_splits(int *s_split, const int *__restrict__ split_r,
                                             const int *__restrict__ split_a,
                                             const int *__restrict__ split_b, int t0, int t1) {
    const int n = t1 - t0 + 1;
    for (int i = threadIdx.x; i < n; i += kBlock) {
        s_split[3 * i] = split_r[t0 + i];
        s_split[3 * i + 1] = split_a[t0 + i];
        s_split[3 * i + 2] = split_b[t0 + i];
    }
}

// Every lane reads the same words, so the split is moved to scalar registers.
__device__ __forceinline__ TileSplit lds_split(const int *s_split, int i) {
    auto u = [&](int k) { return __builtin_amdgcn_readfirstlane(s_split[3 * i + k]); };
    return TileSplit{u(0), u(1), u(2), u(3), u(4), u(5)};
}

// A staged tile in LDS is one word array `s_cr` of n + 1 words, n = na + nb + (r1 - r0)
// (at most kTile + 1: the pair rule adds one B entry to a tile): A's coordinates at
// [0, na), B's at [na, na + nb), then the tile's row words s_row = s_cr + na + nb, where
// s_row[k] = (max(posA[r0+k], a0) - a0) | (max(posB[r0+k], b0) - b0) << 16 for k < nr =
// r1 - r0 + 1 (s_row[0] is 0: a0 and b0 lie in row r0).  Values, when the level has them, are
// in s_val at the coordinates' indices.  Entries and rows share the array because a tile's
// items are its entries plus its row ends: a tile of many short rows holds few entries.
//
// Slot k of the n staged words (k >= 1 for rows) is loaded into two registers: A's (or B's)
// coordinate and value bits, or row r0 + 1 + (k - na - nb)'s two offsets.  Lane `tid` loads
// slots tid + j * kBlock, j < kSlots, one tile ahead; slot kSlots * kBlock (a tile of
// kTile + 1 words) is loaded when the tile is staged.
constexpr int kSlots = kTile / kBlock;
constexpr int kCap = kTile + 2;  // n + 1 words
static_assert(kSlots * kBlock == kTile, "a tile is a whole number of slot rounds");

struct Slots {
    int x[kSlots];  // coordinate, or posA of a row
    int y[kSlots];  // value bits, or posB of a row
};

// Global addresses of slot k (0 <= k < n) of the tile `sp`: x from px[off], y from py[off].
__device__ __forceinline__ void slot_source(int k, const TileSplit &sp, int na, int nab,
                                            const int *__restrict__ pa,
                                            const int *__restrict__ ca, const int *__restrict__ va,
                                            const int *__restrict__ pb,
                                            const int *__restrict__ cb, const int *__restrict__ vb,
                                            const int *&px, const int *&py, int &off) {
    if (k < na) {
        px = ca;
        py = va;
        off = sp.a0 + k;
    } else if (k < nab) {
        px = cb;
        py = vb;
        off = sp.b0 + (k - na);
    } else {
        px = pa;
        py = pb;
        off = sp.r0 + 1 + (k - nab);
    }
}

// Loads are issued unconditionally (lanes past the end re-read the last slot) and nothing is
// computed from them until they are stored to LDS, so a whole tile's loads are in flight at
// once.
__device__ __forceinline__ void fetch_slots(Slots &st, const TileSplit &sp,
                                            const int *__restrict__ pa, const int *__restrict__ ca,
                                            const float *__restrict__ va,
                                            const int *__restrict__ pb, const int *__restrict__ cb,
                                            const float *__restrict__ vb, int tid) {
    const int na = sp.a1 - sp.a0, nab = na + (sp.b1 - sp.b0), n = nab + (sp.r1 - sp.r0);
    if (n == 0) return;  // uniform
    const int *vai = reinterpret_cast<const int *>(va);
    const int *vbi = reinterpret_cast<const int *>(vb);
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
        const int k = min(tid + j * kBlock, n - 1);
        const int *px, *py;
        int off;
        slot_source(k, sp, na, nab, pa, ca, vai, pb, cb, vbi, px, py, off);
        st.x[j] = px[off];
        st.y[j] = py[off];
    }
}

// Row-start bins: row k >= 1 of the tile starts at item
// x_k = (a0 + b0 + r0 - tile_lo) + ra_k + rb_k + k counted from the tile's lane grid
// tile_lo = tile * kTile, so it is the row of every lane L >= ceil(x_k / kItemsPerLane) until a
// later row starts.  It is recorded as atomicMax(s_bin[L], tag << 16 | k) for that first L
// (if L < kBlock); after a barrier, lane_first_row turns the bins into each lane's first row
// with one workgroup max-scan, replacing a per-lane binary search over the tile's rows.  The
// tag (distinct per staged tile of a workgroup, increasing) makes stale entries of earlier
// tiles lose every max and read as "no row", so the bins are never cleared.
__device__ __forceinline__ void stage_slot(int k, int x, int y, const TileSplit &sp, int nab,
                                           int *s_cr, float *s_val, unsigned *s_bin,
                                           unsigned tag, int tile_lo) {
    if (k < nab) {
        s_cr[k] = x;
        s_val[k] = __int_as_float(y);
    } else {
        const int kr = k - nab + 1;  // tile row
        const unsigned ra = static_cast<unsigned>(max(x, sp.a0) - sp.a0);
        const unsigned rb = static_cast<unsigned>(max(y, sp.b0) - sp.b0);
        s_cr[nab + kr] = static_cast<int>(ra | (rb << 16));
        const int xi = (sp.a0 + sp.b0 + sp.r0 - tile_lo) + static_cast<int>(ra + rb) + kr;
        const int lane = max(1, (xi + kItemsPerLane - 1) / kItemsPerLane);
        if (lane < kBlock) atomicMax(&s_bin[lane], (tag << 16) | static_cast<unsigned>(kr));
    }
}

__device__ __forceinline__ void stage_slots(const Slots &st, const TileSplit &sp, int *s_cr,
                                            float *s_val, int tid,
                                            const int *__restrict__ pa, const int *__restrict__ ca,
                                            const float *__restrict__ va,
                                            const int *__restrict__ pb, const int *__restrict__ cb,
                                            const float *__restrict__ vb,
                                            unsigned *s_bin, unsigned tag, int tile_lo) {
    const int na = sp.a1 - sp.a0, nab = na + (sp.b1 - sp.b0), n = nab + (sp.r1 - sp.r0);
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
        const int k = tid + j * kBlock;
        if (k < n) stage_slot(k, st.x[j], st.y[j], sp, nab, s_cr, s_val, s_bin, tag, tile_lo);
    }
    if (tid == 0) {
        s_cr[nab] = 0;  // row 0's word
        if (n > kSlots * kBlock) {  // the tile's last slot (rare): loaded now
            const int k = kSlots * kBlock;
            const int *px, *py;
            int off;
            slot_source(k, sp, na, nab, pa, ca, reinterpret_cast<const int *>(va), pb, cb,
                        reinterpret_cast<const int *>(vb), px, py, off);
            const int x = px[off];
            const int y = py[off];
            stage_slot(k, x, y, sp, nab, s_cr, s_val, s_bin, tag, tile_lo);
        }
    }
}

// This lane's first row (tile-local) from the row-start bins of the tile staged with `tag`
// (see stage_slot): the largest row recorded at or before this lane.  Call after the barrier
// that ends the staging.  No barrier: each wave reads the earlier waves' bins itself (at most
// three per lane) and takes their maximum along with its own running maximum.
__device__ __forceinline__ int lane_first_row(const unsigned *s_bin, unsigned tag, int tid) {
    auto row_at = [&](int i) {
        const unsigned v = s_bin[i];
        return (v >> 16) == tag ? static_cast<int>(v & 0xffffu) : 0;
    };
    const int w = tid / dev::kWave, l = tid % dev::kWave;
    int before = 0;
    for (int j = 0; j < w; ++j) before = max(before, row_at(j * dev::kWave + l));  // uniform
    before = __builtin_amdgcn_readlane(dev::wave_inclusive_max_dpp(before), dev::kWave - 1);
    return max(before, dev::wave_inclusive_max_dpp(row_at(tid)));
}

// ---- one lane's walk -------------------------------------------------------------------

// Result of walking a lane's items: outputs in registers (step s fills slot s when bit s of
// `valid` is set), the steps that were row ends, and the first row the lane touched.
template <int STEPS>
struct LaneOut {
    int crd[STEPS];
    float val[STEPS];
    unsigned valid, row_ends;
    int first_row;
};

// One lane's walk, from its first row (tile-local, given by the row-start bins): its split in
// the row is found by a merge-path search.
__device__ __forceinline__ void walk_lane(LaneOut<kItemsPerLane + 1> &out, const TileSplit &sp,
                                          int tile, const int *s_crd, const float *s_val,
                                          const unsigned *s_row, int tid, int row) {
    constexpr int kSteps = kItemsPerLane + 1;
    constexpr int kMax = INT_MAX;  // head sentinel: row exhausted on that side
    const int r0 = sp.r0, a0 = sp.a0, b0 = sp.b0, r1 = sp.r1, a1 = sp.a1, b1 = sp.b1;
    const int na = a1 - a0, nr = r1 - r0 + 1;
    auto A = [&](int x) { return s_crd[x - a0]; };
    auto B = [&](int y) { return s_crd[na + y - b0]; };
    auto row_a = [&](int k) { return a0 + static_cast<int>(s_row[k] & 0xffffu); };
    auto row_b = [&](int k) { return b0 + static_cast<int>(s_row[k] >> 16); };

    const int tile_lo = tile * kTile;
    const int tile_start = a0 + b0 + r0;  // item index of the tile's first item
    const int tile_end = a1 + b1 + r1;    // one past its last item
    const int g_lo = tid == 0 ? tile_start : tile_lo + tid * kItemsPerLane;
    const int steps = tid == kBlock - 1 ? tile_end - g_lo
                                        : min(tile_lo + (tid + 1) * kItemsPerLane, tile_end) - g_lo;
    int k = 0, a = a0, b = b0;
    if (tid > 0 && g_lo < tile_end) {
        k = row;
        const int aS = row_a(k), bS = row_b(k);
        const int aE = k < nr - 1 ? row_a(k + 1) : a1;
        const int bE = k < nr - 1 ? row_b(k + 1) : b1;
        const int D = g_lo - (r0 + k);
        int slo = max(aS, D - bE), shi = min(aE, D - bS);
        while (slo < shi) {
            const int mid = (slo + shi) >> 1;
            if (A(mid) <= B(D - 1 - mid)) {
                slo = mid + 1;
            } else {
                shi = mid;
            }
        }
        a = slo;
        b = D - slo;
    }
    out.first_row = r0 + k;
    // From here positions are indices into the staged arrays: A's entries at [0, na), B's at
    // [na, na + nb).  A tile holds at most kTile + 1 entries (the pair rule adds one), so
    // every index read below, one past a row's last entry included, is < kCap.
    const int nb = b1 - b0;
    auto end_a = [&](int kk) { return kk < nr - 1 ? static_cast<int>(s_row[kk + 1] & 0xffffu) : na; };
    auto end_b = [&](int kk) {
        return na + (kk < nr - 1 ? static_cast<int>(s_row[kk + 1] >> 16) : nb);
    };
    int ia = a - a0, ib = na + b - b0;
    int iae = end_a(k), ibe = end_b(k);
    int last_a = ia > static_cast<int>(s_row[k] & 0xffffu) ? s_crd[ia - 1] : -1;
    int xa = ia < iae ? s_crd[ia] : kMax;
    int xb = ib < ibe ? s_crd[ib] : kMax;
    unsigned valid = 0, row_ends = 0;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        out.crd[s] = 0;
        out.val[s] = 0.0f;
        if (s < steps) {
            if (xa == kMax && xb == kMax) {  // row end
                // (reads at indices always inside the staged arrays, then selects: no nested
                // branches, each waiting for its own read)
                row_ends |= 1u << s;
                ++k;
                const unsigned rn = s_row[min(k + 1, nr - 1)];
                const int ha = s_crd[ia], hb = s_crd[ib];
                const bool last_row = k >= nr - 1;
                iae = last_row ? na : static_cast<int>(rn & 0xffffu);
                ibe = na + (last_row ? nb : static_cast<int>(rn >> 16));
                last_a = -1;
                xa = ia < iae ? ha : kMax;
                xb = ib < ibe ? hb : kMax;
            } else {
                const bool take_a = xa <= xb;
                const bool pair = take_a && xa == xb;
                out.crd[s] = min(xa, xb);
                const float own = s_val[take_a ? ia : ib];
                const float vb = s_val[ib];  // read even when unpaired: no branch
                out.val[s] = pair ? own + vb : own;
                const bool emit = take_a || last_a != xb;
                valid |= static_cast<unsigned>(emit) << s;
                if (take_a) last_a = xa;
                ia += take_a;
                ib += !take_a;
                const int np = take_a ? ia : ib;  // reload the head that advanced
                const bool in = np < (take_a ? iae : ibe);
                const int h0 = s_crd[np];  // always read (np < kCap), then mask
                const int h = in ? h0 : kMax;
                xa = take_a ? h : xa;
                xb = take_a ? xb : h;
            }
        }
    }
    out.valid = valid;
    out.row_ends = row_ends;
}

// ---- kernels ---------------------------------------------------------------------------

// Chunk of tiles owned by workgroup w: [w*chunk, min((w+1)*chunk, num_tiles)).
__device__ __forceinline__ void chunk_range(int num_tiles, int chunk, int &t0, int &t1) {
    t0 = blockIdx.x * chunk;
    t1 = min(t0 + chunk, num_tiles);
}

template <int WAVES, typename T>
__device__ __forceinline__ T block_sum(T v, T *s_wave) {
    v = dev::wave_sum(v);
    if (dev::lane() == 0) s_wave[threadIdx.x / dev::kWave] = v;
    __syncthreads();
    T all = 0;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) all += s_wave[i];
    __syncthreads();
    return all;
}

// ---- pair count: the union's count pass ----------------------------------------------
//
// A union tile's output count is na + nb - pairs, and an equal A/B pair never straddles
// tiles, so the count pass only has to find the pairs.  In every row of the tile where both
// operands have entries, each entry of the side with fewer entries (A on a tie) is searched
// in the other side's range of the row (binary search in LDS).  Rows where one side is empty
// cost only their offsets; a row heavy in one operand costs the light side's entries times
// log2 of the heavy side's length.  At C2 (Zipf rows, independent operands) that is 2.4e5
// searches for 3.4e7 items.
//
// Staging reads 16-byte granules: the tile's A range then its B range of coordinates, each
// cut at its array's 16-byte boundaries (a granule holding one element of the range lies in
// the same page as that element, so reading all of it never leaves mapped memory; the extra
// elements are never used), and the row offsets of up to kRowBlock + 1 rows per pass.

// Offset of each array's base address from a 16-byte boundary, in elements (0..3).
struct Misalign {
    int ca, cb, pa, pb;
};

// A 16-byte granule as a native vector (HIP's int4 is a struct over a union, which keeps
// arrays of it in scratch memory).
typedef int grain_t __attribute__((ext_vector_type(4)));

constexpr int kGrains = 4;      // coordinate granules per lane: 4096 entries >= tile + padding
constexpr int kRowGrains = 2;   // row-offset granules per lane per operand: 2048 offsets
constexpr int kRowBlock = kRowGrains * 4 * kBlock - 4;  // rows per pass (their ends included)
constexpr int kGrainCap = kGrains * 4 * kBlock;

__device__ __forceinline__ int grain_first(int lo, int mis) { return ((lo + mis) & ~3) - mis; }
__device__ __forceinline__ int grain_count(int lo, int hi, int mis) {
    return hi > lo ? (hi - grain_first(lo, mis) + 3) >> 2 : 0;
}

// Where a tile's coordinates land in LDS: granule q at s[4q .. 4q + 3], A's granules first;
// A's entry a0 at index offA, B's entry b0 at offB.
struct GrainLayout {
    int firstA, nga, firstB, ngb, offA, offB;
};

__device__ __forceinline__ GrainLayout grain_layout(const TileSplit &sp, int misA, int misB) {
    GrainLayout g;
    g.firstA = grain_first(sp.a0, misA);
    g.nga = grain_count(sp.a0, sp.a1, misA);
    g.firstB = grain_first(sp.b0, misB);
    g.ngb = grain_count(sp.b0, sp.b1, misB);
    g.offA = sp.a0 - g.firstA;
    g.offB = 4 * g.nga + (sp.b0 - g.firstB);
    return g;
}

struct TileGrains {
    grain_t v[kGrains];
};

// Loads are issued unconditionally (lanes past the end re-read the last granule) so that a
// whole tile's loads are in flight at once.
__device__ __forceinline__ void fetch_grains(TileGrains &tg, const GrainLayout &g,
                                             const int *__restrict__ xa,
                                             const int *__restrict__ xb, int tid) {
    const int n = g.nga + g.ngb;
    if (n == 0) return;  // uniform
#pragma unroll
    for (int j = 0; j < kGrains; ++j) {
        const int q = min(tid + j * kBlock, n - 1);
        const int *src = q < g.nga ? xa + g.firstA + 4 * q : xb + g.firstB + 4 * (q - g.nga);
        tg.v[j] = *reinterpret_cast<const grain_t *>(src);
    }
}

__device__ __forceinline__ void store_grains(const TileGrains &tg, const GrainLayout &g,
                                             int *s, int tid) {
    const int n = g.nga + g.ngb;
#pragma unroll
    for (int j = 0; j < kGrains; ++j) {
        const int q = tid + j * kBlock;
        if (q < n) *reinterpret_cast<grain_t *>(s + 4 * q) = tg.v[j];
    }
}

// Row offsets of rows [lo, hi) of both operands (at most kRowBlock + 1 rows).
struct RowGrains {
    grain_t a[kRowGrains], b[kRowGrains];
};

__device__ __forceinline__ void fetch_row_grains(RowGrains &rg, const int *__restrict__ pa,
                                                 const int *__restrict__ pb, int lo, int hi,
                                                 const Misalign &mis, int tid) {
    const int fa = grain_first(lo, mis.pa), na = grain_count(lo, hi, mis.pa);
    const int fb = grain_first(lo, mis.pb), nb = grain_count(lo, hi, mis.pb);
#pragma unroll
    for (int j = 0; j < kRowGrains; ++j) {
        const int qa = min(tid + j * kBlock, na - 1), qb = min(tid + j * kBlock, nb - 1);
        rg.a[j] = *reinterpret_cast<const grain_t *>(pa + fa + 4 * qa);
        rg.b[j] = *reinterpret_cast<const grain_t *>(pb + fb + 4 * qb);
    }
}

// Tile-local starts of rows [lo, hi): s_ra[k] = max(pa[lo + k] - a0, 0), likewise s_rb.
__device__ __forceinline__ void store_row_grains(const RowGrains &rg, int lo, int hi,
                                                 const Misalign &mis, int a0, int b0,
                                                 unsigned short *s_ra, unsigned short *s_rb,
                                                 int tid) {
    const int fa = grain_first(lo, mis.pa), fb = grain_first(lo, mis.pb);
    const int n = hi - lo;
#pragma unroll
    for (int j = 0; j < kRowGrains; ++j) {
        const int q = tid + j * kBlock;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int ka = fa + 4 * q + e - lo, kb = fb + 4 * q + e - lo;
            if (ka >= 0 && ka < n) s_ra[ka] = static_cast<unsigned short>(max(rg.a[j][e] - a0, 0));
            if (kb >= 0 && kb < n) s_rb[kb] = static_cast<unsigned short>(max(rg.b[j][e] - b0, 0));
        }
    }
}

// LDS of the pair count.
struct PairShared {
    int crd[kGrainCap];
    unsigned short ra[kRowBlock + 4], rb[kRowBlock + 4];
    int mpre[kRowBlock + 1];
    int wave[kBlock / dev::kWave];
    unsigned wsum[kBlock / dev::kWave];
};

// Running totals of a pair-count workgroup.
struct PairTotals {
    unsigned found;    // this lane's pairs since the last flush
    unsigned entries;  // entries of both operands since the last flush (uniform)
    unsigned total;    // the workgroup's output count (thread 0)
};

// One tile of the pair count: stage it from registers (tg, rg), refill the registers with
// tile `t_next`'s loads (split `nsp`, if `has_next`), then count its pairs.
__device__ __forceinline__ void pair_tile(
    PairShared &sh, int t, int t_last, const TileSplit &sp, const GrainLayout &g,
    TileGrains &tg, RowGrains &rg, bool has_next, const TileSplit &nsp,
    const int *__restrict__ pa, const int *__restrict__ ca, const int *__restrict__ pb,
    const int *__restrict__ cb, const Misalign &mis, int write_chunk,
    unsigned *__restrict__ chunk_count, PairTotals &acc, int tid) {
    const int na = sp.a1 - sp.a0, nb = sp.b1 - sp.b0, nr = sp.r1 - sp.r0 + 1;
    const int offA = g.offA, offB = g.offB;
    store_grains(tg, g, sh.crd, tid);
    store_row_grains(rg, sp.r0, min(sp.r0 + kRowBlock + 1, sp.r1 + 1), mis, sp.a0, sp.b0, sh.ra,
                     sh.rb, tid);
    if (has_next) {  // uniform: tile t_next's loads, in flight during the next two tiles
        const GrainLayout ng = grain_layout(nsp, mis.ca, mis.cb);
        fetch_grains(tg, ng, ca, cb, tid);
        fetch_row_grains(rg, pa, pb, nsp.r0, min(nsp.r0 + kRowBlock + 1, nsp.r1 + 1), mis, tid);
    }
    // this lane's first item in the write kernel, relative to the tile's first item
    const int tile_start = sp.a0 + sp.b0 + sp.r0, tile_end = sp.a1 + sp.b1 + sp.r1;
    const int g_lo = tid == 0 ? tile_start : t * kTile + tid * kItemsPerLane;
    const int rel = g_lo - tile_start;
    // this lane's items in the write kernel (for the walk count)
    const int steps = tid == kBlock - 1
                          ? tile_end - g_lo
                          : min(t * kTile + (tid + 1) * kItemsPerLane, tile_end) - g_lo;
    __syncthreads();
    for (int kb = 0; kb < nr; kb += kRowBlock) {  // one pass unless nr > kRowBlock
        const int nrb = min(kRowBlock, nr - kb);
        if (kb > 0) {
            // Further rows of a tile with more than kRowBlock rows: staged here, with plain
            // loads (rare: such a tile holds few entries).
            __syncthreads();
            const int cnt = min(nrb + 1, nr - kb);
            for (int k = tid; k < cnt; k += kBlock) {
                sh.ra[k] = static_cast<unsigned short>(max(pa[sp.r0 + kb + k] - sp.a0, 0));
                sh.rb[k] = static_cast<unsigned short>(max(pb[sp.r0 + kb + k] - sp.b0, 0));
            }
            __syncthreads();
        }
        // Per row: searches to do = the smaller side's entries when both sides have some.
        constexpr int kR = (kRowBlock + kBlock - 1) / kBlock;
        const int per = (nrb + kBlock - 1) / kBlock;  // rows per lane, contiguous
        int m[kR];
        int mine = 0;
#pragma unroll
        for (int i = 0; i < kR; ++i) {
            m[i] = 0;
            const int k = tid * per + i;
            if (i < per && k < nrb) {
                const bool last = kb + k + 1 == nr;
                const int la = (last ? na : sh.ra[k + 1]) - sh.ra[k];
                const int lb = (last ? nb : sh.rb[k + 1]) - sh.rb[k];
                m[i] = (la > 0 && lb > 0) ? min(la, lb) : 0;
                mine += m[i];
            }
        }
        int work = 0;
        int run = dev::block_exclusive_sum<kBlock, int, false>(mine, sh.wave, work);
#pragma unroll
        for (int i = 0; i < kR; ++i) {
            const int k = tid * per + i;
            if (i < per && k < nrb) sh.mpre[k] = run;
            run += m[i];
        }
        __syncthreads();
        // Tiles with many searches (both operands dense in the same rows) count their pairs
        // with a merge walk of each lane's write-kernel items instead (single-pass tiles).
        const bool walk = nr <= kRowBlock && work >= kWalkMin;
        for (int j = walk ? work : tid; j < work; j += kBlock) {
            int lo = 0, hi = nrb - 1;  // the row: last k with mpre[k] <= j
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (sh.mpre[mid] <= j) {
                    lo = mid;
                } else {
                    hi = mid - 1;
                }
            }
            const int k = lo;
            const bool last = kb + k + 1 == nr;
            const int sa = sh.ra[k], ea = last ? na : sh.ra[k + 1];
            const int sb = sh.rb[k], eb = last ? nb : sh.rb[k + 1];
            const int nth = j - sh.mpre[k];
            int x, base, l, h;
            if (ea - sa <= eb - sb) {
                x = sh.crd[offA + sa + nth];
                base = offB;
                l = sb;
                h = eb;
            } else {
                x = sh.crd[offB + sb + nth];
                base = offA;
                l = sa;
                h = ea;
            }
            const int end = h;
            while (l < h) {  // first position >= x
                const int mid = (l + h) >> 1;
                if (sh.crd[base + mid] < x) {
                    l = mid + 1;
                } else {
                    h = mid;
                }
            }
            acc.found += (l < end && sh.crd[base + l] == x) ? 1u : 0u;
        }
        // The write kernel's start of this lane: the row (last k whose first item is at or
        // before it), then the merge-path split of the row's A and B entries before it (ties:
        // A first).
        if (walk && g_lo < tile_end) {
            int lo = 0, hi = nrb - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (sh.ra[mid] + sh.rb[mid] + kb + mid <= rel) {
                    lo = mid;
                } else {
                    hi = mid - 1;
                }
            }
            const int k = lo;
            const bool last = kb + k + 1 == nr;
            const int aS = sh.ra[k], aE = last ? na : sh.ra[k + 1];
            const int bS = sh.rb[k], bE = last ? nb : sh.rb[k + 1];
            const int D = rel - (kb + k);  // entries of the tile before the item
            int slo = max(aS, D - bE), shi = min(aE, D - bS);
            while (slo < shi) {
                const int mid = (slo + shi) >> 1;
                if (sh.crd[offA + mid] <= sh.crd[offB + D - 1 - mid]) {
                    slo = mid + 1;
                } else {
                    shi = mid;
                }
            }
            {  // (kb == 0) count the pairs among this lane's items: a pair at its A
                constexpr int kEnd = INT_MAX;  // head of an exhausted row side
                auto end_a = [&](int r) { return r + 1 < nr ? static_cast<int>(sh.ra[r + 1]) : na; };
                auto end_b = [&](int r) { return r + 1 < nr ? static_cast<int>(sh.rb[r + 1]) : nb; };
                int r = k, ia = slo, ib = D - slo;
                int iae = end_a(r), ibe = end_b(r);
                int xa = ia < iae ? sh.crd[offA + ia] : kEnd;
                int xb = ib < ibe ? sh.crd[offB + ib] : kEnd;
                unsigned pairs = 0;
                // (reads at indices inside the staged arrays, then selects: no nested
                // branches, each waiting for its own read)
                auto crd_at = [&](int x) { return sh.crd[min(x, kGrainCap - 1)]; };
#pragma unroll
                for (int st = 0; st < kItemsPerLane + 1; ++st) {
                    if (st < steps) {
                        if (xa == kEnd && xb == kEnd) {  // row end
                            ++r;
                            const int rn = min(r + 1, nr - 1);
                            const int an = sh.ra[rn], bn = sh.rb[rn];
                            const int ha = crd_at(offA + ia), hb = crd_at(offB + ib);
                            const bool last_row = r + 1 >= nr;
                            iae = last_row ? na : an;
                            ibe = last_row ? nb : bn;
                            xa = ia < iae ? ha : kEnd;
                            xb = ib < ibe ? hb : kEnd;
                        } else {
                            const bool take_a = xa <= xb;
                            pairs += (take_a && xa == xb) ? 1u : 0u;
                            ia += take_a;
                            ib += !take_a;
                            const bool in = take_a ? ia < iae : ib < ibe;
                            const int h0 = crd_at(take_a ? offA + ia : offB + ib);
                            const int h = in ? h0 : kEnd;
                            xa = take_a ? h : xa;
                            xb = take_a ? xb : h;
                        }
                    }
                }
                acc.found += pairs;
            }
        }
    }
    acc.entries += static_cast<unsigned>(na + nb);
    if (t == t_last || (t + 1) % write_chunk == 0) {  // uniform: end of a write chunk
        const unsigned pairs = block_sum<kBlock / dev::kWave>(acc.found, sh.wsum);
        if (tid == 0) {
            const unsigned c = acc.entries - pairs;
            atomicAdd(&chunk_count[t / write_chunk], c);
            acc.total += c;
        }
        acc.found = 0;
        acc.entries = 0;
    }
    __syncthreads();  // every lane is done with this tile's LDS
}

// Output counts of a union level (na + nb - pairs per tile), added into
// chunk_count[tile / write_chunk] (zeroed by the partition kernel): the counts of the write
// kernel's chunks, whose grid is chosen independently of this kernel's (`chunk` tiles per
// workgroup here, two tiles in flight).  Their sum, the result length, goes to `length_out`
// from the last workgroup.
__global__ __launch_bounds__(kBlock) void pair_count_kernel(
    const int *__restrict__ pa, const int *__restrict__ ca, const int *__restrict__ pb,
    const int *__restrict__ cb, Misalign mis, int num_tiles, int chunk, int write_chunk,
    const int *__restrict__ split_r, const int *__restrict__ split_a,
    const int *__restrict__ split_b, unsigned *__restrict__ chunk_count,
    unsigned long long *__restrict__ done, int64_t *__restrict__ length_out) {
    __shared__ PairShared sh;
    __shared__ int s_split[3 * (kMaxChunk + 1)];

    const int tid = threadIdx.x;
    int t0, t1;
    chunk_range(num_tiles, chunk, t0, t1);
    if (t0 >= t1) {
        if (tid == 0) dev::add_to_total(0u, done, length_out);
        return;
    }
    stage_splits(s_split, split_r, split_a, split_b, t0, t1);
    __syncthreads();
    // Two tiles in flight: tiles t0 + 2i go through (tg0, rg0), t0 + 2i + 1 through (tg1, rg1).
    TileGrains tg0, tg1;
    RowGrains rg0, rg1;
    TileSplit sp0 = lds_split(s_split, 0);
    TileSplit sp1 = lds_split(s_split, t0 + 1 < t1 ? 1 : 0);
    GrainLayout g0 = grain_layout(sp0, mis.ca, mis.cb);
    GrainLayout g1 = grain_layout(sp1, mis.ca, mis.cb);
    fetch_grains(tg0, g0, ca, cb, tid);
    fetch_row_grains(rg0, pa, pb, sp0.r0, min(sp0.r0 + kRowBlock + 1, sp0.r1 + 1), mis, tid);
    if (t0 + 1 < t1) {
        fetch_grains(tg1, g1, ca, cb, tid);
        fetch_row_grains(rg1, pa, pb, sp1.r0, min(sp1.r0 + kRowBlock + 1, sp1.r1 + 1), mis, tid);
    }
    PairTotals acc{0u, 0u, 0u};
    for (int t = t0; t < t1; t += 2) {
        const bool n0 = t + 2 < t1, n1 = t + 3 < t1;
        const TileSplit nsp0 = lds_split(s_split, n0 ? t + 2 - t0 : 0);
        pair_tile(sh, t, t1 - 1, sp0, g0, tg0, rg0, n0, nsp0, pa, ca, pb, cb, mis, write_chunk,
                  chunk_count, acc, tid);
        sp0 = nsp0;
        g0 = grain_layout(sp0, mis.ca, mis.cb);
        if (t + 1 < t1) {
            const TileSplit nsp1 = lds_split(s_split, n1 ? t + 3 - t0 : 0);
            pair_tile(sh, t + 1, t1 - 1, sp1, g1, tg1, rg1, n1, nsp1, pa, ca, pb, cb, mis,
                      write_chunk, chunk_count, acc, tid);
            sp1 = nsp1;
            g1 = grain_layout(sp1, mis.ca, mis.cb);
        }
    }
    if (tid == 0) dev::add_to_total(acc.total, done, length_out);
}

// Writes the result's pos, crd and val.  Every lane finds its start from the tile's row-start
// bins and a search inside its row.
__global__ __launch_bounds__(kBlock) void walk_write_kernel(
    const int *__restrict__ pa, const int *__restrict__ ca, const float *__restrict__ va,
    const int *__restrict__ pb, const int *__restrict__ cb, const float *__restrict__ vb,
    int num_tiles, int chunk, const int *__restrict__ split_r, const int *__restrict__ split_a,
    const int *__restrict__ split_b, const unsigned *__restrict__ chunk_count,
    int *__restrict__ pc, int *__restrict__ cc, float *__restrict__ vc) {
    constexpr int kSteps = kItemsPerLane + 1;
    constexpr int kLoads = (kCap + kBlock - 1) / kBlock;  // outputs per lane in the stores
    __shared__ int s_cr[kCap];  // coordinates then row words (see slot staging)
    __shared__ float s_val[kCap];
    __shared__ int s_wave[kBlock / dev::kWave];
    __shared__ int s_split[3 * (kMaxChunk + 1)];
    __shared__ unsigned s_bin[kBlock];  // row-start bins (see stage_slot)

    const int tid = threadIdx.x;
    int t0, t1;
    chunk_range(num_tiles, chunk, t0, t1);
    if (t0 >= t1) return;
    s_bin[tid] = 0u;
    stage_splits(s_split, split_r, split_a, split_b, t0, t1);

    // Offset of this chunk: the counts of every earlier chunk.
    int before = 0, base = 0;
    for (int i = tid; i < static_cast<int>(blockIdx.x); i += kBlock) before += chunk_count[i];
    (void)dev::block_exclusive_sum<kBlock>(before, s_wave, base);
    if (blockIdx.x == 0 && tid == 0) pc[0] = 0;

    TileSplit sp = lds_split(s_split, 0);  // (the exclusive sum above ended with a barrier)
    Slots st;
    fetch_slots(st, sp, pa, ca, va, pb, cb, vb, tid);
    stage_slots(st, sp, s_cr, s_val, tid, pa, ca, va, pb, cb, vb, s_bin, 1u, t0 * kTile);
    __syncthreads();
    TileSplit nsp = lds_split(s_split, t0 + 1 < t1 ? 1 : 0);
    int row = lane_first_row(s_bin, 1u, tid);
    for (int t = t0; t < t1; ++t) {
        fetch_slots(st, nsp, pa, ca, va, pb, cb, vb, tid);
        const TileSplit nsp2 = lds_split(s_split, t + 2 < t1 ? t + 2 - t0 : t + 1 < t1 ? t + 1 - t0 : t - t0);
        LaneOut<kSteps> lo;
        const unsigned *s_row =
            reinterpret_cast<const unsigned *>(s_cr) + (sp.a1 - sp.a0) + (sp.b1 - sp.b0);
        walk_lane(lo, sp, t, s_cr, s_val, s_row, tid, row);

        int tile_total = 0;
        // (the scan's barrier also means every lane is done reading this tile's LDS inputs;
        // s_wave is next written after this tile's later barriers)
        const int offset = dev::block_exclusive_sum<kBlock, int, false>(
            static_cast<int>(__popc(lo.valid)), s_wave, tile_total);

        int o = offset, r = lo.first_row;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            if (lo.row_ends & (1u << s)) {
                pc[r + 1] = base + o;
                ++r;
            }
            if (lo.valid & (1u << s)) {
                s_cr[o] = lo.crd[s];
                s_val[o] = lo.val[s];
                ++o;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int q = tid + j * kBlock;
            if (q < tile_total) {
                cc[base + q] = s_cr[q];
                vc[base + q] = s_val[q];
            }
        }
        base += tile_total;
        __syncthreads();  // staged outputs consumed
        if (t + 1 < t1) {
            const unsigned tag = static_cast<unsigned>(t + 2 - t0);
            stage_slots(st, nsp, s_cr, s_val, tid, pa, ca, va, pb, cb, vb, s_bin, tag,
                        (t + 1) * kTile);
            __syncthreads();
            row = lane_first_row(s_bin, tag, tid);
        }
        sp = nsp;
        nsp = nsp2;
    }
}

// ---- host ------------------------------------------------------------------------------

// Offset of an int32 array's base from a 16-byte boundary, in elements; int32 arrays must
// be 4-byte aligned.  A null (empty) array counts as aligned.
int misalign(const void *p, int *out) {
    const uintptr_t v = reinterpret_cast<uintptr_t>(p);
    if (v & 3u) return NACHO_ERR_INVALID_ARGUMENT;
    *out = static_cast<int>((v & 15u) >> 2);
    return NACHO_OK;
}

// The union of the allocation-free csr_add: scratch of a few bytes per tile from `call`'s
// arena.
int walk_union(Call &call, int rows, const LevelOperand &A, const LevelOperand &B,
               const LevelResult &Z, long long *out_len) {
    const long long total = static_cast<long long>(A.len) + B.len + rows;
    const int num_tiles = total > 0 ? static_cast<int>((total + kTile - 1) / kTile) : 1;
    int *splits = nullptr;
    unsigned *counts = nullptr;
    NACHO_TRY(call.scratch_n(3 * (static_cast<size_t>(num_tiles) + 1), &splits));
    int *split_r = splits, *split_a = splits + num_tiles + 1, *split_b = splits + 2 * (num_tiles + 1);
    // Grids: as many workgroups of a kernel as stay resident, each owning a contiguous chunk
    // of tiles.
    int resident = 0, count_resident = 0;
    NACHO_TRY(resident_grid(reinterpret_cast<const void *>(walk_write_kernel), kBlock, &resident));
    NACHO_TRY(resident_grid(reinterpret_cast<const void *>(pair_count_kernel), kBlock,
                            &count_resident));
    // (more workgroups than resident when a chunk reaches kMaxChunk: still correct)
    const int chunk = std::min((num_tiles + resident - 1) / resident, kMaxChunk);
    const int count_chunk = std::min((num_tiles + count_resident - 1) / count_resident, kMaxChunk);
    const int grid = (num_tiles + chunk - 1) / chunk;
    const int count_grid = (num_tiles + count_chunk - 1) / count_chunk;
    NACHO_TRY(call.scratch_n(static_cast<size_t>(grid) + 4 + 2 * dev::kTotalWords, &counts));
    // 64-bit accumulator of the length total (8-byte aligned words after the counts).
    unsigned long long *done =
        reinterpret_cast<unsigned long long *>(counts + ((grid + 2) & ~1));
    int64_t *length_out = nullptr;
    NACHO_TRY(call.length_word(&length_out));
    Misalign mis{};
    NACHO_TRY(misalign(A.crd, &mis.ca));
    NACHO_TRY(misalign(B.crd, &mis.cb));
    NACHO_TRY(misalign(A.pos, &mis.pa));
    NACHO_TRY(misalign(B.pos, &mis.pb));
    const hipStream_t s = call.stream();
    csr_partition_kernel<kTile><<<partition_blocks(num_tiles), kPartBlock, 0, s>>>(
        A.pos, A.crd, B.pos, B.crd, rows, static_cast<int>(total), num_tiles, split_r, split_a,
        split_b, done, counts, grid, 1);
    NACHO_TRY_HIP(hipGetLastError());
    pair_count_kernel<<<count_grid, kBlock, 0, s>>>(A.pos, A.crd, B.pos, B.crd, mis, num_tiles,
                                                    count_chunk, chunk, split_r, split_a,
                                                    split_b, counts, done, length_out);
    NACHO_TRY_HIP(hipGetLastError());
    NACHO_TRY(call.mark_length());
    walk_write_kernel<<<grid, kBlock, 0, s>>>(A.pos, A.crd, A.val, B.pos, B.crd, B.val, num_tiles,
                                              chunk, split_r, split_a, split_b, counts, Z.pos,
                                              Z.crd, Z.val);
    NACHO_TRY_HIP(hipGetLastError());
    int64_t len = 0;
    NACHO_TRY(call.wait_length(&len));
    *out_len = len;
    return NACHO_OK;
}

// Bytes of scratch walk_union takes for `items` merge items (entries of both operands plus
// rows).
size_t walk_arena_bytes(long long items) {
    const long long tiles = items > 0 ? (items + kTile - 1) / kTile : 1;
    // splits (3 per boundary), chunk counts (at most one per tile) plus the ticket words,
    // the length word, and 256-byte alignment of each piece
    return static_cast<size_t>(12 * (tiles + 1) + 4 * (tiles + 6) + 8 * dev::kTotalWords + 8 +
                               4 * 256);
}

}  // namespace

bool bad_csr(const nacho_csr *t) {
    if (!t || t->dim_i_size < 0 || t->dim_j_size < 0 || t->dim_j_length < 0) return true;
    if (!t->dim_j_offsets) return true;
    if (t->dim_j_length > 0 && (!t->dim_j_indices || !t->values)) return true;
    return false;
}

int csr_binary(bool intersect, const nacho_csr *a, const nacho_csr *b, nacho_csr *z,
               int32_t num_blocks, int32_t threads_per_block, void *stream,
               const nacho_allocator *alloc, const char *kernel_name) {
    if (!z) return NACHO_ERR_INVALID_ARGUMENT;
    *z = nacho_csr{};
    NACHO_TRY(check_launch_hints(num_blocks, threads_per_block));
    if (bad_csr(a) || bad_csr(b)) return NACHO_ERR_INVALID_ARGUMENT;
    if (a->dim_i_size != b->dim_i_size || a->dim_j_size != b->dim_j_size) {
        return NACHO_ERR_INVALID_ARGUMENT;
    }
    const int rows = a->dim_i_size;
    const long long nnz_a = a->dim_j_length, nnz_b = b->dim_j_length;
    if (nnz_a + nnz_b + rows > static_cast<long long>(INT_MAX) - 2 * kTile) {
        return NACHO_ERR_INDEX_OVERFLOW;
    }
    const long long cap = intersect ? (nnz_a < nnz_b ? nnz_a : nnz_b) : nnz_a + nnz_b;

    Call call(stream, alloc);
    int *pc = nullptr, *cc = nullptr;
    float *vc = nullptr;
    NACHO_TRY(call.result_n(static_cast<size_t>(rows) + 1, &pc));
    NACHO_TRY(call.result_n(static_cast<size_t>(cap), &cc));
    NACHO_TRY(call.result_n(static_cast<size_t>(cap), &vc));

    const LevelOperand A{a->dim_j_offsets, a->dim_j_indices, a->values, a->dim_j_length, nullptr};
    const LevelOperand B{b->dim_j_offsets, b->dim_j_indices, b->values, b->dim_j_length, nullptr};
    const LevelResult Z{pc, cc, vc, nullptr, nullptr};
    long long nnz = 0;
    NACHO_TRY(merge_level(call, intersect, true, false, rows, extent_bits(a->dim_j_size), A, B, Z,
                          &nnz, kernel_name));
    if (nnz > cap) return NACHO_ERR_MALFORMED_INPUT;
    if (nnz == 0) {
        // Empty result: zeroed offsets, no coordinate/value buffers
        // (stitch_and_generate.cpp:168-220 for the intersection early exit).
        call.drop_result(cc);
        call.drop_result(vc);
        cc = nullptr;
        vc = nullptr;
    }
    z->dim_i_size = rows;
    z->dim_j_size = a->dim_j_size;
    z->dim_j_offsets = pc;
    z->dim_j_length = static_cast<int32_t>(nnz);
    z->dim_j_indices = cc;
    z->values = vc;
    z->nnz = static_cast<int32_t>(nnz);
    call.commit();
    return NACHO_OK;
}

// ---- allocation-free csr_add ------------------------------------------------------------
// Scratch of nacho_gpu_csr_add_f32_noalloc: a file-scope device array, one copy per GPU,
// held for the life of the process.  Host code never passes `scratch` itself to a kernel
// (in host code the name is a stand-in, not a device address): it looks up each device's
// address once with hipGetSymbolAddress and uses that.
constexpr size_t kNoAllocScratchBytes = size_t{8} << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;

// One GPU's `scratch`: its device address (looked up on the first call there) and the lock
// that one call holds from its first launch until its last kernel has finished.
struct ScratchSlot {
    std::mutex busy;
    void *address = nullptr;
};

int scratch_slot(ScratchSlot **out) {
    static std::mutex lookup;
    static ScratchSlot slots[kMaxDevices];
    int device = 0;
    NACHO_TRY_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) return NACHO_ERR_INVALID_ARGUMENT;
    std::lock_guard<std::mutex> lock(lookup);
    ScratchSlot &slot = slots[device];
    if (!slot.address) {
        void *p = nullptr;
        NACHO_TRY_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return NACHO_ERR_INTERNAL;
        slot.address = p;
    }
    *out = &slot;
    return NACHO_OK;
}

// Waits for the stream when the call leaves, on every exit path, so that no kernel of the
// call still reads `scratch` once the slot's lock is released.
struct StreamDrain {
    hipStream_t stream;
    ~StreamDrain() { (void)hipStreamSynchronize(stream); }
};

int csr_add_noalloc(const nacho_csr *a, const nacho_csr *b, nacho_csr *z, int32_t num_blocks,
                    int32_t threads_per_block, void *stream) {
    if (!z) return NACHO_ERR_INVALID_ARGUMENT;
    int *pc = z->dim_j_offsets, *cc = z->dim_j_indices;
    float *vc = z->values;
    const long long capacity = z->dim_j_length;
    z->dim_j_length = 0;
    z->nnz = 0;
    NACHO_TRY(check_launch_hints(num_blocks, threads_per_block));
    if (bad_csr(a) || bad_csr(b)) return NACHO_ERR_INVALID_ARGUMENT;
    if (a->dim_i_size != b->dim_i_size || a->dim_j_size != b->dim_j_size) {
        return NACHO_ERR_INVALID_ARGUMENT;
    }
    const int rows = a->dim_i_size;
    const long long nnz_a = a->dim_j_length, nnz_b = b->dim_j_length;
    const long long items = nnz_a + nnz_b + rows;
    if (items > static_cast<long long>(INT_MAX) - 2 * kTile) return NACHO_ERR_INDEX_OVERFLOW;
    if (!pc || capacity < nnz_a + nnz_b || (capacity > 0 && (!cc || !vc))) {
        return NACHO_ERR_INVALID_ARGUMENT;
    }
    if (items > NACHO_NOALLOC_MAX_ITEMS) return NACHO_ERR_SCRATCH_TOO_SMALL;
    if (walk_arena_bytes(items) > kNoAllocScratchBytes) return NACHO_ERR_INTERNAL;
    ScratchSlot *slot = nullptr;
    NACHO_TRY(scratch_slot(&slot));
    // Calls on one GPU take turns: the lock is held until the call's kernels have drained
    // (StreamDrain runs after Call's destructor, before the lock is released).
    std::lock_guard<std::mutex> hold(slot->busy);
    StreamDrain drain{static_cast<hipStream_t>(stream)};
    Call call(stream, slot->address, kNoAllocScratchBytes);
    const LevelOperand A{a->dim_j_offsets, a->dim_j_indices, a->values, a->dim_j_length, nullptr};
    const LevelOperand B{b->dim_j_offsets, b->dim_j_indices, b->values, b->dim_j_length, nullptr};
    const LevelResult Z{pc, cc, vc, nullptr, nullptr};
    long long nnz = 0;
    NACHO_TRY(walk_union(call, rows, A, B, Z, &nnz));
    if (nnz > nnz_a + nnz_b) return NACHO_ERR_MALFORMED_INPUT;
    z->dim_i_size = rows;
    z->dim_j_size = a->dim_j_size;
    z->dim_j_length = static_cast<int32_t>(nnz);
    z->nnz = static_cast<int32_t>(nnz);
    return NACHO_OK;
}

}  // namespace csr
}  // namespace nacho

extern "C" {

int nacho_gpu_csr_add_f32_noalloc(const nacho_csr *a, const nacho_csr *b, nacho_csr *z,
                                  int32_t num_blocks, int32_t threads_per_block,
                                  void *stream) {
    return nacho::csr::csr_add_noalloc(a, b, z, num_blocks, threads_per_block, stream);
}


int nacho_gpu_csr_add_f32(const nacho_csr *a, const nacho_csr *b, nacho_csr *z,
                          int32_t num_blocks, int32_t threads_per_block, void *stream,
                          const nacho_allocator *alloc) {
    return nacho::csr::csr_binary(false, a, b, z, num_blocks, threads_per_block, stream, alloc,
                                  "csr_add: partition+count+write");
}

int nacho_gpu_csr_mul_f32(const nacho_csr *a, const nacho_csr *b, nacho_csr *z,
                          int32_t num_blocks, int32_t threads_per_block, void *stream,
                          const nacho_allocator *alloc) {
    return nacho::csr::csr_binary(true, a, b, z, num_blocks, threads_per_block, stream, alloc,
                                  "csr_mul: partition+count+write");
}

}  // extern "C"
