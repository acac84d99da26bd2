// Tile boundaries of a merged row sequence, shared by the level merge (level_merge.hip) and
// the allocation-free csr_add (csr_merge.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "device_utils.hpp"
#include "runtime.hpp"

namespace nacho {
namespace csr {

constexpr int kPartBlock = 64;  // threads per workgroup of the partition kernel
// Lanes that search one tile boundary together: each round of the searches costs one
// dependent load and narrows the range (kPartLanes + 1)-fold; wider groups spend more
// divergent loads per round.
constexpr int kPartLanes = 8;

inline int partition_blocks(int num_tiles) {
    return static_cast<int>(
        ceil_div((static_cast<size_t>(num_tiles) + 1) * kPartLanes, kPartBlock));
}

// The work is the merged sequence of every row's A entries, B entries and one row-end item,
// cut into tiles.  G lanes together find the split of diagonal `diag`: its row, then the
// merge-path split inside the row (ties: A first).  An equal A/B pair is never split across
// tiles: the boundary takes its B entry too (the reference's balancing step,
// partition.cpp:964-983), so a tile holds at most one entry more than its items.
template <int G>
__device__ __forceinline__ void find_split(const int *__restrict__ pa,
                                           const int *__restrict__ ca,
                                           const int *__restrict__ pb,
                                           const int *__restrict__ cb, int rows, int diag,
                                           int &r, int &a, int &b) {
    // Largest row r in [0, rows] with S(r) <= diag (S(0) = 0).
    r = dev::group_last_true<G>(0, rows, [&](int x) { return pa[x] + pb[x] + x <= diag; });
    if (r == rows) {
        a = pa[rows];
        b = pb[rows];
        return;
    }
    // Merge-path split of the row at a + b == D (ties: A first): a is one past the last
    // x in [lo, hi) with A[x] <= B[D - 1 - x], then the pair rule.
    const int D = diag - r;
    const int aS = pa[r], aE = pa[r + 1], bS = pb[r], bE = pb[r + 1];
    const int lo = max(aS, D - bE), hi = min(aE, D - bS);
    a = dev::group_last_true<G>(lo - 1, hi - 1,
                                [&](int x) { return ca[x] <= cb[D - 1 - x]; }) + 1;
    b = D - a;
    if (a > aS && b < bE && ca[a - 1] == cb[b]) ++b;
}

// Tile boundaries t in [0, num_tiles] (diagonals min(t * TILE, total)), kPartLanes lanes each.
// Boundary 0 also zeroes the ticket counters that the next kernel's length total uses, and
// the first n_counts boundaries zero the chunk counts (n_counts <= num_tiles + 1,
// count_stride words apart).
template <int TILE>
__global__ __launch_bounds__(kPartBlock) void csr_partition_kernel(
    const int *__restrict__ pa, const int *__restrict__ ca, const int *__restrict__ pb,
    const int *__restrict__ cb, int rows, int total, int num_tiles, int *__restrict__ split_r,
    int *__restrict__ split_a, int *__restrict__ split_b, unsigned long long *__restrict__ done,
    unsigned *__restrict__ zero_counts, int n_counts, int count_stride) {
    const int t = (static_cast<int>(blockIdx.x) * kPartBlock + static_cast<int>(threadIdx.x)) /
                  kPartLanes;
    if (t > num_tiles) return;  // whole lane groups
    const bool lead = threadIdx.x % kPartLanes == 0;
    if (lead && t == 0) dev::zero_total(done);  // accumulator of the kernel that totals the length
    if (lead && t < n_counts) zero_counts[t * count_stride] = 0u;
    const long long d64 = static_cast<long long>(t) * TILE;
    int r, a, b;
    find_split<kPartLanes>(pa, ca, pb, cb, rows, d64 > total ? total : static_cast<int>(d64), r,
                           a, b);
    if (lead) {
        split_r[t] = r;
        split_a[t] = a;
        split_b[t] = b;
    }
}

struct TileSplit {
    int r0, a0, b0, r1, a1, b1;
};

__device__ __forceinline__ TileSplit load_split(const int *__restrict__ split_r,
                                                const int *__restrict__ split_a,
                                                const int *__restrict__ split_b, int tile) {
    return TileSplit{split_r[tile], split_a[tile], split_b[tile],
                     split_r[tile + 1], split_a[tile + 1], split_b[tile + 1]};
}

}  // namespace csr
}  // namespace nacho
