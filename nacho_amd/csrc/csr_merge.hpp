// Level merge shared by the CSR, COO, DCSR and CSF3 entry points (see level_merge.hip).
#pragma once

#include <cstdint>

#include "runtime.hpp"

namespace nacho {
namespace csr {

// One operand level: `pos` has rows + 1 entries (pos[0] == 0) indexing `crd`/`val`
// (`len` entries).  `next` (optional) is the offsets array of the level below, indexed by
// this level's positions (len + 1 entries); when null, child pointers are the positions.
struct LevelOperand {
    const int *pos;
    const int *crd;
    const float *val;
    int len;
    const int *next;
};

// Result buffers, sized by the caller for the worst case: pos rows + 1, crd/val (and row)
// the union (or intersection) bound, child_a/child_b that bound + 1.
struct LevelResult {
    int *pos;
    int *crd;
    float *val;
    int *child_a;
    int *child_b;
    // Value levels only, optional: the row of every output (a COO result's i coordinate).
    int *row = nullptr;
    // Union value levels only, optional: each output coordinate c is stored split, as
    // c >> low_bits to crd and c & (2^low_bits - 1) to crd_low (a COO3 result's j and k).
    int *crd_low = nullptr;
    int low_bits = 0;
    // Intersection value levels only, optional: the level's inner product instead of its
    // result.  Σ a·b over the pairs (each product one binary32 multiply, as the result's
    // values) is summed in binary64 in a fixed order, rounded once and stored to this device
    // float; pos, crd and val are then not written (they may be null), *out_len is 0, and
    // the host does not wait for the device.
    float *dot = nullptr;
};

// Headroom merge_level keeps below INT_MAX for its item count (entries of both operands plus
// rows): it refuses larger levels with NACHO_ERR_INDEX_OVERFLOW.  Callers that choose between
// it and another path keep 2 * kLevelTileSlack.
constexpr long long kLevelItemSlack = 7680;
constexpr long long kLevelTileSlack = 4096;
static_assert(kLevelItemSlack <= 2 * kLevelTileSlack, "what callers route here is taken");

// Merge A and B row by row: union (or intersection) of each row's coordinates, with values
// (a+b / a*b / copies) when `values`, or with child pointers when `child` (unions only).
// Coordinates are ordered as int32 numbers; those of the extent lie in [0, 2^crd_bits),
// crd_bits <= 31, and others are merged as well, by a slow walk.  Writes Z.pos for every row and
// returns the result length in *out_len.  The call's kernel timer (if enabled) brackets all of
// the level's kernels under `kernel_name`.
//
// With `length_pending`, the host does not wait for the length: *length_pending is set,
// *out_len is left alone, and the caller, having queued what it has to on the stream, reads
// the length with call.wait_length before any other level merge of the call (and collects
// the level's timer with call.collect_timer before starting another).
int merge_level(Call &call, bool intersect, bool values, bool child, int rows, int crd_bits,
                const LevelOperand &A, const LevelOperand &B, const LevelResult &Z,
                long long *out_len, const char *kernel_name, bool *length_pending = nullptr);

// Bits of coordinates below `extent` (at least 1).
inline int extent_bits(int extent) {
    return extent > 2 ? 32 - __builtin_clz(static_cast<unsigned>(extent - 1)) : 1;
}

// Σ v[0, n) summed in binary64 in a fixed order and rounded once to the device float *out
// (kernels queued on the call's stream; v may be null when n is 0).
int sum_values(Call &call, const float *v, long long n, float *out);

// A CSR descriptor that no entry point can take (negative sizes, missing buffers).
bool bad_csr(const nacho_csr *t);

}  // namespace csr
}  // namespace nacho
