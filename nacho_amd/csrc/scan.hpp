// Device-wide exclusive prefix sums of int64 counts (scan.hip).
#pragma once

#include <cstdint>

#include "runtime.hpp"

namespace nacho {
namespace scan {

// out[i] = in[0] + ... + in[i-1] for i in [0, n]; out has n + 1 entries (out[n] = total) and is
// not `in`.  `total` (optional): a pinned host word (Call::value_word) that also gets it.
struct Job {
    const int64_t *in;
    int64_t n;
    int64_t *out;
    int64_t *total = nullptr;
};

// Up to kMaxJobs independent scans at once: one launch when every input is short, two or three
// otherwise.  Runs on the call's stream; scratch comes from the call.
constexpr int kMaxJobs = 4;
int exclusive_scans(Call &call, const Job *jobs, int count);

int exclusive_scan_i64(Call &call, const int64_t *in, int64_t n, int64_t *out,
                       int64_t *total = nullptr);

}  // namespace scan
}  // namespace nacho
