// Device-wide exclusive prefix sums of int64 counts — the 64-bit replacement for the CUB
// DeviceScan::InclusiveSum calls of the reference's generated code
// (stitch_and_generate_gpu.cpp:412-446, 717-740), whose int32 counters overflow on the
// SpGEMM configuration (6.0e9 products).
//
// Two launches: every chunk's sum, then every chunk's scan, whose workgroup adds up the sums
// of the chunks before its own (at most kSummedChunks words, read from L2) instead of waiting
// for a launch that scans them, and whose last chunk stores the total.  Inputs of more chunks have
// their sums scanned by a launch in between: what the workgroups read of them otherwise grows
// with the square.  Inputs of up to kDirectChunks chunks need the last launch only: its
// workgroups add up the entries before their own.  Against four launches (sums, their scan,
// chunks, total), or one of a single workgroup up to 32,768 entries (10.8 us), 8 to 10 us less
// per scan on MI355X; above kSummedChunks, a product of 128M rows 24.2 -> 20.5 ms a call.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_utils.hpp"
#include "scan.hpp"

namespace nacho {
namespace scan {

constexpr int kBlock = 256;
constexpr int kPerThread = 16;
constexpr int kChunk = kBlock * kPerThread;
constexpr unsigned kDirectChunks = 4;  // a launch costs about as much as reading 3 chunks
constexpr unsigned kSummedChunks = 2048;
constexpr int kSumsBlock = 1024;

struct Jobs {
    const int64_t *in[kMaxJobs];
    int64_t *out[kMaxJobs];
    int64_t *total[kMaxJobs];
    int64_t n[kMaxJobs];
    unsigned first[kMaxJobs + 1];  // first chunk of each job; [count] = all chunks
    int count;
};

// The job of chunk `b`, and the chunk's number in it.
__device__ __forceinline__ int job_of(const Jobs &jobs, unsigned b, unsigned &chunk) {
    int j = 0;
    while (j + 1 < jobs.count && b >= jobs.first[j + 1]) ++j;
    chunk = b - jobs.first[j];
    return j;
}

__global__ __launch_bounds__(kBlock) void chunk_sums_kernel(Jobs jobs,
                                                            int64_t *__restrict__ sums) {
    __shared__ int64_t s_wave[kBlock / dev::kWave];
    unsigned chunk;
    const int job = job_of(jobs, blockIdx.x, chunk);
    const int64_t *__restrict__ in = jobs.in[job];
    const int64_t n = jobs.n[job];
    const int64_t base = static_cast<int64_t>(chunk) * kChunk;
    int64_t v = 0;
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int64_t i = base + threadIdx.x + static_cast<int64_t>(j) * kBlock;
        if (i < n) v += in[i];
    }
    int64_t total = 0;
    (void)dev::block_exclusive_sum<kBlock>(v, s_wave, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Workgroup j: the sums of job j's chunks become those of the chunks before each.
__global__ __launch_bounds__(kSumsBlock) void scan_sums_kernel(Jobs jobs,
                                                               int64_t *__restrict__ sums) {
    __shared__ int64_t s_wave[kSumsBlock / dev::kWave];
    const unsigned first = jobs.first[blockIdx.x], end = jobs.first[blockIdx.x + 1];
    int64_t carry = 0;
    for (unsigned c0 = first; c0 < end; c0 += kSumsBlock) {  // uniform
        const unsigned c = c0 + threadIdx.x;
        const int64_t v = c < end ? sums[c] : 0;
        int64_t total = 0;
        const int64_t before = dev::block_exclusive_sum<kSumsBlock>(v, s_wave, total);
        if (c < end) sums[c] = carry + before;
        carry += total;
    }
}

// sums: the chunks' sums, those of the chunks before (`scanned`), or null (few chunks).
__global__ __launch_bounds__(kBlock) void scan_chunks_kernel(Jobs jobs,
                                                             const int64_t *__restrict__ sums,
                                                             bool scanned) {
    __shared__ int64_t s_wave[kBlock / dev::kWave];
    unsigned chunk;
    const int job = job_of(jobs, blockIdx.x, chunk);
    const int64_t *__restrict__ in = jobs.in[job];
    int64_t *__restrict__ out = jobs.out[job];
    const int64_t n = jobs.n[job];
    const int64_t base = static_cast<int64_t>(chunk) * kChunk;
    // blocked arrangement: thread t owns elements [t*kPerThread, (t+1)*kPerThread)
    int64_t v[kPerThread];
    int64_t mine = 0;
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int64_t i = base + static_cast<int64_t>(threadIdx.x) * kPerThread + j;
        v[j] = i < n ? in[i] : 0;
        mine += v[j];
    }
    int64_t before = 0, carry = 0;
    if (scanned) {  // uniform
        carry = sums[blockIdx.x];
    } else if (chunk > 0) {
        if (!sums) {
#pragma unroll 8
            for (int64_t i = threadIdx.x; i < base; i += kBlock) before += in[i];
        } else {
            for (unsigned c = threadIdx.x; c < chunk; c += kBlock) {
                before += sums[jobs.first[job] + c];
            }
        }
        (void)dev::block_exclusive_sum<kBlock>(before, s_wave, carry);
    }
    int64_t total = 0;
    int64_t run = carry + dev::block_exclusive_sum<kBlock>(mine, s_wave, total);
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int64_t i = base + static_cast<int64_t>(threadIdx.x) * kPerThread + j;
        if (i < n) out[i] = run;
        run += v[j];
    }
    if (blockIdx.x + 1 == jobs.first[job + 1] && threadIdx.x == 0) {
        out[n] = carry + total;
        if (jobs.total[job]) dev::store_system(jobs.total[job], carry + total);
    }
}

int exclusive_scans(Call &call, const Job *jobs, int count) {
    if (count < 1 || count > kMaxJobs) return NACHO_ERR_INVALID_ARGUMENT;
    Jobs j{};
    j.count = count;
    bool direct = true;    // every input is a few chunks
    bool scanned = false;  // some input is many
    int64_t chunks = 0;
    for (int k = 0; k < count; ++k) {
        j.in[k] = jobs[k].in;
        j.out[k] = jobs[k].out;
        j.total[k] = jobs[k].total;
        j.n[k] = jobs[k].n;
        j.first[k] = static_cast<unsigned>(chunks);
        const int64_t c = jobs[k].n > 0 ? (jobs[k].n + kChunk - 1) / kChunk : 1;
        direct = direct && c <= kDirectChunks;
        scanned = scanned || c > kSummedChunks;
        chunks += c;
        if (chunks > INT32_MAX) return NACHO_ERR_INDEX_OVERFLOW;
    }
    j.first[count] = static_cast<unsigned>(chunks);
    const hipStream_t s = call.stream();
    int64_t *sums = nullptr;
    if (!direct) {
        NACHO_TRY(call.scratch_n(static_cast<size_t>(chunks), &sums));
        chunk_sums_kernel<<<static_cast<unsigned>(chunks), kBlock, 0, s>>>(j, sums);
        NACHO_TRY_HIP(hipGetLastError());
        if (scanned) {
            scan_sums_kernel<<<static_cast<unsigned>(count), kSumsBlock, 0, s>>>(j, sums);
            NACHO_TRY_HIP(hipGetLastError());
        }
    }
    scan_chunks_kernel<<<static_cast<unsigned>(chunks), kBlock, 0, s>>>(j, sums, scanned);
    NACHO_TRY_HIP(hipGetLastError());
    return NACHO_OK;
}

int exclusive_scan_i64(Call &call, const int64_t *in, int64_t n, int64_t *out, int64_t *total) {
    const Job job{in, n, out, total};
    return exclusive_scans(call, &job, 1);
}

}  // namespace scan
}  // namespace nacho
