// egx_xfer.h -- host arrays to and from the device through pinned chunks.
#pragma once

#include <cstdint>
#include <memory>
#include <vector>

#include "egx_common.h"

namespace egx {

// Host arrays to device memory on stream s; returns when they are there.
struct Upload {
    void* dev;
    const void* host;
    size_t bytes;
};
int upload(const std::vector<Upload>& jobs, hipStream_t s);

// One result vector on its way to the caller: n values at dev, written to
// host as doubles: plain doubles, or (packed) floats x that become
// x * (1 / sum), or 1 / n when sum is not positive -- the arithmetic of the
// device's FP64 output (k_pr_output), bit for bit.
struct Fetch {
    const void* dev;
    double* host;
    int64_t n;
    bool packed;
    double sum;
    const double* sum_at = nullptr;  // instead of sum: pinned, written by work queued before the values'
    int32_t* words = nullptr;        // (download) packed 4-byte words, copied here as they are
};

// Whether the values of a fetch, which are behind longer work, are about to
// land: soon(of), asked again and again while one thread waits.  Without it
// they are taken to land now.
struct Due {
    bool (*soon)(const void* of) = nullptr;
    const void* of = nullptr;
};

// All of `jobs`, whose values are written by work queued on s; returns when
// the callers' arrays hold them.
int fetch(const std::vector<Fetch>& jobs, hipStream_t s, const Due& due = Due{});

// 4-byte words at dev, written by work queued on s, to host as they are.
int download(const void* dev, int32_t* host, int64_t n, hipStream_t s);

// A small result that its last kernel writes to pinned memory itself, which
// saves the launch that carries it there: begin() gives the memory (false:
// too large, or none to be had), the kernel ends in raise_flag(), finish()
// waits for it and hands the values (f.dev is not read) to the caller.
class DirectFetch {
  public:
    DirectFetch();
    ~DirectFetch();
    DirectFetch(const DirectFetch&) = delete;
    DirectFetch& operator=(const DirectFetch&) = delete;
    bool begin(size_t bytes, hipStream_t s);
    int finish(const Fetch& f);
    char* to = nullptr;
    uint32_t* count = nullptr;
    uint32_t* flag = nullptr;

  private:
    struct State;
    std::unique_ptr<State> st_;
};

// The end of a kernel that writes to the host: all threads of every
// workgroup take part.  The last workgroup knows that the others' writes are
// out (each thread fences before its workgroup counts), raises the flag, and
// leaves the count at 0 for the next use.
__device__ __forceinline__ void raise_flag(uint32_t* count, uint32_t* flag) {
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (atomicAdd(count, 1u) + 1u == gridDim.x) {
        atomicExch(count, 0u);
        __hip_atomic_store(flag, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace egx
