// egx_xfer.h -- host arrays to and from the device through pinned chunks.
#pragma once

#include <cstdint>
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
};

// All of `jobs`, whose values are written by work queued on s; returns when
// the callers' arrays hold them.
int fetch(const std::vector<Fetch>& jobs, hipStream_t s);

}  // namespace egx
