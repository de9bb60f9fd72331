// The walk of a score tile along k, which the entry takes as 64 bits (with a
// zero k stride any k fits memory): how many elements are left is counted in 64
// bits, the length of a chunk in 32. Internal header; no HIP call, so that a CPU
// program can include it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ofh {

template <int BK>
struct KChunks {
    int64_t left;  // k elements from the current chunk on
    __host__ __device__ explicit KChunks(int64_t k) : left(k) {}
    __host__ __device__ bool any() const { return left > 0; }
    __host__ __device__ bool more() const { return left > BK; }  // a chunk follows the current one
    __host__ __device__ int len() const { return left < BK ? (int)left : BK; }
    __host__ __device__ void next() { left -= BK; }
};

}  // namespace ofh
