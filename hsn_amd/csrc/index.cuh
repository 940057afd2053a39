// The sparse-round ops' index and flag arrays as the caller holds them (include/hsn_ops.h's width
// bits of the dtype code): the kernels read either width, which costs a uniform branch a load
// against two launches an array to narrow it first (4.4 + 2.5 us each; 22 of them took 77 us of a
// 4096-slot round's 468).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hsn {

struct Idx {
    const void* p;
    int wide;  // int64_t, clamped into [-1, 2^31 - 1] as it is read; else int32_t
    __device__ __forceinline__ int operator[](int64_t i) const {
        if (!wide) return static_cast<const int32_t*>(p)[i];
        const int64_t v = static_cast<const int64_t*>(p)[i];
        return v < -1 ? -1 : v > 0x7fffffff ? 0x7fffffff : static_cast<int>(v);
    }
};

struct Flags {
    const void* p;
    int bytes;  // one byte a flag (bool); else int32_t
    __device__ __forceinline__ bool operator[](int64_t i) const {
        return bytes ? static_cast<const uint8_t*>(p)[i] != 0 : static_cast<const int32_t*>(p)[i] != 0;
    }
};

}  // namespace hsn
