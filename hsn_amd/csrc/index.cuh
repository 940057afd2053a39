// The sparse-round ops' index and flag arrays as the caller holds them (include/hsn_ops.h's width
// bits of the dtype code): the kernels read either width instead of two launches an array that
// narrow it first (4.4 + 2.5 us each; 22 of them took 77 us of a 4096-slot round's 468).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace hsn {

// The kernels' instantiations: kNarrow int32_t indices and flags, kWide int64_t indices and flags of
// a byte, kMixed any other mix, told at run time. A width known to the compiler keeps a loop's loads
// together: told at run time, by a branch a load, the messages took 1.03 to 1.16 times the int32
// kernels' time (more with more edges) and grad_V 1.35 times without the branch, two loads an index.
enum Widths : int { kNarrow, kWide, kMixed };

// (an instantiation carries what it reads and no more: with the width beside the pointer the int32
// kernels' code moved by a few words, and the messages' serial loop took 1.1 times as long)
__device__ __forceinline__ int clamped_index(int64_t v) {
    return v < -1 ? -1 : v > 0x7fffffff ? 0x7fffffff : static_cast<int>(v);
}
template <int W>
struct Idx {
    const void* p;
    int wide;  // int64_t, clamped into [-1, 2^31 - 1] as it is read; else int32_t
    __device__ __forceinline__ int operator[](int64_t i) const {
        return wide ? clamped_index(static_cast<const int64_t*>(p)[i]) : static_cast<const int32_t*>(p)[i];
    }
};
template <>
struct Idx<kNarrow> {
    const int32_t* p;
    __device__ __forceinline__ int operator[](int64_t i) const { return p[i]; }
};
template <>
struct Idx<kWide> {
    const int64_t* p;
    __device__ __forceinline__ int operator[](int64_t i) const { return clamped_index(p[i]); }
};

template <int W>
struct Flags {
    const void* p;
    int bytes;  // one byte a flag (bool); else int32_t
    __device__ __forceinline__ bool operator[](int64_t i) const {
        return bytes ? static_cast<const uint8_t*>(p)[i] != 0 : static_cast<const int32_t*>(p)[i] != 0;
    }
};
template <>
struct Flags<kNarrow> {
    const int32_t* p;
    __device__ __forceinline__ bool operator[](int64_t i) const { return p[i] != 0; }
};
template <>
struct Flags<kWide> {
    const uint8_t* p;
    __device__ __forceinline__ bool operator[](int64_t i) const { return p[i] != 0; }
};

// An array in one instantiation's type (`wide`: its own width bit).
template <int W>
inline Idx<W> index_array(const void* p, bool wide) {
    if constexpr (W == kNarrow) return {static_cast<const int32_t*>(p)};
    else if constexpr (W == kWide) return {static_cast<const int64_t*>(p)};
    else return {p, wide ? 1 : 0};
}
template <int W>
inline Flags<W> flag_array(const void* p, bool bytes) {
    if constexpr (W == kNarrow) return {static_cast<const int32_t*>(p)};
    else if constexpr (W == kWide) return {static_cast<const uint8_t*>(p)};
    else return {p, bytes ? 1 : 0};
}

// Calls f with the instantiation for these bits: `all` are the width bits of the arrays the call has.
template <class F>
inline void by_widths(int bits, int all, const F& f) {
    if ((bits & all) == 0) f(std::integral_constant<int, kNarrow>{});
    else if ((bits & all) == all) f(std::integral_constant<int, kWide>{});
    else f(std::integral_constant<int, kMixed>{});
}

}  // namespace hsn
