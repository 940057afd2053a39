// The RMS candidate: a prologue normalises the candidate input once (the only cross-column
// quantity of the round, computed from inputs only), an epilogue applies the norm's VJP.
//
// Both are bound by HBM: the prologue reads and writes [slots, d], the epilogue reads two and
// writes one. For d a multiple of 4 up to 256 and rows aligned to four elements, L lanes hold a
// slot, four columns each, so a wavefront's access covers 64 / L whole rows in 16-byte (fp32) or
// 8-byte (bf16) pieces, kU of them in flight; the epilogue sums the gain's gradient on the way,
// a partial a workgroup and a small launch over the partials. Other d and unaligned rows take the
// row-a-wavefront kernels. At 32768 slots of d 64 in fp32: prologue 6.1 us (9.5 a row a wavefront),
// epilogue with the gain's gradient 6.2 + 3.7 us (9.8 and 76.7: that pass ran in d workgroups, each
// reading one column with a stride of d).
#pragma once

#include <hip/hip_runtime.h>

#include "abi_util.h"
#include "common.cuh"
#include "dpp.cuh"
#include "sweep.cuh"

namespace hsn {
namespace rms {

// ynorm[s, x] = y[s, x] * inv[s] * w[x],  inv[s] = rsqrt(mean_x y^2 + eps): a wavefront per slot
template <typename IN>
__global__ __launch_bounds__(256) void rms_prologue(const IN* y, const float* w, IN* ynorm,
                                                    float* inv, int64_t slots, int d, float eps) {
    const int64_t s = int64_t(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (s >= slots) return;
    const int lane = lane_id();
    float sum = 0.0f;
    for (int x = lane; x < d; x += kWave) {
        const float v = to_f32(y[s * d + x]);
        sum += v * v;
    }
    for (int m = 1; m < kWave; m <<= 1) sum += __shfl_xor(sum, m, kWave);
    const float r = rsqrtf(sum / static_cast<float>(d) + eps);
    if (lane == 0) inv[s] = r;
    for (int x = lane; x < d; x += kWave) store_f32(ynorm, s * d + x, to_f32(y[s * d + x]) * r * w[x]);
}

// dL/dw[x] = sum over slots of dpre[x] y[x] inv (one workgroup per column, fixed-shape tree)
template <typename IN>
__global__ __launch_bounds__(256) void rms_weight_grad(const IN* y, const IN* dpre, const float* inv,
                                                       float* dw, int64_t slots, int d) {
    __shared__ float part[256];
    const int x = blockIdx.x;
    float acc = 0.0f;
    for (int64_t s = threadIdx.x; s < slots; s += blockDim.x)
        acc += to_f32(dpre[s * d + x]) * to_f32(y[s * d + x]) * inv[s];
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) dw[x] = part[0];
}

// dy[x] = inv w[x] dpre[x] - inv^3 y[x] / d * sum_x' dpre[x'] w[x'] y[x'], in place over dpre
template <typename IN>
__global__ __launch_bounds__(256) void rms_input_grad(const IN* y, IN* dy, const float* inv,
                                                      const float* w, int64_t slots, int d) {
    const int64_t s = int64_t(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (s >= slots) return;
    const int lane = lane_id();
    const float r = inv[s];
    float dot = 0.0f;
    for (int x = lane; x < d; x += kWave) dot += to_f32(dy[s * d + x]) * w[x] * to_f32(y[s * d + x]);
    for (int m = 1; m < kWave; m <<= 1) dot += __shfl_xor(dot, m, kWave);
    const float k3 = r * r * r * dot / static_cast<float>(d);
    for (int x = lane; x < d; x += kWave) {
        const float v = r * w[x] * to_f32(dy[s * d + x]) - k3 * to_f32(y[s * d + x]);
        store_f32(dy, s * d + x, v);
    }
}

// ---- four columns a lane ----

constexpr int kU = 4;  // row groups of a wavefront in flight

struct Four {
    float v[4];
};
__device__ __forceinline__ Four load4(const float* p) {
    const float4 q = *reinterpret_cast<const float4*>(p);
    return Four{{q.x, q.y, q.z, q.w}};
}
__device__ __forceinline__ Four load4(const bf16_t* p) {
    const uint2 q = *reinterpret_cast<const uint2*>(p);
    return Four{{__uint_as_float(q.x << 16), __uint_as_float(q.x & 0xffff0000u),
                 __uint_as_float(q.y << 16), __uint_as_float(q.y & 0xffff0000u)}};
}
__device__ __forceinline__ void store4(float* p, const Four& f) {
    *reinterpret_cast<float4*>(p) = make_float4(f.v[0], f.v[1], f.v[2], f.v[3]);
}
__device__ __forceinline__ void store4(bf16_t* p, const Four& f) {
    bf16_t e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = from_f32<bf16_t>(f.v[i]);
    uint2 q;
    __builtin_memcpy(&q, e, 8);
    *reinterpret_cast<uint2*>(p) = q;
}

// ynorm[s, x] = y[s, x] * inv[s] * w[x],  inv[s] = rsqrt(mean_x y^2 + eps): L lanes a slot
template <typename IN, int L>
__global__ __launch_bounds__(256) void prologue4(const IN* y, const float* w, IN* ynorm, float* inv,
                                                 int64_t slots, int d, float eps) {
    constexpr int R = kWave / L;  // slots a wavefront's access covers
    const int lane = lane_id(), c = 4 * (lane % L);
    const int64_t s0 = (int64_t(blockIdx.x) * 4 + threadIdx.x / kWave) * kU * R + lane / L;
    const bool in = c < d;
    Four g{}, q[kU];
    if (in)
#pragma unroll
        for (int i = 0; i < 4; ++i) g.v[i] = w[c + i];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
        const int64_t s = s0 + u * R;
        q[u] = in && s < slots ? load4(y + s * d + c) : Four{};
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
        const int64_t s = s0 + u * R;
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) sum += q[u].v[i] * q[u].v[i];
        sum = group_sum<L>(sum);
        const float r = rsqrtf(sum / static_cast<float>(d) + eps);
        if (s >= slots) continue;
        if (lane % L == 0) inv[s] = r;
#pragma unroll
        for (int i = 0; i < 4; ++i) q[u].v[i] = q[u].v[i] * r * g.v[i];
        if (in) store4(ynorm + s * d + c, q[u]);
    }
}

// dy[x] = inv w[x] dpre[x] - inv^3 y[x] / d * sum_x' dpre[x'] w[x'] y[x'], in place over dpre, and
// with `part` the workgroup's share of dL/dw[x] = sum over slots of dpre[x] y[x] inv: its slots
// [blockIdx.x * per, + per), the lanes' sums added in lane order.
template <typename IN, int L>
__global__ __launch_bounds__(256) void vjp4(const IN* y, IN* dy, const float* inv, const float* w,
                                            float* part, int64_t slots, int64_t per, int d) {
    constexpr int R = kWave / L, kRows = 4 * R;
    __shared__ float red[kRows][4 * L + 1];
    const int lane = lane_id(), wv = threadIdx.x / kWave, c = 4 * (lane % L);
    const bool in = c < d;
    const int64_t end = min(slots, (int64_t(blockIdx.x) + 1) * per);
    Four g{}, acc{};
    if (in)
#pragma unroll
        for (int i = 0; i < 4; ++i) g.v[i] = w[c + i];
    for (int64_t s0 = int64_t(blockIdx.x) * per + wv * R + lane / L; s0 - lane / L < end; s0 += kU * kRows) {
        Four q[kU], p[kU];
        float r[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int64_t s = s0 + u * kRows;
            const bool ok = in && s < end;
            q[u] = ok ? load4(y + s * d + c) : Four{};
            p[u] = ok ? load4(dy + s * d + c) : Four{};
            r[u] = s < end ? inv[s] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int64_t s = s0 + u * kRows;
            float dot = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) dot += p[u].v[i] * g.v[i] * q[u].v[i];
            dot = group_sum<L>(dot);
            const float k3 = r[u] * r[u] * r[u] * dot / static_cast<float>(d);
            Four o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o.v[i] = r[u] * g.v[i] * p[u].v[i] - k3 * q[u].v[i];
                acc.v[i] += p[u].v[i] * q[u].v[i] * r[u];
            }
            if (in && s < end) store4(dy + s * d + c, o);
        }
    }
    if (!part) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wv * R + lane / L][c + i] = acc.v[i];
    __syncthreads();
    for (int x = threadIdx.x; x < d; x += 256) {
        float s = 0.0f;
        for (int i = 0; i < kRows; ++i) s += red[i][x];
        part[int64_t(blockIdx.x) * d + x] = s;
    }
}

// dL/dw from the workgroups' shares: 16 columns a workgroup, 16 runs of shares a column, added in
// run order.
static __global__ __launch_bounds__(256) void weight_sum(const float* part, float* dw, int parts, int d) {
    __shared__ float red[16][17];
    const int x = blockIdx.x * 16 + threadIdx.x % 16, g = threadIdx.x / 16;
    float s = 0.0f;
    if (x < d) {
#pragma unroll 8
        for (int i = g; i < parts; i += 16) s += part[int64_t(i) * d + x];
    }
    red[g][threadIdx.x % 16] = s;
    __syncthreads();
    if (g == 0 && x < d) {
        float t = 0.0f;
        for (int i = 0; i < 16; ++i) t += red[i][threadIdx.x % 16];
        dw[x] = t;
    }
}

// ---- host side ----

inline bool rows_of_four(const void* a, const void* b, int d, size_t elem) {
    return d % 4 == 0 && d <= 256 && reinterpret_cast<uintptr_t>(a) % (4 * elem) == 0 &&
           reinterpret_cast<uintptr_t>(b) % (4 * elem) == 0;
}
// Calls f with the lanes a slot takes: the power of two from 4 that covers d / 4 columns.
template <class F>
inline void by_lanes(int d, const F& f) {
    if (d <= 16) f(std::integral_constant<int, 4>{});
    else if (d <= 32) f(std::integral_constant<int, 8>{});
    else if (d <= 64) f(std::integral_constant<int, 16>{});
    else if (d <= 128) f(std::integral_constant<int, 32>{});
    else f(std::integral_constant<int, 64>{});
}

template <typename IN>
inline void launch_prologue(const IN* y, const float* w, IN* ynorm, float* inv, int64_t slots, int d,
                            float eps, hipStream_t st) {
    if (rows_of_four(y, ynorm, d, sizeof(IN)))
        by_lanes(d, [&](auto l) {
            constexpr int L = decltype(l)::value;
            const int64_t per = 4 * kU * (kWave / L);
            hipLaunchKernelGGL((prologue4<IN, L>), dim3(static_cast<unsigned>((slots + per - 1) / per)),
                               dim3(256), 0, st, y, w, ynorm, inv, slots, d, eps);
        });
    else
        hipLaunchKernelGGL((rms_prologue<IN>), dim3(static_cast<unsigned>((slots + 3) / 4)), dim3(256), 0,
                           st, y, w, ynorm, inv, slots, d, eps);
    HSN_HIP(hipGetLastError());
}

// `scratch`: the prologue's ynorm, not read any more, takes the workgroups' shares (a workgroup
// has at least 64 slots where there is more than one, so they fit).
template <typename IN>
inline void launch_vjp(const IN* y, IN* dy, const float* inv, const float* w, float* dw, IN* scratch,
                       int64_t slots, int d, hipStream_t st) {
    if (rows_of_four(y, dy, d, sizeof(IN)) && slots >= 2) {
        by_lanes(d, [&](auto l) {
            constexpr int L = decltype(l)::value;
            const int64_t step = 4 * (kWave / L);
            int64_t per = (slots + 1023) / 1024;
            per = (per + step - 1) / step * step;
            if (per < 64) per = 64;
            const int parts = static_cast<int>((slots + per - 1) / per);
            float* part = dw ? reinterpret_cast<float*>(scratch) : nullptr;
            hipLaunchKernelGGL((vjp4<IN, L>), dim3(parts), dim3(256), 0, st, y, dy, inv, w, part, slots,
                               per, d);
            HSN_HIP(hipGetLastError());
            if (dw)
                hipLaunchKernelGGL(weight_sum, dim3((d + 15) / 16), dim3(256), 0, st, part, dw, parts, d);
        });
    } else {
        if (dw)
            hipLaunchKernelGGL((rms_weight_grad<IN>), dim3(d), dim3(256), 0, st, y, dy, inv, dw, slots, d);
        hipLaunchKernelGGL((rms_input_grad<IN>), dim3(static_cast<unsigned>((slots + 3) / 4)), dim3(256), 0,
                           st, y, dy, inv, w, slots, d);
    }
    HSN_HIP(hipGetLastError());
}

}  // namespace rms
}  // namespace hsn
