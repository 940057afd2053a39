// The window's sweeps cell by cell (gfx950). Each cell's updates form a chain in time; chains of
// different cells are independent but for the summary q, which adds every slot's delta of a
// position. So the state needs no shared memory: a wavefront walks one cell's chain with the
// cell's d columns in its lanes (column x in lane x % 64, register x / 64), and every load and
// store is a whole row of a [B, T, K, d] tensor (d * sizeof(io) contiguous bytes), against the
// S-column pieces of the time-chunked sweeps (sweep.cuh), whose slices shrink as K grows.
//
//   row_lists     (row): the row's decisions as per-cell event lists (CSR): ptr[N + 1], then
//                 the events (t << 8 | k) of each cell in time order, then the padded slots in
//                 time order. Counts by LDS atomics (integers: any order), ranks within a block
//                 of positions from a bit per position per cell (popcount below t):
//                 deterministic. By ranges of cells (row_lists_ranges) where the row allows.
//   chain_fwd     (row, group of cells; a wavefront per cell): h_old, h_sel, the end state, the
//                 ages, each valid slot's delta h_sel - h_old in fp32 where the rows are bf16
//                 or omitted; the row maximum of |h| per position from each cell's value on the
//                 intervals between its events (LDS atomic max), a table per group.
//   summary_delta (row, position): D[t] = the sum of the valid slots' deltas; the row maximum,
//                 the largest of the groups'.
//   summary_scan_fwd (row, 64 columns): q before and after every position, a scan over time
//                 of D / N with the resets.
//   summary_scan_bwd (row, 64 columns): the summary cotangent R, a reverse scan in fp64, as the
//                 per-position share R / N and d_q0.
//   chain_bwd     (row, group of cells): the reverse chains of the cotangent A with the
//                 activations' VJPs; d_h0.
//
// Reference: the forward restates python/hsn/kernels/native.py:244-303 and
// python/hsn/model/state.py:267-324 per position (python/hsn/train/compile.py:1296-1344); the
// backward restates python/hsn/train/split.py:128-174 with the carried state
// (python/hsn/train/state_gradient.py:402-416). A reset at r zeroes the state before position
// r reads it (forward) and the cotangents after position r is processed (backward): for a
// cell's consecutive events t' < t, the chain restarts from zero exactly when a reset lies in
// (t', t], i.e. when the first reset after t' is at or before t. Padded slots gather cell 0
// (h_old shows cell 0 before the position's update, h_sel after it) and get exact zeros in the
// backward.
#pragma once

#include <stddef.h>

#include <type_traits>

#include "sweep.cuh"

namespace hsn {
namespace chain {

constexpr int kMaxV = 4;   // columns per lane: d <= 256
constexpr int kMaxK = 255;  // slots per position (the event's slot field is 8 bits)
constexpr int kEvWin = 64;  // events per window: one event per lane

// ------------------------------------------------------------------------------------------
// The per-row event lists
// ------------------------------------------------------------------------------------------

constexpr int kListThreads = 1024;
constexpr int kListU = 8;  // slots per thread and block of positions

// positions per block of the rank pass (a multiple of 32): a bit per position per cell in at most
// 64 KiB, and at most 2048 slots unless one word of positions has more (32 K <= 8160 slots, within
// the kListU * kListThreads a block's threads hold)
__host__ __device__ inline int list_block(int N, int T, int K) {
    int P = 32;
    while (P < T && int64_t(N) * (2 * P / 32) * 4 <= 65536 && 2 * P * K <= 2048) P *= 2;
    return P;
}
// the scan partials' words: the 16 wavefronts' and the row's total, or a prefix per word of the
// block's padded-slot bits and their total
__host__ __device__ inline int list_partials(int P, int K) {
    const int pkw = (P * K + 31) / 32 + 1;
    return pkw > 65 ? pkw : 65;
}
__host__ __device__ inline int list_words(int N, int T, int K) {  // LDS words of row_lists
    const int P = list_block(N, T, K);
    return 2 * N + N * (P / 32) + (P * K + 31) / 32 + list_partials(P, K) + 4;
}

struct ListArgs {
    const int32_t* slots;  // [B, T, K]: the cell, or -1 on a padded slot
    int32_t* ptr;          // [B, N + 1]
    int32_t* ev;           // [B, T * K]
    int B, T, N, K;
};

__device__ __forceinline__ int slot_cell(const int32_t* slots, int64_t i, int N) {
    const int c = slots[i];
    return c >= 0 && c < N ? c : -1;
}

static __global__ __launch_bounds__(kListThreads) void row_lists(ListArgs a) {
    extern __shared__ uint32_t lds_u[];
    const int b = blockIdx.x;
    const int tid = threadIdx.x;
    const int T = a.T, N = a.N, K = a.K;
    const int P = list_block(N, T, K), PW = P / 32;
    int* cnt = reinterpret_cast<int*>(lds_u);  // [N]: counts, then the events placed so far
    int* base = cnt + N;                       // [N]: the list starts
    uint32_t* mask = reinterpret_cast<uint32_t*>(base + N);  // [N][PW]
    const int PKW = (P * K + 31) / 32;
    uint32_t* pmask = mask + N * PW;                  // [PKW]: the block's padded slots
    int* wsum = reinterpret_cast<int*>(pmask + PKW);  // scan partials
    int* misc = wsum + list_partials(P, K);           // [0]: padded slots placed so far
    const int64_t row = int64_t(b) * T * K;
    for (int c = tid; c < N; c += kListThreads) cnt[c] = 0;
    if (tid == 0) misc[0] = 0;
    __syncthreads();
    const int n_slots = T * K;
    for (int i0 = tid; i0 < n_slots; i0 += kListThreads * kListU) {  // kListU loads in flight
        int cs[kListU];
#pragma unroll
        for (int u = 0; u < kListU; ++u) {
            const int i = i0 + u * kListThreads;
            cs[u] = i < n_slots ? slot_cell(a.slots, row + i, N) : -1;
        }
#pragma unroll
        for (int u = 0; u < kListU; ++u)
            if (cs[u] >= 0) atomicAdd(&cnt[cs[u]], 1);
    }
    __syncthreads();
    // exclusive scan of the counts (a chunk of cells per thread, then the chunks' prefix)
    const int per = (N + kListThreads - 1) / kListThreads;
    const int c0 = min(N, tid * per), c1 = min(N, c0 + per);
    int s = 0;
    for (int c = c0; c < c1; ++c) s += cnt[c];
    const int lane = tid & 63, wv = tid >> 6;
    int incl = s;
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(incl, o, 64);
        if (lane >= o) incl += u;
    }
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    if (tid == 0) {
        int acc = 0;
        for (int w = 0; w < kListThreads / 64; ++w) {
            const int v = wsum[w];
            wsum[w] = acc;
            acc += v;
        }
        wsum[kListThreads / 64] = acc;  // the row's valid events
    }
    __syncthreads();
    int run = wsum[wv] + incl - s;
    for (int c = c0; c < c1; ++c) {
        const int v = cnt[c];
        base[c] = run;
        cnt[c] = 0;
        a.ptr[int64_t(b) * (N + 1) + c] = run;
        run += v;
    }
    const int n_valid = wsum[kListThreads / 64];
    if (tid == 0) a.ptr[int64_t(b) * (N + 1) + N] = n_valid;
    int32_t* ev = a.ev + row;
    // blocks of P positions (P * K <= kListU * kListThreads slots): a thread's slots of the next
    // block are loaded while the current one is ranked
    int cur[kListU], nxt[kListU];
    auto fetch = [&](int t0, int (&cs)[kListU]) __attribute__((always_inline)) {
        const int n = min(P, T - t0) * K;
#pragma unroll
        for (int u = 0; u < kListU; ++u) {
            const int i = tid + u * kListThreads;
            cs[u] = t0 < T && i < n ? slot_cell(a.slots, row + int64_t(t0) * K + i, N) : -2;
        }
    };
    fetch(0, cur);
    for (int t0 = 0; t0 < T; t0 += P) {
        const int pn = min(P, T - t0);
        fetch(t0 + P, nxt);
        __syncthreads();
        for (int i = tid; i < N * PW; i += kListThreads) mask[i] = 0u;
        for (int i = tid; i < PKW; i += kListThreads) pmask[i] = 0u;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kListU; ++u) {
            const int i = tid + u * kListThreads, c = cur[u];
            if (c == -2) continue;  // past the block
            const int tl = i / K;
            if (c >= 0) atomicOr(&mask[c * PW + (tl >> 5)], 1u << (tl & 31));
            else atomicOr(&pmask[i >> 5], 1u << (i & 31));
        }
        __syncthreads();
        if (tid < 64) {  // the padded slots' exclusive prefix per word, in wsum (wavefront 0)
            int acc = 0;
            for (int w0 = 0; w0 < PKW; w0 += 64) {
                const int w = w0 + tid;
                const int v = w < PKW ? __popc(pmask[w]) : 0;
                int incl = v;
                for (int o = 1; o < 64; o <<= 1) {
                    const int u = __shfl_up(incl, o, 64);
                    if (tid >= o) incl += u;
                }
                if (w < PKW) wsum[w] = acc + incl - v;
                acc += __shfl(incl, 63, 64);
            }
            if (tid == 0) wsum[PKW] = acc;  // the block's padded slots
        }
        __syncthreads();
        const int pad0 = misc[0];
#pragma unroll
        for (int u = 0; u < kListU; ++u) {
            const int i = tid + u * kListThreads, c = cur[u];
            if (c == -2) continue;
            const int tl = i / K, k = i - tl * K;
            const int t = t0 + tl;
            if (c >= 0) {
                int rank = cnt[c];
                const uint32_t* m = mask + c * PW;
                for (int w = 0; w < (tl >> 5); ++w) rank += __popc(m[w]);
                rank += __popc(m[tl >> 5] & ((1u << (tl & 31)) - 1u));
                ev[base[c] + rank] = (t << 8) | k;
            } else {
                const int r = wsum[i >> 5] + __popc(pmask[i >> 5] & ((1u << (i & 31)) - 1u));
                ev[n_valid + pad0 + r] = (t << 8) | k;
            }
        }
        (void)pn;
        __syncthreads();
        for (int c = tid; c < N; c += kListThreads) {
            int v = 0;
            for (int w = 0; w < PW; ++w) v += __popc(mask[c * PW + w]);
            cnt[c] += v;
        }
        if (tid == 0) misc[0] = pad0 + wsum[PKW];
#pragma unroll
        for (int u = 0; u < kListU; ++u) cur[u] = nxt[u];
    }
}

// The same lists by (row, range of cells): a wavefront takes its share of the row's positions in
// order. It counts its slots of each of the range's cells (two 16-bit counts a word), the counts'
// prefix over the cells and the wavefronts gives every wavefront its own place in each cell's list,
// and it places its slots position by position (a position's cells are distinct; a wavefront's LDS
// operations complete in order) by the counts' old values. The range's part of the row's list is put
// together in LDS and written in order; the last range's goes on with the padded slots. A row of
// T K <= 32768 slots, so offsets are 16 bits. Bound by the instructions a slot (every range reads the
// row's slots twice), hence ranges only as far as they fill the chip. The LDS operations of a step's
// positions are issued without a wait between: with one, B256 T1024 N4096 K32 took 90 us instead
// of 37, two ranges a row and sixteen wavefronts.
constexpr int kRangeSlots = 32768;

__host__ __device__ inline int range_waves(int N) { return N > 2048 ? 8 : 16; }
__host__ __device__ inline int range_cells(int B, int N) {  // cells a range, even
    int R = 1;
    while (int64_t(B) * R < 256 && N / (2 * R) >= 64) R *= 2;
    const int NR = (N + R - 1) / R;
    return NR + (NR & 1);
}
__host__ __device__ inline int range_words(int W, int NR, int T, int K) {  // LDS words
    return W * (NR / 2) + (T * K + 1) / 2 + 3 * W + 2;
}

// SUB: positions a step, at most 64 / K.
template <int W, int SUB>
__global__ __launch_bounds__(64 * W) void row_lists_ranges(ListArgs a, int NR) {
    extern __shared__ uint32_t lds_u[];
    constexpr int kThreads = 64 * W;
    const int b = blockIdx.y, z = blockIdx.x;
    const int tid = threadIdx.x, lane = lane_id(), w = uniform(tid / 64);
    const int T = a.T, N = a.N, K = a.K, NW = NR / 2;
    const uint32_t c_lo = z * NR, c_hi = min(N, int(c_lo) + NR), span = c_hi - c_lo;
    const bool last = int(c_hi) == N;
    uint32_t* const cnt = lds_u;  // [W][NW]
    uint16_t* const stage = reinterpret_cast<uint16_t*>(cnt + W * NW);  // [T K]
    int* const under = reinterpret_cast<int*>(cnt + W * NW + (T * K + 1) / 2);  // [W]: lower ranges' slots
    int* const pads = under + W;  // [W]: padded slots
    int* const wsum = pads + W;   // [W]: the scan's partials
    const int per = (T + W - 1) / W;
    const int s_lo = min(T, w * per) * K, s_n = min(T, (w + 1) * per) * K - s_lo;
    const int32_t* const slots = a.slots + int64_t(b) * T * K + s_lo;
    for (int i = tid; i < W * NW; i += kThreads) cnt[i] = 0u;
    __syncthreads();
    uint32_t* const mine = cnt + w * NW;
    int lo = 0, pad = 0;
    constexpr int kU = 8;  // loads in flight
    for (int s0 = 0; s0 < s_n; s0 += 64 * kU) {
        uint32_t cs[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) cs[u] = slots[min(s0 + 64 * u + lane, s_n - 1)];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            if (s0 + 64 * u >= s_n) break;
            const bool here = s0 + 64 * u + lane < s_n;
            const uint32_t rel = cs[u] - c_lo;
            if (z > 0) lo += here && cs[u] < c_lo ? 1 : 0;
            if (last) pad += here && cs[u] >= uint32_t(N) ? 1 : 0;
            if (here && rel < span) atomicAdd(&mine[rel >> 1], (rel & 1u) ? 0x10000u : 1u);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo += __shfl_xor(lo, o, 64);
        pad += __shfl_xor(pad, o, 64);
    }
    if (lane == 0) under[w] = lo, pads[w] = pad;
    __syncthreads();
    // consecutive words of two cells a thread: the wavefronts' prefix, then the cells'
    const int each = (NW + kThreads - 1) / kThreads, i0 = tid * each, i1 = min(NW, i0 + each);
    int own = 0;
    for (int i = i0; i < i1; ++i) {
        uint32_t run = 0u;
#pragma unroll
        for (int v = 0; v < W; ++v) run += cnt[v * NW + i];
        own += (run & 0xffffu) + (run >> 16);
    }
    int incl = own;
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(incl, o, 64);
        if (lane >= o) incl += u;
    }
    if (lane == 63) wsum[w] = incl;
    int first = 0;  // the row's events in lower ranges
#pragma unroll
    for (int v = 0; v < W; ++v) first += under[v];
    __syncthreads();
    int at = incl - own, total = 0;
#pragma unroll
    for (int v = 0; v < W; ++v) {
        at += v < w ? wsum[v] : 0;
        total += wsum[v];
    }
    int32_t* const ptr = a.ptr + int64_t(b) * (N + 1);
    for (int i = i0; i < i1; ++i) {
        uint32_t n[W], run = 0u;
#pragma unroll
        for (int v = 0; v < W; ++v) n[v] = cnt[v * NW + i];
#pragma unroll
        for (int v = 0; v < W; ++v) run += n[v];
        const int n0 = run & 0xffffu, n1 = run >> 16;
        uint32_t place = uint32_t(at) | (uint32_t(at + n0) << 16);
#pragma unroll
        for (int v = 0; v < W; ++v) {
            cnt[v * NW + i] = place;
            place += n[v];
        }
        const uint32_t c = c_lo + 2 * i;
        if (c < c_hi) ptr[c] = first + at;
        if (c + 1 < c_hi) ptr[c + 1] = first + at + n0;
        at += n0 + n1;
    }
    if (last && tid == 0) ptr[N] = first + total;
    int pad_at = total, n_out = total;
    if (last) {
#pragma unroll
        for (int v = 0; v < W; ++v) {
            pad_at += v < w ? pads[v] : 0;
            n_out += pads[v];
        }
    }
    __syncthreads();
    const int step = SUB * K;  // whole positions, at most 64 slots
    const int sub = SUB > 1 ? lane / K : 0;
    constexpr int kV = SUB >= 8 ? 1 : 8 / SUB;  // steps in flight
    for (int s0 = 0; s0 < s_n; s0 += step * kV) {
        uint32_t cs[kV], old[kV][SUB];
#pragma unroll
        for (int u = 0; u < kV; ++u) cs[u] = slots[min(s0 + step * u + lane, s_n - 1)];
#pragma unroll
        for (int u = 0; u < kV; ++u) {
            const bool here = lane < step && s0 + step * u + lane < s_n;
            const uint32_t rel = cs[u] - c_lo;
#pragma unroll
            for (int j = 0; j < SUB; ++j)
                if (here && rel < span && (SUB == 1 || sub == j))
                    old[u][j] = atomicAdd(&mine[rel >> 1], (rel & 1u) ? 0x10000u : 1u);
        }
#pragma unroll
        for (int u = 0; u < kV; ++u) {
            const int s = s0 + step * u + lane;
            const bool here = lane < step && s < s_n;
            const uint32_t rel = cs[u] - c_lo;
            uint32_t o = old[u][0];
#pragma unroll
            for (int j = 1; j < SUB; ++j) o = sub == j ? old[u][j] : o;
            if (here && rel < span)
                stage[(rel & 1u) ? o >> 16 : o & 0xffffu] = static_cast<uint16_t>(s_lo + s);
            if (last) {
                const bool out = here && cs[u] >= uint32_t(N);
                const uint64_t m = ballot(out);
                if (out) stage[pad_at + lanes_below(m)] = static_cast<uint16_t>(s_lo + s);
                pad_at += __popcll(m);
            }
        }
    }
    __syncthreads();
    int32_t* const ev = a.ev + int64_t(b) * T * K + first;
    const uint32_t inv = 0xffffffffu / uint32_t(K) + 1u;  // s / K for s < 2^15: exact (K = 1: 0)
    for (int i = tid; i < n_out; i += kThreads) {
        const uint32_t s = stage[i], t = K > 1 ? __umulhi(s, inv) : s;
        ev[i] = static_cast<int32_t>((t << 8) | (s - t * K));
    }
}

// ------------------------------------------------------------------------------------------
// Shared pieces of the chain kernels
// ------------------------------------------------------------------------------------------

constexpr int kChainWaves = 8;
constexpr int kChainThreads = 64 * kChainWaves;

// The row's reset table in LDS: nr[p] = the first reset at or after position p (T: none),
// p = 0..T, and the last reset of the row (-1: none), returned. `bits` [TW] and `nx` [TW + 1]
// are scratch.
__device__ __forceinline__ int reset_table(const uint8_t* reset_row, int T, int* nr,
                                           uint32_t* bits, int* nx, int tid, int nthreads) {
    const int TW = (T + 31) / 32;
    for (int t0 = 0; t0 < T; t0 += nthreads) {  // every wavefront ballots its 64 positions
        const int t = t0 + tid;
        const bool r = t < T && reset_row != nullptr && reset_row[t] != 0;
        const uint64_t m = ballot(r);
        if ((tid & 63) == 0 && t < T) {
            const int w = t / 32;
            bits[w] = static_cast<uint32_t>(m);
            if (w + 1 < TW) bits[w + 1] = static_cast<uint32_t>(m >> 32);
        }
    }
    __syncthreads();
    if (tid == 0) {
        int next = T;
        nx[TW] = T;
        for (int w = TW - 1; w >= 0; --w) {  // nx[w]: the first reset in words >= w
            const uint32_t v = bits[w];
            next = v ? w * 32 + __builtin_ctz(v) : next;
            nx[w] = next;
        }
        int last = -1;
        for (int w = TW - 1; w >= 0 && last < 0; --w)
            if (bits[w]) last = w * 32 + 31 - __builtin_clz(bits[w]);
        nr[T + 1] = last;  // passed on through LDS
    }
    __syncthreads();
    for (int p = tid; p <= T; p += nthreads) {
        if (p == T) {
            nr[T] = T;
        } else {
            const int w = p / 32;
            const uint32_t above = bits[w] & (0xffffffffu << (p & 31));  // positions >= p
            nr[p] = above ? w * 32 + __builtin_ctz(above) : nx[w + 1];
        }
    }
    __syncthreads();
    return nr[T + 1];
}

// (row, group) of a chain workgroup from the grid (8, G, B/8) (or (1, G, B)): the rows with the
// same blockIdx.x share an XCD, so a row's lists and shares stay in one L2.
__device__ __forceinline__ void group_coords(int& b, int& g) {
    b = blockIdx.x * gridDim.z + blockIdx.z;
    g = blockIdx.y;
}
inline dim3 chain_grid(int B, int G) {
    const int x = B % 8 == 0 ? 8 : 1;
    return dim3(x, G, B / x);
}

// LDS words of a chain workgroup: nr [T + 2], the reset bits [TW], their word table [TW + 1],
// the row maxima [T], the next cell to take, the group's list starts [C + 1], its staged events
// [stage] and its cells in the order they are taken [C].
__host__ __device__ inline int chain_words(int T, int C, int stage) {
    const int TW = (T + 31) / 32;
    return (T + 2) + TW + (TW + 1) + T + 1 + (C + 1) + stage + C;
}

// The group's cells heaviest first (most events; ties by cell), into order[0 .. nc): the
// wavefronts take cells in this order, so the long chains start first and the workgroup's
// wavefronts finish together (a workgroup holds its CU slot until its last wavefront ends).
// cptr must be visible to every thread; ends with a barrier.
__device__ __forceinline__ void heavy_first(const int* cptr, int nc, int* order, int tid,
                                            int nthreads) {
    for (int i = tid; i < nc; i += nthreads) {
        const int ni = cptr[i + 1] - cptr[i];
        int rank = 0;
        for (int j = 0; j < nc; ++j) {
            const int nj = cptr[j + 1] - cptr[j];
            rank += (nj > ni || (nj == ni && j < i)) ? 1 : 0;
        }
        order[rank] = i;
    }
    __syncthreads();
}

// The wavefront maximum of the bit patterns of |h| over the cell's columns (a NaN above +inf).
template <int V>
__device__ __forceinline__ uint32_t cell_abs_max(const float (&h)[V], int lane, int d) {
    uint32_t m = 0u;
#pragma unroll
    for (int v = 0; v < V; ++v) m = umax(m, lane + 64 * v < d ? abs_bits(h[v]) : 0u);
    return wave_max_from_groups<1>(m);
}

// The row maxima over positions [p0, p1) from one cell's value (bits): the first 64 positions
// inline (intervals are mostly shorter than a wavefront), the rest out of line.
__device__ __attribute__((noinline)) void max_interval_tail(uint32_t* hm, int p0, int p1,
                                                           uint32_t val, int lane) {
    for (int p = p0 + lane; p < p1; p += 64) atomicMax(&hm[p], val);
}
__device__ __forceinline__ void max_interval(uint32_t* hm, int p0, int p1, uint32_t val,
                                             int lane) {
    if (p0 + lane < p1) atomicMax(&hm[p0 + lane], val);
    if (unlikely(uniform(p1 - p0) > 64)) max_interval_tail(hm, p0 + 64, p1, val, lane);
}

// ------------------------------------------------------------------------------------------
// Forward chains
// ------------------------------------------------------------------------------------------

struct FwdArgs {
    const void* y;  // [B, T, K, d] io: the candidate's pre-activation (the RMS prologue's output)
    const void* g;  // the write gate's pre-activation
    const int32_t* ptr;  // the lists: [B, N + 1], [B, T * K]
    const int32_t* ev;
    const uint8_t* reset;  // [B, T] (null: none)
    const float* h0;       // [B, N, d]
    const int64_t* age0;   // [B, N] (with age_T)
    const int64_t* pos0;   // [B] (with pos_T)
    void* h_old;           // [B, T, K, d] io (optional)
    void* h_sel;           // (optional)
    float* delta;          // [B, T, K, d] fp32: h_sel - h_old of the valid slots (optional)
    uint32_t* hm_groups;   // [B, T, G]: each group's row maximum per position, |h| bits
                           // (optional: with the row maxima)
    float* h_T;            // [B, N, d] (optional)
    int64_t* age_T;        // [B, N] (optional)
    int64_t* pos_T;        // [B] (optional)
    int B, T, N, d, K;
    int C, stage;  // cells per workgroup, staged events per workgroup
    int heavy;     // chain_fwd4: cells of more events are walked alone
};

template <typename IO, int V>
__device__ __forceinline__ void fetch_rows(IO (&yv)[V], IO (&gv)[V], rsrc_t ry, rsrc_t rg,
                                           const uint32_t (&voff)[V], uint32_t so, bool in) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const uint32_t vo = in ? voff[v] : kOob;
        yv[v] = bload<IO>(ry, vo, so);
        gv[v] = bload<IO>(rg, vo, so);
    }
}

// The age of cell c at the window's end: its last event's position (-1: none) and the row's last reset.
__device__ __forceinline__ void end_age(const FwdArgs& a, int b, int c, int tprev, int lrT) {
    int64_t age;
    if (tprev >= 0 && tprev >= lrT) age = (a.T - 1) - tprev;
    else if (lrT >= 0) age = a.T - lrT;
    else age = a.age0[int64_t(b) * a.N + c] + a.T;
    a.age_T[int64_t(b) * a.N + c] = age;
}

// What a wavefront that walks one cell at a time holds of its row and its columns (lane + 64 v).
template <int V>
struct FwdRow {
    int b, pc0, nst, lrT, pad_begin;  // staged events: cev[0 .. nst) is ev[pc0 ..)
    const int32_t* ev;
    const int *cev, *nr;
    uint32_t* hm;
    rsrc_t ry, rg, rho, rhs, rdl;
    uint32_t srow, srow4, voff[V], voff4[V];
};
template <typename IO, int V>
__device__ __forceinline__ void column_offsets(int d, uint32_t (&voff)[V], uint32_t (&voff4)[V]) {
    const int lane = lane_id();
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const bool in = lane + 64 * v < d;
        voff[v] = in ? uint32_t(lane + 64 * v) * sizeof(IO) : kOob;
        voff4[v] = in ? uint32_t(lane + 64 * v) * 4u : kOob;
    }
}

// Cell c, whose events are the row's list from e_beg to e_end, by the whole wavefront; cell 0 takes the
// row's padded slots too (PADS: the caller has none, this is it, or look).
enum Pads { kNoPads, kPadCell, kPadsMaybe };
template <typename IO, int V, int NB, bool DELTA, bool HMAX, Pads PADS>
__device__ __forceinline__ void walk_cell(const FwdArgs& a, const FwdRow<V>& r, int c, int e_beg, int e_end) {
    const int lane = lane_id();
    const int T = a.T, N = a.N, d = a.d, K = a.K, n_slots = T * K;
    float h[V];
    const float* h0c = a.h0 + (int64_t(r.b) * N + c) * d;
#pragma unroll
    for (int v = 0; v < V; ++v) h[v] = lane + 64 * v < d ? h0c[lane + 64 * v] : 0.0f;
    float hold_last[V];  // the state before the latest event (cell 0's padded slots)
#pragma unroll
    for (int v = 0; v < V; ++v) hold_last[v] = 0.0f;
    uint32_t vprev = HMAX ? cell_abs_max<V>(h, lane, d) : 0u;
    int tprev = -1, s = 0;
    int nrprev = r.nr[0];  // the first reset after the latest event
    // cell 0's padded slots at positions below `limit`, in time order (a window of 64 of
    // them in the lanes)
    int pp = r.pad_begin, pwb = -1, pwv = 0;
    auto flush = [&](int limit) __attribute__((always_inline)) {
        while (pp < n_slots) {
            if (pwb < 0 || pp >= pwb + kEvWin) {
                pwb = pp;
                pwv = lane < n_slots - pp ? r.ev[pp + lane] : 0x7fffffff;
            }
            const int off = pp - pwb;
            const uint64_t below = ballot(lane >= off && (pwv >> 8) < limit);
            const int n = __popcll(below);
            for (int i = 0; i < n; ++i) {
                const int q = __builtin_amdgcn_readlane(pwv, off + i);
                const int t = q >> 8;
                const uint32_t so = uint32_t(t * K + (q & 255)) * r.srow;
                const bool same = t == tprev;
                const bool zero = nrprev <= t;
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    const float now = zero ? 0.0f : h[v];
                    bstore_f32<IO>(same ? hold_last[v] : now, r.rho, r.voff[v], so);
                    bstore_f32<IO>(same ? h[v] : now, r.rhs, r.voff[v], so);
                }
            }
            pp += n;
            if (off + n < kEvWin) break;  // the next one is at or after `limit`
        }
    };
    const bool pad_here = PADS == kPadCell || (PADS == kPadsMaybe && c == 0 && r.pad_begin < n_slots);
    // one event: position t, its slot's byte offsets (so: storage rows, so4: fp32 rows) and
    // the first reset after t
    auto update = [&](auto pad_c, int t, uint32_t so, uint32_t so4, int nrq, const IO (&yv)[V],
                      const IO (&gv)[V]) __attribute__((always_inline)) {
        constexpr bool kPad = decltype(pad_c)::value;
        const bool zero = nrprev <= t;  // a reset since the cell's last event
        if constexpr (HMAX) max_interval(r.hm, s, min(t, nrprev), vprev, lane);
        if constexpr (kPad) flush(t);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const float hold = zero ? 0.0f : h[v];
            const float bg = fast_sigmoid(to_f32(gv[v]));
            const float cand = fast_tanh(to_f32(yv[v]));
            const float hn = (1.0f - bg) * hold + bg * cand;
            bstore_f32<IO>(hold, r.rho, r.voff[v], so);
            bstore_f32<IO>(hn, r.rhs, r.voff[v], so);
            if constexpr (DELTA) bstore(hn - hold, r.rdl, r.voff4[v], so4);
            if constexpr (kPad) hold_last[v] = hold;
            h[v] = hn;
        }
        if constexpr (HMAX) vprev = cell_abs_max<V>(h, lane, d);
        s = t;
        tprev = t;
        nrprev = nrq;
        if constexpr (kPad) flush(t + 1);
    };
    // windows of 64 events (one per lane), in batches of NB with two batches in flight; a
    // window's positions, slot offsets and next resets are computed for all its events at
    // once (lane i: event i) and read per event with readlane
    auto walk = [&](auto staged_c, auto pad_c) __attribute__((always_inline)) {
        constexpr bool kStaged = decltype(staged_c)::value;
        for (int w0 = e_beg; w0 < e_end; w0 += kEvWin) {
            const int m = min(kEvWin, e_end - w0);
            int evw;
            if constexpr (kStaged) evw = lane < m ? r.cev[w0 - r.pc0 + lane] : 0;
            else evw = lane < m ? r.ev[w0 + lane] : 0;
            const int tw = evw >> 8;
            const int slw = tw * K + (evw & 255);
            const uint32_t sow = uint32_t(slw) * r.srow;
            const uint32_t so4w = uint32_t(slw) * r.srow4;
            const int nrw = lane < m ? r.nr[tw + 1] : T;
            IO ya[NB][V], ga[NB][V], yb[NB][V], gb[NB][V];
            auto fetch = [&](int j, IO (&yv)[NB][V], IO (&gv)[NB][V])
                             __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const uint32_t so = __builtin_amdgcn_readlane(sow, min(j + i, kEvWin - 1));
                    fetch_rows<IO, V>(yv[i], gv[i], r.ry, r.rg, r.voff, so, j + i < m);
                }
            };
            auto step = [&](int j, const IO (&yv)[NB][V], const IO (&gv)[NB][V])
                            __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    if (j + i < m) {
                        const int idx = j + i;
                        update(pad_c, __builtin_amdgcn_readlane(tw, idx),
                               __builtin_amdgcn_readlane(sow, idx),
                               DELTA ? __builtin_amdgcn_readlane(so4w, idx) : 0u,
                               __builtin_amdgcn_readlane(nrw, idx), yv[i], gv[i]);
                    }
                }
            };
            fetch(0, ya, ga);
            for (int j = 0; j < m; j += 2 * NB) {
                fetch(j + NB, yb, gb);
                step(j, ya, ga);
                if (j + NB >= m) break;
                fetch(j + 2 * NB, ya, ga);
                step(j + NB, yb, gb);
            }
        }
    };
    if constexpr (PADS == kPadCell) {
        walk(std::false_type{}, std::true_type{});
    } else {
        if (PADS == kPadsMaybe && pad_here) walk(std::false_type{}, std::true_type{});
        else if (e_end - r.pc0 <= r.nst) walk(std::true_type{}, std::false_type{});
        else walk(std::false_type{}, std::false_type{});
    }
    if (PADS != kNoPads && pad_here) flush(T);
    if constexpr (HMAX) max_interval(r.hm, s, min(T, nrprev), vprev, lane);
    const bool cleared = nrprev < T;  // a reset after the cell's last event
    if (a.h_T) {
        float* hTc = a.h_T + (int64_t(r.b) * N + c) * d;
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (lane + 64 * v < d) hTc[lane + 64 * v] = cleared ? 0.0f : h[v];
    }
    if (a.age_T && lane == 0) end_age(a, r.b, c, tprev, r.lrT);
}

template <typename IO, int V, int NB, bool DELTA, bool HMAX>
__global__ __launch_bounds__(kChainThreads) void chain_fwd(FwdArgs a) {
    extern __shared__ uint32_t lds_u[];
    int b, g;
    group_coords(b, g);
    const int tid = threadIdx.x, lane = lane_id();
    const int T = a.T, N = a.N, d = a.d, K = a.K;
    const int TW = (T + 31) / 32;
    int* nr = reinterpret_cast<int*>(lds_u);             // [T + 2]
    uint32_t* rbits = lds_u + (T + 2);                   // [TW]
    int* nx = reinterpret_cast<int*>(rbits + TW);        // [TW + 1]
    uint32_t* hm = reinterpret_cast<uint32_t*>(nx + TW + 1);  // [T]
    int* next = reinterpret_cast<int*>(hm + T);          // [1]
    int* cptr = next + 1;                                // [C + 1]
    int* cev = cptr + a.C + 1;                           // [stage]
    int* order = cev + a.stage;                          // [C]
    const int c_begin = g * a.C, c_end = min(N, c_begin + a.C);
    const int nc = c_end - c_begin;
    const int32_t* ptr = a.ptr + int64_t(b) * (N + 1);
    const int32_t* ev = a.ev + int64_t(b) * T * K;
    // the group's list starts and its first `stage` events, staged once for every wavefront
    const int pc0 = ptr[c_begin];
    const int nst = min(ptr[c_end] - pc0, a.stage);
    for (int i = tid; i <= nc; i += kChainThreads) cptr[i] = ptr[c_begin + i];
    for (int i = tid; i < nst; i += kChainThreads) cev[i] = ev[pc0 + i];
    for (int p = tid; p < T; p += kChainThreads) hm[p] = 0u;
    if (tid == 0) next[0] = 0;
    const int lrT = reset_table(a.reset ? a.reset + int64_t(b) * T : nullptr, T, nr, rbits, nx,
                                tid, kChainThreads);
    heavy_first(cptr, nc, order, tid, kChainThreads);
    const int64_t slot0 = int64_t(b) * T * K;
    const uint32_t row_bytes = uint32_t(T) * K * d * sizeof(IO);
    FwdRow<V> r;
    r.b = b, r.pc0 = pc0, r.nst = nst, r.lrT = lrT, r.pad_begin = ptr[N];
    r.ev = ev, r.cev = cev, r.nr = nr, r.hm = hm;
    r.ry = make_rsrc(static_cast<const IO*>(a.y) + slot0 * d, row_bytes);
    r.rg = make_rsrc(static_cast<const IO*>(a.g) + slot0 * d, row_bytes);
    r.rho = make_rsrc(a.h_old ? static_cast<IO*>(a.h_old) + slot0 * d : nullptr, a.h_old ? row_bytes : 0u);
    r.rhs = make_rsrc(a.h_sel ? static_cast<IO*>(a.h_sel) + slot0 * d : nullptr, a.h_sel ? row_bytes : 0u);
    r.rdl = make_rsrc(a.delta ? a.delta + slot0 * d : nullptr, a.delta ? uint32_t(T) * K * d * 4u : 0u);
    r.srow = uint32_t(d) * sizeof(IO), r.srow4 = uint32_t(d) * 4u;
    column_offsets<IO, V>(d, r.voff, r.voff4);

    for (;;) {
        int slot = lane == 0 ? atomicAdd(next, 1) : 0;
        slot = __builtin_amdgcn_readfirstlane(slot);
        if (slot >= nc) break;
        const int ci = uniform(order[slot]);
        const int c = c_begin + ci;
        const int e_beg = uniform(cptr[ci]), e_end = uniform(cptr[ci + 1]);
        walk_cell<IO, V, NB, DELTA, HMAX, kPadsMaybe>(a, r, c, e_beg, e_end);
    }
    if (a.pos_T && g == 0 && tid == 0) a.pos_T[b] = lrT >= 0 ? int64_t(T - lrT) : a.pos0[b] + T;
    if (HMAX) {  // the group's maxima, reduced over the groups by summary_delta
        __syncthreads();
        const int G = gridDim.y;
        uint32_t* hg = a.hm_groups + int64_t(b) * T * G + g;
        for (int p = tid; p < T; p += kChainThreads) hg[int64_t(p) * G] = hm[p];
    }
}

// ------------------------------------------------------------------------------------------
// The summary: the valid slots' delta sum per position, then a scan over time
// ------------------------------------------------------------------------------------------

struct DeltaArgs {
    const void* h_old;    // [B, T, K, d] io (PAIR)
    const void* h_sel;
    const float* delta;   // [B, T, K, d] fp32 (not PAIR)
    const int32_t* slots; // [B, T, K]
    float* D;             // [B, T, d]
    const uint32_t* hm_groups;  // [B, T, G] (optional)
    float* h_max;         // [B, T]: the maximum over the groups (with hm_groups)
    int B, T, N, d, K, G;
};

// A wavefront per (row, position), lanes over the columns: D[t] = the sum over the position's
// valid slots, in slot order, of h_sel - h_old as stored (PAIR: fp32 rows, the forward's own
// values) or of the chains' fp32 deltas (bf16 rows, or an omitted h_old / h_sel).
template <typename IO, int V, bool PAIR>
__global__ __launch_bounds__(256) void summary_delta(DeltaArgs a) {
    const int pos = blockIdx.x * 4 + uniform(threadIdx.x / 64);
    const int b = blockIdx.y;
    if (pos >= a.T) return;
    const int lane = lane_id();
    const int d = a.d, K = a.K;
    const int64_t slot0 = (int64_t(b) * a.T + pos) * K;
    const rsrc_t r1 = PAIR ? make_rsrc(static_cast<const IO*>(a.h_sel) + slot0 * d, uint32_t(K) * d * sizeof(IO))
                           : make_rsrc(a.delta + slot0 * d, uint32_t(K) * d * 4u);
    const rsrc_t r0 = make_rsrc(PAIR ? static_cast<const IO*>(a.h_old) + slot0 * d : nullptr,
                                PAIR ? uint32_t(K) * d * sizeof(IO) : 0u);
    constexpr uint32_t E = PAIR ? sizeof(IO) : 4u;
    uint32_t voff[V];
#pragma unroll
    for (int v = 0; v < V; ++v) voff[v] = lane + 64 * v < d ? uint32_t(lane + 64 * v) * E : kOob;
    float D[V];
#pragma unroll
    for (int v = 0; v < V; ++v) D[v] = 0.0f;
    constexpr int kU = 8;
    for (int k64 = 0; k64 < K; k64 += 64) {
        const uint64_t okm = ballot(k64 + lane < K && slot_cell(a.slots, slot0 + k64 + lane, a.N) >= 0);
        for (int k0 = 0; k0 < min(64, K - k64); k0 += kU) {
            float s1[kU][V], s0[kU][V];
#pragma unroll
            for (int i = 0; i < kU; ++i) {
                const int k = k64 + k0 + i;
                const bool ok = k0 + i < 64 && ((okm >> min(k0 + i, 63)) & 1ull) && k < K;
                const uint32_t so = uint32_t(min(k, K - 1)) * d * E;
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    const uint32_t vo = ok ? voff[v] : kOob;
                    if constexpr (PAIR) {
                        s1[i][v] = to_f32(bload<IO>(r1, vo, so));
                        s0[i][v] = to_f32(bload<IO>(r0, vo, so));
                    } else {
                        s1[i][v] = bload<float>(r1, vo, so);
                        s0[i][v] = 0.0f;
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < kU; ++i)
#pragma unroll
                for (int v = 0; v < V; ++v) D[v] += PAIR ? s1[i][v] - s0[i][v] : s1[i][v];
        }
    }
    float* Dp = a.D + (int64_t(b) * a.T + pos) * d;
#pragma unroll
    for (int v = 0; v < V; ++v)
        if (lane + 64 * v < d) Dp[lane + 64 * v] = D[v];
    if (a.hm_groups) {  // the row maximum: the largest of the groups' (|h| bits, NaN above inf)
        const uint32_t* hg = a.hm_groups + (int64_t(b) * a.T + pos) * a.G;
        uint32_t m = 0u;
        for (int g = lane; g < a.G; g += 64) m = umax(m, hg[g]);
        m = wave_max_from_groups<1>(m);
        if (lane == 0) a.h_max[int64_t(b) * a.T + pos] = __uint_as_float(m);
    }
}

constexpr int kScanWaves = 16;

struct ScanArgs {
    // forward: D [B, T, d] fp32 -> q_pre, q_post [B, T, d] io (optional), q_T [B, d] from q0
    const float* D;
    const float* q0;
    void* q_pre;
    void* q_post;
    float* q_T;
    // backward: dq_pre, dq_post [B, T, d] io (optional), dq_T [B, d] (optional) -> the share
    // R / N [B, T, d] fp32 and d_q0 [B, d] (optional)
    const void* dq_pre;
    const void* dq_post;
    const float* dq_T;
    float* share;
    float* dq0;
    const uint8_t* reset;  // [B, T] (optional)
    int B, T, d;
    DivN divn;
};

// (row, 64 columns): 16 wavefronts over consecutive ranges of 32 positions, in rounds of 512
// positions. A range maps the summary q to (reset in range ? 0 : q) + c, c its D / N sum after
// its last reset; the wavefronts exchange (reset, c) through LDS, each folds the earlier ones'
// into its start value and replays its positions in the reference's order per position
// (python/hsn/kernels/native.py:302 with state.py:267-283): q_pre[t] = (reset[t] ? 0 : q),
// q_post[t] = q_pre[t] + D[t] / N. Rows of [., T, d] tensors are buffer resources: a lane's
// column is its voffset, the position a uniform soffset (kept inside the row: only the voffset
// masks an access).
template <typename IO>
__global__ __launch_bounds__(64 * kScanWaves) void summary_scan_fwd(ScanArgs a) {
    __shared__ int rss[kScanWaves];
    __shared__ float cx[kScanWaves][64];
    const int b = blockIdx.y, z = blockIdx.x;
    const int lane = lane_id(), w = uniform(threadIdx.x / 64);
    const int x = z * 64 + lane;
    const bool col = x < a.d;
    const int T = a.T, d = a.d;
    const DivN divn = a.divn;
    const int64_t row = int64_t(b) * T * d;
    const rsrc_t rD = make_rsrc(a.D + row, uint32_t(T) * d * 4u);
    const rsrc_t rqa = make_rsrc(a.q_pre ? static_cast<IO*>(a.q_pre) + row : nullptr,
                                 a.q_pre ? uint32_t(T) * d * sizeof(IO) : 0u);
    const rsrc_t rqb = make_rsrc(a.q_post ? static_cast<IO*>(a.q_post) + row : nullptr,
                                 a.q_post ? uint32_t(T) * d * sizeof(IO) : 0u);
    const uint32_t vo4 = col ? uint32_t(x) * 4u : kOob, vo = col ? uint32_t(x) * sizeof(IO) : kOob;
    float q = col ? a.q0[int64_t(b) * d + x] : 0.0f;
    constexpr int kR = 32;
    for (int r0 = 0; r0 < T; r0 += kR * kScanWaves) {
        const int t0 = r0 + w * kR;
        float Dv[kR];
#pragma unroll
        for (int j = 0; j < kR; ++j) {  // past T: the lane offset masks the load (reads 0)
            const bool in = t0 + j < T;
            Dv[j] = bload<float>(rD, in ? vo4 : kOob, uint32_t(in ? t0 + j : 0) * d * 4u);
        }
        const uint32_t rsm = static_cast<uint32_t>(ballot(
            lane < kR && t0 + lane < T && a.reset != nullptr && a.reset[int64_t(b) * T + t0 + lane] != 0));
        float c = 0.0f;
#pragma unroll
        for (int j = 0; j < kR; ++j) {
            if ((rsm >> j) & 1u) c = 0.0f;
            c += divn(Dv[j]);
        }
        if (lane == 0) rss[w] = rsm != 0u ? 1 : 0;
        cx[w][lane] = c;
        __syncthreads();
        float qs = q;  // this range's start value
        for (int j = 0; j < w; ++j) qs = (rss[j] ? 0.0f : qs) + cx[j][lane];
        float qe = qs;  // the round's end value
        for (int j = w; j < kScanWaves; ++j) qe = (rss[j] ? 0.0f : qe) + cx[j][lane];
        float qq = qs;
#pragma unroll
        for (int j = 0; j < kR; ++j) {  // past T: the lane offset drops the stores
            const bool in = t0 + j < T;
            const uint32_t so = uint32_t(in ? t0 + j : 0) * d * sizeof(IO);
            const uint32_t vj = in ? vo : kOob;
            if ((rsm >> j) & 1u) qq = 0.0f;
            bstore_f32<IO>(qq, rqa, vj, so);
            qq = qq + divn(Dv[j]);
            bstore_f32<IO>(qq, rqb, vj, so);
        }
        q = qe;
        __syncthreads();  // before the next round reuses the exchange
    }
    if (a.q_T && w == 0 && col) a.q_T[int64_t(b) * d + x] = q;
}

// The reverse scan of the summary cotangent (python/hsn/train/split.py:154-173): latest first,
// R += dq_post[t]; share[t] = R / N; R += dq_pre[t]; a reset at t zeroes R after it. In fp64
// (so the ranges' composition rounds no differently from a sequential sum), each share rounded
// once to fp32.
template <typename IO>
__global__ __launch_bounds__(64 * kScanWaves) void summary_scan_bwd(ScanArgs a) {
    __shared__ int rss[kScanWaves];
    __shared__ double cx[kScanWaves][64];
    const int b = blockIdx.y, z = blockIdx.x;
    const int lane = lane_id(), w = uniform(threadIdx.x / 64);
    const int x = z * 64 + lane;
    const bool col = x < a.d;
    const int T = a.T, d = a.d;
    const DivN divn = a.divn;
    const int64_t row = int64_t(b) * T * d;
    const rsrc_t rpa = make_rsrc(a.dq_pre ? static_cast<const IO*>(a.dq_pre) + row : nullptr,
                                 a.dq_pre ? uint32_t(T) * d * sizeof(IO) : 0u);
    const rsrc_t rpb = make_rsrc(a.dq_post ? static_cast<const IO*>(a.dq_post) + row : nullptr,
                                 a.dq_post ? uint32_t(T) * d * sizeof(IO) : 0u);
    const rsrc_t rsh = make_rsrc(a.share + row, uint32_t(T) * d * 4u);
    const uint32_t vo4 = col ? uint32_t(x) * 4u : kOob, vo = col ? uint32_t(x) * sizeof(IO) : kOob;
    double R = (col && a.dq_T) ? double(a.dq_T[int64_t(b) * d + x]) : 0.0;
    constexpr int kR = 16;  // two values per position, within 128 registers
    const int span = kR * kScanWaves;
    const int rounds = (T + span - 1) / span;
    for (int rr = rounds - 1; rr >= 0; --rr) {
        const int t0 = rr * span + w * kR;
        float va[kR], vb[kR];
#pragma unroll
        for (int j = 0; j < kR; ++j) {  // past T: the lane offset masks the loads (reads 0)
            const bool in = t0 + j < T;
            const uint32_t so = uint32_t(in ? t0 + j : 0) * d * sizeof(IO);
            va[j] = to_f32(bload<IO>(rpa, in ? vo : kOob, so));
            vb[j] = to_f32(bload<IO>(rpb, in ? vo : kOob, so));
        }
        const uint32_t rsm = static_cast<uint32_t>(ballot(
            lane < kR && t0 + lane < T && a.reset != nullptr && a.reset[int64_t(b) * T + t0 + lane] != 0));
        double c = 0.0;  // this range's map on R, latest first: R -> (reset ? 0 : R) + c
#pragma unroll
        for (int j = kR - 1; j >= 0; --j) {
            c += double(vb[j]);
            c += double(va[j]);
            if ((rsm >> j) & 1u) c = 0.0;
        }
        if (lane == 0) rss[w] = rsm != 0u ? 1 : 0;
        cx[w][lane] = c;
        __syncthreads();
        double Rs = R;  // R entering this range: the later ranges' maps applied
        for (int j = kScanWaves - 1; j > w; --j) Rs = (rss[j] ? 0.0 : Rs) + cx[j][lane];
        double Re = Rs;
        for (int j = w; j >= 0; --j) Re = (rss[j] ? 0.0 : Re) + cx[j][lane];
        double Rr = Rs;
#pragma unroll
        for (int j = kR - 1; j >= 0; --j) {
            Rr += double(vb[j]);
            const bool in = t0 + j < T;
            bstore(static_cast<float>(divn(Rr)), rsh, in ? vo4 : kOob, uint32_t(in ? t0 + j : 0) * d * 4u);
            Rr += double(va[j]);
            if ((rsm >> j) & 1u) Rr = 0.0;
        }
        R = Re;
        __syncthreads();
    }
    if (a.dq0 && w == 0 && col) a.dq0[int64_t(b) * d + x] = static_cast<float>(R);
}

// ------------------------------------------------------------------------------------------
// Backward chains
// ------------------------------------------------------------------------------------------

struct BwdArgs {
    const void* y;      // [B, T, K, d] io: the candidate's pre-activation (RMS: normalised)
    const void* g;      // the gate's pre-activation
    const void* h_old;
    const void* dsel;   // optional
    const int32_t* ptr;
    const int32_t* ev;
    const uint8_t* reset;
    const float* share;  // [B, T, d]
    const float* dh_T;   // optional [B, N, d]
    void* dy;
    void* dg;
    float* dh0;  // optional
    int B, T, N, d, K;
    int C, stage, heavy;
};

// The backward's FwdRow.
template <int V>
struct BwdRow {
    int b, pc0, nst;
    const int32_t* ev;
    const int *cev, *nr;
    rsrc_t ry, rg, rho, rds, rdy, rdg, rsh;
    uint32_t srow, srow4, voff[V], voff4[V];
};

// Per cell, latest event first (python/hsn/train/split.py:154-173): with the cotangent A of the
// cell's state after the event and the share R / N of its position, g = A + d_h_sel + R / N;
// dc = b g, db = (c - h_old) g, then through c = tanh(y) and b = sigmoid(gate); the state before
// the event gets (1 - b)(A + d_h_sel) - b R / N (h_old enters the summary's delta with -1 / N).
template <typename IO, int V, int NB>
__device__ __forceinline__ void walk_cell(const BwdArgs& a, const BwdRow<V>& r, int c, int e_beg, int e_end) {
    const int lane = lane_id();
    const int T = a.T, N = a.N, d = a.d, K = a.K;
    struct Rows {
        IO y[NB][V], g[NB][V], h[NB][V], s[NB][V];
        float r[NB][V];
    };
    const bool staged = e_end - r.pc0 <= r.nst;
    float A[V];
    {  // the end cotangent, cut by a reset after the cell's last event
        const int t_last = e_end > e_beg
                               ? (uniform(staged ? r.cev[e_end - 1 - r.pc0] : r.ev[e_end - 1]) >> 8)
                               : -1;
        const bool cut = r.nr[t_last + 1] < T;
        const float* dhc = a.dh_T ? a.dh_T + (int64_t(r.b) * N + c) * d : nullptr;
#pragma unroll
        for (int v = 0; v < V; ++v)
            A[v] = (dhc && !cut && lane + 64 * v < d) ? dhc[lane + 64 * v] : 0.0f;
    }
    int tnext = T;  // the later event's position
    int t_first = T;
    auto walk = [&](auto staged_c) __attribute__((always_inline)) {
        constexpr bool kStaged = decltype(staged_c)::value;
        for (int w1 = e_end; w1 > e_beg; w1 -= kEvWin) {
            const int m = min(kEvWin, w1 - e_beg);
            const int w0 = w1 - m;
            int evw;
            if constexpr (kStaged) evw = lane < m ? r.cev[w0 - r.pc0 + lane] : 0;
            else evw = lane < m ? r.ev[w0 + lane] : 0;
            // the window's positions, slot offsets, share offsets and next resets, for all
            // its events at once (lane i: event i), read per event with readlane
            const int tw = evw >> 8;
            const uint32_t sow = uint32_t(tw * K + (evw & 255)) * r.srow;
            const uint32_t stw = uint32_t(tw) * r.srow4;
            const int nrw = lane < m ? r.nr[tw + 1] : T;
            Rows qa, qb;
            // batch j holds window indices [j - NB + 1, j], fetched latest first
            auto fetch = [&](int j, Rows& q) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int idx = j - i;
                    const uint32_t so = __builtin_amdgcn_readlane(sow, max(idx, 0));
                    const uint32_t st = __builtin_amdgcn_readlane(stw, max(idx, 0));
                    const bool in = idx >= 0;
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        const uint32_t vo = in ? r.voff[v] : kOob;
                        q.y[i][v] = bload<IO>(r.ry, vo, so);
                        q.g[i][v] = bload<IO>(r.rg, vo, so);
                        q.h[i][v] = bload<IO>(r.rho, vo, so);
                        q.s[i][v] = bload<IO>(r.rds, vo, so);
                        q.r[i][v] = bload<float>(r.rsh, in ? r.voff4[v] : kOob, st);
                    }
                }
            };
            auto step = [&](int j, const Rows& q) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int idx = j - i;
                    if (idx >= 0) {
                        const int t = __builtin_amdgcn_readlane(tw, idx);
                        const int nrq = __builtin_amdgcn_readlane(nrw, idx);
                        const uint32_t so = __builtin_amdgcn_readlane(sow, idx);
                        const bool zero = nrq <= tnext && tnext < T;  // a reset in (t, tnext]
#pragma unroll
                        for (int v = 0; v < V; ++v) {
                            const float carried = (zero ? 0.0f : A[v]) + to_f32(q.s[i][v]);
                            const float share = q.r[i][v];
                            const float gg = carried + share;
                            const float bg = fast_sigmoid(to_f32(q.g[i][v]));
                            const float cc = fast_tanh(to_f32(q.y[i][v]));
                            const float dc = bg * gg * (1.0f - cc * cc);
                            const float db = (cc - to_f32(q.h[i][v])) * gg * (bg * (1.0f - bg));
                            bstore_f32<IO>(dc, r.rdy, r.voff[v], so);
                            bstore_f32<IO>(db, r.rdg, r.voff[v], so);
                            A[v] = (1.0f - bg) * carried - bg * share;
                        }
                        tnext = t;
                    }
                }
            };
            fetch(m - 1, qa);
            for (int j = m - 1; j >= 0; j -= 2 * NB) {
                fetch(j - NB, qb);
                step(j, qa);
                if (j - NB < 0) break;
                fetch(j - 2 * NB, qa);
                step(j - NB, qb);
            }
        }
    };
    if (staged) walk(std::true_type{});
    else walk(std::false_type{});
    t_first = tnext;
    if (a.dh0) {  // the start state's cotangent: cut by a reset at or before the first event
        const bool z = r.nr[0] <= min(t_first, T - 1);
        float* d0 = a.dh0 + (int64_t(r.b) * N + c) * d;
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (lane + 64 * v < d) d0[lane + 64 * v] = z ? 0.0f : A[v];
    }
}

template <typename IO, int V, int NB>
__global__ __launch_bounds__(kChainThreads) void chain_bwd(BwdArgs a) {
    extern __shared__ uint32_t lds_u[];
    int b, g;
    group_coords(b, g);
    const int tid = threadIdx.x, lane = lane_id();
    const int T = a.T, N = a.N, d = a.d, K = a.K;
    const int TW = (T + 31) / 32;
    int* nr = reinterpret_cast<int*>(lds_u);
    uint32_t* rbits = lds_u + (T + 2);
    int* nx = reinterpret_cast<int*>(rbits + TW);
    int* next = nx + TW + 1 + T;  // the layout of chain_fwd (no row maxima used)
    int* cptr = next + 1;
    int* cev = cptr + a.C + 1;
    int* order = cev + a.stage;
    const int c_begin = g * a.C, c_end = min(N, c_begin + a.C);
    const int nc = c_end - c_begin;
    const int32_t* ptr = a.ptr + int64_t(b) * (N + 1);
    const int32_t* ev = a.ev + int64_t(b) * T * K;
    const int pc0 = ptr[c_begin];
    const int nst = min(ptr[c_end] - pc0, a.stage);
    for (int i = tid; i <= nc; i += kChainThreads) cptr[i] = ptr[c_begin + i];
    for (int i = tid; i < nst; i += kChainThreads) cev[i] = ev[pc0 + i];
    if (tid == 0) next[0] = 0;
    reset_table(a.reset ? a.reset + int64_t(b) * T : nullptr, T, nr, rbits, nx, tid, kChainThreads);
    heavy_first(cptr, nc, order, tid, kChainThreads);
    const int64_t slot0 = int64_t(b) * T * K;
    const uint32_t row_bytes = uint32_t(T) * K * d * sizeof(IO);
    BwdRow<V> r;
    r.b = b, r.pc0 = pc0, r.nst = nst, r.ev = ev, r.cev = cev, r.nr = nr;
    r.ry = make_rsrc(static_cast<const IO*>(a.y) + slot0 * d, row_bytes);
    r.rg = make_rsrc(static_cast<const IO*>(a.g) + slot0 * d, row_bytes);
    r.rho = make_rsrc(static_cast<const IO*>(a.h_old) + slot0 * d, row_bytes);
    r.rds = make_rsrc(a.dsel ? static_cast<const IO*>(a.dsel) + slot0 * d : nullptr, a.dsel ? row_bytes : 0u);
    r.rdy = make_rsrc(static_cast<IO*>(a.dy) + slot0 * d, row_bytes);
    r.rdg = make_rsrc(static_cast<IO*>(a.dg) + slot0 * d, row_bytes);
    r.rsh = make_rsrc(a.share + int64_t(b) * T * d, uint32_t(T) * d * 4u);
    r.srow = uint32_t(d) * sizeof(IO), r.srow4 = uint32_t(d) * 4u;
    column_offsets<IO, V>(d, r.voff, r.voff4);
    const int n_slots = T * K;
    const int pad_begin = ptr[N];

    for (;;) {
        int slot = lane == 0 ? atomicAdd(next, 1) : 0;
        slot = __builtin_amdgcn_readfirstlane(slot);
        if (slot >= nc) break;
        const int ci = uniform(order[slot]);
        const int c = c_begin + ci;
        const int e_beg = uniform(cptr[ci]), e_end = uniform(cptr[ci + 1]);
        walk_cell<IO, V, NB>(a, r, c, e_beg, e_end);
    }
    if (g == 0) {  // exact zeros on the row's padded slots, every wavefront a share
        const int wv = tid >> 6;
        for (int pw = pad_begin + wv * kEvWin; pw < n_slots; pw += kEvWin * kChainWaves) {
            const int m = min(kEvWin, n_slots - pw);
            const int pe = lane < m ? ev[pw + lane] : 0;
            for (int i = 0; i < m; ++i) {
                const int q = __builtin_amdgcn_readlane(pe, i);
                const uint32_t so = uint32_t((q >> 8) * K + (q & 255)) * r.srow;
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    bstore_f32<IO>(0.0f, r.rdy, r.voff[v], so);
                    bstore_f32<IO>(0.0f, r.rdg, r.voff[v], so);
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// The chains, several cells a wavefront (chain_fwd4, chain_bwd4)
// ------------------------------------------------------------------------------------------
//
// For d a multiple of 4 up to 128 and rows aligned to four elements, a cell's columns lie in L
// lanes, four a lane (16-byte accesses of fp32 rows, 8-byte ones of bf16), and a wavefront walks
// 64 / L cells side by side, so one instruction serves an event of each. The cells are taken
// heaviest first, so neighbours hold about as many events; a lane whose cell has no event left
// masks its accesses. A cell of more than kHeavy events is walked by a wavefront alone, a column a
// lane: side by side, the longest chain of a workgroup takes each event at the pace of four cells'
// instructions (N 4096 with a Zipf bias, 1024 events in the heaviest cells: forward 2.18 ms, all
// cells side by side, 1.64 with the heavy ones alone).
//
// What bounds it is a cell's chain of loads, with 64 / L cells' rows in flight a wavefront. Measured
// (us, forward and backward; one cell a wavefront in brackets): B64 T512 N1024 d64 K16 bf16 96 and
// 106 (128 and 133); B128 T128 N512 d128 K8 fp32 70 and 101 (80 and 123), 67 and 93 being their
// bytes at a copy's 5.03 TB/s; B256 T1024 N4096 d64 K32 bf16 Zipf 1681 and 1717 (1734 forward; the backward
// on one card 1804 against 1786: a few cells' serial chains, which nothing beside them shortens, but 1472
// against 1661 for evenly popular cells). Four wavefronts a workgroup instead of eight 109 and 120 at the
// first shape, batches of four events 97 and 116. The cells a workgroup and the events up to which a
// cell is walked beside others follow from the shape (quad_cells, quad_heavy in chain.hip).
//
// The row maxima are marked per interval between a cell's events on three scales (positions, 16
// and 256 of them), at most five LDS atomics an interval instead of one a position and wavefront;
// cells without an event keep one maximum a wavefront.

constexpr int kQuadWaves = 8;
constexpr int kQuadThreads = 64 * kQuadWaves;
constexpr int kHeavy = 64;  // and the limit of FwdArgs / BwdArgs::heavy
constexpr int NB = 2;  // events of a cell in a batch, two batches in flight

struct RawB { uint32_t v[2]; };  // four bf16
struct RawF { uint32_t v[4]; };  // four fp32
template <typename IO>
using Raw = std::conditional_t<sizeof(IO) == 4, RawF, RawB>;

__device__ __forceinline__ RawF load_raw(rsrc_t r, uint32_t vo, const float*) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, vo, 0u, 0);
    return RawF{{v[0], v[1], v[2], v[3]}};
}
__device__ __forceinline__ RawB load_raw(rsrc_t r, uint32_t vo, const bf16_t*) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, vo, 0u, 0);
    return RawB{{static_cast<uint32_t>(v[0]), static_cast<uint32_t>(v[1])}};
}
__device__ __forceinline__ float lane_of(const RawF& q, int i) { return __uint_as_float(q.v[i]); }
__device__ __forceinline__ float lane_of(const RawB& q, int i) {
    return __uint_as_float(i & 1 ? q.v[i / 2] & 0xffff0000u : q.v[i / 2] << 16);
}
__device__ __forceinline__ void store4(const float (&x)[4], rsrc_t r, uint32_t vo, const float*) {
    decltype(__builtin_amdgcn_raw_buffer_load_b128(r, 0u, 0u, 0)) v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __float_as_uint(x[i]);
    __builtin_amdgcn_raw_buffer_store_b128(v, r, vo, 0u, 0);
}
__device__ __forceinline__ void store4(const float (&x)[4], rsrc_t r, uint32_t vo, const bf16_t*) {
    decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0u, 0u, 0)) v;
    v[0] = uint32_t(from_f32<bf16_t>(x[0]).bits) | uint32_t(from_f32<bf16_t>(x[1]).bits) << 16;
    v[1] = uint32_t(from_f32<bf16_t>(x[2]).bits) | uint32_t(from_f32<bf16_t>(x[3]).bits) << 16;
    __builtin_amdgcn_raw_buffer_store_b64(v, r, vo, 0u, 0);
}

// LDS words of a quad workgroup: chain_words, the maxima's two coarse scales and the order's bins.
constexpr int kLightBins = 65, kHeavyBins = 72, kOrderBins = kHeavyBins + kLightBins;
__host__ __device__ inline int coarse_words(int T) { return (T + 15) / 16 + (T + 255) / 256; }
__host__ __device__ inline int quad_words(int T, int C, int stage) {
    return chain_words(T, C, stage) + coarse_words(T) + kOrderBins;
}

// The group's cells by events, most first, into order[0 .. nc): exactly by their number up to kHeavy of
// them, by a quarter of a power of two above; within a bin in any order, on which nothing depends (a
// cell's chain is its own, the maxima are integers'). A counting sort: heavy_first compares every
// pair of cells, 10 us of a workgroup of 1024. cptr must be visible to every thread; ends with a barrier.
__device__ __forceinline__ void order_cells(const int* cptr, int nc, int* order, int* bins, int tid) {
    auto bin = [&](int i) __attribute__((always_inline)) {
        const int n = cptr[i + 1] - cptr[i];
        if (n <= kHeavy) return kHeavyBins + kHeavy - n;
        const int e = 31 - __builtin_clz(n);  // 6 .. 23 (T < 2^23)
        return kHeavyBins - 1 - (4 * (e - 6) + ((n >> (e - 2)) & 3));
    };
    for (int i = tid; i < kOrderBins; i += kQuadThreads) bins[i] = 0;
    __syncthreads();
    for (int i = tid; i < nc; i += kQuadThreads) atomicAdd(&bins[bin(i)], 1);
    __syncthreads();
    if (tid < kWave) {  // the bins' first places
        constexpr int kPer = (kOrderBins + kWave - 1) / kWave;
        int n[kPer], own = 0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            n[i] = kPer * tid + i < kOrderBins ? bins[kPer * tid + i] : 0;
            own += n[i];
        }
        int at = own;
        for (int o = 1; o < kWave; o <<= 1) {
            const int u = __shfl_up(at, o, kWave);
            if (tid >= o) at += u;
        }
        at -= own;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (kPer * tid + i < kOrderBins) bins[kPer * tid + i] = at;
            at += n[i];
        }
    }
    __syncthreads();
    for (int i = tid; i < nc; i += kQuadThreads) order[atomicAdd(&bins[bin(i)], 1)] = i;
    __syncthreads();
}

// val into the maxima of positions [p0, p1), by the L lanes of a group.
template <int L>
__device__ __forceinline__ void mark_run(uint32_t* tab, int p0, int p1, uint32_t val, int l) {
    for (int p = p0 + l; p < p1; p += L) atomicMax(&tab[p], val);
}
template <int L>
__device__ __forceinline__ void mark(uint32_t* hm, uint32_t* hc, uint32_t* hs, int p0, int p1,
                                     uint32_t val, int l) {
    if (p0 >= p1 || val == 0u) return;
    const int a = min(p1, (p0 + 15) & ~15);
    mark_run<L>(hm, p0, a, val, l);
    if (a >= p1) return;
    const int b = p1 & ~15;  // [a, b) is whole blocks of 16
    mark_run<L>(hm, b, p1, val, l);
    const int c0 = a / 16, c1 = b / 16, ca = min(c1, (c0 + 15) & ~15);
    mark_run<L>(hc, c0, ca, val, l);
    if (ca >= c1) return;
    const int cb = c1 & ~15;
    mark_run<L>(hc, cb, c1, val, l);
    mark_run<L>(hs, ca / 16, cb / 16, val, l);
}

// The cells of more than `heavy` events (at most kHeavy): the first of the order.
__device__ __forceinline__ int heavy_cells(const int* cptr, const int* order, int nc, int heavy) {
    int lo = 0, hi = nc;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1, ci = order[mid];
        if (cptr[ci + 1] - cptr[ci] > heavy) lo = mid + 1;
        else hi = mid;
    }
    return uniform(lo);
}

template <typename IO, int L, bool DELTA, bool HMAX>
__global__ __launch_bounds__(kQuadThreads, 5) void chain_fwd4(FwdArgs a) {
    extern __shared__ uint32_t lds_u[];
    constexpr int Q = kWave / L;
    int b, g;
    group_coords(b, g);
    const int tid = threadIdx.x, lane = lane_id(), l = lane % L, gq = lane / L;
    const int T = a.T, N = a.N, d = a.d, K = a.K;
    const int TW = (T + 31) / 32;
    int* nr = reinterpret_cast<int*>(lds_u);                  // [T + 2]
    uint32_t* rbits = lds_u + (T + 2);                        // [TW]
    int* nx = reinterpret_cast<int*>(rbits + TW);             // [TW + 1]
    uint32_t* hm = reinterpret_cast<uint32_t*>(nx + TW + 1);  // [T]
    int* next = reinterpret_cast<int*>(hm + T);               // [1]
    int* cptr = next + 1;                                     // [C + 1]
    int* cev = cptr + a.C + 1;                                // [stage]
    int* order = cev + a.stage;                               // [C]
    uint32_t* hc = reinterpret_cast<uint32_t*>(order + a.C);  // [(T + 15) / 16]
    uint32_t* hs = hc + (T + 15) / 16;                        // [(T + 255) / 256]
    int* bins = reinterpret_cast<int*>(hs + (T + 255) / 256);  // [kOrderBins]
    const int c_begin = g * a.C, c_end = min(N, c_begin + a.C);
    const int nc = c_end - c_begin;
    const int32_t* ptr = a.ptr + int64_t(b) * (N + 1);
    const int32_t* ev = a.ev + int64_t(b) * T * K;
    const int pc0 = ptr[c_begin];
    const int nst = min(ptr[c_end] - pc0, a.stage);
    const int pad_begin = ptr[N];
    for (int i = tid; i <= nc; i += kQuadThreads) cptr[i] = ptr[c_begin + i];
    for (int i = tid; i < nst; i += kQuadThreads) cev[i] = ev[pc0 + i];
    if constexpr (HMAX) {
        for (int p = tid; p < T; p += kQuadThreads) hm[p] = 0u;
        for (int p = tid; p < coarse_words(T); p += kQuadThreads) hc[p] = 0u;
    }
    if (tid == 0) next[0] = 0;
    const int lrT = reset_table(a.reset ? a.reset + int64_t(b) * T : nullptr, T, nr, rbits, nx,
                                tid, kQuadThreads);
    order_cells(cptr, nc, order, bins, tid);
    const int64_t slot0 = int64_t(b) * T * K;
    const uint32_t row_bytes = uint32_t(T) * K * d * sizeof(IO);
    const IO* kind = nullptr;
    const rsrc_t ry = make_rsrc(static_cast<const IO*>(a.y) + slot0 * d, row_bytes);
    const rsrc_t rg = make_rsrc(static_cast<const IO*>(a.g) + slot0 * d, row_bytes);
    const rsrc_t rho = make_rsrc(a.h_old ? static_cast<IO*>(a.h_old) + slot0 * d : nullptr,
                                 a.h_old ? row_bytes : 0u);
    const rsrc_t rhs = make_rsrc(a.h_sel ? static_cast<IO*>(a.h_sel) + slot0 * d : nullptr,
                                 a.h_sel ? row_bytes : 0u);
    const rsrc_t rdl = make_rsrc(a.delta ? a.delta + slot0 * d : nullptr,
                                 a.delta ? uint32_t(T) * K * d * 4u : 0u);
    const int n_slots = T * K;
    const bool pads = pad_begin < n_slots;  // cell 0 then also writes the padded slots: by itself
    const bool cin = 4 * l < d;
    const uint32_t ocol = uint32_t(4 * l) * sizeof(IO), ocol4 = uint32_t(4 * l) * 4u;
    const uint32_t srow = uint32_t(d) * sizeof(IO), srow4 = uint32_t(d) * 4u;
    const rsrc_t rh0 = make_rsrc(a.h0 + int64_t(b) * N * d, uint32_t(N) * srow4);
    const rsrc_t rhT = make_rsrc(a.h_T ? a.h_T + int64_t(b) * N * d : nullptr,
                                 a.h_T ? uint32_t(N) * srow4 : 0u);
    const int nr0 = nr[0];

    // one cell by the whole wavefront (walk_cell): the cells of more than a.heavy events, whose chain a
    // wavefront of several cells would walk more slowly, and cell 0 where the row has padded slots
    constexpr int V = L <= 16 ? 1 : 2;
    FwdRow<V> r;
    r.b = b, r.pc0 = pc0, r.nst = nst, r.lrT = lrT, r.pad_begin = pad_begin;
    r.ev = ev, r.cev = cev, r.nr = nr, r.hm = hm;
    r.ry = ry, r.rg = rg, r.rho = rho, r.rhs = rhs, r.rdl = rdl;
    r.srow = srow, r.srow4 = srow4;
    column_offsets<IO, V>(d, r.voff, r.voff4);
    auto single = [&](auto pad_cell, int ci) __attribute__((always_inline)) {
        constexpr Pads kPads = decltype(pad_cell)::value ? kPadCell : kNoPads;
        walk_cell<IO, V, 4, DELTA, HMAX, kPads>(a, r, c_begin + ci, uniform(cptr[ci]), uniform(cptr[ci + 1]));
    };

    const int heavy = heavy_cells(cptr, order, nc, a.heavy);
    if (pads && g == 0 && tid < kWave) single(std::true_type{}, 0);  // first: it has the padded slots too
    uint32_t idle = 0u;  // the largest |h| of the cells without an event (this lane's columns)
    for (;;) {
        int item = lane == 0 ? atomicAdd(next, 1) : 0;  // a heavy cell, or the next Q light ones
        item = __builtin_amdgcn_readfirstlane(item);
        if (item < heavy) {
            const int ci = uniform(order[item]);
            if (!(pads && c_begin + ci == 0)) single(std::false_type{}, ci);
            continue;
        }
        const int slot = heavy + (item - heavy) * Q;
        if (slot >= nc) break;
        const int my = slot + gq;
        const int ci = my < nc ? order[my] : 0;
        const int c = c_begin + ci;
        const bool has = my < nc && !(pads && c == 0);
        const int e0 = has ? cptr[ci] : 0;
        const int n = has ? cptr[ci + 1] - e0 : 0;
        // heaviest first, so the first group's cell has the most events (the lone cell 0 aside)
        int nmax = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) nmax = max(nmax, __builtin_amdgcn_readlane(n, q * L));
        const uint32_t oh = has && cin ? uint32_t(c) * srow4 + ocol4 : kOob;
        float h[4];
        {
            const RawF raw = load_raw(rh0, oh, static_cast<const float*>(nullptr));
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = lane_of(raw, i);
        }
        if (nmax == 0) {  // uniform: no cell of the wavefront has an event
            if constexpr (HMAX)
#pragma unroll
                for (int i = 0; i < 4; ++i) idle = umax(idle, abs_bits(h[i]));
            const bool cleared = nr0 < T;
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = cleared ? 0.0f : h[i];
            store4(h, rhT, oh, static_cast<const float*>(nullptr));
            if (a.age_T && l == 0 && has) end_age(a, b, c, -1, lrT);
            continue;
        }
        auto abs_max = [&]() __attribute__((always_inline)) {
            uint32_t m = 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i) m = umax(m, abs_bits(h[i]));
            return group_max<L>(m);
        };
        uint32_t vprev = 0u;
        int tprev = -1, s = 0, nrprev = nr0;
        struct Batch {
            Raw<IO> y[NB], g[NB];
            int t[NB], sl[NB], nr[NB];
        };
        auto walk = [&](auto staged_c) __attribute__((always_inline)) {
            constexpr bool kStaged = decltype(staged_c)::value;
            auto fetch = [&](int j, Batch& q) __attribute__((always_inline)) {
                int e[NB];
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int at = e0 + min(j + i, max(n - 1, 0));
                    if constexpr (kStaged) e[i] = n > 0 ? cev[at - pc0] : 0;
                    else e[i] = n > 0 ? ev[at] : 0;
                }
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const bool in = j + i < n;
                    q.t[i] = e[i] >> 8;
                    q.sl[i] = q.t[i] * K + (e[i] & 255);
                    q.nr[i] = nr[q.t[i] + 1];
                    const uint32_t vo = in && cin ? uint32_t(q.sl[i]) * srow + ocol : kOob;
                    q.y[i] = load_raw(ry, vo, kind);
                    q.g[i] = load_raw(rg, vo, kind);
                }
            };
            auto step = [&](int j, const Batch& q) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    if (j + i >= nmax) break;  // uniform
                    const bool in = j + i < n;
                    const int t = q.t[i];
                    const bool zero = nrprev <= t;  // a reset since the cell's last event
                    if constexpr (HMAX)
                        if (in) mark<L>(hm, hc, hs, s, min(t, nrprev), vprev, l);
                    const uint32_t vo = in && cin ? uint32_t(q.sl[i]) * srow + ocol : kOob;
                    float hold[4], hn[4], dl[4];
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        hold[x] = zero ? 0.0f : h[x];
                        const float bg = fast_sigmoid(lane_of(q.g[i], x));
                        const float cand = fast_tanh(lane_of(q.y[i], x));
                        hn[x] = (1.0f - bg) * hold[x] + bg * cand;
                        dl[x] = hn[x] - hold[x];
                    }
                    store4(hold, rho, vo, kind);
                    store4(hn, rhs, vo, kind);
                    if constexpr (DELTA)
                        store4(dl, rdl, in && cin ? uint32_t(q.sl[i]) * srow4 + ocol4 : kOob,
                               static_cast<const float*>(nullptr));
#pragma unroll
                    for (int x = 0; x < 4; ++x) h[x] = in ? hn[x] : h[x];
                    if constexpr (HMAX) {
                        const uint32_t v = abs_max();
                        vprev = in ? v : vprev;
                    }
                    s = in ? t : s;
                    tprev = in ? t : tprev;
                    nrprev = in ? q.nr[i] : nrprev;
                }
            };
            Batch qa, qb;
            fetch(0, qa);
            if constexpr (HMAX) vprev = abs_max();  // the start state's, once its load is back
            for (int j = 0; j < nmax; j += 2 * NB) {
                fetch(j + NB, qb);
                step(j, qa);
                if (j + NB >= nmax) break;
                fetch(j + 2 * NB, qa);
                step(j + NB, qb);
            }
        };
        if (ballot(has && e0 + n - pc0 > nst) == 0ull) walk(std::true_type{});
        else walk(std::false_type{});
        if constexpr (HMAX)
            if (has) mark<L>(hm, hc, hs, s, min(T, nrprev), vprev, l);
        const bool cleared = nrprev < T;  // a reset after the cell's last event
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = cleared ? 0.0f : h[i];
        store4(h, rhT, oh, static_cast<const float*>(nullptr));
        if (a.age_T && l == 0 && has) end_age(a, b, c, tprev, lrT);
    }
    if constexpr (HMAX) {
        const uint32_t v = wave_max_from_groups<1>(idle);
        if (lane < L) mark<L>(hm, hc, hs, 0, min(T, nr0), v, l);
    }
    if (a.pos_T && g == 0 && tid == 0) a.pos_T[b] = lrT >= 0 ? int64_t(T - lrT) : a.pos0[b] + T;
    if constexpr (HMAX) {  // the group's maxima, reduced over the groups by summary_delta
        __syncthreads();
        const int G = gridDim.y;
        uint32_t* hg = a.hm_groups + int64_t(b) * T * G + g;
        for (int p = tid; p < T; p += kQuadThreads)
            hg[int64_t(p) * G] = umax(hm[p], umax(hc[p / 16], hs[p / 256]));
    }
}

template <typename IO, int L>
__global__ __launch_bounds__(kQuadThreads, sizeof(IO) == 4 ? 4 : 5) void chain_bwd4(BwdArgs a) {
    extern __shared__ uint32_t lds_u[];
    constexpr int Q = kWave / L;
    int b, g;
    group_coords(b, g);
    const int tid = threadIdx.x, lane = lane_id(), l = lane % L, gq = lane / L;
    const int T = a.T, N = a.N, d = a.d, K = a.K;
    const int TW = (T + 31) / 32;
    int* nr = reinterpret_cast<int*>(lds_u);
    uint32_t* rbits = lds_u + (T + 2);
    int* nx = reinterpret_cast<int*>(rbits + TW);
    int* next = nx + TW + 1 + T;  // the layout of chain_fwd4 (no row maxima used)
    int* cptr = next + 1;
    int* cev = cptr + a.C + 1;
    int* order = cev + a.stage;
    int* bins = order + a.C + coarse_words(T);
    const int c_begin = g * a.C, c_end = min(N, c_begin + a.C);
    const int nc = c_end - c_begin;
    const int32_t* ptr = a.ptr + int64_t(b) * (N + 1);
    const int32_t* ev = a.ev + int64_t(b) * T * K;
    const int pc0 = ptr[c_begin];
    const int nst = min(ptr[c_end] - pc0, a.stage);
    for (int i = tid; i <= nc; i += kQuadThreads) cptr[i] = ptr[c_begin + i];
    for (int i = tid; i < nst; i += kQuadThreads) cev[i] = ev[pc0 + i];
    if (tid == 0) next[0] = 0;
    reset_table(a.reset ? a.reset + int64_t(b) * T : nullptr, T, nr, rbits, nx, tid, kQuadThreads);
    order_cells(cptr, nc, order, bins, tid);
    const int64_t slot0 = int64_t(b) * T * K;
    const uint32_t row_bytes = uint32_t(T) * K * d * sizeof(IO);
    const IO* kind = nullptr;
    const float* f32 = nullptr;
    const rsrc_t ry = make_rsrc(static_cast<const IO*>(a.y) + slot0 * d, row_bytes);
    const rsrc_t rg = make_rsrc(static_cast<const IO*>(a.g) + slot0 * d, row_bytes);
    const rsrc_t rho = make_rsrc(static_cast<const IO*>(a.h_old) + slot0 * d, row_bytes);
    const rsrc_t rds = make_rsrc(a.dsel ? static_cast<const IO*>(a.dsel) + slot0 * d : nullptr,
                                 a.dsel ? row_bytes : 0u);
    const rsrc_t rdy = make_rsrc(static_cast<IO*>(a.dy) + slot0 * d, row_bytes);
    const rsrc_t rdg = make_rsrc(static_cast<IO*>(a.dg) + slot0 * d, row_bytes);
    const rsrc_t rsh = make_rsrc(a.share + int64_t(b) * T * d, uint32_t(T) * d * 4u);
    const bool cin = 4 * l < d;
    const uint32_t ocol = uint32_t(4 * l) * sizeof(IO), ocol4 = uint32_t(4 * l) * 4u;
    const uint32_t srow = uint32_t(d) * sizeof(IO), srow4 = uint32_t(d) * 4u;
    const rsrc_t rdhT = make_rsrc(a.dh_T ? a.dh_T + int64_t(b) * N * d : nullptr,
                                  a.dh_T ? uint32_t(N) * srow4 : 0u);
    const rsrc_t rdh0 = make_rsrc(a.dh0 ? a.dh0 + int64_t(b) * N * d : nullptr,
                                  a.dh0 ? uint32_t(N) * srow4 : 0u);
    const int nr0 = nr[0];

    constexpr int V = L <= 16 ? 1 : 2;
    BwdRow<V> r;
    r.b = b, r.pc0 = pc0, r.nst = nst, r.ev = ev, r.cev = cev, r.nr = nr;
    r.ry = ry, r.rg = rg, r.rho = rho, r.rds = rds, r.rdy = rdy, r.rdg = rdg, r.rsh = rsh;
    r.srow = srow, r.srow4 = srow4;
    column_offsets<IO, V>(d, r.voff, r.voff4);
    auto single = [&](int ci) __attribute__((always_inline)) {  // a heavy cell, as in chain_fwd4
        walk_cell<IO, V, 4>(a, r, c_begin + ci, uniform(cptr[ci]), uniform(cptr[ci + 1]));
    };
    const int heavy = heavy_cells(cptr, order, nc, a.heavy);

    for (;;) {
        int item = lane == 0 ? atomicAdd(next, 1) : 0;  // a heavy cell, or the next Q light ones
        item = __builtin_amdgcn_readfirstlane(item);
        if (item < heavy) {
            single(uniform(order[item]));
            continue;
        }
        const int slot = heavy + (item - heavy) * Q;
        if (slot >= nc) break;
        const int my = slot + gq;
        const bool has = my < nc;
        const int ci = has ? order[my] : 0;
        const int c = c_begin + ci;
        const int e0 = has ? cptr[ci] : 0;
        const int n = has ? cptr[ci + 1] - e0 : 0;
        const int nmax = __builtin_amdgcn_readfirstlane(n);  // heaviest first: the first group's
        const bool staged = ballot(has && e0 + n - pc0 > nst) == 0ull;
        const uint32_t oh = has && cin ? uint32_t(c) * srow4 + ocol4 : kOob;
        float A[4];
        {  // the end cotangent, cut by a reset after the cell's last event
            const int last = n > 0 ? (staged ? cev[e0 + n - 1 - pc0] : ev[e0 + n - 1]) >> 8 : -1;
            const bool cut = nr[last + 1] < T;
            const RawF raw = load_raw(rdhT, cut ? kOob : oh, f32);
#pragma unroll
            for (int i = 0; i < 4; ++i) A[i] = lane_of(raw, i);
        }
        int tnext = T;  // the later event's position
        struct Batch {
            Raw<IO> y[NB], g[NB], h[NB], s[NB];
            RawF r[NB];
            int t[NB], sl[NB], nr[NB];
        };
        auto walk = [&](auto staged_c) __attribute__((always_inline)) {
            constexpr bool kStaged = decltype(staged_c)::value;
            // step j of a cell is its event n - 1 - j: latest first
            auto fetch = [&](int j, Batch& q) __attribute__((always_inline)) {
                int e[NB];
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int at = e0 + max(n - 1 - (j + i), 0);
                    if constexpr (kStaged) e[i] = n > 0 ? cev[at - pc0] : 0;
                    else e[i] = n > 0 ? ev[at] : 0;
                }
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const bool in = j + i < n && cin;
                    q.t[i] = e[i] >> 8;
                    q.sl[i] = q.t[i] * K + (e[i] & 255);
                    q.nr[i] = nr[q.t[i] + 1];
                    const uint32_t vo = in ? uint32_t(q.sl[i]) * srow + ocol : kOob;
                    q.g[i] = load_raw(rg, vo, kind);
                    q.s[i] = load_raw(rds, vo, kind);
                    q.r[i] = load_raw(rsh, in ? uint32_t(q.t[i]) * srow4 + ocol4 : kOob, f32);
                    q.y[i] = load_raw(ry, vo, kind);
                    q.h[i] = load_raw(rho, vo, kind);
                }
            };
            auto step = [&](int j, const Batch& q) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    if (j + i >= nmax) break;  // uniform
                    const bool in = j + i < n;
                    const bool zero = q.nr[i] <= tnext && tnext < T;  // a reset in (t, tnext]
                    const uint32_t vo = in && cin ? uint32_t(q.sl[i]) * srow + ocol : kOob;
                    float dc[4], db[4];
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        const float carried = (zero ? 0.0f : A[x]) + lane_of(q.s[i], x);
                        const float share = lane_of(q.r[i], x);
                        const float gg = carried + share;
                        const float bg = fast_sigmoid(lane_of(q.g[i], x));
                        const float cc = fast_tanh(lane_of(q.y[i], x));
                        dc[x] = bg * gg * (1.0f - cc * cc);
                        db[x] = (cc - lane_of(q.h[i], x)) * gg * (bg * (1.0f - bg));
                        const float An = (1.0f - bg) * carried - bg * share;
                        A[x] = in ? An : A[x];
                    }
                    store4(dc, rdy, vo, kind);
                    store4(db, rdg, vo, kind);
                    tnext = in ? q.t[i] : tnext;
                }
            };
            Batch qa, qb;
            fetch(0, qa);
            for (int j = 0; j < nmax; j += 2 * NB) {
                fetch(j + NB, qb);
                step(j, qa);
                if (j + NB >= nmax) break;
                fetch(j + 2 * NB, qa);
                step(j + NB, qb);
            }
        };
        if (nmax > 0) {
            if (staged) walk(std::true_type{});
            else walk(std::false_type{});
        }
        // the start state's cotangent: cut by a reset at or before the first event
        const bool z = nr0 <= min(tnext, T - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) A[i] = z ? 0.0f : A[i];
        store4(A, rdh0, oh, f32);
    }
    const int n_slots = T * K, pad_begin = ptr[N];
    if (g == 0) {  // exact zeros on the row's padded slots, a lane group a slot
        const float zero[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int p = pad_begin + tid / L; p < n_slots; p += kQuadThreads / L) {
            const int q = ev[p];
            const uint32_t vo = cin ? uint32_t((q >> 8) * K + (q & 255)) * srow + ocol : kOob;
            store4(zero, rdy, vo, kind);
            store4(zero, rdg, vo, kind);
        }
    }
}

}  // namespace chain
}  // namespace hsn
