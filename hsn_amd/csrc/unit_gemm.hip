// The grouped unit MLP as products over the pairs in unit order (include/hsn_ops.h
// hsn_grouped_unit_mlp_{fwd,bwd}_ws; the same contract as hsn_grouped_unit_mlp_{fwd,bwd}, with a
// workspace).
//
//   unit_order  (one workgroup): the pairs in unit order (a stable counting sort of unit_idx),
//               every unit's first row, and the row tiles of 32 rows and the blocks of RB rows
//               laid end to end unit after unit. Integer work in a fixed order.
//   gm_hidden   (row tile, 64 hidden columns): z1 = v W1[j] + b1[j], stored once rounded, and
//               gelu(z1) of the unrounded z1 in fp32.
//   gm_out      (row tile, 64 columns): gelu(z1) W2[j] + b2[j].
//   gm_dz       (row tile, 64 hidden columns): dz1 = (dout W2[j]^T) gelu'(z1) and gelu(z1), fp32.
//   gm_dv       (row tile, 64 input columns): dz1 W1[j]^T.
//   gm_dw       (64 x 64 tile of W1[j] or W2[j], block of the unit's rows): v^T dz1 and
//               gelu(z1)^T dout with the column sums (the bias gradients); a unit of more than
//               one block leaves fp32 partial sums, which gm_dw_sum adds in block order.
//
// Every product is v_mfma_f32_16x16x4_f32 on operands widened to fp32 (16-bit inputs multiply
// exactly, dz1 and gelu(z1) stay fp32), 2 P (4d H + H d) FLOP a pass against some 150 TFLOP/s. What
// bounds it at P 8192: the loads between a step's products (matrix busy 0.39 in gm_hidden, 0.49 in
// gm_dv, 0.30 in gm_dw, 0.15 to 0.17 in the others); at P 256: each launch's serial steps on few
// workgroups. A tile of 32 rows reuses a unit's weights 32 times; the kernels over 16 pairs a workgroup
// (units.hip) read them once a 16 pairs, and their weight gradients walk all of a unit's pairs in one
// workgroup a tile, 16 pairs a step. Forward and backward together, M 8, d 64, H 512 (us): P 8192 bf16
// 971 -> 229; P 256 fp32 77 -> 52, the forward of few pairs by units.hip (few_pairs below). Of the 971 and
// 77, 19 and 11 are launches that narrowed the indices: unit_order reads either width.
#include <algorithm>
#include <type_traits>

#include "common.cuh"

#include "../../include/hsn_ops.h"
#include "abi_util.h"
#include "unit_math.cuh"

namespace hsn {
hipError_t allow_lds_raw(const void* kernel, size_t lds);

namespace ugemm {

using units::gelu;
using units::gelu_grad;

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kMaxUnits = 1024;  // LDS counts of a unit per wavefront of unit_order: 64 KiB
constexpr int kRT = 32;  // rows of a row tile
constexpr int kNT = 64;  // columns of a tile
constexpr int kKC = 64;  // reduction indices a step
// Measured (P 8192, M 8, d 64, H 512, bf16 | P 256, fp32; us): 32 rows and 64 indices hidden 44.5 |
// 11.1, out 23.7 | 11.7, dv 38.9 | 11.5; 64 rows 43.1, 28.9, 40.9 (and 28.1 against 24.5 for
// hidden at P 4096 in fp32); 32 indices 43.5 | 11.5, 24.3 | 12.7, 37.9 | 12.8. Two steps of rows
// in flight instead of one changed nothing.

// Four consecutive elements, widened (a 16-byte load of fp32, an 8-byte one of 16-bit storage).
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
template <typename T>
__device__ __forceinline__ float4 load4(const T* p) {
    const uint2 raw = *reinterpret_cast<const uint2*>(p);
    T e[4];
    __builtin_memcpy(e, &raw, 8);
    return make_float4(to_f32(e[0]), to_f32(e[1]), to_f32(e[2]), to_f32(e[3]));
}
__device__ __forceinline__ float4 zero4() { return make_float4(0.0f, 0.0f, 0.0f, 0.0f); }

// ------------------------------------------------------------------------------------------
// The pairs in unit order
// ------------------------------------------------------------------------------------------

struct Order {
    int32_t* perm;   // [P]: the pair of a row (pairs with a unit outside the bank have no row)
    int32_t* first;  // [M + 1]: a unit's first row
    int32_t* tile;   // [tiles]: a row tile's unit, or -1 past the last
    int32_t* row0;   // [tiles]: its first row
    int32_t* block;  // [blocks]: a weight-gradient block's unit, or -1 past the last
    int32_t* bfirst; // [M + 1]: a unit's first block (every unit has one, also without pairs)
    int32_t* pfirst; // [M]: the first partial sum of a unit of more than one block
    int P, M, tiles, RB, blocks;
};

template <typename I, int kSortWaves>
__global__ __launch_bounds__(64 * kSortWaves) void unit_order(const I* unit_idx, Order o) {
    extern __shared__ int lds_i[];
    int* cnt = lds_i;                      // [kSortWaves][M]: counts, then the next row
    int* part = cnt + kSortWaves * o.M;    // [4][kSortWaves]
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int P = o.P, M = o.M;
    for (int i = tid; i < kSortWaves * M; i += 64 * kSortWaves) cnt[i] = 0;
    __syncthreads();
    // a wavefront's range in batches of kU loads in flight; the last batch stays in registers
    // between the passes (all of the range up to 8192 pairs)
    constexpr int kU = 8;
    const int per = ((P + kSortWaves - 1) / kSortWaves + 63) / 64 * 64;
    const int p0 = w * per, p1 = min(P, p0 + per);
    int u[kU];
    auto fetch = [&](int p) __attribute__((always_inline)) {
        I raw[kU];
#pragma unroll
        for (int i = 0; i < kU; ++i) raw[i] = p + 64 * i + lane < p1 ? unit_idx[p + 64 * i + lane] : I(-1);
#pragma unroll
        for (int i = 0; i < kU; ++i) u[i] = raw[i] >= 0 && raw[i] < I(M) ? static_cast<int>(raw[i]) : -1;
    };
    for (int p = p0; p < p1; p += 64 * kU) {
        fetch(p);
#pragma unroll
        for (int i = 0; i < kU; ++i)
            if (u[i] >= 0) atomicAdd(&cnt[w * M + u[i]], 1);  // integers: any order
    }
    __syncthreads();
    // a unit a thread: its count over the wavefronts' ranges, then the units' prefix
    int n = 0;
    if (tid < M)
        for (int q = 0; q < kSortWaves; ++q) n += cnt[q * M + tid];
    const int nt = (n + kRT - 1) / kRT;
    const int nb = tid < M ? max(1, (n + o.RB - 1) / o.RB) : 0;
    const int np = nb > 1 ? nb : 0;  // partial sums
    int in = n, it = nt, ib = nb, ip = np;
    for (int s = 1; s < 64; s <<= 1) {
        const int a = __shfl_up(in, s, 64), b = __shfl_up(it, s, 64), c = __shfl_up(ib, s, 64),
                  e = __shfl_up(ip, s, 64);
        if (lane >= s) in += a, it += b, ib += c, ip += e;
    }
    if (lane == 63)
        part[w] = in, part[kSortWaves + w] = it, part[2 * kSortWaves + w] = ib, part[3 * kSortWaves + w] = ip;
    __syncthreads();
    int before = 0, tbefore = 0, bbefore = 0, pbefore = 0, all = 0, ball = 0;
    for (int q = 0; q < kSortWaves; ++q) {
        if (q < w)
            before += part[q], tbefore += part[kSortWaves + q], bbefore += part[2 * kSortWaves + q],
                pbefore += part[3 * kSortWaves + q];
        all += part[kSortWaves + q];
        ball += part[2 * kSortWaves + q];
    }
    if (tid < M) {
        const int f = before + in - n, t = tbefore + it - nt, bl = bbefore + ib - nb;
        o.first[tid] = f;
        o.bfirst[tid] = bl;
        o.pfirst[tid] = pbefore + ip - np;
        if (tid == M - 1) o.first[M] = f + n, o.bfirst[M] = bl + nb;
        int at = f;
        for (int q = 0; q < kSortWaves; ++q) {
            const int c = cnt[q * M + tid];
            cnt[q * M + tid] = at;
            at += c;
        }
        for (int q = 0; q < nt; ++q) o.tile[t + q] = tid, o.row0[t + q] = f + q * kRT;
        for (int q = 0; q < nb; ++q) o.block[bl + q] = tid;
    }
    for (int q = all + tid; q < o.tiles; q += 64 * kSortWaves) o.tile[q] = -1;
    for (int q = ball + tid; q < o.blocks; q += 64 * kSortWaves) o.block[q] = -1;
    __syncthreads();
    // every wavefront its own range and counters: a lane's row is its unit's next row plus the
    // lanes below it with the same unit
    for (int p = p0; p < p1; p += 64 * kU) {
        if (per > 64 * kU) fetch(p);
#pragma unroll
        for (int i = 0; i < kU; ++i) {
            if (p + 64 * i >= p1) break;
            const int ui = u[i];
            const int base = ui >= 0 ? cnt[w * M + ui] : 0;
            int rank = 0, n_same = 0;
            for (uint64_t left = ballot(ui >= 0); left != 0ull;) {
                const int ul = __builtin_amdgcn_readlane(ui, __builtin_ctzll(left));
                const uint64_t same = ballot(ui == ul);
                if (ui == ul) rank = lanes_below(same), n_same = __popcll(same);
                left &= ~same;
            }
            if (ui >= 0) {
                o.perm[base + rank] = p + 64 * i + lane;
                if (rank == n_same - 1) cnt[w * M + ui] = base + n_same;
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// ------------------------------------------------------------------------------------------
// A tile product
// ------------------------------------------------------------------------------------------

// acc += A [X x K] B [K x 64] by four wavefronts, each its X/2 x 32 quarter, the reduction in
// steps of KC through LDS with the next step's rows in registers while a step multiplies; a step's
// sum is added to the total at its end (one running sum over all of K was twice as far from the
// 64-bit result at K = 512), and with PARTS 4 a step keeps four sums, an index of every four each, so
// that K = 64 is four runs of 16 (by_reduction). An operand whose memory runs along the reduction (along() true) is kept [x][KC + 4] and read as
// 16 bytes, one that runs along the columns [KC][X + 4] and read as words: lane group g of a
// wavefront takes the reduction's indices 4 g .. 4 g + 3 of each 16, the same on both sides.
// The loaders give four consecutive elements, zero outside the operand: (x, k .. k + 3), or
// (x .. x + 3, k).
template <int X, int KC, bool ALONG>
__host__ __device__ constexpr int tile_words() {
    return ALONG ? X * (KC + 4) : KC * (X + 4);
}
template <int X, int KC, bool ALONG>
__device__ __forceinline__ int tile_x(int e) { return ALONG ? e / (KC / 4) : 4 * (e % (X / 4)); }
template <int X, int KC, bool ALONG>
__device__ __forceinline__ int tile_k(int e) { return ALONG ? 4 * (e % (KC / 4)) : e / (X / 4); }
template <int X, int KC, bool ALONG>
__device__ __forceinline__ int tile_at(int e) {
    return ALONG ? (e / (KC / 4)) * (KC + 4) + 4 * (e % (KC / 4))
                 : (e / (X / 4)) * (X + 4) + 4 * (e % (X / 4));
}

template <int X, int KC, bool ALONG, int NF>
__device__ __forceinline__ void fragment(const float* t, int x0, int s, int lr, int g,
                                         float (&f)[NF][4]) {
#pragma unroll
    for (int q = 0; q < NF; ++q) {
        const int x = x0 + 16 * q + lr;
        if constexpr (ALONG) {
            const float4 v = *reinterpret_cast<const float4*>(t + x * (KC + 4) + 16 * s + 4 * g);
            f[q][0] = v.x, f[q][1] = v.y, f[q][2] = v.z, f[q][3] = v.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) f[q][i] = t[(16 * s + 4 * g + i) * (X + 4) + x];
        }
    }
}

template <int RT, int KC, bool AALONG, bool BALONG, int PARTS = 1, class LA, class LB, class Step>
__device__ __forceinline__ void tile_product(const LA& la, const LB& lb, int K, float* As, float* Bs,
                                             v4f (&acc)[RT / 32][2], const Step& each) {
    constexpr int NA = RT * KC / 4 / 256, NB = kNT * KC / 4 / 256, TM = RT / 32;
    static_assert(PARTS == 1 || PARTS == 4, "the step's sums are added pairwise");
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, g = lane >> 4;
    const int xm = (w >> 1) * (RT / 2), xn = (w & 1) * 32;
    struct Rows {
        float4 a[NA], b[NB];
    };
    auto fetch = [&](int k0, Rows& q) __attribute__((always_inline)) {
        if (k0 >= K) return;  // uniform
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int e = tid + 256 * i;
            q.a[i] = la(tile_x<RT, KC, AALONG>(e), k0 + tile_k<RT, KC, AALONG>(e));
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int e = tid + 256 * i;
            q.b[i] = lb(tile_x<kNT, KC, BALONG>(e), k0 + tile_k<kNT, KC, BALONG>(e));
        }
    };
    auto step = [&](int k0, Rows& q) __attribute__((always_inline)) {
        __syncthreads();  // the previous step's reads are done
#pragma unroll
        for (int i = 0; i < NA; ++i)
            *reinterpret_cast<float4*>(As + tile_at<RT, KC, AALONG>(tid + 256 * i)) = q.a[i];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            *reinterpret_cast<float4*>(Bs + tile_at<kNT, KC, BALONG>(tid + 256 * i)) = q.b[i];
            each(q.b[i]);
        }
        __syncthreads();
        fetch(k0 + KC, q);
        v4f part[PARTS][TM][2] = {};
#pragma unroll
        for (int s = 0; s < KC / 16; ++s) {
            float fa[TM][4], fb[2][4];
            fragment<RT, KC, AALONG, TM>(As, xm, s, lr, g, fa);
            fragment<kNT, KC, BALONG, 2>(Bs, xn, s, lr, g, fb);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int m = 0; m < TM; ++m)
#pragma unroll
                    for (int n = 0; n < 2; ++n)
                        part[i % PARTS][m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            fa[m][i], fb[n][i], part[i % PARTS][m][n], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                if constexpr (PARTS == 4)
                    part[0][m][n] = (part[0][m][n] + part[1][m][n]) + (part[2][m][n] + part[3][m][n]);
                acc[m][n] += part[0][m][n];
            }
    };
    Rows next;
    fetch(0, next);
    for (int k0 = 0; k0 < K; k0 += KC) step(k0, next);
}
struct NoStep {
    __device__ __forceinline__ void operator()(const float4&) const {}
};

// The result element of register r: row xm + 16 m + 4 g + r, column xn + 16 n + lr.
template <int RT, class F>
__device__ __forceinline__ void each_result(const v4f (&acc)[RT / 32][2], const F& f) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, g = lane >> 4;
#pragma unroll
    for (int m = 0; m < RT / 32; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                f((w >> 1) * (RT / 2) + 16 * m + 4 * g + r, (w & 1) * 32 + 16 * n + lr, acc[m][n][r]);
}

// ------------------------------------------------------------------------------------------
// Products over row tiles
// ------------------------------------------------------------------------------------------

// Grids keep gridDim.x a multiple of the 8 XCDs, so workgroups of equal x % 8 run on one of them:
// each XCD takes a run of neighbouring tiles (or blocks), whose rows and unit weights stay in its
// L2 for all of their column tiles.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_run(int x) { return (x % kXcds) * (gridDim.x / kXcds) + x / kXcds; }
inline int pad_xcds(int n) { return (n + kXcds - 1) / kXcds * kXcds; }

struct RowArgs {
    const int32_t *perm, *first, *tile, *row0;
    int d, H;
};

// The workgroup's row tile: its unit (-1: past the last), first row and rows; the rows' pairs
// into LDS (0 past the last row, never stored).
__device__ __forceinline__ int row_tile(const RowArgs& a, int* rows, int& r0, int& n) {
    const int t = xcd_run(blockIdx.x);
    const int j = a.tile[t];
    if (j < 0) return j;
    r0 = a.row0[t];
    n = min(kRT, a.first[j + 1] - r0);
    if (int(threadIdx.x) < kRT) rows[threadIdx.x] = int(threadIdx.x) < n ? a.perm[r0 + threadIdx.x] : 0;
    __syncthreads();
    return j;
}

template <typename T, int PARTS>
__global__ __launch_bounds__(256) void gm_hidden(RowArgs a, const T* v, const T* W1, const T* b1,
                                                 T* hidden, float* act) {
    __shared__ __align__(16) float As[tile_words<kRT, kKC, true>()];
    __shared__ __align__(16) float Bs[tile_words<kNT, kKC, false>()];
    __shared__ int rows[kRT];
    int r0, n;
    const int j = row_tile(a, rows, r0, n);
    if (j < 0) return;
    const int in = 4 * a.d, H = a.H, h0 = blockIdx.y * kNT;
    const T* W = W1 + int64_t(j) * in * H;
    v4f acc[kRT / 32][2] = {};
    tile_product<kRT, kKC, true, false, PARTS>(
        [&](int x, int k) { return x < n && k < in ? load4(v + int64_t(rows[x]) * in + k) : zero4(); },
        [&](int x, int k) { return k < in && h0 + x < H ? load4(W + int64_t(k) * H + h0 + x) : zero4(); },
        in, As, Bs, acc, NoStep{});
    each_result<kRT>(acc, [&](int x, int c, float s) {
        const int h = h0 + c;
        if (x >= n || h >= H) return;
        const float z = s + to_f32(b1[int64_t(j) * H + h]);
        store_f32(hidden, int64_t(rows[x]) * H + h, z);
        act[int64_t(r0 + x) * H + h] = gelu(z);
    });
}

template <typename T, int PARTS>
__global__ __launch_bounds__(256) void gm_out(RowArgs a, const float* act, const T* W2, const T* b2,
                                              T* out) {
    __shared__ __align__(16) float As[tile_words<kRT, kKC, true>()];
    __shared__ __align__(16) float Bs[tile_words<kNT, kKC, false>()];
    __shared__ int rows[kRT];
    int r0, n;
    const int j = row_tile(a, rows, r0, n);
    if (j < 0) return;
    const int d = a.d, H = a.H, o0 = blockIdx.y * kNT;
    const T* W = W2 + int64_t(j) * H * d;
    const float* A = act + int64_t(r0) * H;
    v4f acc[kRT / 32][2] = {};
    tile_product<kRT, kKC, true, false, PARTS>(
        [&](int x, int k) { return x < n && k < H ? load4(A + int64_t(x) * H + k) : zero4(); },
        [&](int x, int k) { return k < H && o0 + x < d ? load4(W + int64_t(k) * d + o0 + x) : zero4(); },
        H, As, Bs, acc, NoStep{});
    each_result<kRT>(acc, [&](int x, int c, float s) {
        const int o = o0 + c;
        if (x < n && o < d) store_f32(out, int64_t(rows[x]) * d + o, s + to_f32(b2[int64_t(j) * d + o]));
    });
}

template <typename T, int PARTS>
__global__ __launch_bounds__(256) void gm_dz(RowArgs a, const T* dout, const T* W2, const T* hidden,
                                             float* dz, float* act) {
    __shared__ __align__(16) float As[tile_words<kRT, kKC, true>()];
    __shared__ __align__(16) float Bs[tile_words<kNT, kKC, true>()];
    __shared__ int rows[kRT];
    int r0, n;
    const int j = row_tile(a, rows, r0, n);
    if (j < 0) return;
    const int d = a.d, H = a.H, h0 = blockIdx.y * kNT;
    const T* W = W2 + (int64_t(j) * H + h0) * d;
    float z[kRT / 32][2][4];  // the saved z1 of this thread's results, in flight with the product
    {
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, g = lane >> 4;
#pragma unroll
        for (int m = 0; m < kRT / 32; ++m)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int x = (w >> 1) * (kRT / 2) + 16 * m + 4 * g + r, h = h0 + (w & 1) * 32 + 16 * q + lr;
                    z[m][q][r] = x < n && h < H ? to_f32(hidden[int64_t(rows[x]) * H + h]) : 0.0f;
                }
    }
    v4f acc[kRT / 32][2] = {};
    tile_product<kRT, kKC, true, true, PARTS>(
        [&](int x, int k) { return x < n && k < d ? load4(dout + int64_t(rows[x]) * d + k) : zero4(); },
        [&](int x, int k) { return h0 + x < H && k < d ? load4(W + int64_t(x) * d + k) : zero4(); },
        d, As, Bs, acc, NoStep{});
#pragma unroll
    for (int m = 0; m < kRT / 32; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[m][q][r] *= gelu_grad(z[m][q][r]), z[m][q][r] = gelu(z[m][q][r]);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, g = lane >> 4;
#pragma unroll
    for (int m = 0; m < kRT / 32; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int x = (w >> 1) * (kRT / 2) + 16 * m + 4 * g + r, h = h0 + (w & 1) * 32 + 16 * q + lr;
                if (x < n && h < H) {
                    dz[int64_t(r0 + x) * H + h] = acc[m][q][r];
                    act[int64_t(r0 + x) * H + h] = z[m][q][r];
                }
            }
}

template <typename T, int PARTS>
__global__ __launch_bounds__(256) void gm_dv(RowArgs a, const float* dz, const T* W1, T* dv) {
    __shared__ __align__(16) float As[tile_words<kRT, kKC, true>()];
    __shared__ __align__(16) float Bs[tile_words<kNT, kKC, true>()];
    __shared__ int rows[kRT];
    int r0, n;
    const int j = row_tile(a, rows, r0, n);
    if (j < 0) return;
    const int in = 4 * a.d, H = a.H, c0 = blockIdx.y * kNT;
    const T* W = W1 + (int64_t(j) * in + c0) * H;
    const float* A = dz + int64_t(r0) * H;
    v4f acc[kRT / 32][2] = {};
    tile_product<kRT, kKC, true, true, PARTS>(
        [&](int x, int k) { return x < n && k < H ? load4(A + int64_t(x) * H + k) : zero4(); },
        [&](int x, int k) { return c0 + x < in && k < H ? load4(W + int64_t(x) * H + k) : zero4(); },
        H, As, Bs, acc, NoStep{});
    each_result<kRT>(acc, [&](int x, int c, float s) {
        if (x < n && c0 + c < in) store_f32(dv, int64_t(rows[x]) * in + c0 + c, s);
    });
}

// ------------------------------------------------------------------------------------------
// The weight gradients
// ------------------------------------------------------------------------------------------

struct DwArgs {
    const int32_t *perm, *first, *block, *bfirst, *pfirst;
    float* part;  // [2 (P / RB)][unit_floats]: the partial sums (W1, b1, W2, b2) of the split units' blocks
    int d, H, RB;
    __host__ __device__ int64_t unit_floats() const {
        return int64_t(4) * d * H + H + int64_t(H) * d + d;
    }
    __host__ __device__ int tiles1() const { return (4 * d + 63) / 64 * ((H + 63) / 64); }
    __host__ __device__ int tiles2() const { return (H + 63) / 64 * ((d + 63) / 64); }
};

// Workgroup (tile, block of RB rows of a unit). Tiles below tiles1() are W1's (input columns x hidden
// columns), the others W2's (hidden x output columns); a tile in the first row of tiles also
// sums its right operand's columns (the bias gradient).
template <typename T>
__global__ __launch_bounds__(256) void gm_dw(DwArgs a, const T* v, const float* dz, const float* act,
                                             const T* dout, T* dW1, T* db1, T* dW2, T* db2) {
    extern __shared__ __align__(16) float lds_f[];
    float* As = lds_f;
    float* Bs = As + tile_words<64, kKC, false>();
    int* rows = reinterpret_cast<int*>(Bs + tile_words<kNT, kKC, false>());  // [RB]
    const int bl = blockIdx.y, tid = threadIdx.x;
    const int j = a.block[bl];
    if (j < 0) return;  // past the last block
    const int f0 = a.first[j], f1 = a.first[j + 1];
    const int r0 = f0 + (bl - a.bfirst[j]) * a.RB, n = min(a.RB, f1 - r0);
    const bool whole = f1 - f0 <= a.RB;  // one block: the gradient itself
    for (int i = tid; i < n; i += 256) rows[i] = a.perm[r0 + i];
    __syncthreads();
    const int d = a.d, H = a.H, in = 4 * d;
    const bool second = int(blockIdx.x) >= a.tiles1();
    const int t = second ? int(blockIdx.x) - a.tiles1() : int(blockIdx.x);
    const int nc = second ? d : H;   // columns of the gradient
    const int nr = second ? H : in;  // its rows
    const int ct = (nc + 63) / 64, x0 = t / ct * 64, c0 = t % ct * 64;
    v4f acc[2][2] = {};
    float4 sum = zero4();
    auto add = [&](const float4& q) { sum.x += q.x, sum.y += q.y, sum.z += q.z, sum.w += q.w; };
    if (second)
        tile_product<64, kKC, false, false>(
            [&](int x, int k) { return k < n && x0 + x < nr ? load4(act + int64_t(r0 + k) * H + x0 + x) : zero4(); },
            [&](int x, int k) { return k < n && c0 + x < nc ? load4(dout + int64_t(rows[k]) * d + c0 + x) : zero4(); },
            n, As, Bs, acc, add);
    else
        tile_product<64, kKC, false, false>(
            [&](int x, int k) { return k < n && x0 + x < nr ? load4(v + int64_t(rows[k]) * in + x0 + x) : zero4(); },
            [&](int x, int k) { return k < n && c0 + x < nc ? load4(dz + int64_t(r0 + k) * H + c0 + x) : zero4(); },
            n, As, Bs, acc, add);
    float* part = a.part + int64_t(a.pfirst[j] + (bl - a.bfirst[j])) * a.unit_floats() +
                  (second ? int64_t(in) * H + H : 0);
    T* dW = second ? dW2 + int64_t(j) * H * d : dW1 + int64_t(j) * in * H;
    each_result<64>(acc, [&](int x, int c, float q) {
        if (x0 + x >= nr || c0 + c >= nc) return;
        const int64_t at = int64_t(x0 + x) * nc + c0 + c;
        if (whole) store_f32(dW, at, q);
        else part[at] = q;
    });
    if (x0 == 0) {  // the columns' sums: 16 threads hold a column group's, added in their order
        __syncthreads();
        float4* red = reinterpret_cast<float4*>(As);
        red[tid] = sum;
        __syncthreads();
        if (tid < 64 && c0 + tid < nc) {
            float q = 0.0f;
            for (int i = 0; i < 16; ++i) q += As[4 * (16 * i + tid / 4) + (tid & 3)];
            if (whole) store_f32(second ? db2 : db1, int64_t(j) * nc + c0 + tid, q);
            else part[int64_t(nr) * nc + c0 + tid] = q;
        }
    }
}

// The units of more than one block: their partial sums in block order, rounded once.
template <typename T>
__global__ __launch_bounds__(256) void gm_dw_sum(DwArgs a, T* dW1, T* db1, T* dW2, T* db2) {
    const int j = blockIdx.y;
    const int p0 = a.pfirst[j], blocks = a.bfirst[j + 1] - a.bfirst[j];
    if (blocks <= 1) return;
    const int64_t u = a.unit_floats(), n1 = int64_t(4) * a.d * a.H, n2 = int64_t(a.H) * a.d;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < u; i += int64_t(gridDim.x) * 256) {
        float q = 0.0f;
        for (int s = 0; s < blocks; ++s) q += a.part[int64_t(p0 + s) * u + i];
        if (i < n1) store_f32(dW1, j * n1 + i, q);
        else if (i < n1 + a.H) store_f32(db1, int64_t(j) * a.H + (i - n1), q);
        else if (i < n1 + a.H + n2) store_f32(dW2, j * n2 + (i - n1 - a.H), q);
        else store_f32(db2, int64_t(j) * a.d + (i - n1 - a.H - n2), q);
    }
}

// ------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------

// Rows a weight-gradient workgroup sums: every unit's at once where the units' tiles fill the
// 256 CUs (twice a unit's mean share, so that only an uneven unit is split), else enough blocks
// for about two workgroups a CU; a block's pairs are kept in LDS. Splitting every unit for four
// workgroups a CU measured 57.5 + 14.4 us (the partial sums' pass) against 68 + 4.6 at P 8192,
// M 8, d 64, H 512 in bf16, and 30.0 + 12.5 against 31.2 at P 4096 in fp32.
int block_rows(int P, int M, int d, int H) {
    const DwArgs a{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, d, H, 0};
    const int64_t tiles = a.tiles1() + a.tiles2();
    const int64_t want = M * tiles >= 256 ? 2 * int64_t(P) / M : P * tiles / 512;
    return static_cast<int>(std::min<int64_t>(4096, std::max<int64_t>(256, (want + 63) / 64 * 64)));
}

inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

struct Layout {
    size_t perm, first, tile, row0, block, bfirst, pfirst, act, dz, part, bytes;
    int tiles, RB, blocks;
};
Layout layout(int P, int M, int d, int H, bool backward) {
    Layout L{};
    L.tiles = pad_xcds(P / kRT + std::min(P, M));
    L.RB = block_rows(P, M, d, H);
    L.blocks = P / L.RB + M;
    size_t at = 0;
    auto take = [&](size_t n) { const size_t r = at; at = align256(at + n); return r; };
    L.perm = take(size_t(P) * 4);
    L.first = take(size_t(M + 1) * 4);
    L.tile = take(size_t(L.tiles) * 4);
    L.row0 = take(size_t(L.tiles) * 4);
    L.block = take(size_t(L.blocks) * 4);
    L.bfirst = take(size_t(M + 1) * 4);
    L.pfirst = take(size_t(M) * 4);
    L.act = take(size_t(P) * H * 4);
    if (backward) {
        L.dz = take(size_t(P) * H * 4);
        const DwArgs a{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, d, H, L.RB};
        // a unit of n > RB pairs has at most 2 (n / RB) blocks; the others write their gradients
        L.part = take(size_t(2) * (P / L.RB) * a.unit_floats() * 4);
    }
    L.bytes = at;
    return L;
}

// The shapes the products take: four elements a load along every operand's rows.
bool takes(int P, int M, int d, int H) {
    return P >= 1 && M >= 1 && M <= kMaxUnits && d >= 4 && d % 4 == 0 && d <= 256 && H >= 4 &&
           H % 4 == 0 && (H + 63) / 64 <= 65535 && P / block_rows(P, M, d, H) + M <= 65535;
}
// Forwards that the kernels without a workspace are faster at: they have no pairs to order first and a
// quarter of the reduction a wavefront. Measured (us, without and with a workspace), fp32: P 256, M 8: d
// 64, H 512 21 and 28; d 64, H 64 17 and 20; P 64, M 32, d 128, H 512 29 and 37; but P 1024, M 8, d 64,
// H 512 32 and 31, P 16, M 32, d 16, H 64 17 and 13, and from 128 units on up to 2 to 3 times. 16-bit
// storage, where they go through a row's hidden tiles in turn: P 256, M 8: d 64, H 64 13 and 23, H 128 21
// and 24, d 128, H 64 21 and 30; P 2048, M 8, d 16, H 64 15 and 18; but d 16, H 512 40 and 28, and P 8192,
// M 16, d 16, H 64 51 and 29.
bool few_pairs(int P, int M, int d, int H, int dtype) {
    if (M > 32) return false;
    if (dtype == HSN_DTYPE_F32) return P <= 512 && int64_t(d) * H >= std::max(1024, 256 * M);
    return P <= 2048 && (H <= 64 || (H <= 128 && d <= 64));
}
bool aligned4(std::initializer_list<const void*> ptrs, size_t elem) {
    for (const void* p : ptrs)
        if (reinterpret_cast<uintptr_t>(p) % (4 * elem) != 0) return false;
    return true;
}

void order_pairs(const void* unit_idx, int index_bits, const Layout& L, char* ws, int P, int M,
                 hipStream_t st) {
    const Order o{reinterpret_cast<int32_t*>(ws + L.perm), reinterpret_cast<int32_t*>(ws + L.first),
                  reinterpret_cast<int32_t*>(ws + L.tile), reinterpret_cast<int32_t*>(ws + L.row0),
                  reinterpret_cast<int32_t*>(ws + L.block), reinterpret_cast<int32_t*>(ws + L.bfirst),
                  reinterpret_cast<int32_t*>(ws + L.pfirst), P, M, L.tiles, L.RB, L.blocks};
    // One wavefront for up to 128 pairs and 64 units: 2.8 us against sixteen wavefronts' 4.7 (P 64, M 8);
    // a step of 64 pairs goes through its units in turn, so more pairs than two steps do not gain
    // (P 512, M 32: the forward 41 us against 33).
    const int waves = P <= 128 && M <= 64 ? 1 : 16;
    const size_t lds = (size_t(waves) * M + 4 * waves) * 4;
    auto launch = [&](auto kernel, auto* idx) {
        if (lds > 64 * 1024) HSN_HIP(allow_lds_raw(reinterpret_cast<const void*>(kernel), lds));
        hipLaunchKernelGGL(kernel, dim3(1), dim3(64 * waves), lds, st, idx, o);
        HSN_HIP(hipGetLastError());
    };
    auto by_waves = [&](auto* idx) {
        using I = std::remove_const_t<std::remove_pointer_t<decltype(idx)>>;
        if (waves == 1) launch(&unit_order<I, 1>, idx);
        else launch(&unit_order<I, 16>, idx);
    };
    if (index_bits == 64) by_waves(static_cast<const int64_t*>(unit_idx));
    else by_waves(static_cast<const int32_t*>(unit_idx));
}

RowArgs row_args(const Layout& L, char* ws, int d, int H) {
    return RowArgs{reinterpret_cast<int32_t*>(ws + L.perm), reinterpret_cast<int32_t*>(ws + L.first),
                   reinterpret_cast<int32_t*>(ws + L.tile), reinterpret_cast<int32_t*>(ws + L.row0), d, H};
}

// The row tiles' sums a step (tile_product) by the reduction's length. Errors against 64 bits in
// fp32, the kernels without a workspace, one sum, four (P 2000): z1 at d 16 (K 64) 0.88e-7, 1.46e-7,
// 0.87e-7, at d 32 (K 128) 1.13e-7, 1.49e-7, 0.91e-7; out at H 64 1.75e-7, 2.20e-7, 1.32e-7. Beyond
// K = 128 one sum a step is no further off than those kernels (z1 at d 64 1.51e-7 both), and four
// cost registers: P 8192, d 64, H 512 in bf16 hidden 45.7 -> 52.1 us, dv 39.4 -> 47.7.
template <class F>
void by_reduction(int K, const F& f) {
    if (K <= 128) f(std::integral_constant<int, 4>{});
    else f(std::integral_constant<int, 1>{});
}

template <typename T>
struct Forward {
    static void run(const void* v, const void* unit_idx, int index_bits, const void* W1, const void* b1,
                    const void* W2, const void* b2, void* hidden, void* out, char* ws, int P, int M,
                    int d, int H, hipStream_t st) {
        const Layout L = layout(P, M, d, H, false);
        order_pairs(unit_idx, index_bits, L, ws, P, M, st);
        const RowArgs a = row_args(L, ws, d, H);
        float* act = reinterpret_cast<float*>(ws + L.act);
        by_reduction(4 * d, [&](auto parts) {
            hipLaunchKernelGGL((gm_hidden<T, decltype(parts)::value>), dim3(L.tiles, (H + 63) / 64), dim3(256), 0, st, a,
                               static_cast<const T*>(v), static_cast<const T*>(W1),
                               static_cast<const T*>(b1), static_cast<T*>(hidden), act);
        });
        HSN_HIP(hipGetLastError());
        by_reduction(H, [&](auto parts) {
            hipLaunchKernelGGL((gm_out<T, decltype(parts)::value>), dim3(L.tiles, (d + 63) / 64), dim3(256), 0, st, a, act,
                               static_cast<const T*>(W2), static_cast<const T*>(b2), static_cast<T*>(out));
        });
        HSN_HIP(hipGetLastError());
    }
};

template <typename T>
struct Backward {
    static void run(const void* v, const void* unit_idx, int index_bits, const void* W1, const void* W2,
                    const void* hidden, const void* dout, void* dv, void* dW1, void* db1, void* dW2,
                    void* db2, char* ws, int P, int M, int d, int H, hipStream_t st) {
        const Layout L = layout(P, M, d, H, true);
        order_pairs(unit_idx, index_bits, L, ws, P, M, st);
        const RowArgs ra = row_args(L, ws, d, H);
        float *act = reinterpret_cast<float*>(ws + L.act), *dz = reinterpret_cast<float*>(ws + L.dz);
        by_reduction(d, [&](auto parts) {
            hipLaunchKernelGGL((gm_dz<T, decltype(parts)::value>), dim3(L.tiles, (H + 63) / 64), dim3(256), 0, st, ra,
                               static_cast<const T*>(dout), static_cast<const T*>(W2),
                               static_cast<const T*>(hidden), dz, act);
        });
        HSN_HIP(hipGetLastError());
        by_reduction(H, [&](auto parts) {
            hipLaunchKernelGGL((gm_dv<T, decltype(parts)::value>), dim3(L.tiles, (4 * d + 63) / 64), dim3(256), 0, st, ra, dz,
                               static_cast<const T*>(W1), static_cast<T*>(dv));
        });
        HSN_HIP(hipGetLastError());
        const DwArgs a{reinterpret_cast<int32_t*>(ws + L.perm), reinterpret_cast<int32_t*>(ws + L.first),
                       reinterpret_cast<int32_t*>(ws + L.block), reinterpret_cast<int32_t*>(ws + L.bfirst),
                       reinterpret_cast<int32_t*>(ws + L.pfirst), reinterpret_cast<float*>(ws + L.part),
                       d, H, L.RB};
        const size_t lds = (tile_words<64, kKC, false>() + tile_words<kNT, kKC, false>() + L.RB) * 4;  // <= 50 KiB
        auto kernel = &gm_dw<T>;
        hipLaunchKernelGGL(kernel, dim3(a.tiles1() + a.tiles2(), L.blocks), dim3(256), lds, st, a,
                           static_cast<const T*>(v), dz, act, static_cast<const T*>(dout),
                           static_cast<T*>(dW1), static_cast<T*>(db1), static_cast<T*>(dW2),
                           static_cast<T*>(db2));
        HSN_HIP(hipGetLastError());
        if (P > L.RB) {
            hipLaunchKernelGGL((gm_dw_sum<T>), dim3(64, M), dim3(256), 0, st, a, static_cast<T*>(dW1),
                               static_cast<T*>(db1), static_cast<T*>(dW2), static_cast<T*>(db2));
            HSN_HIP(hipGetLastError());
        }
    }
};

template <template <typename> class Fn, typename... Args>
void by_dtype(int dtype, Args&&... args) {
    if (dtype == HSN_DTYPE_F32) Fn<float>::run(args...);
    else if (dtype == HSN_DTYPE_F16) Fn<_Float16>::run(args...);
    else Fn<bf16_t>::run(args...);
}

void check(const char* who, int P, int M, int d, int H, int dtype, int index_bits, const void* ws,
           int64_t ws_bytes, bool backward) {
    const std::string f(who);
    HSN_REQUIRE(takes(P, M, d, H), HSN_ERR_INVALID_ARGUMENT,
                f + ": need P >= 1, 1 <= M <= 1024, d a multiple of 4 up to 256 and H a multiple of 4 "
                    "(hsn_grouped_unit_mlp_workspace gives 0 for other shapes)");
    HSN_REQUIRE(int64_t(M) * 4 * d * H <= INT32_MAX && int64_t(P) * H <= INT32_MAX &&
                    int64_t(P) * 4 * d <= INT32_MAX,
                HSN_ERR_SIZE_OVERFLOW, f + ": an element count exceeds INT32_MAX");
    HSN_REQUIRE(dtype == HSN_DTYPE_F32 || dtype == HSN_DTYPE_F16 || dtype == HSN_DTYPE_BF16,
                HSN_ERR_UNSUPPORTED_DTYPE, f + ": unknown dtype code");
    HSN_REQUIRE(index_bits == 32 || index_bits == 64, HSN_ERR_INVALID_ARGUMENT,
                f + ": index_bits must be 32 or 64");
    HSN_REQUIRE(ws && reinterpret_cast<uintptr_t>(ws) % 256 == 0 &&
                    ws_bytes >= int64_t(layout(P, M, d, H, backward).bytes),
                HSN_ERR_INVALID_ARGUMENT,
                f + ": the workspace must be 256-byte aligned and hold hsn_grouped_unit_mlp_workspace bytes");
}

}  // namespace ugemm
}  // namespace hsn

using namespace hsn;

extern "C" int hsn_grouped_unit_mlp_workspace(int P, int M, int d, int H, int dtype, int backward,
                                              int64_t* bytes) {
    HSN_ABI_BEGIN
    HSN_REQUIRE(bytes != nullptr, HSN_ERR_INVALID_ARGUMENT, "hsn_grouped_unit_mlp_workspace: bytes is NULL");
    const bool fits = ugemm::takes(P, M, d, H) && (backward || !ugemm::few_pairs(P, M, d, H, dtype)) && int64_t(M) * 4 * d * H <= INT32_MAX &&
                      int64_t(P) * H <= INT32_MAX && int64_t(P) * 4 * d <= INT32_MAX;
    *bytes = fits ? static_cast<int64_t>(ugemm::layout(P, M, d, H, backward != 0).bytes) : 0;
    HSN_ABI_END
}

extern "C" int hsn_grouped_unit_mlp_fwd_ws(const void* v, const void* unit_idx, int index_bits,
                                           const void* W1, const void* b1, const void* W2,
                                           const void* b2, void* hidden_saved, void* out, int P, int M,
                                           int d, int H, int dtype, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
    HSN_ABI_BEGIN
    const char* who = "hsn_grouped_unit_mlp_fwd_ws";
    ugemm::check(who, P, M, d, H, dtype, index_bits, workspace, workspace_bytes, false);
    HSN_REQUIRE(v && unit_idx && W1 && b1 && W2 && b2 && hidden_saved && out, HSN_ERR_INVALID_ARGUMENT,
                std::string(who) + ": a pointer is NULL");
    HSN_REQUIRE(ugemm::aligned4({v, W1, W2}, dtype == HSN_DTYPE_F32 ? 4 : 2), HSN_ERR_INVALID_ARGUMENT,
                std::string(who) + ": v, W1 and W2 must be aligned to four elements");
    ugemm::by_dtype<ugemm::Forward>(dtype, v, unit_idx, index_bits, W1, b1, W2, b2, hidden_saved, out,
                                    static_cast<char*>(workspace), P, M, d, H, as_stream(stream));
    HSN_ABI_END
}

extern "C" int hsn_grouped_unit_mlp_bwd_ws(const void* v, const void* unit_idx, int index_bits,
                                           const void* W1, const void* W2, const void* hidden_saved,
                                           const void* grad_out, void* grad_v, void* grad_W1,
                                           void* grad_b1, void* grad_W2, void* grad_b2, int P, int M,
                                           int d, int H, int dtype, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
    HSN_ABI_BEGIN
    const char* who = "hsn_grouped_unit_mlp_bwd_ws";
    ugemm::check(who, P, M, d, H, dtype, index_bits, workspace, workspace_bytes, true);
    HSN_REQUIRE(v && unit_idx && W1 && W2 && hidden_saved && grad_out && grad_v && grad_W1 && grad_b1 &&
                    grad_W2 && grad_b2,
                HSN_ERR_INVALID_ARGUMENT, std::string(who) + ": a pointer is NULL");
    HSN_REQUIRE(ugemm::aligned4({v, W1, W2, grad_out}, dtype == HSN_DTYPE_F32 ? 4 : 2),
                HSN_ERR_INVALID_ARGUMENT,
                std::string(who) + ": v, W1, W2 and grad_out must be aligned to four elements");
    ugemm::by_dtype<ugemm::Backward>(dtype, v, unit_idx, index_bits, W1, W2, hidden_saved, grad_out,
                                     grad_v, grad_W1, grad_b1, grad_W2, grad_b2,
                                     static_cast<char*>(workspace), P, M, d, H, as_stream(stream));
    HSN_ABI_END
}
