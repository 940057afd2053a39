// The cell-chain path of hsn_win_forward / hsn_win_backward (chain.cuh): the path choice, the
// workspace layout and the launchers.
#include <algorithm>
#include <atomic>
#include <initializer_list>
#include <string>
#include <type_traits>

#include "abi_util.h"
#include "chain.cuh"
#include "evmap.cuh"
#include "chain_host.h"

namespace hsn {

namespace {

std::atomic<int> g_path{kPathAuto};

constexpr size_t kAlign = 256;
inline size_t align_up(size_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

// Cells per workgroup: the smallest power of two from 16 that brings the grid to about 2048
// workgroups (eight per CU of the 256-CU chip), at most N.
inline int chain_cells(int B, int N) {
    int C = 16;
    while (C < N && int64_t(B) * ((N + C - 1) / C) > 2048) C *= 2;
    return C < N ? C : N;
}

// The same for the kernels that walk several cells a wavefront. Eight cells, a wavefront each, while
// their workgroups are no more than two a CU (one where a cell has eight events or more on average);
// else 32 and more, so that most wavefronts have cells side by side, up to 1024; 16 where 32 would leave
// the chip idle. One workgroup a CU for cells of many events: a heavy cell's chain waits for the CU's
// other wavefronts (not above d = 64, where only two cells walk side by side: B32 T512 N1024 K16 d128
// bf16 evenly 146 + 164 us, two a CU 146 + 139). Measured (us, forward and backward of a window: the
// kernel of one cell a wavefront, 32 cells or more and two workgroups a CU whatever the shape, this):
//   B1 T1024 N64 K8 d64 bf16 123 + 121, 184 + 181, 82 + 77; B8 T512 N128 K8 d128 71 + 70, 87 + 92, 54 + 49;
//   B16 T512 N512 K8 d64 58 + 47, 54 + 37, 54 + 37; with Zipf popularity B64 T512 N1024 K16 d64 355 + 241,
//   259 + 222, 231 + 186, and evenly 212 + 148, 164 + 125, 162 + 122 (two a CU 160 + 122); evenly
//   B64 T512 N64 K8 d64 99 + 75, 139 + 103, 95 + 70 (eight cells, two a CU 91 + 65, but Zipf 185 + 143
//   against 166 + 129).
inline int quad_cells(int B, int T, int N, int d, int K) {
    const bool many = int64_t(T) * K >= int64_t(8) * N;
    auto groups = [&](int C) { return int64_t(B) * ((N + C - 1) / C); };
    int C = 8;
    if (groups(8) > (many ? 256 : 512)) {
        C = groups(32) >= 160 ? 32 : 16;
        while (C < N && C < 1024 && groups(C) > (many && d <= 64 ? 256 : 512)) C *= 2;
    }
    return C < N ? C : N;
}

// Events up to which a cell is walked beside others: none where every cell has a wavefront; 64 where
// the cells have 8 to 32 on average and a workgroup more than 16 of them, else 24. A longer chain, alone, takes each event at half the time,
// but the wavefront's other lanes are lost. Measured, 24 against 64 (us): mean 1 to 4, Zipf: B256 T64
// N128 K8 d64 67 + 44 and 85 + 60, B11 T66 N1655 K3 d16 49 + 28 and 60 + 38; mean 8, normal: B64 T512
// N1024 K16 d64 184 + 141 and 168 + 128; mean 32, evenly: B64 T512 N128 K8 d64 106 + 75 and 94 + 63; mean 64
// (half of the cells on either side of 64): B64 T512 N64 K8 d64 95 + 70 and 124 + 79; 16 cells, Zipf: B64
// T64 N64 K16 d128 58 + 46 and 69 + 62.
inline int quad_heavy(int T, int N, int K, int C) {
    const int64_t events = int64_t(T) * K;
    if (C <= 8) return 0;
    return C > 16 && events >= int64_t(8) * N && events <= int64_t(32) * N ? chain::kHeavy : 24;
}

// Events staged in LDS per workgroup: twice the group's expected count, 256..8192.
inline int chain_stage(int T, int N, int K, int C) {
    const int64_t expect = int64_t(C) * T * K / N;
    int64_t s = (2 * expect + 63) / 64 * 64;
    if (s < 256) s = 256;
    if (s > 8192) s = 8192;
    return static_cast<int>(s);
}

}  // namespace

int path_setting() { return g_path.load(std::memory_order_relaxed); }
void set_path_setting(int path) { g_path.store(path, std::memory_order_relaxed); }

bool slice_takes(int op, int B, int T, int N, int d, int K, const char** why) {
    Geometry g;
    const bool fwd = op == HSN_OP_FORWARD || op == HSN_OP_CELL_UPDATE;
    const int t = op == HSN_OP_CELL_UPDATE ? 1 : T;
    const bool ok = fwd ? choose_geometry(B, t, N, d, K, fwd_lds_bytes, g)
                        : choose_geometry(B, t, N, d, K, bwd_lds_bytes, g);
    if (!ok && why)
        *why = fwd ? "no state slice fits the LDS with one slot per lane (N or K too large)"
                   : "no cotangent slice fits the LDS with one slot per lane (N or K too large)";
    return ok;
}

bool chain_takes(int B, int T, int N, int d, int K, const char** why) {
    const char* r = nullptr;
    if (d > 64 * chain::kMaxV) r = "the cell chains take d <= 256";
    else if (K > chain::kMaxK) r = "the cell chains take K <= 255";
    else if (T >= (1 << 23)) r = "the cell chains take T < 2^23";
    else if (int64_t(chain::list_words(N, T, K)) * 4 > kLdsMax) r = "the row lists do not fit the LDS (N too large)";
    else {
        const int C = chain_cells(B, N);
        if (int64_t(chain::chain_words(T, C, chain_stage(T, N, K, C))) * 4 > kLdsMax)
            r = "the chains' reset table does not fit the LDS (T too large)";
    }
    if (r && why) *why = r;
    return r == nullptr;
}

bool evmap_takes(int op, int B, int T, int N, int d, int K, size_t elem, const char** why) {
    (void)B;
    const char* r = nullptr;
    if (op != HSN_OP_FORWARD && op != HSN_OP_BACKWARD) r = "the event maps take the window forward and backward";
    else if (elem != 4) r = "the event maps take fp32 rows only";
    else if (d % evmap::kS != 0) r = "the event maps take d a multiple of 8";
    else if (T > evmap::kChunks * evmap::kP) r = "the event maps take T <= 256";
    else if (K > evmap::kK) r = "the event maps take K <= 8";
    else if ((op == HSN_OP_FORWARD ? evmap::fwd_layout(N).bytes : evmap::bwd_layout(N).bytes) > size_t(kLdsMax))
        r = "the event maps' tables of N cells do not fit the LDS";
    else if ((int64_t(T) + 32) * K * d * 4 >= (int64_t(1) << 31)) r = "the event maps take (T + 32) K d * 4 < 2^31 bytes a row";
    if (r && why) *why = r;
    return r == nullptr;
}

// MI355X's compute units: the event maps' grid in one round
constexpr int64_t kEvmapOneRound = 256;

int choose_path(int op, int B, int T, int N, int d, int K, size_t elem) {
    const char* why_s = nullptr;
    const char* why_c = nullptr;
    const char* why_e = nullptr;
    const int setting = path_setting();
    const bool any = setting == kPathAuto;
    const bool e_ok = (any || setting == kPathEvmap) && evmap_takes(op, B, T, N, d, K, elem, &why_e);
    if (setting == kPathEvmap && !e_ok)
        throw AbiError{HSN_ERR_INVALID_ARGUMENT, std::string("(event-map path) ") + why_e};
    // The event maps first where they take the shape and their grid of B d / 8 workgroups (one
    // a CU: the maps hold most of the LDS) runs in one round on MI355X's 256 CUs: every
    // workgroup carries a fixed cost (the tables, the walk over all N cells), which a single
    // round pays once. Measured: B32 T256 N256 d64 K8 fp32 (256 workgroups) 28.2 + 28.3 us
    // against the slices' 30.2 + 29.0; B128 T128 N512 d128 K8 fp32 (2048, eight rounds) 213 +
    // 240 us against the chains' 127 + 139.
    if (e_ok && (setting == kPathEvmap || int64_t(B) * (d / evmap::kS) <= kEvmapOneRound))
        return kPathEvmap;
    const bool s_ok = (any || setting == kPathSlice) && slice_takes(op, B, T, N, d, K, &why_s);
    const bool c_ok = (any || setting == kPathChain) && chain_takes(B, T, N, d, K, &why_c);
    if (!s_ok && !c_ok) {
        std::string msg;
        if (setting == kPathSlice) msg = std::string("(slice path) ") + why_s;
        else if (setting == kPathChain) msg = std::string("(chain path) ") + why_c;
        else msg = std::string(why_s) + "; and " + why_c;
        throw AbiError{HSN_ERR_INVALID_ARGUMENT, msg};
    }
    if (!c_ok) return kPathSlice;
    if (!s_ok) return kPathChain;
    // Both slices and chains take it: the slices where a wavefront's piece of a slot row is a
    // full 32-byte sector and the state slice (N * S words) leaves room for chunks of the row in
    // LDS; the chains where the piece would be narrower (K large against d) or the slice large
    // (N large). Measured on MI355X: slices at B32 T256 N256 d64 K8 fp32 (S 8, 68 against 95 us
    // per step), chains at B64 T512 N1024 d64 K16 bf16 (S 4: 0.45 against 1.62 ms) and B128 T128
    // N512 d128 K8 fp32 (S 8, N S 4096: 0.31 against 0.43 ms).
    Geometry g;
    const bool fwd = op == HSN_OP_FORWARD;
    if (fwd) choose_geometry(B, T, N, d, K, fwd_lds_bytes, g);
    else choose_geometry(B, T, N, d, K, bwd_lds_bytes, g);
    return size_t(g.S) * elem >= 32 && int64_t(N) * g.S <= 2048 ? kPathSlice : kPathChain;
}

WorkspaceLayout workspace_layout(int op, int B, int T, int N, int d, int K, size_t elem,
                                 int cand_norm) {
    WorkspaceLayout L;
    const int path = choose_path(op, B, T, N, d, K, elem);
    L.chain = path == kPathChain;
    L.evmap = path == kPathEvmap;
    const int64_t slots = int64_t(B) * T * K;
    size_t at = 0;
    if (L.chain) {
        L.ptr = at;
        at = align_up(at + size_t(B) * (N + 1) * 4);
        L.ev = at;
        at = align_up(at + size_t(slots) * 4);
        L.sum = at;
        at = align_up(at + size_t(B) * T * d * 4);
        if (op == HSN_OP_FORWARD) {
            L.delta = at;
            at = align_up(at + size_t(slots) * d * 4);
            const int C = std::min(chain_cells(B, N), quad_cells(B, T, N, d, K));
            L.hmax = at;
            at = align_up(at + size_t(B) * T * ((N + C - 1) / C) * 4);
        }
    }
    L.rms = at;
    if (cand_norm) at = align_up(at + rms_inv_offset(slots, d, elem) + 4 * size_t(slots));
    L.bytes = at;
    return L;
}

namespace {

void build_lists(const int32_t* slots, int32_t* ptr, int32_t* ev, int B, int T, int N, int K,
                 hipStream_t st) {
    chain::ListArgs la{slots, ptr, ev, B, T, N, K};
    const int NR = chain::range_cells(B, N), W = chain::range_waves(NR);
    const size_t range_lds = size_t(chain::range_words(W, NR, T, K)) * 4;
    // By ranges of cells where a position's slots fit a wavefront (its order is what places the
    // slots) and the row's list fits the LDS beside the counts. Measured (us) against the whole row
    // a workgroup: B64 T512 N1024 K16 9.6 (20.2), B256 T1024 N4096 K32 37 (105), B128 T128 N512 K8
    // 5.8 (7.7), B32 T8192 N1024 K4 43 (170), B8 T64 N64 K4 5.8 (7.0), B1024 T64 N128 K4 18 (24).
    if (K <= 64 && int64_t(T) * K <= chain::kRangeSlots && range_lds <= size_t(kLdsMax)) {
        auto launch = [&](auto waves, auto sub) {
            constexpr int kW = decltype(waves)::value, kSub = decltype(sub)::value;
            auto k = chain::row_lists_ranges<kW, kSub>;
            HSN_HIP(allow_lds(k, range_lds));
            hipLaunchKernelGGL(k, dim3((N + NR - 1) / NR, B), dim3(64 * kW), range_lds, st, la, NR);
        };
        auto by_sub = [&](auto waves) {
            if (K > 32) launch(waves, std::integral_constant<int, 1>{});
            else if (K > 16) launch(waves, std::integral_constant<int, 2>{});
            else if (K > 8) launch(waves, std::integral_constant<int, 4>{});
            else launch(waves, std::integral_constant<int, 8>{});
        };
        if (W == 8) by_sub(std::integral_constant<int, 8>{});
        else by_sub(std::integral_constant<int, 16>{});
        HSN_HIP(hipGetLastError());
        return;
    }
    const size_t lds = size_t(chain::list_words(N, T, K)) * 4;
    HSN_HIP(allow_lds(chain::row_lists, lds));
    hipLaunchKernelGGL(chain::row_lists, dim3(B), dim3(chain::kListThreads), lds, st, la);
    HSN_HIP(hipGetLastError());
}

template <typename IO, int V>
void launch_chain_fwd(const chain::FwdArgs& a, size_t lds, hipStream_t st) {
    constexpr int NB = 4;  // measured: 4 ahead of 8 and 16 (most cells hold a few events)
    auto k = a.delta ? (a.hm_groups ? chain::chain_fwd<IO, V, NB, true, true>
                                    : chain::chain_fwd<IO, V, NB, true, false>)
                     : (a.hm_groups ? chain::chain_fwd<IO, V, NB, false, true>
                                    : chain::chain_fwd<IO, V, NB, false, false>);
    HSN_HIP(allow_lds(k, lds));
    hipLaunchKernelGGL(k, chain::chain_grid(a.B, (a.N + a.C - 1) / a.C),
                       dim3(chain::kChainThreads), lds, st, a);
    HSN_HIP(hipGetLastError());
}

template <typename IO, int V>
void launch_chain_bwd(const chain::BwdArgs& a, size_t lds, hipStream_t st) {
    auto k = chain::chain_bwd<IO, V, 4>;
    HSN_HIP(allow_lds(k, lds));
    hipLaunchKernelGGL(k, chain::chain_grid(a.B, (a.N + a.C - 1) / a.C),
                       dim3(chain::kChainThreads), lds, st, a);
    HSN_HIP(hipGetLastError());
}

// The kernels that walk several cells a wavefront take d a multiple of 4 up to 128 and rows aligned to
// four elements (every access is four columns of a row). Above 128 a wavefront has one cell's columns
// only, and a cell walked alone does not fit the registers that its bounds leave (B8 T256 N128 K8 d256
// bf16, Zipf: 203 + 890 us against chain_fwd's and chain_bwd's 149 + 159).
template <typename IO>
bool takes_four(int d, std::initializer_list<const void*> rows) {
    if (d % 4 != 0 || d > 128) return false;
    for (const void* p : rows)
        if (reinterpret_cast<uintptr_t>(p) % (4 * sizeof(IO)) != 0) return false;
    return true;
}
template <class F>
void by_lanes(int d, const F& f) {
    if (d <= 16) f(std::integral_constant<int, 4>{});
    else if (d <= 32) f(std::integral_constant<int, 8>{});
    else if (d <= 64) f(std::integral_constant<int, 16>{});
    else f(std::integral_constant<int, 32>{});
}
template <typename IO>
void launch_chain_fwd4(const chain::FwdArgs& a, hipStream_t st) {
    const size_t lds = size_t(chain::quad_words(a.T, a.C, a.stage)) * 4;
    by_lanes(a.d, [&](auto lanes) {
        constexpr int L = decltype(lanes)::value;
        auto k = a.delta ? (a.hm_groups ? chain::chain_fwd4<IO, L, true, true>
                                        : chain::chain_fwd4<IO, L, true, false>)
                         : (a.hm_groups ? chain::chain_fwd4<IO, L, false, true>
                                        : chain::chain_fwd4<IO, L, false, false>);
        HSN_HIP(allow_lds(k, lds));
        hipLaunchKernelGGL(k, chain::chain_grid(a.B, (a.N + a.C - 1) / a.C),
                           dim3(chain::kQuadThreads), lds, st, a);
    });
    HSN_HIP(hipGetLastError());
}
template <typename IO>
void launch_chain_bwd4(const chain::BwdArgs& a, hipStream_t st) {
    const size_t lds = size_t(chain::quad_words(a.T, a.C, a.stage)) * 4;
    by_lanes(a.d, [&](auto lanes) {
        constexpr int L = decltype(lanes)::value;
        auto k = chain::chain_bwd4<IO, L>;
        HSN_HIP(allow_lds(k, lds));
        hipLaunchKernelGGL(k, chain::chain_grid(a.B, (a.N + a.C - 1) / a.C),
                           dim3(chain::kQuadThreads), lds, st, a);
    });
    HSN_HIP(hipGetLastError());
}

template <typename IO, int V>
void launch_delta(const chain::DeltaArgs& a, bool pair, hipStream_t st) {
    const dim3 grid((a.T + 3) / 4, a.B);
    if (pair) hipLaunchKernelGGL((chain::summary_delta<IO, V, true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((chain::summary_delta<IO, V, false>), grid, dim3(256), 0, st, a);
    HSN_HIP(hipGetLastError());
}

// Whether the several-cells kernels' LDS holds the row (T large).
template <typename Args>
bool quad_fits(const Args& a) {
    const int C = quad_cells(a.B, a.T, a.N, a.d, a.K);
    return int64_t(chain::quad_words(a.T, C, chain_stage(a.T, a.N, a.K, C))) * 4 <= kLdsMax;
}

template <typename IO>
void forward_io(chain::FwdArgs& fa, chain::DeltaArgs& da, const chain::ScanArgs& sa, bool pair,
                hipStream_t st) {
    const bool four = takes_four<IO>(fa.d, {fa.y, fa.g, fa.h_old, fa.h_sel}) &&
                      takes_four<float>(fa.d, {fa.h0, fa.h_T, fa.delta}) &&
                      int64_t(fa.N) * fa.d * 4 < (int64_t(1) << 31) && quad_fits(fa);
    fa.C = four ? quad_cells(fa.B, fa.T, fa.N, fa.d, fa.K) : chain_cells(fa.B, fa.N);
    fa.stage = chain_stage(fa.T, fa.N, fa.K, fa.C);
    fa.heavy = quad_heavy(fa.T, fa.N, fa.K, fa.C);
    da.G = (fa.N + fa.C - 1) / fa.C;
    const size_t lds = size_t(chain::chain_words(fa.T, fa.C, fa.stage)) * 4;
    const int V = (fa.d + 63) / 64;
    if (four) launch_chain_fwd4<IO>(fa, st);
    switch (V) {
        case 1: if (!four) launch_chain_fwd<IO, 1>(fa, lds, st); launch_delta<IO, 1>(da, pair, st); break;
        case 2: if (!four) launch_chain_fwd<IO, 2>(fa, lds, st); launch_delta<IO, 2>(da, pair, st); break;
        case 3: if (!four) launch_chain_fwd<IO, 3>(fa, lds, st); launch_delta<IO, 3>(da, pair, st); break;
        default: if (!four) launch_chain_fwd<IO, 4>(fa, lds, st); launch_delta<IO, 4>(da, pair, st); break;
    }
    hipLaunchKernelGGL((chain::summary_scan_fwd<IO>), dim3((fa.d + 63) / 64, fa.B),
                       dim3(64 * chain::kScanWaves), 0, st, sa);
    HSN_HIP(hipGetLastError());
}

template <typename IO>
void backward_io(chain::BwdArgs& ba, const chain::ScanArgs& sa, hipStream_t st) {
    const bool four = takes_four<IO>(ba.d, {ba.y, ba.g, ba.h_old, ba.dsel, ba.dy, ba.dg}) &&
                      takes_four<float>(ba.d, {ba.share, ba.dh_T, ba.dh0}) &&
                      int64_t(ba.N) * ba.d * 4 < (int64_t(1) << 31) && quad_fits(ba);
    ba.C = four ? quad_cells(ba.B, ba.T, ba.N, ba.d, ba.K) : chain_cells(ba.B, ba.N);
    ba.stage = chain_stage(ba.T, ba.N, ba.K, ba.C);
    ba.heavy = quad_heavy(ba.T, ba.N, ba.K, ba.C);
    const size_t lds = size_t(chain::chain_words(ba.T, ba.C, ba.stage)) * 4;
    hipLaunchKernelGGL((chain::summary_scan_bwd<IO>), dim3((ba.d + 63) / 64, ba.B),
                       dim3(64 * chain::kScanWaves), 0, st, sa);
    HSN_HIP(hipGetLastError());
    if (four) return launch_chain_bwd4<IO>(ba, st);
    const int V = (ba.d + 63) / 64;
    switch (V) {
        case 1: launch_chain_bwd<IO, 1>(ba, lds, st); break;
        case 2: launch_chain_bwd<IO, 2>(ba, lds, st); break;
        case 3: launch_chain_bwd<IO, 3>(ba, lds, st); break;
        default: launch_chain_bwd<IO, 4>(ba, lds, st); break;
    }
}

}  // namespace

void chain_forward(const void* y, const void* gate_pre, int io_dtype, const uint8_t* reset,
                   const int32_t* slots, const float* h0, const float* q0, const int64_t* age0,
                   const int64_t* pos0, void* q_pre, void* q_post, void* h_sel, void* h_old,
                   float* h_max, float* h_T, float* q_T, int64_t* age_T, int64_t* pos_T, int B,
                   int T, int N, int d, int K, char* ws, const WorkspaceLayout& L,
                   hipStream_t st) {
    int32_t* ptr = reinterpret_cast<int32_t*>(ws + L.ptr);
    int32_t* ev = reinterpret_cast<int32_t*>(ws + L.ev);
    float* D = reinterpret_cast<float*>(ws + L.sum);
    // the summary reads the fp32 rows themselves; else the chains' fp32 deltas (bf16 rows are
    // rounded: summing them would leave q off the mean of h by up to a rounding of |h|)
    const bool pair = io_dtype == HSN_DTYPE_F32 && h_sel && h_old;
    float* delta = pair ? nullptr : reinterpret_cast<float*>(ws + L.delta);
    build_lists(slots, ptr, ev, B, T, N, K, st);
    chain::FwdArgs fa{};
    fa.y = y, fa.g = gate_pre, fa.ptr = ptr, fa.ev = ev, fa.reset = reset;
    fa.h0 = h0, fa.age0 = age0, fa.pos0 = pos0;
    fa.h_old = h_old, fa.h_sel = h_sel, fa.delta = delta;
    uint32_t* hm_groups = h_max ? reinterpret_cast<uint32_t*>(ws + L.hmax) : nullptr;
    fa.hm_groups = hm_groups, fa.h_T = h_T, fa.age_T = age_T, fa.pos_T = pos_T;
    fa.B = B, fa.T = T, fa.N = N, fa.d = d, fa.K = K;
    chain::DeltaArgs da{};
    da.h_old = h_old, da.h_sel = h_sel, da.delta = delta, da.slots = slots, da.D = D;
    da.hm_groups = hm_groups, da.h_max = h_max;
    da.B = B, da.T = T, da.N = N, da.d = d, da.K = K;
    chain::ScanArgs sa{};
    sa.D = D, sa.q0 = q0, sa.q_pre = q_pre, sa.q_post = q_post, sa.q_T = q_T;
    sa.reset = reset, sa.B = B, sa.T = T, sa.d = d, sa.divn = make_divn(N);
    if (io_dtype == HSN_DTYPE_F32) forward_io<float>(fa, da, sa, pair, st);
    else forward_io<bf16_t>(fa, da, sa, pair, st);
}

void chain_backward(const void* y, const void* gate_pre, const void* h_old, int io_dtype,
                    const int32_t* slots, const uint8_t* reset, const void* d_q_pre,
                    const void* d_q_post, const void* d_h_sel, const float* d_h_T,
                    const float* d_q_T, void* dy, void* dgate, float* d_h0, float* d_q0, int B,
                    int T, int N, int d, int K, char* ws, const WorkspaceLayout& L,
                    hipStream_t st) {
    int32_t* ptr = reinterpret_cast<int32_t*>(ws + L.ptr);
    int32_t* ev = reinterpret_cast<int32_t*>(ws + L.ev);
    float* share = reinterpret_cast<float*>(ws + L.sum);
    build_lists(slots, ptr, ev, B, T, N, K, st);
    chain::ScanArgs sa{};
    sa.dq_pre = d_q_pre, sa.dq_post = d_q_post, sa.dq_T = d_q_T, sa.share = share, sa.dq0 = d_q0;
    sa.reset = reset, sa.B = B, sa.T = T, sa.d = d, sa.divn = make_divn(N);
    chain::BwdArgs ba{};
    ba.y = y, ba.g = gate_pre, ba.h_old = h_old, ba.dsel = d_h_sel, ba.ptr = ptr, ba.ev = ev;
    ba.reset = reset, ba.share = share, ba.dh_T = d_h_T, ba.dy = dy, ba.dg = dgate, ba.dh0 = d_h0;
    ba.B = B, ba.T = T, ba.N = N, ba.d = d, ba.K = K;
    if (io_dtype == HSN_DTYPE_F32) backward_io<float>(ba, sa, st);
    else backward_io<bf16_t>(ba, sa, st);
}

}  // namespace hsn

extern "C" int hsn_win_set_path(int path) {
    HSN_ABI_BEGIN
    HSN_REQUIRE(path == hsn::kPathAuto || path == hsn::kPathSlice || path == hsn::kPathChain ||
                    path == hsn::kPathEvmap,
                HSN_ERR_INVALID_ARGUMENT, "hsn_win_set_path: path must be 0 (auto), 1, 2 or 3");
    hsn::set_path_setting(path);
    HSN_ABI_END
}

extern "C" int hsn_win_path(int op, int B, int T, int N, int d, int K, int io_dtype, int* path) {
    HSN_ABI_BEGIN
    HSN_REQUIRE(path != nullptr, HSN_ERR_INVALID_ARGUMENT, "hsn_win_path: path is NULL");
    HSN_REQUIRE(op == HSN_OP_FORWARD || op == HSN_OP_BACKWARD, HSN_ERR_INVALID_ARGUMENT,
                "hsn_win_path: op must be HSN_OP_FORWARD or HSN_OP_BACKWARD");
    HSN_REQUIRE(B >= 1 && T >= 1 && N >= 1 && d >= 1 && K >= 1 && K <= N,
                HSN_ERR_INVALID_ARGUMENT, "hsn_win_path: bad dimensions");
    HSN_REQUIRE(io_dtype == HSN_DTYPE_F32 || io_dtype == HSN_DTYPE_BF16,
                HSN_ERR_UNSUPPORTED_DTYPE, "hsn_win_path: io_dtype must be f32 or bf16");
    *path = hsn::choose_path(op, B, T, N, d, K, io_dtype == HSN_DTYPE_F32 ? 4 : 2);
    HSN_ABI_END
}

extern "C" int hsn_win_workspace_bytes(int op, int B, int T, int N, int d, int K, int io_dtype,
                                       int cand_norm, int64_t* bytes) {
    HSN_ABI_BEGIN
    HSN_REQUIRE(bytes != nullptr, HSN_ERR_INVALID_ARGUMENT, "hsn_win_workspace_bytes: bytes is NULL");
    HSN_REQUIRE(op == HSN_OP_FORWARD || op == HSN_OP_BACKWARD, HSN_ERR_INVALID_ARGUMENT,
                "hsn_win_workspace_bytes: op must be HSN_OP_FORWARD or HSN_OP_BACKWARD");
    HSN_REQUIRE(B >= 1 && T >= 1 && N >= 1 && d >= 1 && K >= 1 && K <= N,
                HSN_ERR_INVALID_ARGUMENT, "hsn_win_workspace_bytes: bad dimensions");
    HSN_REQUIRE(io_dtype == HSN_DTYPE_F32 || io_dtype == HSN_DTYPE_BF16,
                HSN_ERR_UNSUPPORTED_DTYPE, "hsn_win_workspace_bytes: io_dtype must be f32 or bf16");
    HSN_REQUIRE(hsn::check_elems({int64_t(B) * T * K * d, int64_t(B) * N * d}),
                HSN_ERR_SIZE_OVERFLOW, "hsn_win_workspace_bytes: a tensor is too large");
    *bytes = static_cast<int64_t>(hsn::workspace_layout(op, B, T, N, d, K,
                                                        io_dtype == HSN_DTYPE_F32 ? 4 : 2,
                                                        cand_norm ? 1 : 0)
                                      .bytes);
    HSN_ABI_END
}
