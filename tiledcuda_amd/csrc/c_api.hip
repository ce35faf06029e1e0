// Implementation of the C-ABI declared in include/tcu_c_api.h: argument checks, shape
// dispatch and kernel launches. No device memory is allocated here and no stream is
// synchronised (but for tcu_lstm_persistent_status, whose purpose it is); errors become status codes plus a
// thread-local message.
#include "tcu_c_api.h"

#include "kernels/b2b_gemm_fwd.hpp"
#include "kernels/b2b_gemm_stream.hpp"
#include "kernels/flash_attn_fwd.hpp"
#include "kernels/flash_attn_keys.hpp"
#include "kernels/flash_attn_tile_w64.hpp"
#include "kernels/flash_attn_w64_k32.hpp"
#include "kernels/flash_attn_w64.hpp"
#include "kernels/gemm_direct.hpp"
#include "kernels/gemm_pipelined.hpp"
#include "kernels/gemm_ragged.hpp"
#include "kernels/gemm_w128.hpp"
#include "kernels/gemm_w128k.hpp"
#include "kernels/lstm_direct.hpp"
#include "kernels/lstm_fwd.hpp"
#include "kernels/lstm_layer.hpp"
#include "kernels/lstm_ragged.hpp"
#include "kernels/lstm_recurrent.hpp"
#include "kernels/mod.hpp"

#include <climits>
#include <cstdlib>
#include <mutex>
#include <set>
#include <algorithm>
#include <string>
#include <tuple>
#include <type_traits>
#include <utility>

using namespace tiledcuda;
using namespace tiledcuda::kernels;
namespace tl = tiledcuda::cell::tile_layout;

namespace {

thread_local std::string g_last_error;

// kernels whose dynamic-LDS limit has already been raised, per device
std::mutex g_attr_mutex;
std::set<std::pair<const void*, int>> g_attr_done;

int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}

int hip_fail(hipError_t e, const char* what) {
    return fail(TCU_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

/// The kernels that the thread's last launches ran (host functions; tcu_recent_kernel names them).
constexpr unsigned kRecentKernels = 4;
thread_local const void* g_recent_kernels[kRecentKernels];
thread_local unsigned g_launches = 0;

/// Launch with dynamic LDS; raises the limit when the kernel needs more than the default. The kernel's parameter types
/// are taken from the kernel pointer and every argument is converted to its parameter's type before its address goes
/// into the argument array: an argument of another width or a wrong count is a compile error, not a garbled launch.
template <typename... Params, typename... Args>
int launch(void (*kernel)(Params...), dim3 grid, dim3 block, int lds_bytes, hipStream_t stream, Args&&... args) {
    static_assert(sizeof...(Params) == sizeof...(Args), "launch: argument count differs from the kernel's parameter count");
    static_assert((std::is_convertible_v<Args&&, Params> && ...), "launch: an argument does not convert to its parameter's type");
    if (lds_bytes > kMaxLdsBytes) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "kernel needs more LDS than a CU has");
    if (lds_bytes > 48 * 1024) {
        // once per kernel function (and per device: the attribute is per device)
        int device = 0;
        (void)hipGetDevice(&device);
        const auto key = std::make_pair(reinterpret_cast<const void*>(kernel), device);
        bool known;
        {
            std::lock_guard<std::mutex> lock(g_attr_mutex);
            known = g_attr_done.count(key) != 0;
        }
        if (!known) {
            // (every instantiation is launched with one fixed size; asking for the CU's whole LDS would be refused
            // for a kernel that also has static LDS)
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
            if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
            std::lock_guard<std::mutex> lock(g_attr_mutex);
            g_attr_done.insert(key);
        }
    }
    // the launch's own return value: an error left behind earlier by unrelated code of the calling thread is neither
    // reported as this launch's nor cleared
    std::tuple<std::remove_cv_t<Params>...> params(std::forward<Args>(args)...);
    void* argv[sizeof...(Params) + 1];
    [&]<size_t... kIs>(std::index_sequence<kIs...>) {
        ((argv[kIs] = static_cast<void*>(&std::get<kIs>(params))), ...);
    }(std::index_sequence_for<Params...>{});
    hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, argv, size_t(lds_bytes), stream);
    if (e != hipSuccess) return hip_fail(e, "kernel launch");
    g_recent_kernels[g_launches++ % kRecentKernels] = reinterpret_cast<const void*>(kernel);
    return TCU_OK;
}

/// Adds which of the T step launches of an LSTM layer failed to the message (steps before it are enqueued).
int lstm_step_failed(int rc, int t, int T) {
    return fail(rc, g_last_error + " (LSTM step " + std::to_string(t) + " of " + std::to_string(T) +
                        "; the steps before it were enqueued)");
}

bool positive(std::initializer_list<int> v) {
    for (int x : v)
        if (x <= 0) return false;
    return true;
}

/// The kernels move 16 bytes per lane (vector loads, direct-to-LDS loads, vector stores): operands must start on a
/// 16-byte boundary (null = absent optional operand is fine here; required ones are checked for null separately).
bool aligned16(std::initializer_list<const void*> v) {
    for (const void* p : v)
        if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return false;
    return true;
}

// ---------------------------------------------------------------------------- static scratch
// Device memory owned by the library for the entry point that may not allocate (tcu_lstm_f16_noalloc): every device
// the library runs on holds one copy of this array, at its own address, until the process ends. In host code the
// array's name is only a handle for hipGetSymbolAddress, never a device address.
constexpr unsigned long long kScratchBytes = 64ull << 20;
constexpr unsigned long long kPersistentSyncBytes = 4096;  // synchronisation words in front of the pre-activations
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

/// Device address of `scratch` on the current device, looked up once per device.
int scratch_address(void** out) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (device < 0 || device >= kMaxDevices) return fail(TCU_ERR_HIP, "device ordinal beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!ptr || reinterpret_cast<uintptr_t>(ptr) % 256 != 0)
            return fail(TCU_ERR_HIP, "hipGetSymbolAddress(scratch) returned an unusable address");
        g_scratch_ptr[device] = ptr;
    }
    *out = g_scratch_ptr[device];
    return TCU_OK;
}

// ---------------------------------------------------------------------------- scatter_nd
/// Whether p is ordinary (coarse-grained) memory of the current device. Packed f16 atomics are carried out in its L2s; on
/// host, managed, fine-grained and other devices' memory, which a caller may hand over as well, they need not be.
bool plain_device_memory(const void* p) {
    hipPointerAttribute_t attr{};
    if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
        (void)hipGetLastError();  // a caller that checks its own launches later must not find this one's error
        return false;
    }
    int device = -1;
    return attr.type == hipMemoryTypeDevice && !attr.isManaged && attr.allocationFlags == 0 &&
           hipGetDevice(&device) == hipSuccess && attr.device == device;
}

// ---------------------------------------------------------------------------- GEMM
template <typename OutType, int kM, int kN, int kK, int kTM, int kTN, int kChunkK, typename WarpLayout>
int launch_simple_gemm(const __half* A, const __half* B, OutType* C, hipStream_t stream) {
    using Shape = GemmShape<kM, kN, kK>;
    using Cfg = GemmTraits<__half, OutType, Shape, kTM, kTN, WarpLayout, kChunkK>;
    auto kernel = &simple_gemm<__half, OutType, kM, kN, kK, kTM, kTN, typename Cfg::IteratorA, typename Cfg::RegA,
                               typename Cfg::ALoader, typename Cfg::IteratorB, typename Cfg::RegB,
                               typename Cfg::BLoader, typename Cfg::GlobalC, typename Cfg::RegC,
                               typename Cfg::CStorer>;
    return launch(kernel, dim3(kM / kTM, kN / kTN), dim3(Cfg::kThreads), 0, stream, A, B, C);
}

template <typename OutType, int kM, int kN, int kK, int kTM, int kTN, int kTK, int kRK, typename WarpLayout>
int launch_all_mem_gemm(const __half* A, const __half* B, OutType* C, hipStream_t stream) {
    using Cfg = KeGemmTraits<__half, OutType, GemmShape<kM, kN, kK>, GemmShape<kTM, kTN, kTK>, kRK, WarpLayout>;
    auto kernel =
        &gemm<__half, OutType, kM, kN, kK, kTM, kTN, kTK, typename Cfg::GIteratorA, typename Cfg::SIteratorA,
              typename Cfg::SharedA, typename Cfg::RegA, typename Cfg::G2SLoaderA, typename Cfg::S2RLoaderA,
              typename Cfg::GIteratorB, typename Cfg::SIteratorB, typename Cfg::SharedB, typename Cfg::RegB,
              typename Cfg::G2SLoaderB, typename Cfg::S2RLoaderB, typename Cfg::GlobalC, typename Cfg::SharedC,
              typename Cfg::RegC, typename Cfg::R2SStorerC, typename Cfg::S2GStorerC>;
    return launch(kernel, dim3(kM / kTM, kN / kTN), dim3(Cfg::kThreads), Cfg::kShmBytes, stream, A, B, C);
}

using PipeLarge = PipelinedGemmTraits<256, 256, 64, 4, 2, 2>;  // 8 wavefronts, 2 per SIMD
using PipeMid = PipelinedGemmTraits<128, 128, 64, 2, 2, 2>;
using PipeSmall = PipelinedGemmTraits<64, 64, 64, 2, 2, 2>;
using PipeSmallRing = PipelinedGemmTraits<64, 64, 64, 2, 2, 4>;  // 4-stage ring, 64 KiB of LDS: 2 workgroups per CU
using PipeTallRing = PipelinedGemmTraits<96, 64, 64, 2, 2, 4>;   // the same, 80 KiB
using PipeWideRing = PipelinedGemmTraits<96, 96, 64, 2, 3, 4>;   // 6 wavefronts, 96 KiB: one workgroup per CU

/// Which tile the pipelined kernel takes for a shape, and what the launch is expected to cost. A launch runs
/// ceil(tiles / capacity) rounds of workgroups, capacity = 256 CUs x the workgroups of that size a CU holds (1, 2, 4),
/// and a round costs K / 1024 x 25.5, 16 or 13 us for 256 x 256, 128 x 128 and 64 x 64 tiles (measured on full rounds at
/// K = 1024 .. 4096); the larger tile wins a tie. With few 64 x 64 tiles per CU there is no neighbour workgroup to hide
/// the latency of a tile's loads behind: then the same tile with a 4-stage ring (3 tiles in flight, 2 workgroups per
/// CU) is the choice: 4.2 us per K / 1024 with at most one workgroup per CU (1024^2 x 8192: 36.7 us), 5.8 with two, 7 per
/// round beyond.
enum PipeConfig { kPipeLarge, kPipeMid, kPipeSmall, kPipeSmallRing };
struct PipePlan {
    PipeConfig config;
    double us;
};
PipePlan pipelined_plan(int M, int N, int K) {
    const auto tiles = [&](int tile) { return (long)((M + tile - 1) / tile) * ((N + tile - 1) / tile); };
    const auto rounds = [&](int tile, int per_cu) { return double((tiles(tile) + 256l * per_cu - 1) / (256l * per_cu)); };
    const double large = rounds(256, 1) * 25.5, mid = rounds(128, 2) * 16.0, small = rounds(64, 4) * 13.0;
    const double ring = tiles(64) <= 256 ? 4.2 : tiles(64) <= 512 ? 5.8 : rounds(64, 2) * 7.0;
    const double least_small = small < ring ? small : ring;
    PipePlan plan;
    if (large <= mid && large <= least_small) plan = {kPipeLarge, large};
    else if (mid <= least_small) plan = {kPipeMid, mid};
    else if (small <= ring) plan = {kPipeSmall, small};
    else plan = {kPipeSmallRing, ring};
    plan.us = 2.5 + plan.us * K / 1024.0;
    return plan;
}

/// The pipelined kernel for M, N, K any multiples of 16, with the tile of pipelined_plan(). Edge tiles (rows clamped,
/// stores guarded, the K tail zeroed in LDS) are compiled in only where the shape is not a whole number of the chosen
/// tiles. ldb other than K and words to clear: f32 results only; wide_ring: f16 results only.
template <typename OutType>
int gemm_pipelined_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream,
                            int ldc = 0, int ldb = 0, unsigned int* zero_words = nullptr, int zero_count = 0, bool wide_ring = false) {
    if (ldc == 0) ldc = N;
    if (ldb == 0) ldb = K;
    if (M % 16 != 0 || N % 16 != 0 || K % 16 != 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM shapes are whole 16 x 16 tiles: M, N and K must be multiples of 16");
    if ((long)ldb * 512 >= (1l << 32))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "pipelined GEMM addresses a tile's rows with 32-bit offsets: K < 2^23");
    auto go = [&](auto traits) {
        using Traits = decltype(traits);
        const long grid = (long)((M + Traits::kBM - 1) / Traits::kBM) * ((N + Traits::kBN - 1) / Traits::kBN);
        if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM: too many tiles for one launch");
        if constexpr (std::is_same_v<OutType, float>)
            if (ldb != K || zero_count > 0)
                return launch(&gemm_pipelined<Traits, OutType, true, true>, dim3(unsigned(grid)), dim3(Traits::kThreads),
                              Traits::template lds_bytes<OutType>(), stream, A, B, C, M, N, K, ldb, ldc, zero_words, zero_count);
        if (M % Traits::kBM == 0 && N % Traits::kBN == 0 && K % Traits::kBK == 0)
            return launch(&gemm_pipelined<Traits, OutType, false>, dim3(unsigned(grid)), dim3(Traits::kThreads),
                          Traits::template lds_bytes<OutType>(), stream, A, B, C, M, N, K, ldb, ldc, zero_words, zero_count);
        return launch(&gemm_pipelined<Traits, OutType, true>, dim3(unsigned(grid)), dim3(Traits::kThreads),
                      Traits::template lds_bytes<OutType>(), stream, A, B, C, M, N, K, ldb, ldc, zero_words, zero_count);
    };
    if constexpr (std::is_same_v<OutType, __half>)
        if (wide_ring) return go(PipeWideRing{});
    switch (pipelined_plan(M, N, K).config) {
        case kPipeLarge: return go(PipeLarge{});
        case kPipeMid: return go(PipeMid{});
        case kPipeSmall: return go(PipeSmall{});
        default: break;
    }
    // the ring, f16 results, more than one 64 x 64 tile per CU, M not whole tiles: tiles of 96 x 64 where there is at most one of them
    // per CU. us, 64 x 64 -> 96 x 64: 1040^2 x 2064: 19.2 -> 15.1; 1312 x 784 x 2832: 24.7 -> 19.0; 624 x 1984 x 1344: 10.0, 10.1 (of 60 such
    // sizes 57 are as short or shorter, on average by 11 %, and 3 longer, at most by 2.5 %: 2544 x 448 x 3936: 23.7, 24.3). Whole tiles
    // have no edges to lose (832 x 1664 x 1152: 8.9, 9.4), f32 results, 32 bytes per lane and row, gain at long K only (1184 x 1120 x
    // 672: 8.1, 8.3), a single step of K nothing (1968 x 768 x 64: 3.4, 3.5).
    if constexpr (std::is_same_v<OutType, __half>) {
        const long small = (long)((M + 63) / 64) * ((N + 63) / 64), tall = (long)((M + 95) / 96) * ((N + 63) / 64);
        if (M % 64 != 0 && K >= 256 && small > 256 && small <= 512 && tall <= 256) return go(PipeTallRing{});
    }
    return go(PipeSmallRing{});
}

template <typename OutType>
int gemm_w128_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream,
                       int lda = 0, int ldb = 0, int ldc = 0, unsigned int* zero_words = nullptr, int zero_count = 0) {
    using T = GemmW128Traits;
    if (lda == 0) lda = K;
    if (ldb == 0) ldb = K;
    if (ldc == 0) ldc = N;
    if (M % 16 != 0 || N % 16 != 0 || K % 16 != 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD GEMM needs M, N and K in multiples of 16");
    if ((long)std::max(lda, ldb) * 2 * T::kBM >= (1l << 32))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD GEMM addresses a 256-row panel with 32-bit offsets");
    if (M % T::kBM == 0 && N % T::kBN == 0 && K % T::kBK == 0)
        return launch(&gemm_w128<OutType>, dim3((M / T::kBM) * (N / T::kBN)), dim3(T::kThreads), T::kLdsBytes, stream, A, B,
                      C, M, N, K, lda, ldb, ldc, zero_words, zero_count);
    // edge tiles: rows beyond M or N loaded from the last valid row, stores guarded, a partial last tile of K zero-filled
    const long grid = (long)((M + T::kBM - 1) / T::kBM) * ((N + T::kBN - 1) / T::kBN);
    if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM: too many tiles for one launch");
    return launch(&gemm_w128<OutType, T, true>, dim3(unsigned(grid)), dim3(T::kThreads), T::kLdsBytes, stream, A, B, C, M, N,
                  K, lda, ldb, ldc, zero_words, zero_count);
}

/// gemm_w128 with 256 x 128 workgroup tiles: for products with too few 256 x 256 tiles to fill the chip and too many
/// 128 x 128 tiles for one round of the K-splitting kernel.
template <typename OutType>
int gemm_w128_narrow_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream,
                              int ldc = 0) {
    using T = GemmW128TraitsN<4>;
    if (ldc == 0) ldc = N;
    if (M % 16 != 0 || N % 16 != 0 || K % T::kBK != 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD GEMM with 256 x 128 tiles needs M and N in "
                                               "multiples of 16 and K % 64 == 0");
    if ((long)K * 2 * T::kBM >= (1l << 32))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD GEMM addresses a 256-row panel with 32-bit offsets");
    if (M % T::kBM == 0 && N % T::kBN == 0)
        return launch(&gemm_w128<OutType, T>, dim3((M / T::kBM) * (N / T::kBN)), dim3(T::kThreads), T::kLdsBytes, stream, A,
                      B, C, M, N, K, K, K, ldc, static_cast<unsigned int*>(nullptr), 0);
    // edge tiles: rows beyond M or N loaded from the last valid row, stores guarded
    const long grid = (long)((M + T::kBM - 1) / T::kBM) * ((N + T::kBN - 1) / T::kBN);
    if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM: too many tiles for one launch");
    return launch(&gemm_w128<OutType, T, true>, dim3(unsigned(grid)), dim3(T::kThreads), T::kLdsBytes, stream, A, B, C, M, N,
                  K, K, K, ldc, static_cast<unsigned int*>(nullptr), 0);
}

template <typename OutType, typename T>
int launch_gemm_w128k(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream, int ldc) {
    const long grid = (long)((M + T::kBM - 1) / T::kBM) * ((N + T::kBN - 1) / T::kBN);
    if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM: too many tiles for one launch");
    // edge tiles: rows beyond M or N loaded from the last valid row, stores guarded per 16 x 16 block; with a tail in K also
    // where M and N are whole tiles
    const bool whole = M % T::kBM == 0 && N % T::kBN == 0;
    auto kernel = K % T::kBK != 0 ? &gemm_w128k<OutType, true, T, true> : whole ? &gemm_w128k<OutType, false, T> : &gemm_w128k<OutType, true, T>;
    return launch(kernel, dim3(unsigned(grid)), dim3(T::kThreads), T::kLdsBytes, stream, A, B, C, M, N, K, K, K, ldc,
                  static_cast<unsigned int*>(nullptr), 0);
}

template <typename OutType>
int gemm_w128k_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream,
                        int ldc = 0) {
    using T = GemmW128kTraits;
    if (ldc == 0) ldc = N;
    if (M % 16 != 0 || N % 16 != 0 || K % 16 != 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the K-splitting one-wavefront-per-SIMD GEMM needs M, N and K in multiples of 16");
    if ((long)K * 2 * T::kBM >= (1l << 32))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the K-splitting GEMM addresses a 128-row panel with 32-bit offsets");
    // All workgroups run at once (one per CU), so the launch takes as long as one tile: when 128 x 128 tiles would
    // leave a quarter of the CUs idle and 128 x 96 tiles still fit one round, the smaller tile is the shorter launch
    const long rows = (M + 127) / 128;
    const long tiles128 = rows * ((N + 127) / 128), tiles96 = rows * ((N + 95) / 96);
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        cus = 0;
    if (cus > 0 && tiles128 <= (3l * cus) / 4 && tiles96 <= cus)
        return launch_gemm_w128k<OutType, GemmW128kTraitsN<6>>(A, B, C, M, N, K, stream, ldc);
    return launch_gemm_w128k<OutType, T>(A, B, C, M, N, K, stream, ldc);
}

template <typename OutType, int kM, int kN, int kK, int kTM, int kTN, typename WarpLayout>
int launch_tile_pipelined(const __half* A, const __half* B, OutType* C, hipStream_t stream) {
    using Traits = PipelinedGemmTileTraits<__half, OutType, GemmShape<kM, kN, kK>, kTM, kTN, WarpLayout>;
    auto kernel = &gemm_tile_pipelined<__half, OutType, Traits>;
    return launch(kernel, dim3((kM / kTM) * (kN / kTN)), dim3(Traits::kThreads), Traits::kShmBytes, stream, A, B, C);
}

/// The pipelined kernel composed from tile-library functors has compile-time shapes, like every kernel written against
/// the tile API: the instantiations below are the benchmark shape and the shapes its tests use.
template <typename OutType>
int gemm_tile_pipelined_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream) {
    using W42 = tl::RowMajor<4, 2>;
    using W22 = tl::RowMajor<2, 2>;
    if (M == 4096 && N == 4096 && K == 4096) return launch_tile_pipelined<OutType, 4096, 4096, 4096, 256, 256, W42>(A, B, C, stream);
    if (M == 1024 && N == 1024 && K == 1024) return launch_tile_pipelined<OutType, 1024, 1024, 1024, 256, 256, W42>(A, B, C, stream);
    if (M == 512 && N == 768 && K == 192) return launch_tile_pipelined<OutType, 512, 768, 192, 128, 128, W22>(A, B, C, stream);
    if (M == 256 && N == 256 && K == 64) return launch_tile_pipelined<OutType, 256, 256, 64, 64, 64, W22>(A, B, C, stream);
    return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the tile-API pipelined GEMM is instantiated for 4096^3, 1024^3, 512x768x192 "
                                           "and 256x256x64");
}

template <typename OutType, int kM, int kN, int kK>
int launch_tile_w128(const __half* A, const __half* B, OutType* C, hipStream_t stream) {
    using Traits = ScheduledGemmTileTraits<__half, OutType, GemmShape<kM, kN, kK>>;
    auto kernel = &gemm_tile_w128<__half, OutType, Traits>;
    return launch(kernel, dim3((kM / Traits::kTM) * (kN / Traits::kTN)), dim3(Traits::kThreads), Traits::kShmBytes, stream,
                  A, B, C);
}

/// The one-wavefront-per-SIMD kernel composed from tile-library functors: compile-time shapes, as above.
template <typename OutType>
int gemm_tile_w128_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream) {
    if (M == 4096 && N == 4096 && K == 4096) return launch_tile_w128<OutType, 4096, 4096, 4096>(A, B, C, stream);
    if (M == 1024 && N == 1024 && K == 1024) return launch_tile_w128<OutType, 1024, 1024, 1024>(A, B, C, stream);
    if (M == 512 && N == 768 && K == 192) return launch_tile_w128<OutType, 512, 768, 192>(A, B, C, stream);
    if (M == 256 && N == 256 && K == 64) return launch_tile_w128<OutType, 256, 256, 64>(A, B, C, stream);
    return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the tile-API one-wavefront-per-SIMD GEMM is instantiated for 4096^3, 1024^3, "
                                           "512x768x192 and 256x256x64");
}

/// M or N a little above a multiple of 256: edge tiles of 256 x 256 cost a whole extra round of workgroups for a
/// sliver of output. When the cost model says so, the product is computed as three launches on disjoint parts of C:
/// the leading block of whole 256 x 256 tiles by the one-wavefront-per-SIMD kernel, the columns beyond it (all rows)
/// and the rows beyond it (the leading columns) by the pipelined kernel with small tiles. Same order of the sum
/// everywhere, so the result is bit for bit that of one launch. Returns kPlanNotTaken when the plain launch is the
/// better plan.
constexpr int kPlanNotTaken = INT_MIN;
double gemm_w128_us(long tiles, int K);
template <typename OutType>
int gemm_main_and_strips(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream,
                         double other_us) {
    using T = GemmW128Traits;
    const int Mm = M / T::kBM * T::kBM, Nm = N / T::kBN * T::kBN;
    if ((Mm == M && Nm == N) || K % T::kBK != 0 || (long)K * 512 >= (1l << 32)) return kPlanNotTaken;
    const long tiles = (long)(Mm / T::kBM) * (Nm / T::kBN);
    if (tiles < 128) return kPlanNotTaken;
    const double main_us = gemm_w128_us(tiles, K);
    const double right_us = N > Nm ? 2.0 + pipelined_plan(M, N - Nm, K).us : 0.0;
    const double bottom_us = M > Mm ? 2.0 + pipelined_plan(M - Mm, Nm, K).us : 0.0;
    if (main_us + right_us + bottom_us >= std::min(other_us, pipelined_plan(M, N, K).us)) return kPlanNotTaken;
    int rc = gemm_w128_dispatch<OutType>(A, B, C, Mm, Nm, K, stream, K, K, N);
    if (rc == TCU_OK && N > Nm) rc = gemm_pipelined_dispatch<OutType>(A, B + size_t(Nm) * K, C + Nm, M, N - Nm, K, stream, N);
    if (rc == TCU_OK && M > Mm)
        rc = gemm_pipelined_dispatch<OutType>(A + size_t(Mm) * K, B, C + size_t(Mm) * N, M - Mm, Nm, K, stream, N);
    return rc;
}

/// Whether AUTO sends an unsplit product to the kernel whose wavefronts split K: about one 128 x 128 tile per CU and a
/// long enough K (2048^3: 21.9 against 26.8 us for the LDS-bound 64 x 64-per-wavefront tilings, 1536 x 1536 x 4096: 26.6
/// against 38.5 us, 2048 x 2048 x 1536: 19.8 against 22.6 us); with a short K its reduction through LDS costs more than
/// it saves. A K that is not a multiple of 128 costs the last step in full; the kernels it would go to instead lose as much
/// (1808 x 1808 x 1040: 20.8 -> 15.8 us, 2064 x 1040 x 1072: 15.6 -> 14.5, 1552 x 1552 x 1600: 18.4 -> 15.7, 2048 x 2048 x 4112:
/// 74.0 -> 39.3, 1040 x 1040 x 8208: 67.4 -> 50.2, 176 x 7104 x 13104: 159 -> 115), but for a short K in multiples of 64 (2000 x
/// 2000 x 1088: 16.0 against 16.4), and where half or more of a tile would lie beyond M or N (48 x 11968 x 12864: 102 us
/// against 77, 15936 x 32 x 12816: 128 against 93, 64 x 13200 x 7856: 78 against 71).
bool gemm_w128k_is_the_choice(int M, int N, int K) {
    if (M % 16 != 0 || N % 16 != 0 || K % 16 != 0 || K < 1024 || (long)K * 256 >= (1l << 32)) return false;
    if (K % 128 != 0 && (M <= 64 || N <= 64)) return false;
    if (K % 128 == 64 && K < 1536) return false;
    const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
    // the fewer tiles, the longer K has to be (1408 x 1280 x 4096, 110 tiles: 24.7 against 26.1 us; 1536 x 1280 x 2048, 120:
    // 15.6 against 14.2; 1792^2 x 1024, 196: 11.8 against 13.2; 1536^2 x 1024, 144: 10.3 against 10.0)
    // (512 x 2304 x 8192, 72 tiles: 40.3 against 42.7; 2304 x 640 x 8192, 90: 41.3 against 46.8)
    return tiles >= (K >= 8192 ? 72 : K >= 4096 ? 100 : K >= 1536 ? 128 : 150) && tiles <= 256;
}

/// Whether AUTO sends an unsplit product to the 256 x 128 tile: at most 128 tiles of 256 x 256 (half of the chip or
/// more would idle), 128 x 128 tiles need two rounds of the K-splitting kernel, but 256 x 128 tiles fill one round
/// (2048 x 2560 x 4096: 45.9 against 59.1 us for the pipelined kernel, 3072 x 2560 x 4096: 57.0 against 67.3,
/// 4096 x 2048 x 8192: 106.5 against 134.7 us for 128 tiles of 256 x 256); a short K is left to the pipelined kernel's
/// ring.
bool gemm_narrow_is_the_choice(int M, int N, int K) {
    if (M % 16 != 0 || N % 16 != 0 || K % 64 != 0 || K < 1024 || (long)K * 512 >= (1l << 32)) return false;
    if (gemm_w128k_is_the_choice(M, N, K)) return false;
    const long narrow = (long)((M + 255) / 256) * ((N + 127) / 128);  // with edge tiles where M, N are not whole tiles
    return narrow > 128 && narrow <= 256;
}

/// Expected time of one launch, in us, of the kernels above where AUTO runs them (measured on whole-chip launches): the
/// K-splitting kernel 5 us + 0.95 us per 128 of K with 128 x 128 tiles, 0.75 us with 128 x 96 tiles; the 256 x 128 tile
/// 6 us + per 64 of K 0.70 us with up to 160 tiles, rising to 0.83 us with 256; 256 x 256 tiles 3 us + per 1024 of K
/// 23.5 us for every full round of 256 workgroups and, for a single round of t, 10.6 + 12.9 t / 256 us (the chip is
/// power-limited: fewer busy CUs run at a higher clock) but not below 17 us (what one workgroup needs by itself).
double gemm_w128k_us(int M, int N, int K) {
    const long rows = (M + 127) / 128;
    const long tiles128 = rows * ((N + 127) / 128), tiles96 = rows * ((N + 95) / 96);
    return 5.0 + (tiles128 <= 192 && tiles96 <= 256 ? 0.75 : 0.95) * ((K + 127) / 128);
}

double gemm_narrow_us(int M, int N, int K) {
    const long narrow = (long)((M + 255) / 256) * ((N + 127) / 128);
    return 6.0 + (0.70 + 0.13 * (narrow > 160 ? double(narrow - 160) / 96.0 : 0.0)) * (K / 64);
}

double gemm_w128_us(long tiles, int K) {
    const long full = (tiles - 1) / 256, last = tiles - 256 * full;
    // a last round behind full ones starts unevenly (the XCDs differ by about 4 %) and runs beside their stragglers:
    // 13 to 23 us measured, rising with its fill (8192 x 8448, 7168^2, 6144^2, 2560 x 8192, 6976 x 8192)
    const double fill = last / 256.0;
    const double last_us = full == 0 ? std::max(17.0, 10.6 + 12.9 * fill) : std::min(23.5, 12.0 + 20.0 * fill);
    return 3.0 + (K / 1024.0) * (23.5 * full + last_us);
}

/// Whether a product with f16 results that the K-splitting kernel would take (about one tile of 128 x 128 or 128 x 96 per CU) goes to the
/// pipelined kernel's ring with tiles of 96 x 96 instead: with a K this short the sums over the wavefronts cost more than the fragments
/// that they share save. One workgroup per CU, 2.5 us + per 1024 of K 6.2 us with few of them, 8.4 with 256; a K tail costs the other
/// kernel 1 us. us, K-splitting -> this: 2064 x 1040 x 1072: 13.6 -> 11.4; 576 x 3776 x 1264: 14.2 -> 12.3; 992 x 1952 x 1680: 14.8 -> 15.2 (of
/// 36 such sizes 33 are shorter, on average by 8 %). f32 results take this kernel 1.3 us more and stay (34 sizes, on average as long:
/// 2096 x 1040 x 1424: 16.0, 14.8; 976 x 1936 x 1552: 14.9, 15.9), and so does a longer K (2048 x 1024 x 4096: 26.9, 31.0).
bool gemm_wide_ring_is_the_choice(int M, int N, int K) {
    const long tiles = (long)((M + 95) / 96) * ((N + 95) / 96);
    if (tiles > 256 || (long)K * 512 >= (1l << 32)) return false;
    return 2.5 + (6.2 + 2.2 * double(tiles) / 256.0) * K / 1024.0 < 0.97 * (gemm_w128k_us(M, N, K) + (K % 128 != 0 ? 1.0 : 0.0));
}

/// More than one round of 256 x 256 tiles, the last of them far from full (2560 x 8192: 320 tiles, the last 64 of which
/// cost as much again as the first 256): the leading rows (or columns) whose tiles fill whole rounds go to gemm_w128, the
/// rest of C to the kernel that fills the chip with smaller tiles - the K-splitting kernel (32 to 64 tiles of 256 x 256
/// left), the 256 x 128 tile (65 to 128 left), else the pipelined kernel. Two launches on disjoint parts of C
/// (2560 x 8192 x 4096: 134.6 against 166.3 us, 4352^2 x 4096: 127.8 against 164.1, 3072 x 6144 x 4096: 125.6 against
/// 160.9). M and N in multiples of 16: the split falls on a multiple of 256, every kernel involved has edge tiles.
/// The plan: the best split and what it is expected to cost (1e30: none).
struct GemmRoundsPlan {
    double us;
    int main_rows, main_cols;  // in tiles of 256; one of them is set
};

GemmRoundsPlan gemm_rounds_and_rest_plan(int M, int N, int K) {
    GemmRoundsPlan plan{1e30, 0, 0};
    if (M % 16 != 0 || N % 16 != 0 || K % 64 != 0 || (long)K * 512 >= (1l << 32)) return plan;
    const int tm = (M + 255) / 256, tn = (N + 255) / 256;
    const long tiles = (long)tm * tn;
    if (tiles <= 256 || tiles % 256 == 0) return plan;
    auto rest_us = [&](int Mr, int Nr) {
        if (gemm_w128k_is_the_choice(Mr, Nr, K)) return gemm_w128k_us(Mr, Nr, K);
        if (gemm_narrow_is_the_choice(Mr, Nr, K)) return gemm_narrow_us(Mr, Nr, K);
        return pipelined_plan(Mr, Nr, K).us;
    };
    for (int t = 1; t < tm; ++t) {
        const double us = gemm_w128_us((long)t * tn, K) + 2.0 + rest_us(M - 256 * t, N);
        if (us < plan.us) plan = {us, t, 0};
    }
    for (int t = 1; t < tn; ++t) {
        const double us = gemm_w128_us((long)t * tm, K) + 2.0 + rest_us(M, N - 256 * t);
        if (us < plan.us) plan = {us, 0, t};
    }
    return plan;
}

template <typename OutType>
int gemm_rounds_and_rest(const __half* A, const __half* B, OutType* C, int M, int N, int K, GemmRoundsPlan plan,
                         hipStream_t stream) {
    const int Mm = plan.main_rows ? 256 * plan.main_rows : M, Nm = plan.main_cols ? 256 * plan.main_cols : N;
    int rc = gemm_w128_dispatch<OutType>(A, B, C, Mm, Nm, K, stream, K, K, N);
    if (rc != TCU_OK) return rc;
    const __half* Ar = plan.main_rows ? A + size_t(Mm) * K : A;
    const __half* Br = plan.main_cols ? B + size_t(Nm) * K : B;
    OutType* Cr = plan.main_rows ? C + size_t(Mm) * N : C + Nm;
    const int Mr = plan.main_rows ? M - Mm : M, Nr = plan.main_cols ? N - Nm : N;
    if (gemm_w128k_is_the_choice(Mr, Nr, K)) return gemm_w128k_dispatch<OutType>(Ar, Br, Cr, Mr, Nr, K, stream, N);
    if (gemm_narrow_is_the_choice(Mr, Nr, K)) return gemm_w128_narrow_dispatch<OutType>(Ar, Br, Cr, Mr, Nr, K, stream, N);
    return gemm_pipelined_dispatch<OutType>(Ar, Br, Cr, Mr, Nr, K, stream, N);
}

/// How tcu_gemm_f16_ws runs a product: unsplit (splits == 1), or split over K into `splits` ranges whose f32 partial
/// products come from gemm_w128 (256 x 256 tiles) or from gemm_w128k (128 x 128 tiles: four times the workgroups per
/// range, so a quarter of the ranges - and of the partial products to write and add - fills the chip).
/// Split only if 256 x 256 tiles would leave at least half of the chip idle (at most 128 tiles), K gives every workgroup
/// at least 512 of it (1024 with 128 x 128 tiles), and the split is expected to beat the unsplit launch by 5 %. Expected
/// cost of s ranges (measured, one workgroup per CU at most): 10 us for the two launches and the epilogues + 1.4 us per
/// k-tile of a range + the partial products written and read once (2 x s x M x N x 4 bytes at 5.3 TB/s); of the unsplit
/// launch: pipelined_plan(), or the K-splitting kernel's time where AUTO would run it.
struct GemmSplitPlan {
    int splits;
    bool tiles128;
    double us;
};

/// Expected time of the unsplit launch on few output tiles, apart from the kernel of gemm_direct_plan() and, without `tail`,
/// from the K-splitting kernel where K is not a multiple of its step.
double gemm_unsplit_us(int M, int N, int K, bool tail = true) {
    double us = pipelined_plan(M, N, K).us;
    if (gemm_w128k_is_the_choice(M, N, K) && (tail || K % 128 == 0)) us = std::min(us, gemm_w128k_us(M, N, K));
    if (gemm_narrow_is_the_choice(M, N, K)) us = std::min(us, gemm_narrow_us(M, N, K));
    const long tiles = (long)((M + 255) / 256) * ((N + 255) / 256);
    return tiles > 128 ? std::min(us, gemm_w128_us(tiles, (K + 63) / 64 * 64)) : us;
}

GemmSplitPlan gemm_split_plan(int M, int N, int K) {
    using T = GemmW128Traits;
    GemmSplitPlan plan{1, false, 0.0};
    if (M % 16 != 0 || N % 16 != 0 || K % T::kBK != 0) return plan;
    const bool whole256 = M % T::kBM == 0 && N % T::kBN == 0;  // the 256 x 256 form splits whole tiles only
    const long tiles = (long)((M + T::kBM - 1) / T::kBM) * ((N + T::kBN - 1) / T::kBN);
    const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128);  // (the 128 x 128 form has edge tiles)
    if (tiles > 128) return plan;
    double best_us = 0.95 * gemm_unsplit_us(M, N, K, false);  // (the workspace a caller is told is that of this plan)
    const double plane_us = 2.0 * double(M) * N * 4 / 5.3e6;  // a plane of partial products written and read once
    for (int s = 2; whole256 && s * tiles <= 256 && K % (s * T::kBK) == 0 && K / s >= 512; s *= 2) {
        const double us = 10.0 + 1.4 * (K / s / T::kBK) + s * plane_us;
        if (us < best_us) {
            plan = {s, false, us};
            best_us = us;
        }
    }
    // partial products from the kernel whose wavefronts split K inside the workgroup: 8 us for the two launches, the
    // reduction through LDS and the epilogues + per 128 of a range 0.62 us with up to 128 workgroups, rising to 0.95 us
    // with 256 (their loads share the L2s) - measured on 256^2 x 8192 ... 1024 x 2048 x 16384 with 2 to 16 ranges
    if ((long)K * 256 < (1l << 32)) {
        for (int s = 2; s * tiles128 <= 256 && K % (s * 128) == 0 && K / s >= 512; s *= 2) {
            const long groups = s * tiles128;
            const double per_tile = 0.62 + 0.33 * (groups > 128 ? double(groups - 128) / 128.0 : 0.0);
            const double us = 8.0 + per_tile * (K / s / 128) + s * plane_us;
            if (us < best_us) {
                plan = {s, true, us};
                best_us = us;
            }
        }
    }
    return plan;
}

int gemm_split_count(int M, int N, int K) { return gemm_split_plan(M, N, K).splits; }

/// The tile of the kernel whose 8 wavefronts split K without barriers, and what its launch is expected to cost: 2.4 us + rounds
/// of one workgroup per CU, each as long as its rows take to arrive (95 KB per us and CU) plus 0.1 us per 16 x 16 tile for
/// the sums of the wavefronts, + 0.4 of the time operands and result take at 5.2 TB/s; no less than that whole time; 0.6 us for
/// every round after the first, which a short K does not hide (384 x 448 x 128: three rounds of 1 x 1 tiles 4.5 us, one of 2 x 2
/// 2.9; 3664 x 640 x 1472: three of 4 x 4 22.1, the pipelined kernel 19.8). Within 15 %
/// of the measured times from half a round of workgroups on (with fewer, a CU receives up to 147 KB per us).
struct GemmDirectPlan {
    int ut, rt;
    double us;
};
GemmDirectPlan gemm_direct_plan(int M, int N, int K) {
    GemmDirectPlan plan{0, 0, 1e30};
    if (M % 16 != 0 || N % 16 != 0 || K % 16 != 0 || K >= (1 << 24)) return plan;
    const double once_us = 2.0 * (double(K) * (double(M) + N) + double(M) * N) / 5.2e6;
    for (const auto& [ut, rt] : {std::pair{1, 1}, std::pair{1, 2}, std::pair{2, 1}, std::pair{2, 2}, std::pair{1, 4},
                                 std::pair{4, 1}, std::pair{2, 4}, std::pair{4, 2}, std::pair{4, 4}}) {
        const long groups = (long)((M + 16 * rt - 1) / (16 * rt)) * ((N + 16 * ut - 1) / (16 * ut));
        if (groups > INT_MAX) continue;
        const double cu_us = double((groups + 255) / 256) * (0.1 * ut * rt + 32.0 * (ut + rt) * K / 95e3);
        const double us = 2.4 + std::max(cu_us + 0.4 * once_us, once_us) + 0.6 * double((groups + 255) / 256 - 1);
        if (us < plan.us) plan = {ut, rt, us};
    }
    return plan;
}

/// Whether AUTO runs that kernel rather than another one in a single launch: us, others -> this kernel, 32 x 1024 x 1024:
/// 6.8 -> 2.8; 208 x 464 x 1008: 7.5 -> 3.6; 512^3: 4.4 -> 3.3; 512 x 1024 x 1024: 6.4 -> 5.0; 256 x 4096 x 4096: 21.1 -> 19.5;
/// 1024^3 stays: 6.9 against 7.2.
bool gemm_direct_is_the_choice(int M, int N, int K) { return gemm_direct_plan(M, N, K).us < gemm_unsplit_us(M, N, K); }

/// ... and whether rather than a split over K through a workspace, which takes up to 6 us more than gemm_split_plan() expects
/// when it does not find its operands and planes in the L2s: 32 x 4096 x 4096: 18.1 -> 10.5, 256 x 256 x 8192: 18.1 -> 8.9,
/// 512 x 512 x 8192: 19.4 -> 14.2; 1024 x 1024 x 8192: 29.3 -> 28.3.
bool gemm_split_is_the_choice(int M, int N, int K) {
    const GemmSplitPlan plan = gemm_split_plan(M, N, K);
    return plan.splits > 1 && plan.us + 4.0 <= gemm_direct_plan(M, N, K).us && plan.us < gemm_unsplit_us(M, N, K);
}

template <typename OutType>
int gemm_direct_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream, int ldb = 0,
                         unsigned int* zero_words = nullptr, int zero_count = 0) {
    if (ldb == 0) ldb = K;
    if (M % 16 != 0 || N % 16 != 0 || K % 16 != 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM shapes are whole 16 x 16 tiles: M, N and K must be multiples of 16");
    const GemmDirectPlan plan = gemm_direct_plan(M, N, K);
    if (plan.ut == 0) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the barrier-free GEMM addresses a tile's rows with 32-bit offsets: K < 2^24");
    auto go = [&](auto traits) {
        using T = decltype(traits);
        const long grid = (long)((M + T::kBM - 1) / T::kBM) * ((N + T::kBN - 1) / T::kBN);
        auto kernel = &gemm_direct<T, OutType>;
        if constexpr (std::is_same_v<OutType, float>)  // (the only results that come with a row distance of B or words to clear)
            if (ldb != K || zero_count > 0) kernel = &gemm_direct<T, OutType, true>;
        return launch(kernel, dim3(unsigned(grid)), dim3(T::kThreads), T::kLdsBytes, stream, A, B, C, M, N, K, ldb, zero_words, zero_count);
    };
    switch (10 * plan.ut + plan.rt) {
        case 11: return go(GemmDirectTraits<1, 1>{});
        case 12: return go(GemmDirectTraits<1, 2>{});
        case 21: return go(GemmDirectTraits<2, 1>{});
        case 22: return go(GemmDirectTraits<2, 2>{});
        case 14: return go(GemmDirectTraits<1, 4>{});
        case 41: return go(GemmDirectTraits<4, 1>{});
        case 24: return go(GemmDirectTraits<2, 4>{});
        case 42: return go(GemmDirectTraits<4, 2>{});
        default: return go(GemmDirectTraits<4, 4>{});
    }
}

template <typename OutType>
int gemm_splitk(const __half* A, const __half* B, OutType* C, int M, int N, int K, GemmSplitPlan plan, float* partial,
                hipStream_t stream) {
    using T = GemmW128Traits;
    if ((long)K * 2 * T::kBM >= (1l << 32))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD GEMM addresses a 256-row panel with 32-bit offsets");
    int rc;
    if (plan.tiles128) {
        using Tk = GemmW128kTraits;
        const int tiles = ((M + Tk::kBM - 1) / Tk::kBM) * ((N + Tk::kBN - 1) / Tk::kBN);
        if (M % Tk::kBM == 0 && N % Tk::kBN == 0)
            rc = launch(&gemm_w128k<float, false, Tk>, dim3(tiles, plan.splits), dim3(Tk::kThreads), Tk::kLdsBytes, stream, A,
                        B, partial, M, N, K / plan.splits, K, K, N, static_cast<unsigned int*>(nullptr), 0);
        else  // edge tiles: rows beyond M or N loaded from the last valid row, stores guarded
            rc = launch(&gemm_w128k<float, true, Tk>, dim3(tiles, plan.splits), dim3(Tk::kThreads), Tk::kLdsBytes, stream, A,
                        B, partial, M, N, K / plan.splits, K, K, N, static_cast<unsigned int*>(nullptr), 0);
    } else {
        const int tiles = (M / T::kBM) * (N / T::kBN);
        rc = launch(&gemm_w128<float>, dim3(tiles, plan.splits), dim3(T::kThreads), T::kLdsBytes, stream, A, B, partial, M, N,
                    K / plan.splits, K, K, N, static_cast<unsigned int*>(nullptr), 0);
    }
    if (rc != TCU_OK) return rc;
    const size_t n = size_t(M) * N;
    return launch(&splitk_reduce<OutType>, dim3(unsigned((n / 4 + 255) / 256)), dim3(256), 0, stream,
                  static_cast<const float*>(partial), C, n, plan.splits);
}

template <typename OutType>
int gemm_ragged_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, hipStream_t stream) {
    using T = RaggedGemmTraits;
    if (M % 16 != 0 || N % 16 != 0 || K % 16 != 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM shapes are whole 16 x 16 tiles: M, N and K must be multiples of 16");
    const long grid = (long)((M + T::kBM - 1) / T::kBM) * ((N + T::kBN - 1) / T::kBN);
    if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "GEMM: too many 64 x 64 blocks for one launch");
    return launch(&gemm_ragged<OutType>, dim3(unsigned(grid)), dim3(T::kThreads), 0, stream, A, B, C, M, N, K);
}

template <typename OutType>
int gemm_dispatch(const __half* A, const __half* B, OutType* C, int M, int N, int K, int algo, hipStream_t stream) {
    using W22 = tl::RowMajor<2, 2>;
    switch (algo) {
        case TCU_GEMM_TILE_PIPELINED:
            return gemm_tile_pipelined_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_WAVE128:
            return gemm_w128_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_TILE_WAVE128:
            return gemm_tile_w128_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_WAVE128_KSPLIT:
            if (K % 128 != 0) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the K-splitting one-wavefront-per-SIMD GEMM needs K in multiples of 128");
            return gemm_w128k_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_WAVE128_NARROW:
            return gemm_w128_narrow_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_DIRECT:
            return gemm_direct_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_AUTO:
            // one product of tiles or three: the kernel that takes its operand tiles straight from global memory has the
            // shortest start (48 x 48 x 32: 2.1 us against 2.4; from K = 64 on the next one is as fast). It is also the one
            // whose offsets have 64 bits: every K is accepted there, as it is without the other kernels
            if ((long)M * N < 64 * 64 && (K <= 48 || K >= (1 << 24))) return gemm_ragged_dispatch<OutType>(A, B, C, M, N, K, stream);
            // few output tiles: the kernel that splits K over wavefronts without barriers
            if (gemm_direct_is_the_choice(M, N, K)) return gemm_direct_dispatch<OutType>(A, B, C, M, N, K, stream);
            // where the 256 x 256 tile is the choice anyway, the one-wavefront-per-SIMD kernel is the faster one
            if (M % 256 == 0 && N % 256 == 0 && K % 64 == 0 && (long)(M / 256) * (N / 256) > 128 &&
                (long)K * 512 < (1l << 32)) {
                // ... in one launch, or - where its last round would be far from full and the cost model expects 7 % -
                // on the leading rows or columns, with a second launch of smaller tiles on the rest of C
                const GemmRoundsPlan rounds = gemm_rounds_and_rest_plan(M, N, K);
                if (rounds.us < 0.93 * gemm_w128_us((long)(M / 256) * (N / 256), K))
                    return gemm_rounds_and_rest<OutType>(A, B, C, M, N, K, rounds, stream);
                return gemm_w128_dispatch<OutType>(A, B, C, M, N, K, stream);
            }
            // too few 256 x 256 tiles for the chip, but about one 128 x 128 tile per CU and a long enough K: the
            // kernel whose wavefronts split K (each owns the whole tile)
            if (gemm_w128k_is_the_choice(M, N, K)) {
                if (std::is_same_v<OutType, __half> && gemm_wide_ring_is_the_choice(M, N, K))
                    return gemm_pipelined_dispatch<OutType>(A, B, C, M, N, K, stream, 0, 0, nullptr, 0, true);
                return gemm_w128k_dispatch<OutType>(A, B, C, M, N, K, stream);
            }
            // between the two: 256 x 128 tiles fill one round
            if (gemm_narrow_is_the_choice(M, N, K)) return gemm_w128_narrow_dispatch<OutType>(A, B, C, M, N, K, stream);
            if (M % 16 == 0 && N % 16 == 0) {
                // M or N not multiples of 256: the one-wavefront-per-SIMD kernel with edge tiles, that kernel on the
                // leading block of whole tiles plus the pipelined kernel on the strips beyond it, that kernel on the
                // rows or columns that fill whole rounds plus smaller tiles on the rest, or the pipelined kernel with the
                // tile its cost model picks - whichever is expected to be the shortest
                const long tiles_e = (long)((M + 255) / 256) * ((N + 255) / 256);
                const double edge_us = K % 16 == 0 && tiles_e >= 128 && (long)K * 512 < (1l << 32)
                                           ? gemm_w128_us(tiles_e, (K + 63) / 64 * 64) : 1e30;
                const GemmRoundsPlan rounds = gemm_rounds_and_rest_plan(M, N, K);
                const double rounds_us = rounds.us / 0.93;  // (two launches have to promise 7 % over the other plans)
                const int rc = gemm_main_and_strips<OutType>(A, B, C, M, N, K, stream, std::min(edge_us, rounds_us));
                if (rc != kPlanNotTaken) return rc;
                const double pipelined_us = pipelined_plan(M, N, K).us;
                if (rounds_us < edge_us && rounds_us < pipelined_us)
                    return gemm_rounds_and_rest<OutType>(A, B, C, M, N, K, rounds, stream);
                if (edge_us < pipelined_us) return gemm_w128_dispatch<OutType>(A, B, C, M, N, K, stream);
            }
            [[fallthrough]];
        case TCU_GEMM_PIPELINED:
            return gemm_pipelined_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_RAGGED:
            return gemm_ragged_dispatch<OutType>(A, B, C, M, N, K, stream);
        case TCU_GEMM_GLOBAL_REG:
          if constexpr (std::is_same_v<OutType, float>) {
            if (M == 128 && N == 64 && K == 256)  // the README shape of the reference
                return launch_simple_gemm<OutType, 128, 64, 256, 128, 64, 32, W22>(A, B, C, stream);
            if (M == 1024 && N == 1024 && K == 2048)  // the driver shape of 01_gemm_global_reg/main.cu:105-106
                return launch_simple_gemm<OutType, 1024, 1024, 2048, 256, 128, 64, W22>(A, B, C, stream);
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "global->register GEMM is instantiated for 128x64x256 and "
                                                   "1024x1024x2048 only");
          }
          [[fallthrough]];
        case TCU_GEMM_ALL_MEM:
          if constexpr (std::is_same_v<OutType, float>) {
            if (algo == TCU_GEMM_ALL_MEM && M == 128 && N == 64 && K == 256)
                return launch_all_mem_gemm<OutType, 128, 64, 256, 64, 64, 64, 32, W22>(A, B, C, stream);
            if (algo == TCU_GEMM_ALL_MEM && M == 4096 && N == 4096 && K == 4096)  // the driver shape of 02_gemm_all_mem/main.cu:5-8
                return launch_all_mem_gemm<OutType, 4096, 4096, 4096, 64, 256, 32, 32, W22>(A, B, C, stream);
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "single-stage LDS GEMM is instantiated for 128x64x256 and "
                                                   "4096^3 only");
          }
          return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the reference-style GEMM kernels write f32 only");
        default:
            return fail(TCU_ERR_INVALID_ARGUMENT, "unknown GEMM algo");
    }
}

// ---------------------------------------------------------------------------- b2b GEMM
template <typename OutType, int kN, int kK, int kP, int kTM, int kTN, typename WarpLayout>
int launch_b2b(const __half* A, const __half* B, const __half* C, OutType* D, int M, int batch, hipStream_t stream) {
    using Traits = FusedGemmTraits<__half, float, OutType, FusedGemmShape<0, kN, kK, kP>,
                                   FusedGemmShape<kTM, kTN, kK, kP>, WarpLayout>;
    auto kernel = &KeFusedGemm<__half, OutType, Traits>;
    return launch(kernel, dim3(M / kTM, 1, batch), dim3(Traits::kThreads), Traits::kShmBytes, stream, A, B, C, D, M);
}

template <typename OutType, int kN, int kK = 128, int kP = 128, int kTN = 256, int kWaves = 8>
int launch_b2b_tile_resident(const __half* A, const __half* B, const __half* C, OutType* D, int M, int batch, hipStream_t stream) {
    using Traits = ResidentFusedGemmTraits<__half, OutType, kN, kK, kP, kTN, kWaves>;
    return launch(&b2b_gemm_tile_resident<__half, OutType, Traits>, dim3(M / Traits::kTM, batch), dim3(Traits::kThreads),
                  Traits::kShmBytes, stream, A, B, C, D, M);
}

/// Wavefronts of the kernel that streams the weights past 32 rows per wavefront, and whether AUTO runs it rather than the one with 32
/// rows per workgroup (K = P = 128, N a multiple of 256). Both run rounds of one workgroup per CU; a round takes 1.85 us per
/// 256 columns + 1.7 with 32 rows, per 64 columns 1.65 us + 5.5 with 256 rows (8 wavefronts), 1.3 us + 5 with 128 (4).
struct B2bStreamPlan {
    int waves;
    bool is_the_choice;
};
B2bStreamPlan b2b_stream_plan(int M, int N, int batch) {
    const auto rounds = [&](int rows) { return double(((long)((M + rows - 1) / rows) * batch + 255) / 256); };
    const double resident = rounds(32) * (1.85 * (N / 256) + 1.7);
    const double eight = rounds(256) * (1.65 * (N / 64) + 5.5), four = rounds(128) * (1.3 * (N / 64) + 5.0);
    return {eight <= four ? 8 : 4, std::min(eight, four) < 0.93 * resident};
}

template <int kWaves, typename OutType>
int launch_b2b_stream(const __half* A, const __half* B, const __half* C, OutType* D, int M, int N, int batch, hipStream_t stream) {
    using T = B2bStreamTraits<kWaves, 2>;
    const long grid = (long)((M + T::kTM - 1) / T::kTM) * batch;
    if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "b2b GEMM: too many row blocks for one launch");
    return launch(&b2b_gemm_stream<T, OutType>, dim3(unsigned(grid)), dim3(T::kThreads), T::kLdsBytes, stream, A, B, C, D, M, N, batch);
}

template <typename OutType>
int b2b_dispatch(const __half* A, const __half* B, const __half* C, OutType* D, int M, int N, int K, int P, int batch,
                 int algo, hipStream_t stream) {
    if (algo != TCU_B2B_AUTO && algo != TCU_B2B_TILE_LIBRARY && algo != TCU_B2B_RESIDENT && algo != TCU_B2B_ROWS &&
        algo != TCU_B2B_TILE_RESIDENT && algo != TCU_B2B_STREAM)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_b2b_gemm_f16: unknown algo");
    if (algo == TCU_B2B_TILE_RESIDENT) {
        // the LDS-resident kernel composed from tile-library functors: compile-time N, like every tile-API kernel
        if (K == 128 && P == 128 && M % 32 == 0) {
            if (N == 256) return launch_b2b_tile_resident<OutType, 256>(A, B, C, D, M, batch, stream);
            if (N == 1024) return launch_b2b_tile_resident<OutType, 1024>(A, B, C, D, M, batch, stream);
            if (N == 2048) return launch_b2b_tile_resident<OutType, 2048>(A, B, C, D, M, batch, stream);
        }
        if (K == 64 && P == 64 && M % 32 == 0) {
            if (N == 128) return launch_b2b_tile_resident<OutType, 128, 64, 64, 128, 4>(A, B, C, D, M, batch, stream);
            if (N == 256) return launch_b2b_tile_resident<OutType, 256, 64, 64, 128, 4>(A, B, C, D, M, batch, stream);
        }
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the tile-API LDS-resident b2b kernel is instantiated for K = P = 128 with N in "
                                               "{256, 1024, 2048} and for K = P = 64 with N in {128, 256}, M a multiple of 32");
    }
    // many rows: workgroups that keep both weight blocks for their whole life and walk over blocks of 256 rows
    if (algo == TCU_B2B_ROWS || (algo == TCU_B2B_AUTO && (long)M * batch >= 32768)) {
        if (N == 256 && K == 128 && P == 128 && M % 64 == 0) {
            using T = B2bRowsTraits;
            const int blocks = (M + T::kRowsPerBlock - 1) / T::kRowsPerBlock;
            const int per_item = std::max(1, 256 / batch);  // one workgroup per CU: about 256 in all
            return launch(&b2b_gemm_rows<OutType>, dim3(std::min(blocks, per_item), batch), dim3(T::kThreads), T::kLdsBytes,
                          stream, A, B, C, D, M);
        }
        if (algo == TCU_B2B_ROWS)
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the many-rows b2b kernel takes N = 256, K = P = 128 and M a multiple of 64");
    }
    // long N and many rows: the weights pass once for 128 or 256 rows
    if (algo == TCU_B2B_STREAM || algo == TCU_B2B_AUTO) {
        if (N % 256 == 0 && N > 256 && N < (1 << 23) && K == 128 && P == 128 && M % 32 == 0) {
            const B2bStreamPlan plan = b2b_stream_plan(M, N, batch);
            if (algo == TCU_B2B_STREAM || plan.is_the_choice)
                return plan.waves == 8 ? launch_b2b_stream<8>(A, B, C, D, M, N, batch, stream) : launch_b2b_stream<4>(A, B, C, D, M, N, batch, stream);
        }
        if (algo == TCU_B2B_STREAM)
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the weight-streaming b2b kernel takes K = P = 128, N a multiple of 256 from 512 to "
                                                   "2^23 and M a multiple of 32");
    }
    if (algo != TCU_B2B_TILE_LIBRARY) {
        if (N % 256 == 0 && K == 128 && P == 128 && M % 32 == 0)
            return launch(&b2b_gemm_resident<OutType>, dim3(M / B2bResidentTraits::kTM, batch),
                          dim3(B2bResidentTraits::kThreads), B2bResidentTraits::kLdsBytes, stream, A, B, C, D, M, N);
        if (algo == TCU_B2B_RESIDENT)
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the LDS-resident b2b kernel takes K = P = 128, N a multiple of 256 "
                                                   "and M a multiple of 32");
    }
    // K = P = 64: the LDS-resident composition from tile-library functors is the fast kernel (direct-to-LDS loads, both
    // products split over the wavefronts): 2.2 against 3.0 us at the reference driver's (256, 128, 64, 64)
    if (algo == TCU_B2B_AUTO && K == 64 && P == 64 && M % 32 == 0) {
        if (N == 128) return launch_b2b_tile_resident<OutType, 128, 64, 64, 128, 4>(A, B, C, D, M, batch, stream);
        if (N == 256) return launch_b2b_tile_resident<OutType, 256, 64, 64, 128, 4>(A, B, C, D, M, batch, stream);
    }
    if (N == 256 && K == 128 && P == 128) {
        // 32-row tiles keep all 256 CUs busy up to M * batch = 8192; 64-row tiles beyond that
        if (M % 64 == 0 && (long)M * batch > 16384)
            return launch_b2b<OutType, 256, 128, 128, 64, 64, tl::RowMajor<4, 1>>(A, B, C, D, M, batch, stream);
        if (M % 32 == 0) return launch_b2b<OutType, 256, 128, 128, 32, 64, tl::RowMajor<2, 1>>(A, B, C, D, M, batch, stream);
    }
    if (N == 128 && K == 64 && P == 64 && M % 32 == 0)
        return launch_b2b<OutType, 128, 64, 64, 32, 64, tl::RowMajor<2, 1>>(A, B, C, D, M, batch, stream);
    if (N == 64 && K == 64 && P == 64 && M % 16 == 0)
        return launch_b2b<OutType, 64, 64, 64, 16, 32, tl::RowMajor<1, 1>>(A, B, C, D, M, batch, stream);
    // the rest of the shape list of the reference's driver (examples/cpp/02_fused_two_gemms/fused_gemm.cu:212-259),
    // with its tile shapes and warp layouts
    if (N == 16 && K == 16 && P == 16 && M % 16 == 0)
        return launch_b2b<OutType, 16, 16, 16, 16, 16, tl::RowMajor<1, 1>>(A, B, C, D, M, batch, stream);
    if (N == 32 && K == 16 && P == 32 && M % 16 == 0)
        return launch_b2b<OutType, 32, 16, 32, 16, 16, tl::RowMajor<1, 1>>(A, B, C, D, M, batch, stream);
    if (N == 64 && K == 32 && P == 64 && M % 32 == 0)
        return launch_b2b<OutType, 64, 32, 64, 32, 32, tl::RowMajor<2, 1>>(A, B, C, D, M, batch, stream);
    if (N == 1024 && K == 128 && P == 128 && M % 64 == 0)
        return launch_b2b<OutType, 1024, 128, 128, 64, 64, tl::RowMajor<4, 1>>(A, B, C, D, M, batch, stream);
    if (N == 2048 && K == 128 && P == 128 && M % 64 == 0)
        return launch_b2b<OutType, 2048, 128, 128, 64, 128, tl::RowMajor<4, 1>>(A, B, C, D, M, batch, stream);
    return fail(TCU_ERR_UNSUPPORTED_SHAPE,
                "the tile-library b2b GEMM is instantiated for (N, K, P) in {(16,16,16), (32,16,32), (64,32,64), (64,64,64), "
                "(128,64,64), (256,128,128), (1024,128,128), (2048,128,128)} with M a multiple of its row tile (16 ... 64); "
                "the LDS-resident kernel takes K = P = 128, N % 256 == 0, M % 32 == 0");
}

// ---------------------------------------------------------------------------- attention
template <int kNStatic, int kD, bool kVRowMajor, int kTM, int kTN, typename WarpLayout>
int launch_fa(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, float scale,
              hipStream_t stream) {
    using Traits = FlashAttentionTraits<__half, float, __half, FlashAttentionShape<0, kNStatic, kD, kD>,
                                        FlashAttentionShape<kTM, kTN, kD, kD>, kVRowMajor, WarpLayout>;
    auto kernel = &flash_attention<__half, __half, Traits>;
    return launch(kernel, dim3(M / kTM, 1, batch), dim3(Traits::kThreads), Traits::kShmBytes, stream, Q, K, V, O, M, N,
                  scale);
}

template <int kNStatic, int kD, bool kVRowMajor, int kTM, int kTN, typename WarpLayout>
int launch_fa_pipelined(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, float scale,
                        hipStream_t stream) {
    using Traits = FlashAttentionTraits<__half, float, __half, FlashAttentionShape<0, kNStatic, kD, kD>,
                                        FlashAttentionShape<kTM, kTN, kD, kD>, kVRowMajor, WarpLayout>;
    auto kernel = &flash_attention_pipelined<__half, __half, Traits>;
    return launch(kernel, dim3(M / kTM, 1, batch), dim3(Traits::kThreads), Traits::kShmBytesPipelined, stream, Q, K, V, O,
                  M, N, scale);
}

template <int kD, int kWaves, bool kFused>
int launch_fa_fwd(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, float scale,
                  hipStream_t stream) {
    using Traits = FlashFwdTraits<kD, kWaves, 64>;
    auto kernel = kFused ? &flash_attention_fwd_fused<Traits> : &flash_attention_fwd<Traits>;
    const long grid = (long)((M + Traits::kBM - 1) / Traits::kBM) * batch;
    if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "attention: too many query blocks for one launch");
    return launch(kernel, dim3(unsigned(grid)), dim3(Traits::kThreads), Traits::kLdsBytes, stream, Q, K, V, O, batch, M, N,
                  scale);
}

template <bool kVColMajor>
int launch_fa_w64(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, float scale,
                  hipStream_t stream) {
    using Traits = FlashW64Traits<128>;
    if ((long)N * 256 >= (1l << 32))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD attention kernel addresses a V block with 32-bit offsets");
    return launch(&flash_attention_fwd_w64<Traits, kVColMajor>, dim3(((M + Traits::kBM - 1) / Traits::kBM) * batch),
                  dim3(Traits::kThreads), Traits::kLdsBytes, stream, Q, K, V, O, batch, M, N, scale);
}

template <int kM, int kN>
int launch_fa_tile_w64(const __half* Q, const __half* K, const __half* V, __half* O, int batch, float scale,
                       hipStream_t stream) {
    using Traits = FlashW64TileTraits<__half, kM, kN, 128>;
    return launch(&flash_attention_tile_w64<__half, Traits>, dim3((kM / Traits::kTM) * batch), dim3(Traits::kThreads),
                  Traits::kShmBytes, stream, Q, K, V, O, batch, scale);
}

/// The one-wavefront-per-SIMD kernel composed from tile-library functors: compile-time sequence lengths, like every
/// kernel written against the tile API (the benchmark shape and the shapes its tests use).
int fa_tile_w64_dispatch(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, int Kd,
                         float scale, int v_layout, hipStream_t stream) {
    if (Kd != 128 || v_layout != TCU_V_ROW_MAJOR)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the tile-API one-wavefront-per-SIMD attention kernel takes head size 128 and a row-major V");
    if (M == 2048 && N == 2048) return launch_fa_tile_w64<2048, 2048>(Q, K, V, O, batch, scale, stream);
    if (M == 512 && N == 1024) return launch_fa_tile_w64<512, 1024>(Q, K, V, O, batch, scale, stream);
    if (M == 256 && N == 640) return launch_fa_tile_w64<256, 640>(Q, K, V, O, batch, scale, stream);
    if (M == 256 && N == 320) return launch_fa_tile_w64<256, 320>(Q, K, V, O, batch, scale, stream);
    return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the tile-API one-wavefront-per-SIMD attention kernel is instantiated for "
                                           "(M, N) in {(2048, 2048), (512, 1024), (256, 640), (256, 320)}");
}

/// The one-wavefront-per-SIMD kernel on the 16x16x32 instruction (tile-library functors, run-time M and N, either V
/// layout).
template <int kD, bool kVColMajor>
int launch_fa_w64_k32(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, float scale,
                      hipStream_t stream) {
    using Traits = FlashW64K32Traits<__half, kD, kVColMajor>;
    // one workgroup per CU; a workgroup with more than one item fetches the next one's first operands under the last
    // steps of the current one. Items keep their XCD (item number modulo 8) only if the grid is a multiple of 8.
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 8)
        return fail(TCU_ERR_HIP, "attention: cannot read the number of compute units");
    const long items = (long)((M + Traits::kTM - 1) / Traits::kTM) * batch;
    const long grid = std::min<long>(items, cus - cus % 8);
    return launch(&flash_attention_w64_k32<__half, Traits>, dim3(unsigned(grid)), dim3(Traits::kThreads),
                  Traits::kShmBytes, stream, Q, K, V, O, batch, M, N, scale);
}

int fa_w64_k32_dispatch(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, int Kd,
                        float scale, int v_layout, hipStream_t stream) {
    using Traits = FlashW64K32Traits<__half, 128>;
    if (Kd != 128 && !(Kd == 64 && v_layout == TCU_V_ROW_MAJOR))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the 16x16x32 one-wavefront-per-SIMD attention kernel is instantiated for head size "
                                               "128, and for head size 64 with a row-major V");
    if (N < Traits::kStages * Traits::kTN)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the 16x16x32 one-wavefront-per-SIMD attention kernel needs N >= 320");
    if ((long)N * 256 >= (1l << 32))
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD attention kernel addresses a V block with 32-bit offsets");
    if (Kd == 64) return launch_fa_w64_k32<64, false>(Q, K, V, O, batch, M, N, scale, stream);
    return v_layout == TCU_V_ROW_MAJOR ? launch_fa_w64_k32<128, false>(Q, K, V, O, batch, M, N, scale, stream)
                                       : launch_fa_w64_k32<128, true>(Q, K, V, O, batch, M, N, scale, stream);
}

/// How many wavefronts (of 32 queries) a workgroup of the 8-wavefront kernels has, and what the launch is expected to take (us).
/// More wavefronts share a block of keys (at head size 128 a CU holds one workgroup whatever its size: 96 KiB of LDS; at 64 up to
/// three of 2 or 4 wavefronts share one, and every workgroup per CU after the third costs as much as the next: fitted to 286
/// sizes of up to 30 per CU, 6 % deviation), fewer leave less idle behind M. Queries beyond M cost their wavefronts' idle time
/// only; wavefronts that save no workgroup are not taken (489 heads of 64 x 64 at head size 64: 6.2 us with 2, 6.5 with 4), and there
/// more than divide M have to promise 6 % (64 x 2688 x 128: 16.6 with 4, 18.4 with 8, 5 % ahead in the model). The time per key rises from a few busy CUs to all of them (the chip is power-limited); workgroups of 2 wavefronts start
/// sooner at head size 128 (7 x 1600 x 128: 7.0 us, which the key-splitting kernel takes 7.7 for).
/// Measured, us with 2, 4, 8 wavefronts (the largest that divides M was taken before): 200 x 192 x 512 at head size 128:
/// 44.5, 33.5, 21.8; 100 x 448^2: 39.8, 29.7, 19.1; 40 x 832 x 960: 70.2, 50.3, 29.7; 96 x 576^2 at head size 64: 26.7,
/// 18.4, 26.6; 1848 x 320 x 64 at 64: 54.2, 48.2, 73.3; 300 x 64 x 512 at 128: 31.2, 33.2, 37.8; 36 x 448^2 at 128: 14.4, 14.8, 16.4.
struct AttnWavesPlan {
    int waves;
    double us;
    long groups;
    double partial_us;  // head size 64: with the 6 % of blocks partly beyond M, which measure 2 to 8 % above us
};
AttnWavesPlan attn_waves_plan(int batch, int M, int N, int D) {
    struct Cost {
        int waves;
        double round128, start128;               // head size 128: rounds of one workgroup per CU
        double one, second, third, next, start;  // head size 64, by the number of workgroups per CU
    };
    AttnWavesPlan plan{8, 1e30, 0, 1e30};
    double best = 1e30;
    for (const Cost& c : {Cost{2, 1.0, 2.6, 1.0, 0.36, 0.41, 0.43, 2.1}, Cost{4, 1.05, 3.2, 0.985, 0.415, 0.808, 0.573, 2.45},
                          Cost{8, 1.15, 3.2, 1.05, 1.13, 1.12, 1.11, 3.05}}) {
        const long groups = (long)batch * ((M + 32 * c.waves - 1) / (32 * c.waves)), per_cu = (groups + 255) / 256;
        if (groups == plan.groups) continue;
        const double fill = std::min(1.0, groups / 256.0);
        double us, score;
        if (D == 128) {
            score = c.round128 * double(per_cu);
            us = 1.3 + score * (c.start128 + N * (0.0205 + 0.0055 * fill));
        } else {
            const double rounds = c.one + (per_cu > 1 ? c.second : 0.0) + (per_cu > 2 ? c.third + double(per_cu - 3) * c.next : 0.0);
            us = 1.0 + rounds * (c.start + N * (0.0138 + 0.002 * fill));
            const int whole = M % 256 == 0 ? 8 : M % 128 == 0 ? 4 : 2;
            score = c.waves > whole ? 1.06 * us : us;
        }
        if (score < best) {
            best = score;
            plan = {c.waves, us, groups, D == 128 ? us : score};
        }
    }
    return plan;
}

template <int kD, bool kFused>
int fa_fwd_by_rows(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, float scale,
                   hipStream_t stream) {
    switch (attn_waves_plan(batch, M, N, kD).waves) {
        case 8: return launch_fa_fwd<kD, 8, kFused>(Q, K, V, O, batch, M, N, scale, stream);
        case 4: return launch_fa_fwd<kD, 4, kFused>(Q, K, V, O, batch, M, N, scale, stream);
        default: return launch_fa_fwd<kD, 2, kFused>(Q, K, V, O, batch, M, N, scale, stream);
    }
}

/// Whether the key-splitting kernel runs workgroups of 32 queries instead of 64: where twice as many of them still have a CU each, the
/// shorter chain of a block counts for more than keys that are fetched twice. us, 64 ->
/// 32 queries: head size 128, one head, 64 x 64: 6.1 -> 4.4; 64 x 256: 7.5 -> 5.5; 8 x 256 x 1024: 12.1 -> 9.1; 60 x 128 x 4096: 36.0 -> 34.0; 512 x
/// 16384 with 16 splits: 17.9 -> 15.5; beyond (2 x 2048 x 4096 with 4 splits, 512 workgroups): 20.1 -> 23.3. Head size 64, 64 x 256: 5.1 ->
/// 4.0; 32 x 64 x 1024: 8.3 -> 6.3; 128 x 64 x 1024: 9.0 -> 7.6; two per CU: 22 x 704 x 192: 5.7 -> 6.1, 44 x 320 x 4608: 27.0 -> 29.4.
bool attn_keys_narrow(int batch, int M, int splits) { return (long)batch * splits * (M / 32) <= 256; }

template <int kD, bool kVColMajor>
int launch_fa_keys(const __half* Q, const __half* K, const __half* V, __half* O, float* part, int batch, int M, int N,
                   int splits, float scale, hipStream_t stream) {
    auto go = [&](auto traits) {
        using Traits = decltype(traits);
        const long grid = (long)batch * splits * (M / Traits::kBM);
        if (grid > INT_MAX || N >= (1 << 24)) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "attention: too many query blocks or keys for one launch");
        return launch(&flash_attention_keys<Traits>, dim3(unsigned(grid)), dim3(Traits::kThreads), Traits::kLdsBytes, stream, Q, K, V, O, part,
                      batch, M, N, splits, scale);
    };
    const int rc = attn_keys_narrow(batch, M, splits) ? go(FlashKeysTraits<kD, kVColMajor, 1>{}) : go(FlashKeysTraits<kD, kVColMajor>{});
    if (rc != TCU_OK || splits == 1) return rc;
    const size_t rows = size_t(batch) * M;
    auto combine = splits <= 4 ? &flash_attention_combine<kD, 4> : splits <= 8 ? &flash_attention_combine<kD, 8> : &flash_attention_combine<kD, 16>;
    return launch(combine, dim3(unsigned((rows * kD / 4 + 255) / 256)), dim3(256), 0, stream, static_cast<const float*>(part), O,
                  rows, splits);
}

int fa_keys_dispatch(const __half* Q, const __half* K, const __half* V, __half* O, float* part, int batch, int M, int N, int Kd,
                     int splits, float scale, int v_layout, hipStream_t stream) {
    if (Kd == 128 && v_layout == TCU_V_ROW_MAJOR)
        return launch_fa_keys<128, false>(Q, K, V, O, part, batch, M, N, splits, scale, stream);
    if (Kd == 128) return launch_fa_keys<128, true>(Q, K, V, O, part, batch, M, N, splits, scale, stream);
    if (Kd == 64 && v_layout == TCU_V_ROW_MAJOR)
        return launch_fa_keys<64, false>(Q, K, V, O, part, batch, M, N, splits, scale, stream);
    return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the key-splitting attention kernel is instantiated for head size 128, and for head "
                                           "size 64 with a row-major V");
}

/// Expected time (us) of the key-splitting kernel with `splits` workgroups per 64 queries: rounds of 256 (head size 128) or
/// 512 workgroups (64: two per CU), a fixed part for the queries, the first keys and the merge, and per block of 4 x 32 keys
/// 0.95 us (0.62 at head size 64) plus what the memory adds as more workgroups read keys of their own (M / 64 of them share
/// theirs): 2.3 us with 256 of them, 6.8 TB/s; no less than the L2s take for a full chip (1.05, 1.15 us); with splits the
/// partial outputs written, read and one launch more. Fitted to 14 shapes at both head sizes with keys and values not in
/// any cache (32 x 64 x 8192 at 128 with 1, 2, 4, 8, 16 workgroups: 83, 52, 34, 31, 37 us; 64 x 64 x 4096: 50, 35, 32, 37;
/// 8 x 64 x 8192: 77, 46, 29, 21, 18). The three workgroups of a head of 192 queries (of which an XCD's 32 CUs hold ten heads and a
/// part) do not stay together over a long sequence at head size 128: its keys come from beyond the L2s for each of them, at 9 TB/s
/// (136 x 192 x 5952: 159 us where the sum gives 133; with blocks of 256 queries 142).
double attn_keys_us(int batch, int M, int N, int D, int splits) {
    const long groups = (long)batch * (M / 64) * splits, cap = D == 128 ? 256 : 512;
    const double blocks = double(N) / (128.0 * splits);
    double us = D == 128 ? 1.5 : 1.3;
    for (long left = groups; left > 0; left -= cap) {
        const double at_once = double(std::min(left, cap)), own = at_once * 64.0 / M, fill = at_once / cap;
        const double round = D == 128 ? 5.0 + blocks * std::max(0.95 + 0.0052 * own, 1.05 * fill)
                                      : 3.5 + 1.6 * std::max(0.0, 2.0 * fill - 1.0) + blocks * std::max(0.62 + 0.0035 * own, 1.15 * fill);
        // (a last round behind full ones, two workgroups per CU: a few of them run beside the stragglers, many start late. Measured
        // against the price of a round by itself 0.6 at fill 0.1 (24 x 1536 x 1728: 29.2 us), 1.25 at 0.6 (18 x 2880 x 1920: 40.9))
        us += round * (D == 64 && left < cap && left < groups ? std::min(1.2, 0.5 + 1.1 * fill) : 1.0);
    }
    if (D == 128 && M == 192 && splits == 1) us = std::max(us, 6.5 + double(groups) * N * 512.0 / 9e6);
    return us + (splits == 1 ? 0.0 : 2.4 + (D == 128 ? 0.011 : 0.006) * groups);
}

/// ... with workgroups of 32 queries, of which there is one round (see attn_keys_narrow()): 1.6 us less before and after the blocks (0.8 at
/// head size 64) and two thirds of the time per block.
double attn_keys_narrow_us(int batch, int M, int N, int D, int splits) {
    const double heads = double(batch) * splits, blocks = double(N) / (128.0 * splits), fill = heads * (M / 32) / 256;
    const double us = D == 128 ? 4.9 + blocks * std::max(0.62 + 0.0052 * heads, 1.05 * fill)
                               : 4.0 + blocks * std::max(0.45 + 0.0035 * heads, 0.58 * fill);
    return us + (splits == 1 ? 0.0 : 2.4 + (D == 128 ? 0.011 : 0.006) * heads * (M / 64));
}

/// Expected time (us) of the kernels with 64 queries per wavefront in blocks of 256 (the 16x16x32 one, and the 32x32x16 one
/// where AUTO runs it), one block per CU at a time, and of the 32-queries-per-wavefront kernel. The time per key rises by a
/// fifth from a few busy CUs to all of them (the chip is power-limited). Within 10 % of the measured times.
double attn_w64_us(int batch, int M, int N, int D) {
    const long items = (long)batch * ((M + 255) / 256), rounds = (items + 255) / 256;
    const double fill = double(items) / (256.0 * rounds);
    return 1.3 + rounds * (D == 128 ? 6.0 + N * (0.02 + 0.005 * fill) : 4.0 + N * (0.0135 + 0.0043 * fill));
}
/// (with blocks partly beyond M dearer: 104 x 448 x 2560 at head size 64: 44.8 us, the key-splitting kernel 38.8; 84 x 576 x 2688: 54, 43)
double attn_fused_us(int batch, int M, int N, int D) { return attn_waves_plan(batch, M, N, D).partial_us; }

/// Whether AUTO's choice among the kernels that give wavefronts their own queries is the 16x16x32 one: from 256 whole blocks of
/// 256 queries on (192 with N >= 1024), unless a last round of few blocks makes it longer than the 32-queries-per-wavefront
/// kernel (22 x 2944^2 at head size 64, 264 blocks: 99.8 against 76.3 us; a column-major V has no such alternative). Where that one
/// runs 8 wavefronts it has to promise 10 % (128 x 1024 x 448 at 64, 8 % ahead in the model: 24.2 against 23.0; 716 x 256 x 320: 31.5
/// against 28.1), else 5 (144 x 512 x 448, 7 %: 20.5 against 22.7; 88 x 832 x 320, 12 %: 16.3 against 18.8). More than three rounds of
/// blocks at 64 run at the power limit, where this kernel's fewer instructions count for more than its estimate says: there it may be
/// 18 % behind (509 x 3264 x 576, 6 %: 322 against 367 us; 458 x 576 x 1152, 23 %: 129, 129; 94 x 3456 x 320, 22 %: 49, 44; with 5 %
/// as below three rounds 39 such sizes were up to 19 % above the shorter of the two, so 1 %).
bool attn_k32_is_the_choice(int batch, int M, int N, int D, int v_layout) {
    const long blocks = (long)batch * (M / 256);
    if (N < 320 || !(blocks >= 256 || (blocks >= 192 && N >= 1024))) return false;
    if (v_layout == TCU_V_COL_MAJOR) return true;
    const AttnWavesPlan other = attn_waves_plan(batch, M, N, D);
    const long items = (long)batch * ((M + 255) / 256);
    const double margin = other.waves == 8 ? 1.1 : D == 64 && items > 3 * 256 ? 1.18 : 1.05;
    return attn_w64_us(batch, M, N, D) <= margin * other.us;
}

/// Whether it is the 32x32x16 kernel with 64 queries per wavefront (row-major V).
bool attn_w64_is_the_choice(int batch, int M, int N, int D) {
    const long blocks = (long)batch * (M / 256);
    return D == 128 && N >= 1024 && blocks >= 128 && blocks < 192;
}

/// Expected time of that choice.
double attn_blocks_us(int batch, int M, int N, int D, int v_layout) {
    if (v_layout == TCU_V_COL_MAJOR || attn_k32_is_the_choice(batch, M, N, D, v_layout) || attn_w64_is_the_choice(batch, M, N, D))
        return attn_w64_us(batch, M, N, D);
    return attn_fused_us(batch, M, N, D);
}

/// How many workgroups per 64 queries split the keys in the shortest plan of the key-splitting kernel (at most
/// max_splits <= 16; every wavefront gets a block, one workgroup per CU at most: 32 x 64 x 8192 at head size 64 with 8, 12,
/// 16: 20.8, 24.9, 24.2 us), or 0 where the other kernels are expected to be as fast. A split has to promise 2.5 us more,
/// which the second launch and the workspace cost the host.
int attn_keys_plan(int batch, int M, int N, int D, int v_layout, int max_splits) {
    if ((D != 128 && !(D == 64 && v_layout == TCU_V_ROW_MAJOR)) || N >= (1 << 24)) return 0;
    const long groups = (long)batch * (M / 64);
    if (groups > 4096) return 0;
    // 192 queries, a column-major V, more workgroups than CUs: blocks of 256 queries, whose fourth wavefront idles, need one round
    // per 256 heads (us, key-splitting against blocks: 96 x 192 x 2368: 61.3, 53; 110 x 192 x 4096: 99, 85; 128 x 192 x 10240:
    // 263, 210), unless the second round has a few workgroups only and not too many keys (88 x 192 x 1600: 34.4, 36.6; x 4096: 80,
    // 84; x 10240: 230, 199)
    if (D == 128 && M == 192 && v_layout == TCU_V_COL_MAJOR && (groups > 272 || (groups > 256 && N > 4096))) return 0;
    double best_us = 1e30;
    int best = 0;
    for (int s : {1, 2, 3, 4, 6, 8, 12, 16}) {
        if (s > max_splits || (s > 1 && (s * groups > 256 || N < 128 * s))) break;
        const double us = attn_keys_us(batch, M, N, D, s) + (s > 1 ? 2.5 : 0.0);
        if (us < best_us) {
            best_us = us;
            best = s;
        }
    }
    // the first keys of a few workgroups arrive 0.5 us sooner, those of a full chip 0.3 us later: beside the other kernels
    // that counts (8 x 128 x 192 at 128: 7.5 against 7.9 us, 7 x 1600 x 128: 7.7 against 7.0)
    if (D == 128 && best == 1) best_us += 0.8 * std::min(1.0, groups / 256.0) - 0.55;
    // (the number of splits is that of workgroups of 64 queries: those of 32 shift it by a step at most, within the model's 6 %)
    if (attn_keys_narrow(batch, M, best)) best_us = attn_keys_narrow_us(batch, M, N, D, best) + (best > 1 ? 2.5 : 0.0);
    return best_us < attn_blocks_us(batch, M, N, D, v_layout) ? best : 0;
}

int fa_dispatch(const __half* Q, const __half* K, const __half* V, __half* O, int batch, int M, int N, int Kd, int P,
                float scale, int v_layout, int algo, hipStream_t stream, float* part = nullptr, int splits = 1) {
    using W41 = tl::RowMajor<4, 1>;
    if (Kd != P) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "attention needs the query and value head sizes equal");
    if (M % 64 != 0 || N % 64 != 0) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "attention needs M % 64 == 0 and N % 64 == 0");
    if (algo != TCU_ATTN_AUTO && algo != TCU_ATTN_TILE_LIBRARY && algo != TCU_ATTN_MFMA32 &&
        algo != TCU_ATTN_MFMA32_FUSED && algo != TCU_ATTN_WAVE64 && algo != TCU_ATTN_TILE_WAVE64 &&
        algo != TCU_ATTN_WAVE64_K32 && algo != TCU_ATTN_KEYS)
        return fail(TCU_ERR_INVALID_ARGUMENT, "unknown attention algo");
    if (v_layout != TCU_V_ROW_MAJOR && v_layout != TCU_V_COL_MAJOR) return fail(TCU_ERR_INVALID_ARGUMENT, "unknown v_layout");
    if (algo == TCU_ATTN_TILE_WAVE64) return fa_tile_w64_dispatch(Q, K, V, O, batch, M, N, Kd, scale, v_layout, stream);
    if (algo == TCU_ATTN_WAVE64_K32) return fa_w64_k32_dispatch(Q, K, V, O, batch, M, N, Kd, scale, v_layout, stream);
    if (algo == TCU_ATTN_KEYS) return fa_keys_dispatch(Q, K, V, O, part, batch, M, N, Kd, splits, scale, v_layout, stream);
    if (algo == TCU_ATTN_WAVE64) {
        if (Kd != 128)
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the one-wavefront-per-SIMD attention kernel is instantiated for head size 128");
        return v_layout == TCU_V_ROW_MAJOR ? launch_fa_w64<false>(Q, K, V, O, batch, M, N, scale, stream)
                                           : launch_fa_w64<true>(Q, K, V, O, batch, M, N, scale, stream);
    }
    if (v_layout == TCU_V_ROW_MAJOR && algo != TCU_ATTN_TILE_LIBRARY) {
        if (Kd != 128 && Kd != 64) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "attention is instantiated for head sizes 64 and 128");
        // Few query blocks: the wavefronts split the keys. Enough to fill the chip: the kernels with 64 queries per wavefront.
        // From one block of 256 queries per CU on the chip runs at its power limit, where
        // the 16x16x32 instruction wins, at every sequence length that kernel takes (256 x 512 x 512 x 128: 45.6 against
        // 57.9 us for the 8-wavefront kernel, 1024 x 320 x 320: 117.7 against 203); a half-empty chip runs at full clock,
        // where the 32x32x16 kernel's fewer issue cycles do (long sequences, head size 128: 16 x 2048^2 45.7 against 48.8
        // us; with 192 blocks the 16x16x32 kernel is ahead again, 52.6 against 55.5).
        if (algo == TCU_ATTN_AUTO && attn_keys_plan(batch, M, N, Kd, v_layout, 1) == 1)
            return fa_keys_dispatch(Q, K, V, O, nullptr, batch, M, N, Kd, 1, scale, v_layout, stream);
        if (algo == TCU_ATTN_AUTO && attn_k32_is_the_choice(batch, M, N, Kd, v_layout))
            return fa_w64_k32_dispatch(Q, K, V, O, batch, M, N, Kd, scale, v_layout, stream);
        if (algo == TCU_ATTN_AUTO && attn_w64_is_the_choice(batch, M, N, Kd))
            return launch_fa_w64<false>(Q, K, V, O, batch, M, N, scale, stream);
        if (algo == TCU_ATTN_MFMA32)
            return Kd == 128 ? fa_fwd_by_rows<128, false>(Q, K, V, O, batch, M, N, scale, stream)
                             : fa_fwd_by_rows<64, false>(Q, K, V, O, batch, M, N, scale, stream);
        return Kd == 128 ? fa_fwd_by_rows<128, true>(Q, K, V, O, batch, M, N, scale, stream)
                         : fa_fwd_by_rows<64, true>(Q, K, V, O, batch, M, N, scale, stream);
    }
    if (algo == TCU_ATTN_MFMA32 || algo == TCU_ATTN_MFMA32_FUSED)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the 32x32x16 attention kernels take a row-major V");
    if (v_layout == TCU_V_ROW_MAJOR) {
        // row-major V: the double-buffered composition (direct-to-LDS ring); 32 query rows per wavefront where M allows
        if (Kd == 128 && M % 128 == 0) return launch_fa_pipelined<0, 128, true, 128, 64, W41>(Q, K, V, O, batch, M, N, scale, stream);
        if (Kd == 128) return launch_fa_pipelined<0, 128, true, 64, 64, W41>(Q, K, V, O, batch, M, N, scale, stream);
        if (Kd == 64) return launch_fa_pipelined<0, 64, true, 64, 64, W41>(Q, K, V, O, batch, M, N, scale, stream);
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "attention is instantiated for head sizes 64 and 128");
    }
    // column-major V (the reference op's convention), any N % 64 == 0
    if (Kd != 128) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "column-major V is instantiated for head size 128");
    if (algo == TCU_ATTN_AUTO) {
        // as for a row-major V
        if (attn_keys_plan(batch, M, N, Kd, v_layout, 1) == 1)
            return fa_keys_dispatch(Q, K, V, O, nullptr, batch, M, N, Kd, 1, scale, v_layout, stream);
        if (attn_k32_is_the_choice(batch, M, N, Kd, v_layout))
            return fa_w64_k32_dispatch(Q, K, V, O, batch, M, N, Kd, scale, v_layout, stream);
        return launch_fa_w64<true>(Q, K, V, O, batch, M, N, scale, stream);
    }
    // the kernel composed from tile primitives has the leading dimension of V (= N) as a compile-time constant, like
    // the reference op: one instantiation per N
    switch (N) {
        case 64: return launch_fa<64, 128, false, 64, 64, W41>(Q, K, V, O, batch, M, N, scale, stream);
        case 128: return launch_fa<128, 128, false, 64, 64, W41>(Q, K, V, O, batch, M, N, scale, stream);
        case 256: return launch_fa<256, 128, false, 64, 64, W41>(Q, K, V, O, batch, M, N, scale, stream);
        case 2048: return launch_fa<2048, 128, false, 64, 64, W41>(Q, K, V, O, batch, M, N, scale, stream);
        default:
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the tile-library attention kernel takes a column-major V for N in {64, 128, "
                                                   "256, 2048}");
    }
}

// ---------------------------------------------------------------------------- LSTM
template <int kI, int kH, int kTM, int kTH, int kTK, typename WarpLayout>
int launch_lstm(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0,
                __half* h_all, float* c_out, int T, int B, hipStream_t stream) {
    using Traits = LstmCellTraits<__half, float, kI, kH, kTM, kTH, kTK, WarpLayout>;
    auto kernel = &lstm_cell<__half, Traits>;
    for (int t = 0; t < T; ++t) {
        const __half* x_t = x + size_t(t) * B * kI;
        const __half* h_in = t == 0 ? h0 : h_all + size_t(t - 1) * B * kH;
        const float* c_in = t == 0 ? c0 : c_out;
        __half* h_out = h_all + size_t(t) * B * kH;
        int rc = launch(kernel, dim3(B / kTM, kH / kTH), dim3(Traits::kThreads), Traits::kShmBytes, stream, x_t, h_in,
                        W, bias, c_in, c_out, h_out);
        if (rc != TCU_OK) return lstm_step_failed(rc, t, T);
    }
    return TCU_OK;
}

/// The step kernel for any B, I, H in multiples of 16 addresses its operands with 32-bit byte offsets.
bool lstm_direct_takes(int B, int I, int H) {
    return B % 16 == 0 && I % 16 == 0 && H % 16 == 0 && 8.0 * H * (double(I) + H) < 4294967296.0 &&
           2.0 * B * std::max(I, H) < 4294967296.0;
}

/// Tile of that kernel (16-row tiles of weights x of the batch) for a step over `columns` columns: rounds of one workgroup per
/// CU, each as long as its rows take to arrive (95 KB per us and CU) plus 0.1 us per 16 x 16 tile for the sums of the eight
/// wavefronts and 0.8 us whatever the tile, without which a short sum got many rounds of small tiles (66 sizes with all seven
/// tiles: on average 0.7 % from the best of them, 3.8 before; 1x1, 2x2, 4x4: 768 x 256 and 256 columns, as with a projection:
/// 14.1, 8.1, 6.0; 384 x 128, 128: 5.8, 4.1, 5.5; 1568 x 176, 400 columns: 16.4, 11.9, 9.2, 4x1 8.5). Measured, us per step with
/// 1x1, 2x1, 2x2, 4x1, 4x2, 4x4 tiles: B 80, I 336, H 656: 6.5, 6.1, 4.5, 4.6, 5.2, 6.9;
/// 16, 1024, 1024: 3.9, 4.4, 4.9, 5.4, 6.1, 7.9; 64, 1024, 1024: 8.8, 8.2, 5.7, 5.8, 6.7, 8.9; 240, 368, 592: 12.1, 12.8,
/// 10.0, 8.5, 9.0, 7.4; 256, 1024, 1024: 28, 28, 18, 18, 14, 9.7.
struct LstmTilePlan {
    int ut, rt;
    double us;
};
LstmTilePlan lstm_direct_plan(int B, int H, int columns) {
    LstmTilePlan plan{1, 1, 1e30};
    for (const auto& [ut, rt] : {std::pair{1, 1}, std::pair{1, 2}, std::pair{2, 1}, std::pair{2, 2}, std::pair{4, 1},
                                 std::pair{4, 2}, std::pair{4, 4}}) {
        const long groups = (long)((H + 4 * ut - 1) / (4 * ut)) * ((B + 16 * rt - 1) / (16 * rt));
        const double us = double((groups + 255) / 256) * (0.8 + 0.1 * ut * rt + 32.0 * (ut + rt) * columns / 95e3);
        if (us < plan.us) plan = {ut, rt, us};
    }
    return plan;
}

template <int kUT, int kRT, bool kHoisted>
int launch_lstm_direct_tiles(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0,
                             __half* h_all, float* c_out, int T, int B, int I, int H, const float* pre, hipStream_t stream) {
    using Traits = LstmDirectTraits<kUT, kRT>;
    const long grid = (long)((H + Traits::kUnits - 1) / Traits::kUnits) * ((B + Traits::kRows - 1) / Traits::kRows);
    if (grid > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16: too many tiles for one launch");
    for (int t = 0; t < T; ++t) {
        const __half* h_in = t == 0 ? h0 : h_all + size_t(t - 1) * B * H;
        const float* c_in = t == 0 ? c0 : c_out;
        int rc = launch(&lstm_cell_direct<Traits, kHoisted>, dim3(unsigned(grid)), dim3(Traits::kThreads), Traits::kLdsBytes,
                        stream, x + size_t(t) * B * I, h_in, W, bias, c_in, c_out, h_all + size_t(t) * B * H, B,
                        pre ? pre + size_t(t) * B * 4 * H : nullptr, I, H);
        if (rc != TCU_OK) return lstm_step_failed(rc, t, T);
    }
    return TCU_OK;
}

template <bool kHoisted>
int launch_lstm_direct(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0, __half* h_all,
                       float* c_out, int T, int B, int I, int H, const float* pre, hipStream_t stream) {
    const LstmTilePlan plan = lstm_direct_plan(B, H, kHoisted ? H : I + H);
    auto go = [&](auto ut, auto rt) {
        return launch_lstm_direct_tiles<decltype(ut)::value, decltype(rt)::value, kHoisted>(x, W, bias, h0, c0, h_all, c_out, T,
                                                                                           B, I, H, pre, stream);
    };
    using one = std::integral_constant<int, 1>;
    using two = std::integral_constant<int, 2>;
    using four = std::integral_constant<int, 4>;
    if (plan.ut == 1) return plan.rt == 1 ? go(one{}, one{}) : go(one{}, two{});
    if (plan.ut == 2) return plan.rt == 1 ? go(two{}, one{}) : go(two{}, two{});
    return plan.rt == 1 ? go(four{}, one{}) : plan.rt == 2 ? go(four{}, two{}) : go(four{}, four{});
}

/// The GEMM that computes the input half of the gates of all steps (rows = T * B): with few rows the 128 x 128 tiles of the
/// K-splitting kernel (1024 rows, I and H 1024: 13 against 22 us), else the 256 x 256 ones (tiles128 = 0).
struct LstmProjectionPlan {
    long tiles128;
    double us;
};
LstmProjectionPlan lstm_projection_plan(long rows, int I, int H) {
    const long tiles128 = ((rows + 127) / 128) * ((4l * H + 127) / 128), tiles256 = ((rows + 255) / 256) * ((4l * H + 255) / 256);
    const double us128 = double((tiles128 + 255) / 256) * (5.0 + 0.95 * (I / 128)), us256 = gemm_w128_us(tiles256, I);
    if (us128 < us256 && (long)(I + H) * 256 < (1l << 32)) return {tiles128, us128};
    return {0, us256};
}

/// Expected time of one launch of the step kernel. Beyond the rounds of lstm_direct_plan() it counts the operands that the
/// 32 workgroups of an XCD bring into its L2 (0.7 us per MB and round): many rows of a large batch pass once per round.
double lstm_step_us(int B, int H, int columns) {
    const LstmTilePlan plan = lstm_direct_plan(B, H, columns);
    const long row_blocks = (B + 16 * plan.rt - 1) / (16 * plan.rt), unit_blocks = (H + 4 * plan.ut - 1) / (4 * plan.ut);
    const double mb = 32e-6 * columns * (std::min(32l, row_blocks) * plan.rt + (32 + row_blocks - 1) / row_blocks * plan.ut);
    return 2.2 + double((row_blocks * unit_blocks + 255) / 256) * (0.12 * plan.ut * plan.rt + 2.2e-4 * (plan.ut + plan.rt) * columns + 0.7 * mb);
}

/// Whether AUTO computes the input half of the gates of all steps beforehand where the caller has a workspace for it: the
/// projection runs at the rate of a GEMM (0.83 of its expected time and 3.5 us, with the pre-activations written and read
/// 0.37 us per MB), and a step is left with H of its I + H columns. Both plans within 12 % of the measured times of most of
/// 133 sizes; us, a fused kernel per step against this: T 8, B 64, I 8192, H 4096: 710, 364; 2048, 4096, 256: 378, 198; 1024, 4096,
/// 512: 286, 197; T 16, B 256, I 4096, H 1024: 317, 237; 256, 2048, 1024: 210, 183; 256, 1024, 1024: 151, 157; T 8, B 512, I
/// 512, H 1024: 118, 138. Of 115 more sizes the chosen plan is within 3 % of the shorter for 108, at most 14 % above it
/// (T 4, B 1472, I 1280, H 128: 41, 36).
bool lstm_projection_pays(int T, int B, int I, int H) {
    if (I < 512 || T < 4 || tcu_lstm_workspace_bytes(T, B, I, H) == 0 || (long)T * B > INT_MAX) return false;
    if (!lstm_direct_takes(B, I, H)) return true;  // (the streaming step kernel: half of its bytes are W[:, :I])
    const double projection = 3.5 + 0.83 * lstm_projection_plan((long)T * B, I, H).us + 0.37 * 16e-6 * T * double(B) * H;
    return 1.02 * (projection + T * lstm_step_us(B, H, H)) < T * lstm_step_us(B, H, I + H);
}

int launch_lstm_hoisted(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0, __half* h_all,
                        float* c_out, int T, int B, int I, int H, float* pre, hipStream_t stream) {
    // pre[T * B, 4H] = x[T * B, I] . W[:, :I]^T: the stored [4H, I] operand is the first I columns of W's rows
    const long rows = long(T) * B;
    if (rows > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16_ws: T * B exceeds the 32-bit row count");
    const LstmProjectionPlan plan = lstm_projection_plan(rows, I, H);
    int rc;
    if (plan.tiles128 > 0) {
        using Tk = GemmW128kTraits;
        auto kernel = rows % Tk::kBM == 0 ? &gemm_w128k<float, false, Tk> : &gemm_w128k<float, true, Tk>;
        rc = launch(kernel, dim3(unsigned(plan.tiles128)), dim3(Tk::kThreads), Tk::kLdsBytes, stream, x, W, pre, int(rows), 4 * H, I, I,
                    I + H, 4 * H, static_cast<unsigned int*>(nullptr), 0);
    } else {
        rc = gemm_w128_dispatch<float>(x, W, pre, int(rows), 4 * H, I, stream, I, I + H);
    }
    if (rc != TCU_OK) return rc;
    if (lstm_direct_takes(B, I, H)) return launch_lstm_direct<true>(x, W, bias, h0, c0, h_all, c_out, T, B, I, H, pre, stream);
    using Traits = LstmFwdTraits<>;
    auto kernel = &lstm_cell_fwd<Traits, true>;
    const int grid = (B / Traits::kTM) * (H / Traits::kTH);
    for (int t = 0; t < T; ++t) {
        const __half* x_t = x + size_t(t) * B * I;
        const __half* h_in = t == 0 ? h0 : h_all + size_t(t - 1) * B * H;
        const float* c_in = t == 0 ? c0 : c_out;
        __half* h_out = h_all + size_t(t) * B * H;
        const float* pre_t = pre + size_t(t) * B * 4 * H;
        rc = launch(kernel, dim3(grid), dim3(Traits::kThreads), Traits::kLdsBytes, stream, x_t, h_in, W, bias, c_in,
                    c_out, h_out, B, pre_t, I, H);
        if (rc != TCU_OK) return lstm_step_failed(rc, t, T);
    }
    return TCU_OK;
}

int launch_lstm_ragged(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0,
                       __half* h_all, float* c_out, int T, int B, int I, int H, hipStream_t stream) {
    using Traits = RaggedLstmTraits;
    const dim3 grid((H + Traits::kUnits - 1) / Traits::kUnits, B / Traits::kRows);
    for (int t = 0; t < T; ++t) {
        const __half* x_t = x + size_t(t) * B * I;
        const __half* h_in = t == 0 ? h0 : h_all + size_t(t - 1) * B * H;
        const float* c_in = t == 0 ? c0 : c_out;
        __half* h_out = h_all + size_t(t) * B * H;
        int rc = launch(&lstm_cell_ragged, grid, dim3(Traits::kThreads), 0, stream, x_t, h_in, W, bias, c_in, c_out, h_out,
                        B, I, H);
        if (rc != TCU_OK) return lstm_step_failed(rc, t, T);
    }
    return TCU_OK;
}

int launch_lstm_fwd(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0, __half* h_all,
                    float* c_out, int T, int B, int I, int H, hipStream_t stream) {
    using Traits = LstmFwdTraits<>;
    auto kernel = &lstm_cell_fwd<Traits>;
    const int grid = (B / Traits::kTM) * (H / Traits::kTH);
    for (int t = 0; t < T; ++t) {
        const __half* x_t = x + size_t(t) * B * I;
        const __half* h_in = t == 0 ? h0 : h_all + size_t(t - 1) * B * H;
        const float* c_in = t == 0 ? c0 : c_out;
        __half* h_out = h_all + size_t(t) * B * H;
        int rc = launch(kernel, dim3(grid), dim3(Traits::kThreads), Traits::kLdsBytes, stream, x_t, h_in, W, bias, c_in,
                        c_out, h_out, B, static_cast<const float*>(nullptr), I, H);
        if (rc != TCU_OK) return lstm_step_failed(rc, t, T);
    }
    return TCU_OK;
}

/// The shapes that lstm_layer_xcd takes: T >= 2 (its workgroups count on a second step), H within the registers of an XCD, at most
/// kMaxGroups groups of rows, and the 32-bit offsets of its operands and of the projection's.
int lstm_layer_row_tiles(int B) { return B <= 128 ? 1 : 2; }
bool lstm_layer_takes(int T, int B, int I, int H) {
    if (T < 2 || H > 1024 || (long)T * B > INT_MAX || !lstm_direct_takes(B, I, H)) return false;
    const int rows = 16 * lstm_layer_row_tiles(B);
    return (B + rows - 1) / rows <= LstmLayerTraits<1, 4, 1>::kMaxGroups && (long)(I + H) * 512 < (1l << 32);
}

/// pre[T * B, 4H] = x . W[:, :I]^T in f32 with the kernel that is expected to take least, `sync` cleared on the side.
struct LstmLayerProjection {
    int kernel;  // 0: gemm_direct, 1: gemm_w128k, 2: gemm_w128, 3: gemm_pipelined
    double us;
};
LstmLayerProjection lstm_layer_projection(long rows, int I, int H) {
    const double mb = 16e-6 * double(rows) * H;  // of pre-activations: f32 outputs cost these kernels 0.15 to 0.6 us per MB
    LstmLayerProjection plan{0, gemm_direct_plan(int(rows), 4 * H, I).us + 0.6 * mb};
    const long tiles128 = ((rows + 127) / 128) * ((4l * H + 127) / 128), tiles256 = ((rows + 255) / 256) * ((4l * H + 255) / 256);
    const double us128 = double((tiles128 + 255) / 256) * (5.0 + 0.95 * ((I + 127) / 128)) + 0.3 * mb;
    const double us256 = gemm_w128_us(tiles256, (I + 63) / 64 * 64) + 0.15 * mb, us_pipe = pipelined_plan(int(rows), 4 * H, I).us + 0.4 * mb;
    if (us128 < plan.us) plan = {1, us128};
    if (us256 < plan.us) plan = {2, us256};
    if (us_pipe < plan.us) plan = {3, us_pipe};
    return plan;
}

/// Launches that the layer's steps are divided into, each with its projection before it, so that the pre-activations of one take at
/// most 256 MiB whatever T is (eight times h_all otherwise: 17 GB at T 4096, B 256, H 1024). Every part has 4 steps or more. A part
/// costs what the layer takes before its first step once more, and its pre-activations come from nearer: us, whole -> in parts, T 1024 and
/// B 256, I 1024, H 1024 (16 parts): 6120 -> 6280; 128, 512, 1024 (8): 3220 -> 3200; 80, 336, 656 (4): 2300 -> 2180; 256, 256, 256 (4): 1990 -> 1850.
constexpr unsigned long long kLstmLayerPreBytes = 256ull << 20;
int lstm_layer_parts(int T, int B, int H) {
    const long steps = long(kLstmLayerPreBytes / (16ull * B * H));  // 8 and more: B <= 2048, H <= 1024
    return int((T + steps - 1) / steps);
}

int lstm_layer_rounds(int B) {  // of 8 groups of rows, one per XCD
    const int rows = 16 * lstm_layer_row_tiles(B);
    return ((B + rows - 1) / rows + 7) / 8;
}

/// Expected time of the layer kernel's steps, for every round of 8 groups of rows (measured over 90 sizes, us per step with 16 and 32
/// rows: H 128 0.73, 1.1; 256 0.95, 1.45; 512 1.2, 1.9; 768 1.75, 2.9; 1024 2.05, 3.9).
double lstm_layer_steps_us(int T, int B, int H) {
    static constexpr double kStepUs[5][2] = {{0.73, 1.1}, {0.95, 1.45}, {1.2, 1.9}, {1.75, 2.9}, {2.05, 3.9}};
    const int size = H <= 128 ? 0 : H <= 256 ? 1 : H <= 512 ? 2 : H <= 768 ? 3 : 4;
    return double(lstm_layer_rounds(B)) * T * kStepUs[size][lstm_layer_row_tiles(B) - 1];
}

/// Whether AUTO runs the layer that way: the projection, 1.5 us to the next launch, what the kernel takes before its first step (the
/// weights arrive at 0.9 MB per us and XCD) and its steps against a launch per step. The first sum is the least that was measured;
/// where the two plans are close the second counts (fitted to 500 sizes, T 4 to 32, up to 480 rows, within 7 %): the start of many
/// units, another round's claims. By it 3 of 600 other sizes take longer than a launch per step, at most 8 %; by the first alone 20 of 320, up to 15 %
/// (us, steps, layer: 14 x 480 x 288 x 288: 79, 86; 5 x 368 x 144 x 768: 57, 65). Longer layers gain as much as 32 steps or more: T 1024, B 80,
/// I 336, H 656: 4656, 2311. us, steps
/// -> this: T 16, B 256, I 1024, H 1024: 149 -> 106; 24, 80, 336, 656: 109 -> 75; 20, 16, 416, 80: 60 -> 24; 8, 96, 176, 160: 25 -> 18; not taken: 8,
/// 80, 384, 576: 34, 38; 5, 352, 144, 864: 62, 73; 31, 368, 96, 160: 111, 114. Long inputs stay with lstm_projection_pays().
bool lstm_layer_pays(int T, int B, int I, int H) {
    if (T < 4 || !lstm_layer_takes(T, B, I, H) || lstm_projection_pays(T, B, I, H)) return false;
    const int parts = lstm_layer_parts(T, B, H);
    const double projection = parts * lstm_layer_projection((long)((T + parts - 1) / parts) * B, I, H).us, steps = lstm_layer_steps_us(T, B, H);
    const double fill = (H / 1024.0) * (H / 1024.0);  // of an XCD's registers
    const double layer = std::max(projection + parts * (7.5 + 9.0 * fill) + steps,
                                  1.15 * projection + parts * (5.0 + 16.0 * fill) + 4.0 * (lstm_layer_rounds(B) - 1) + 1.06 * steps);
    return 1.05 * layer < T * lstm_step_us(B, H, I + H);
}

/// What a launch of lstm_layer_xcd may use; other values than these are for tests (tcu_lstm_f16_layer_limited).
struct LstmLayerLimits {
    int workgroups = INT_MAX;
    int takeover_us = -1;  // lstm_layer_takeover_us()
    int max_tries = 1 << 24;  // of 0.5 us and more each
};

/// How long a workgroup waits for the others to start before it takes over the slice of one that has not: twice the time of all steps.
/// The layer's CUs are mostly held by something as short as itself, and a workgroup with two slices fetches the weights of both again
/// in every step, for the rest of the launch. Two layers on two streams, us for both, by the wait (30 us, 200 us; a launch per
/// step): T 24, B 80, I 336, H 656: 149-355, 118; 165; T 64: 757, 263; 397; T 64, B 128, I 512, H 784: 1067, 357; 523.
int lstm_layer_takeover_us(int T, int B, int H) { return int(30.0 + std::min(1e6, 2.0 * lstm_layer_steps_us(T, B, H))); }

template <int kTW, int kKS, int kRT>
int launch_lstm_layer_xcd(const float* pre, const __half* W, const __half* bias, const __half* h0, const float* c0, __half* h_all,
                          float* c_out, int T, int B, int I, int H, unsigned int* sync, const LstmLayerLimits& limits, hipStream_t s) {
    using Traits = LstmLayerTraits<kTW, kKS, kRT>;
    const int peers = (H + Traits::kUnits - 1) / Traits::kUnits;
    const int grid = std::min(limits.workgroups, 8 * peers);
    return launch(&lstm_layer_xcd<Traits>, dim3(unsigned(grid)), dim3(Traits::kThreads), Traits::kLdsBytes, s, pre, W, I + H, I, bias, h0,
                  c0, h_all, c_out, T, B, H, sync,
                  100 * (limits.takeover_us < 0 ? lstm_layer_takeover_us(T, B, H) : limits.takeover_us), limits.max_tries);
}

int launch_lstm_layer_part(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0, __half* h_all,
                           float* c_out, int T, int B, int I, int H, unsigned char* workspace, const LstmLayerLimits& limits,
                           hipStream_t s) {
    auto sync = reinterpret_cast<unsigned int*>(workspace);
    auto pre = reinterpret_cast<float*>(workspace + kPersistentSyncBytes);
    constexpr int kSyncWords = LstmLayerTraits<1, 4, 1>::kSyncWords;
    static_assert(kSyncWords * sizeof(unsigned int) <= kPersistentSyncBytes);
    const int rows = T * B;
    int rc;
    switch (lstm_layer_projection(rows, I, H).kernel) {
        case 0: rc = gemm_direct_dispatch<float>(x, W, pre, rows, 4 * H, I, s, I + H, sync, kSyncWords); break;
        case 1: {
            using Tk = GemmW128kTraits;
            const long tiles = ((rows + 127l) / 128) * ((4l * H + 127) / 128);
            auto kernel = I % Tk::kBK != 0 ? &gemm_w128k<float, true, Tk, true, true> : rows % Tk::kBM == 0 && 4 * H % Tk::kBN == 0
                          ? &gemm_w128k<float, false, Tk, false, true> : &gemm_w128k<float, true, Tk, false, true>;
            rc = launch(kernel, dim3(unsigned(tiles)), dim3(Tk::kThreads), Tk::kLdsBytes, s, x, W, pre, rows, 4 * H, I, I, I + H, 4 * H, sync,
                        kSyncWords);
            break;
        }
        case 2: rc = gemm_w128_dispatch<float>(x, W, pre, rows, 4 * H, I, s, I, I + H, 4 * H, sync, kSyncWords); break;
        default: rc = gemm_pipelined_dispatch<float>(x, W, pre, rows, 4 * H, I, s, 4 * H, I + H, sync, kSyncWords);
    }
    if (rc != TCU_OK) return rc;
    auto go = [&](auto tw, auto ks) {
        constexpr int kTW = decltype(tw)::value, kKS = decltype(ks)::value;
        if (lstm_layer_row_tiles(B) == 1)
            return launch_lstm_layer_xcd<kTW, kKS, 1>(pre, W, bias, h0, c0, h_all, c_out, T, B, I, H, sync, limits, s);
        return launch_lstm_layer_xcd<kTW, kKS, 2>(pre, W, bias, h0, c0, h_all, c_out, T, B, I, H, sync, limits, s);
    };
    using one = std::integral_constant<int, 1>;
    using two = std::integral_constant<int, 2>;
    if (H <= 128) return go(one{}, std::integral_constant<int, 4>{});
    if (H <= 256) return go(one{}, std::integral_constant<int, 8>{});
    if (H <= 512) return go(one{}, std::integral_constant<int, 16>{});
    if (H <= 768) return go(two{}, std::integral_constant<int, 24>{});
    return go(two{}, std::integral_constant<int, 32>{});
}

/// ... in lstm_layer_parts() parts: the states that one ends with are those that the next begins with.
int launch_lstm_layer(const __half* x, const __half* W, const __half* bias, const __half* h0, const float* c0, __half* h_all,
                      float* c_out, int T, int B, int I, int H, unsigned char* workspace, const LstmLayerLimits& limits, hipStream_t s) {
    const int parts = lstm_layer_parts(T, B, H);
    for (int part = 0, t = 0; part < parts; ++part) {
        const int end = int((long)T * (part + 1) / parts);
        const int rc = launch_lstm_layer_part(x + size_t(t) * B * I, W, bias, t == 0 ? h0 : h_all + size_t(t - 1) * B * H, t == 0 ? c0 : c_out,
                                              h_all + size_t(t) * B * H, c_out, end - t, B, I, H, workspace, limits, s);
        if (rc != TCU_OK) return lstm_step_failed(rc, t, T);
        t = end;
    }
    return TCU_OK;
}

/// The weight-stationary recurrence for hidden size kH: 8 * kH / 32 workgroups, kH / 32 per XCD.
template <int kH>
int launch_lstm_recurrent_xcd(const __half* pre, const __half* W, const void* bias, const void* h0, const void* c0, void* h_all,
                              void* c_out, int T, int B, int I, unsigned int* sync, unsigned long long spin_us,
                              long peers_override, hipStream_t s) {
    using Traits = LstmRecurrentTraits<kH>;
    const unsigned int peers = peers_override >= 0 ? unsigned(peers_override) : unsigned(Traits::kCusPerXcd);
    return launch(&lstm_recurrent_xcd<Traits, __half>, dim3(Traits::kGrid), dim3(Traits::kThreads), Traits::kLdsBytes, s, pre,
                  W, I + kH, I, static_cast<const __half*>(bias), static_cast<const __half*>(h0),
                  static_cast<const float*>(c0), static_cast<__half*>(h_all), static_cast<float*>(c_out), T, B, sync,
                  spin_us * 100ull, peers);
}

/// tcu_lstm_f16_layer within `limits`.
int lstm_f16_layer(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all, void* c_out, int T, int B,
                   int I, int H, void* workspace, unsigned long long workspace_bytes, const LstmLayerLimits& limits, void* stream) {
    if (!x || !W || !bias || !h_all || !c_out || !workspace) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_layer: null pointer");
    if (!positive({T, B, I, H})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_layer: sizes must be positive");
    if (!aligned16({x, W, bias, h0, c0, h_all, c_out, workspace}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_layer: operands must be 16-byte aligned");
    const unsigned long long need = tcu_lstm_layer_workspace_bytes(T, B, I, H);
    if (need == 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16_layer: needs T >= 2, B, I and H in multiples of 16, H <= 1024 and B <= 2048");
    if (workspace_bytes < need)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_layer: workspace smaller than tcu_lstm_layer_workspace_bytes()");
    // the kernel marks all of h_all before its first step, and the projection reads all of x before any step is written: a state
    // inside h_all (the last step of an earlier call that wrote the same tensor) or inputs that are its steps (each the output before
    // it) go to the kernels that read and write a step at a time
    auto inside = [&](const void* p, size_t bytes) {
        const auto first = reinterpret_cast<uintptr_t>(p), all_first = reinterpret_cast<uintptr_t>(h_all);
        return p && first < all_first + size_t(T) * B * H * 2 && all_first < first + bytes;
    };
    if (inside(h0, size_t(B) * H * 2) || inside(c0, size_t(B) * H * 4) || inside(x, size_t(T) * B * I * 2))
        return tcu_lstm_f16_algo(x, W, bias, h0, c0, h_all, c_out, T, B, I, H, TCU_LSTM_AUTO, stream);
    return launch_lstm_layer(static_cast<const __half*>(x), static_cast<const __half*>(W), static_cast<const __half*>(bias),
                             static_cast<const __half*>(h0), static_cast<const float*>(c0), static_cast<__half*>(h_all),
                             static_cast<float*>(c_out), T, B, I, H, static_cast<unsigned char*>(workspace), limits,
                             static_cast<hipStream_t>(stream));
}
}  // namespace

extern "C" {

int tcu_version(void) { return 100; }

const char* tcu_recent_kernel(int back) {
    if (back < 0 || unsigned(back) >= kRecentKernels || unsigned(back) >= g_launches) return "";
    const char* name = hipKernelNameRefByPtr(g_recent_kernels[(g_launches - 1 - back) % kRecentKernels], nullptr);
    return name ? name : "";
}

const char* tcu_last_error(void) { return g_last_error.c_str(); }

int tcu_device_count(void) {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess) return fail(TCU_ERR_NO_DEVICE, std::string("hipGetDeviceCount: ") + hipGetErrorString(e));
    return n;
}

int tcu_gemm_f16(const void* A, const void* B, void* C, int M, int N, int K, int out_dtype, int algo, void* stream) {
    if (!A || !B || !C) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16: null pointer");
    if (!positive({M, N, K})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16: sizes must be positive");
    if (!aligned16({A, B, C})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16: operands must be 16-byte aligned");
    auto s = static_cast<hipStream_t>(stream);
    auto a = static_cast<const __half*>(A), b = static_cast<const __half*>(B);
    if (out_dtype == TCU_DTYPE_F32) return gemm_dispatch<float>(a, b, static_cast<float*>(C), M, N, K, algo, s);
    if (out_dtype == TCU_DTYPE_F16) {
        if (algo == TCU_GEMM_GLOBAL_REG || algo == TCU_GEMM_ALL_MEM)
            return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the reference-style GEMM kernels write f32 (their accumulator type)");
        return gemm_dispatch<__half>(a, b, static_cast<__half*>(C), M, N, K, algo, s);
    }
    return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16: out_dtype must be TCU_DTYPE_F32 or TCU_DTYPE_F16");
}

unsigned long long tcu_gemm_workspace_bytes(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const int splits = gemm_split_count(M, N, K);
    return splits > 1 ? (unsigned long long)splits * M * N * sizeof(float) : 0;
}

int tcu_gemm_uses_workspace(int M, int N, int K) {
    return M > 0 && N > 0 && K > 0 && gemm_split_is_the_choice(M, N, K) ? 1 : 0;
}

int tcu_gemm_f16_ws(const void* A, const void* B, void* C, int M, int N, int K, int out_dtype, void* workspace,
                    unsigned long long workspace_bytes, void* stream) {
    const unsigned long long need = (M > 0 && N > 0 && K > 0) ? tcu_gemm_workspace_bytes(M, N, K) : 0;
    if (need == 0 || !workspace) return tcu_gemm_f16(A, B, C, M, N, K, out_dtype, TCU_GEMM_AUTO, stream);
    if (!A || !B || !C) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16_ws: null pointer");
    if (!aligned16({A, B, C, workspace})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16_ws: operands must be 16-byte aligned");
    if (workspace_bytes < need)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16_ws: workspace smaller than tcu_gemm_workspace_bytes()");
    if (!gemm_split_is_the_choice(M, N, K)) return tcu_gemm_f16(A, B, C, M, N, K, out_dtype, TCU_GEMM_AUTO, stream);
    auto a = static_cast<const __half*>(A), b = static_cast<const __half*>(B);
    auto s = static_cast<hipStream_t>(stream);
    auto ws = static_cast<float*>(workspace);
    const GemmSplitPlan plan = gemm_split_plan(M, N, K);
    if (out_dtype == TCU_DTYPE_F32) return gemm_splitk<float>(a, b, static_cast<float*>(C), M, N, K, plan, ws, s);
    if (out_dtype == TCU_DTYPE_F16) return gemm_splitk<__half>(a, b, static_cast<__half*>(C), M, N, K, plan, ws, s);
    return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_gemm_f16_ws: out_dtype must be TCU_DTYPE_F32 or TCU_DTYPE_F16");
}

int tcu_b2b_gemm_f16(const void* A, const void* B, const void* C, void* D, int M, int N, int K, int P, int batch,
                     int out_dtype, void* stream) {
    return tcu_b2b_gemm_f16_algo(A, B, C, D, M, N, K, P, batch, out_dtype, TCU_B2B_AUTO, stream);
}

int tcu_b2b_gemm_f16_algo(const void* A, const void* B, const void* C, void* D, int M, int N, int K, int P, int batch,
                          int out_dtype, int algo, void* stream) {
    if (!A || !B || !C || !D) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_b2b_gemm_f16: null pointer");
    if (!positive({M, N, K, P, batch}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_b2b_gemm_f16: sizes must be positive");
    if (!aligned16({A, B, C, D}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_b2b_gemm_f16: operands must be 16-byte aligned");
    auto s = static_cast<hipStream_t>(stream);
    auto a = static_cast<const __half*>(A), b = static_cast<const __half*>(B), c = static_cast<const __half*>(C);
    if (out_dtype == TCU_DTYPE_F32) return b2b_dispatch<float>(a, b, c, static_cast<float*>(D), M, N, K, P, batch, algo, s);
    if (out_dtype == TCU_DTYPE_F16) return b2b_dispatch<__half>(a, b, c, static_cast<__half*>(D), M, N, K, P, batch, algo, s);
    return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_b2b_gemm_f16: out_dtype must be TCU_DTYPE_F32 or TCU_DTYPE_F16");
}

int tcu_flash_attn_fwd_f16_algo(const void* Q, const void* K, const void* V, void* O, int batch, int M, int N,
                                int Kdim, int P, float scale, int v_layout, int algo, void* stream) {
    if (!Q || !K || !V || !O) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_flash_attn_fwd_f16: null pointer");
    if (!positive({batch, M, N, Kdim, P}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_flash_attn_fwd_f16: sizes must be positive");
    if (!aligned16({Q, K, V, O}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_flash_attn_fwd_f16: operands must be 16-byte aligned");
    return fa_dispatch(static_cast<const __half*>(Q), static_cast<const __half*>(K), static_cast<const __half*>(V),
                       static_cast<__half*>(O), batch, M, N, Kdim, P, scale, v_layout, algo,
                       static_cast<hipStream_t>(stream));
}

int tcu_flash_attn_fwd_f16(const void* Q, const void* K, const void* V, void* O, int batch, int M, int N, int Kdim,
                           int P, float scale, int v_layout, void* stream) {
    return tcu_flash_attn_fwd_f16_algo(Q, K, V, O, batch, M, N, Kdim, P, scale, v_layout, TCU_ATTN_AUTO, stream);
}

unsigned long long tcu_flash_attn_workspace_bytes(int batch, int M, int N, int Kdim, int P, int v_layout) {
    if (!positive({batch, M, N, Kdim, P}) || Kdim != P || M % 64 != 0 || N % 64 != 0) return 0;
    if (v_layout != TCU_V_ROW_MAJOR && v_layout != TCU_V_COL_MAJOR) return 0;
    if (N <= 512) return 0;  // (never split: not worth a plan)
    const int splits = attn_keys_plan(batch, M, N, Kdim, v_layout, 16);
    return splits > 1 ? (unsigned long long)splits * batch * M * (Kdim + 2) * sizeof(float) : 0;
}

int tcu_flash_attn_fwd_f16_ws(const void* Q, const void* K, const void* V, void* O, int batch, int M, int N, int Kdim, int P,
                              float scale, int v_layout, void* workspace, unsigned long long workspace_bytes, void* stream) {
    const unsigned long long need = tcu_flash_attn_workspace_bytes(batch, M, N, Kdim, P, v_layout);
    if (need == 0 || !workspace)
        return tcu_flash_attn_fwd_f16_algo(Q, K, V, O, batch, M, N, Kdim, P, scale, v_layout, TCU_ATTN_AUTO, stream);
    if (!Q || !K || !V || !O) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_flash_attn_fwd_f16_ws: null pointer");
    if (!aligned16({Q, K, V, O, workspace}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_flash_attn_fwd_f16_ws: operands must be 16-byte aligned");
    if (workspace_bytes < need)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_flash_attn_fwd_f16_ws: workspace smaller than tcu_flash_attn_workspace_bytes()");
    return fa_dispatch(static_cast<const __half*>(Q), static_cast<const __half*>(K), static_cast<const __half*>(V),
                       static_cast<__half*>(O), batch, M, N, Kdim, P, scale, v_layout, TCU_ATTN_KEYS,
                       static_cast<hipStream_t>(stream), static_cast<float*>(workspace),
                       attn_keys_plan(batch, M, N, Kdim, v_layout, 16));
}

int tcu_lstm_f16(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                 void* c_out, int T, int B, int I, int H, void* stream) {
    return tcu_lstm_f16_algo(x, W, bias, h0, c0, h_all, c_out, T, B, I, H, TCU_LSTM_AUTO, stream);
}

int tcu_lstm_f16_algo(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                      void* c_out, int T, int B, int I, int H, int algo, void* stream) {
    if (!x || !W || !bias || !h_all || !c_out) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16: null pointer");
    if (!positive({T, B, I, H})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16: sizes must be positive");
    if (!aligned16({x, W, bias, h0, c0, h_all, c_out}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16: operands must be 16-byte aligned");
    auto s = static_cast<hipStream_t>(stream);
    auto xp = static_cast<const __half*>(x), wp = static_cast<const __half*>(W), bp = static_cast<const __half*>(bias);
    auto h0p = static_cast<const __half*>(h0);
    auto c0p = static_cast<const float*>(c0);
    auto hp = static_cast<__half*>(h_all);
    auto cp = static_cast<float*>(c_out);
    if (long(T) * B > INT_MAX) return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16: T * B exceeds the 32-bit row count");
    if (algo != TCU_LSTM_AUTO && algo != TCU_LSTM_TILE_LIBRARY && algo != TCU_LSTM_STREAMING && algo != TCU_LSTM_RAGGED)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16: unknown algo");
    if (B % 16 != 0 || I % 16 != 0 || H % 16 != 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16: shapes are whole 16 x 16 tiles: B, I and H must be multiples of 16");
    if (algo == TCU_LSTM_RAGGED) return launch_lstm_ragged(xp, wp, bp, h0p, c0p, hp, cp, T, B, I, H, s);
    // every shape whose operands 32-bit offsets reach (gigabytes of weights do not fit): per step 4.5 us against 16.6 for the
    // kernel below it at B 80, I 336, H 656, 9.7 against 12.0 for the streaming one at 256, 1024, 1024
    if (algo == TCU_LSTM_AUTO && lstm_direct_takes(B, I, H))
        return launch_lstm_direct<false>(xp, wp, bp, h0p, c0p, hp, cp, T, B, I, H, nullptr, s);
    const bool b64 = B % 64 == 0;
    if (algo != TCU_LSTM_TILE_LIBRARY && b64 && I % 128 == 0 && H % 128 == 0)
        return launch_lstm_fwd(xp, wp, bp, h0p, c0p, hp, cp, T, B, I, H, s);
    if (algo == TCU_LSTM_STREAMING)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "the streaming LSTM kernel needs I % 128 == 0, H % 128 == 0 and B % 64 == 0");
    if (b64) {
        if (I == 1024 && H == 1024)
            return launch_lstm<1024, 1024, 64, 16, 64, tl::RowMajor<4, 1>>(xp, wp, bp, h0p, c0p, hp, cp, T, B, s);
        if (I == 128 && H == 128)
            return launch_lstm<128, 128, 64, 16, 64, tl::RowMajor<4, 1>>(xp, wp, bp, h0p, c0p, hp, cp, T, B, s);
        if (I == 64 && H == 128)
            return launch_lstm<64, 128, 64, 16, 64, tl::RowMajor<4, 1>>(xp, wp, bp, h0p, c0p, hp, cp, T, B, s);
    }
    if (algo == TCU_LSTM_TILE_LIBRARY)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE,
                    "the tile-library LSTM kernel is instantiated for (I, H) in {(1024,1024), (128,128), (64,128)}, B % 64 == 0");
    // every other shape made of whole 16 x 16 tiles: the run-time-shape kernel
    return launch_lstm_ragged(xp, wp, bp, h0p, c0p, hp, cp, T, B, I, H, s);
}

unsigned long long tcu_lstm_workspace_bytes(int T, int B, int I, int H) {
    const bool shape_ok = I > 0 && H > 0 && I % 128 == 0 && H % 128 == 0 && (long)(I + H) * 512 < (1l << 32);
    if (!shape_ok || T <= 0 || B <= 0 || B % 64 != 0 || ((long)T * B) % 256 != 0) return 0;
    return (unsigned long long)T * B * 4 * H * sizeof(float);
}

int tcu_lstm_uses_workspace(int T, int B, int I, int H) { return lstm_projection_pays(T, B, I, H) ? 1 : 0; }

int tcu_lstm_f16_ws(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                    void* c_out, int T, int B, int I, int H, void* workspace, unsigned long long workspace_bytes,
                    void* stream) {
    if (!x || !W || !bias || !h_all || !c_out || !workspace)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_ws: null pointer");
    if (!positive({T, B, I, H})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_ws: sizes must be positive");
    if (!aligned16({x, W, bias, h0, c0, h_all, c_out, workspace}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_ws: operands must be 16-byte aligned");
    const unsigned long long need = tcu_lstm_workspace_bytes(T, B, I, H);
    if (need == 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16_ws: needs I % 128 == 0, H % 128 == 0, B % 64 == 0 and "
                                               "T * B % 256 == 0");
    if (workspace_bytes < need)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_ws: workspace smaller than tcu_lstm_workspace_bytes()");
    auto s = static_cast<hipStream_t>(stream);
    auto xp = static_cast<const __half*>(x), wp = static_cast<const __half*>(W), bp = static_cast<const __half*>(bias);
    auto h0p = static_cast<const __half*>(h0);
    auto c0p = static_cast<const float*>(c0);
    auto hp = static_cast<__half*>(h_all);
    auto cp = static_cast<float*>(c_out);
    auto pre = static_cast<float*>(workspace);
    return launch_lstm_hoisted(xp, wp, bp, h0p, c0p, hp, cp, T, B, I, H, pre, s);
}

unsigned long long tcu_lstm_layer_workspace_bytes(int T, int B, int I, int H) {
    if (!positive({T, B, I, H}) || !lstm_layer_takes(T, B, I, H)) return 0;
    const int parts = lstm_layer_parts(T, B, H);
    return kPersistentSyncBytes + (unsigned long long)((T + parts - 1) / parts) * B * 4 * H * sizeof(float);
}

int tcu_lstm_uses_layer(int T, int B, int I, int H) { return positive({T, B, I, H}) && lstm_layer_pays(T, B, I, H) ? 1 : 0; }

int tcu_lstm_f16_layer(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all, void* c_out,
                       int T, int B, int I, int H, void* workspace, unsigned long long workspace_bytes, void* stream) {
    return lstm_f16_layer(x, W, bias, h0, c0, h_all, c_out, T, B, I, H, workspace, workspace_bytes, LstmLayerLimits{}, stream);
}

int tcu_lstm_f16_layer_limited(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all, void* c_out,
                               int T, int B, int I, int H, void* workspace, unsigned long long workspace_bytes, int max_workgroups,
                               int takeover_us, int max_tries, void* stream) {
    if (max_workgroups < 1 || takeover_us < 0 || takeover_us > 1000000 || max_tries < 0 || max_tries > 1 << 24)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_layer_limited: at least one workgroup, 0 <= takeover_us <= 1000000, 0 <= "
                                              "max_tries <= 2^24");
    return lstm_f16_layer(x, W, bias, h0, c0, h_all, c_out, T, B, I, H, workspace, workspace_bytes, {max_workgroups, takeover_us, max_tries}, stream);
}

unsigned long long tcu_lstm_persistent_workspace_bytes(int T, int B, int I, int H) {
    using Traits = LstmRecurrentTraits<1024>;
    if (T <= 0 || B <= 0 || I <= 0 || (H != 256 && H != 512 && H != 768 && H != 1024)) return 0;
    if (B % Traits::kRows != 0 || B > Traits::kRows * Traits::kXcds || I % 64 != 0) return 0;
    if ((long)T * B % 256 != 0 || (long)T * B > INT_MAX) return 0;
    // the pre-activations of all steps in f16: [T, B, 4H]
    return kPersistentSyncBytes + (unsigned long long)T * B * 4 * H * sizeof(__half);
}

int tcu_lstm_f16_persistent(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                            void* c_out, int T, int B, int I, int H, void* workspace, unsigned long long workspace_bytes,
                            void* stream) {
    using Traits = LstmRecurrentTraits<1024>;
    if (!x || !W || !bias || !h_all || !c_out || !workspace)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_persistent: null pointer");
    if (!positive({T, B, I, H})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_persistent: sizes must be positive");
    if (!aligned16({x, W, bias, h0, c0, h_all, c_out}) || reinterpret_cast<uintptr_t>(workspace) % 128 != 0)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_persistent: operands must be 16-byte aligned, the workspace 128-byte aligned");
    const unsigned long long need = tcu_lstm_persistent_workspace_bytes(T, B, I, H);
    if (need == 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16_persistent: needs H in {256, 512, 768, 1024}, I % 64 == 0, B % 32 == 0, "
                                               "B <= 256 and T * B % 256 == 0");
    if (workspace_bytes < need)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_persistent: workspace smaller than tcu_lstm_persistent_workspace_bytes()");
    // one workgroup per CU, all resident at once, H / 32 per XCD (dealt to the 8 XCDs in turn): at H = 1024 the grid is
    // the chip
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        return fail(TCU_ERR_NO_DEVICE, "tcu_lstm_f16_persistent: no current HIP device");
    if (cus != Traits::kGrid)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16_persistent: written for a device of 256 CUs in 8 XCDs; this one has " +
                                                   std::to_string(cus) + " CUs");
    unsigned long long spin_us = 2000000;  // a wait is microseconds when every workgroup is resident
    long peers = -1;                       // (the number of workgroups per XCD)
    if (const char* e = std::getenv("TCU_LSTM_PERSISTENT_SPIN_US")) spin_us = std::strtoull(e, nullptr, 10);
    if (const char* e = std::getenv("TCU_LSTM_PERSISTENT_PEERS")) peers = long(std::strtoul(e, nullptr, 10));
    auto s = static_cast<hipStream_t>(stream);
    auto sync = static_cast<unsigned int*>(workspace);
    auto pre = reinterpret_cast<__half*>(static_cast<unsigned char*>(workspace) + kPersistentSyncBytes);
    auto xp = static_cast<const __half*>(x), wp = static_cast<const __half*>(W);
    // The projection GEMM writes the pre-activations as f16 (f32 sums rounded once: half the bytes written here and read
    // by the recurrence, where the f32 form of tcu_lstm_f16_ws is bound by the volume of that write) and clears the
    // synchronisation words on the side (its first workgroup): no launch of its own.
    int rc = gemm_w128_dispatch<__half>(xp, wp, pre, T * B, 4 * H, I, s, I, I + H, 0, sync, Traits::kSyncWords);
    if (rc != TCU_OK) return rc;
    switch (H) {
        case 256: return launch_lstm_recurrent_xcd<256>(pre, wp, bias, h0, c0, h_all, c_out, T, B, I, sync, spin_us, peers, s);
        case 512: return launch_lstm_recurrent_xcd<512>(pre, wp, bias, h0, c0, h_all, c_out, T, B, I, sync, spin_us, peers, s);
        case 768: return launch_lstm_recurrent_xcd<768>(pre, wp, bias, h0, c0, h_all, c_out, T, B, I, sync, spin_us, peers, s);
        default: return launch_lstm_recurrent_xcd<1024>(pre, wp, bias, h0, c0, h_all, c_out, T, B, I, sync, spin_us, peers, s);
    }
}

int tcu_lstm_persistent_status(const void* workspace, void* stream) {
    if (!workspace) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_persistent_status: null pointer");
    auto s = static_cast<hipStream_t>(stream);
    unsigned int word = 0;
    hipError_t e = hipStreamSynchronize(s);
    if (e == hipSuccess)
        e = hipMemcpy(&word, static_cast<const unsigned int*>(workspace) + LstmRecurrentTraits<1024>::kErrorWord, sizeof(word),
                      hipMemcpyDeviceToHost);
    if (e != hipSuccess) return fail(TCU_ERR_HIP, std::string("tcu_lstm_persistent_status: ") + hipGetErrorString(e));
    if (word == 1)
        return fail(TCU_ERR_INCOMPLETE, "tcu_lstm_f16_persistent: workgroups that exchange h through an L2 were placed on different XCDs; the outputs are invalid");
    if (word != 0)
        return fail(TCU_ERR_INCOMPLETE, "tcu_lstm_f16_persistent: a workgroup waited for its XCD longer than the limit (the grid "
                                    "was not resident at once); the outputs are invalid");
    return TCU_OK;
}

unsigned long long tcu_lstm_noalloc_max_bytes(void) { return kScratchBytes; }

int tcu_lstm_f16_noalloc(const void* x, const void* W, const void* bias, const void* h0, const void* c0, void* h_all,
                         void* c_out, int T, int B, int I, int H, void* stream) {
    if (!x || !W || !bias || !h_all || !c_out) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_noalloc: null pointer");
    if (!positive({T, B, I, H})) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_noalloc: sizes must be positive");
    if (!aligned16({x, W, bias, h0, c0, h_all, c_out}))
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_lstm_f16_noalloc: operands must be 16-byte aligned");
    const unsigned long long need = tcu_lstm_workspace_bytes(T, B, I, H);
    if (need == 0)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE, "tcu_lstm_f16_noalloc: needs I % 128 == 0, H % 128 == 0, B % 64 == 0 and "
                                               "T * B % 256 == 0");
    if (need > kScratchBytes)
        return fail(TCU_ERR_UNSUPPORTED_SHAPE,
                    "tcu_lstm_f16_noalloc: the gate pre-activations need " + std::to_string(need) +
                        " bytes, more than the library's static scratch buffer of " + std::to_string(kScratchBytes) +
                        " bytes (T * B * 4H * 4 must not exceed it); use tcu_lstm_f16_ws with a caller-owned workspace");
    void* ws = nullptr;
    if (int rc = scratch_address(&ws); rc != TCU_OK) return rc;
    return tcu_lstm_f16_ws(x, W, bias, h0, c0, h_all, c_out, T, B, I, H, ws, kScratchBytes, stream);
}

int tcu_scatter_nd(void* data, const void* updates, const void* indices, const long long* data_dims, int rank,
                   long long n, int k, int dtype, int mode, void* skipped_rows, void* stream) {
    using namespace tiledcuda::kernels;
    if (!data || !updates || !indices || !data_dims) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_scatter_nd: null pointer");
    if (rank <= 0 || rank > kScatterMaxRank || k <= 0 || k > rank)
        return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_scatter_nd: need 0 < k <= rank <= 8");
    if (n < 0) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_scatter_nd: negative row count");
    if (dtype != TCU_DTYPE_F32 && dtype != TCU_DTYPE_F16) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_scatter_nd: dtype must be f32 or f16");
    if (mode != TCU_SCATTER_ASSIGN && mode != TCU_SCATTER_ADD) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_scatter_nd: unknown mode");
    ScatterNdShape shape{};
    int64_t stride = 1;
    for (int d = rank - 1; d >= 0; --d) {
        if (data_dims[d] <= 0) return fail(TCU_ERR_INVALID_ARGUMENT, "tcu_scatter_nd: dimensions must be positive");
        if (d < k) {
            shape.strides[d] = stride;
            shape.dims[d] = data_dims[d];
        }
        stride *= data_dims[d];
    }
    shape.slice = 1;
    for (int d = k; d < rank; ++d) shape.slice *= data_dims[d];
    shape.n = n;
    shape.k = k;
    if (n == 0) return TCU_OK;
    auto s = static_cast<hipStream_t>(stream);
    auto idx = static_cast<const int64_t*>(indices);
    auto bad = static_cast<unsigned int*>(skipped_rows);
    // f16 additions: a word of two elements at a time (see the kernel for both sides measured; slices of one element have no word
    // to themselves: 16384 of them 5.6 us there, 5.1 below)
    if (dtype == TCU_DTYPE_F16 && mode == TCU_SCATTER_ADD && shape.slice > 1 && plain_device_memory(data)) {
        const bool whole = shape.slice % 2 == 0 && reinterpret_cast<uintptr_t>(data) % 4 == 0 && reinterpret_cast<uintptr_t>(updates) % 4 == 0;
        const int64_t per_block = 256 * scatter_pair_pieces(whole);
        const int64_t blocks = (n * scatter_pair_words(whole, shape.slice) + per_block - 1) / per_block;
        return launch(whole ? &scatter_nd_add_pairs<true> : &scatter_nd_add_pairs<false>,
                      dim3(static_cast<unsigned>(std::min<int64_t>(blocks, 1 << 22))), dim3(256), 0, s, static_cast<__half*>(data),
                      static_cast<const __half*>(updates), idx, shape, bad);
    }
    const size_t elem = dtype == TCU_DTYPE_F32 ? 4 : 2;
    const int vec = int(16 / elem);
    const bool vec_ok = mode == TCU_SCATTER_ASSIGN && shape.slice % vec == 0 &&
                        reinterpret_cast<uintptr_t>(data) % 16 == 0 && reinterpret_cast<uintptr_t>(updates) % 16 == 0;
    const int64_t lanes = n * (vec_ok ? shape.slice / vec : shape.slice);
    // enough workgroups to fill the chip several times over; the kernel strides over the rest
    const int64_t want = (lanes + 255) / 256;
    const dim3 grid(static_cast<unsigned>(want < 1 ? 1 : (want > 256 * 64 ? 256 * 64 : want))), block(256);
    auto go = [&](auto* dptr, auto kernel) {
        using T = std::remove_pointer_t<decltype(dptr)>;
        return launch(kernel, grid, block, 0, s, dptr, static_cast<const T*>(updates), idx, shape, bad);
    };
    if (dtype == TCU_DTYPE_F32) {
        auto* d = static_cast<float*>(data);
        if (mode == TCU_SCATTER_ADD) return go(d, &scatter_nd_kernel<float, 1, ScatterMode::kAdd>);
        return vec_ok ? go(d, &scatter_nd_kernel<float, 4, ScatterMode::kAssign>)
                      : go(d, &scatter_nd_kernel<float, 1, ScatterMode::kAssign>);
    }
    auto* d = static_cast<__half*>(data);
    if (mode == TCU_SCATTER_ADD) return go(d, &scatter_nd_kernel<__half, 1, ScatterMode::kAdd>);
    return vec_ok ? go(d, &scatter_nd_kernel<__half, 8, ScatterMode::kAssign>)
                  : go(d, &scatter_nd_kernel<__half, 1, ScatterMode::kAssign>);
}

}  // extern "C"
