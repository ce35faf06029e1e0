// The time loop of the fused LSTM layer in one launch, recurrent weights in registers, for gfx950: same contract as
// kernels/lstm_fwd.hpp, any batch and hidden size in multiples of 16 (H <= 1024, T >= 2), behind the GEMM that computes the input
// half of all steps' gates, pre[T, B, 4H] in f32. (kernels/lstm_recurrent.hpp is the same idea for four hidden sizes on a GPU of
// its own.)
//
// What bounds a launch per step is the launch and the weights that every CU fetches again (109 us for 24 steps of B 80, I 336, H
// 656). Here an XCD owns 16 or 32 rows of the batch and a copy of W[:, I:] in the registers of up to 32 CUs, 16 or 32 hidden units
// each, and h_t goes from CU to CU through that XCD's L2:
//   * h itself says when it is there. Every word of h_all that a workgroup is going to write holds ~0 until then (two f16 NaNs, which
//     the kernel stores as other NaNs), and the readers, past their L1, take a word that is not ~0. A step has no counter, no wait
//     for the acknowledgement of stores and one barrier where h comes in one part;
//   * a wavefront owns 4 units x 4 gates x all columns per tile (the 16 rows of v_mfma_f32_16x16x32_f16's operand): a lane's
//     accumulator holds the four gates of one unit and row, so the cell is updated in registers. The four wavefronts fetch h (a quarter
//     of the rows each, in whole rows: as fragments, 16 rows x 16 bytes per quarter of a load, it came at 16 bytes per clock, so
//     at 45) and share it through LDS;
//   * the pre-activations arrive in LDS a step ahead and are the accumulators' first value.
// No workgroup waits for one that is not running. An XCD's workgroups draw tickets for the slices of the units as they start (the
// XCD is read from the hardware); before step 1 they wait until all slices have filled their words with ~0, and whoever has waited
// `steal_ticks` draws another ticket and works on that slice as well, weights fetched anew per step: slow, and right with a single
// workgroup. Groups of rows are claimed by XCD, and an XCD that is done claims another. So the layer needs no part of the GPU for
// itself. (The waits count their tries all the same. A wavefront that gives one up goes on with cell states of NaN: its units are NaN
// from that step on, and one step later so is all that is computed from them.)
// Measured, kernel alone, us: T 24, B 80, H 656: 55 (6 us until the first workgroups know their rows, 7 for the weights, 1.75 per step:
// 0.45 for h to come back from the L2, 0.2 to LDS, 0.6 for 48 products and their fragments, 0.3 for the cell); 16, 256, 1024: 79
// (20 before the first step, 3.7 per step: the LDS, 64 KB of h in and 256 KB of fragments out, and h itself, 64 KB at 45 bytes per
// clock); 31, 80, 384: 48; 20, 32, 96: 20.
#pragma once

#include <type_traits>

#include "config.hpp"
#include "hip_utils.hpp"
#include "kernels/gemm_pipelined.hpp"  // detail::lds_barrier, load_lds_16B_sbase
#include "kernels/lstm_fwd.hpp"        // detail::sigmoid_fast
#include "util/static_for.hpp"

namespace tiledcuda::kernels {

/// kTW: tiles of 4 units (x 4 gates: the 16 rows of an operand) per wavefront; kKS: 32-column steps of the hidden size (H <= 32 kKS);
/// kRT: 16-row tiles of the batch per XCD.
template <const int kTW_, const int kKS_, const int kRT_>
struct LstmLayerTraits {
    static constexpr int kTW = kTW_, kKS = kKS_, kRT = kRT_;
    static constexpr int kWaves = 4, kThreads = kWaves * kWaveSize;
    static constexpr int kUnits = 16 * kTW, kRows = 16 * kRT;
    static constexpr int kPitch = 64 * kKS;                              // bytes of a row of h in LDS
    static constexpr int kPanelBytes = kRows * kPitch;                   // h_{t-1}; two of them, for even and odd steps
    static constexpr int kParts = kRT * kKS >= 32 && kKS >= 16 ? 2 : 1;  // column ranges of h that arrive one after the other
    static constexpr int kPartSteps = kKS / kParts;
    static constexpr int kLoads = kRT * kKS / 4 / kParts;  // 1 KiB of a part per instruction and wavefront
    static constexpr int kPreBytes = 4096 * kRT * kTW;     // pre-activations of a step; two of them where h comes in one part
    static constexpr int kPreBuffers = kParts == 1 ? 2 : 1;
    static constexpr int kStageBytes = 16 * kPitch;        // a tile of weights on its way in, per wavefront
    static constexpr int kPreOffset = 2 * kPanelBytes > kWaves * kStageBytes ? 2 * kPanelBytes : kWaves * kStageBytes;
    static constexpr int kLdsBytes = kPreOffset + kPreBuffers * kPreBytes;
    static constexpr int kMaxPeers = 32, kXccs = 16, kMaxGroups = 64;
    static constexpr int kSyncWords = 32 * kXccs + kMaxGroups;
    static_assert(kKS % 4 == 0 && 4 * kKS * kTW <= 256 && kLoads * 4 * kParts == kRT * kKS && kLdsBytes <= kMaxLdsBytes - 1024);
    /// Slot (16 bytes: 4 units) of the pre-activations of (gate, row, quad of units).
    HOST_DEVICE static constexpr int pre_key(int row) { return kTW == 1 ? (row >> 2) & 3 : (row >> 1) & 7; }
    HOST_DEVICE static constexpr int pre_slot(int gate, int row, int quad) { return (gate * kRows + row) * 4 * kTW + (quad ^ pre_key(row)); }
};

namespace detail {
using buffer_t = __amdgpu_buffer_rsrc_t;
constexpr unsigned kBufferNone = 0x7ffffff0u;  // an offset beyond every buffer: reads 0
/// 16 bytes past the vector L1 (device scope): data that other CUs write during this launch.
DEVICE u32x4 buffer_fresh(buffer_t b, unsigned off) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 16)); }

/// A pointer that is the same in all lanes, in scalar registers whatever the compiler made of it.
template <typename T>
DEVICE T* uniform(T* p) {
    const auto v = reinterpret_cast<uintptr_t>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane(unsigned(v)), hi = __builtin_amdgcn_readfirstlane(unsigned(v >> 32));
    return reinterpret_cast<T*>(uintptr_t(lo) | uintptr_t(hi) << 32);
}

/// sigmoid(a) * tanh(b) as one quotient, (1 - e) / ((1 + E) (1 + e)) with E = e^-a and e = e^-2|b| <= 1, signed as b: one reciprocal,
/// finite for every finite b, NaN where a or b is.
DEVICE float sigmoid_tanh(float a, float b) {
    const float ea = __expf(-a), eb = __expf(-2.0f * fabsf(b));
    return copysignf((1.0f - eb) * __builtin_amdgcn_rcpf((1.0f + ea) * (1.0f + eb)), b);
}

/// acc = w . h + c and acc += w . h with the weights in AGPRs.
DEVICE void mfma16_weights_in_agprs(f32x4& acc, const f16x8& w, const f16x8& h, const f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %3" : "=&v"(acc) : "a"(w), "v"(h), "v"(c));
}
DEVICE void mfma16_weights_in_agprs(f32x4& acc, const f16x8& w, const f16x8& h) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc) : "a"(w), "v"(h));
}
}  // namespace detail

/// grid = 8 * ceil(H / kUnits) (fewer work as well), block = 256, dynamic LDS = Traits::kLdsBytes; pre [T, B, 4H]; the recurrent
/// block of W starts at column w_col0 of rows of ldw; h0 / c0 may be null (zeros), h0 must not overlap h_all; sync: kSyncWords device
/// words, zero at the launch: per XCD (32 words apart) tickets, the group that its first workgroup found and slices filled, then
/// whose each group of rows is. max_tries: polls of a wait. T >= 2, B <= kMaxGroups * kRows, 4H * ldw below 2^31.
template <typename Traits>
__global__ void __launch_bounds__(Traits::kThreads, 1)
    lstm_layer_xcd(const float* __restrict__ pre, const __half* __restrict__ W, int ldw, int w_col0, const __half* __restrict__ bias,
                   const __half* h0, const float* c0, __half* h_all, float* c_out, int T, int B, int H, unsigned int* sync, int steal_ticks,
                   int max_tries) {
    constexpr int kTW = Traits::kTW, kKS = Traits::kKS, kRT = Traits::kRT, kParts = Traits::kParts, kLoads = Traits::kLoads, kPitch = Traits::kPitch;
    extern __shared__ __align__(1024) unsigned char lds[];
    __shared__ int s_word[2];
    __shared__ unsigned char s_tile[Traits::kMaxPeers];

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_id());
    const int line = lane & 15, g = lane >> 4;
    const int peers = (H + Traits::kUnits - 1) / Traits::kUnits;
    const int groups = (B + Traits::kRows - 1) / Traits::kRows;

    // ---- a ticket of this XCD: slice `ticket` of the units, for every group of rows that the XCD takes; and the group of the XCD's
    // number for it, if no other XCD has it
    const unsigned xcc = __builtin_amdgcn_s_getreg(20 | (0 << 6) | ((4 - 1) << 11));
    unsigned int* const tickets = sync + 32 * xcc;
    unsigned int* const group_word = tickets + 1;
    unsigned int* const ready = tickets + 2;
    unsigned int* const claims = sync + 32 * Traits::kXccs;
    auto claim = [&](int group) {
        unsigned expected = 0;
        __hip_atomic_compare_exchange_strong(claims + group, &expected, xcc + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return expected;  // whose it was
    };
    if (threadIdx.x < 2) {
        int v;
        if (threadIdx.x == 0) {
            v = int(__hip_atomic_fetch_add(tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            s_tile[0] = static_cast<unsigned char>(min(v, Traits::kMaxPeers));
        } else {
            v = -1;
            if (int(xcc) < groups) {
                const unsigned whose = claim(int(xcc));
                if (whose == 0 || whose == xcc + 1) v = int(xcc);
            }
        }
        s_word[threadIdx.x] = v;
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_word[0]) >= peers) return;
    int group = __builtin_amdgcn_readfirstlane(s_word[1]);
    int tiles = 1, served = 0;  // slices held; groups that the XCD has had so far
    int limit = max_tries;      // -1: this wavefront has given up a wait
    __syncthreads();

    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds));
    // ---- this wavefront's weights: tile n is units 16 n + 4 wave .. + 3 of the slice, operand row 4 (unit % 4) + gate
    f16x8 wf[kTW][kKS];
    int loaded = -1;
    auto unit_of = [&](int slice, int n) { return slice * Traits::kUnits + 16 * n + 4 * wave; };
    auto load_weights = [&](int slice) __attribute__((always_inline)) {
        loaded = slice;
        // (few instructions: they run once, as fast as they are fetched)
        const unsigned stage = wave * Traits::kStageBytes;
        const unsigned char* frag[4];  // fragment s: frag[s % 4], 256 (s / 4) bytes on
#pragma unroll
        for (int s = 0; s < 4; ++s) frag[s] = lds + stage + line * kPitch + (((4 * s + g) ^ line) * 16);
        static_for<kTW>([&](auto n) __attribute__((always_inline)) {
            const int unit0 = unit_of(slice, n);
#pragma unroll 1
            for (int j = 0; j < kKS; ++j) {  // (1 KiB each: 16-byte piece p of row r at piece p ^ r)
                const int r = (64 * j + lane) / (4 * kKS), p = ((64 * j + lane) % (4 * kKS)) ^ r;
                const int row = (r & 3) * H + min(unit0 + (r >> 2), H - 1);
                detail::load_lds_16B_sbase(unsigned(row) * (2u * ldw) + (8 * p < H ? 16u * p : 0u), W + w_col0, lds0 + stage + j * 1024);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll 1
            for (int i = H / 8 * 16 + lane; i < 64 * kKS; i += kWaveSize)  // columns beyond H: i / 16 the piece, i % 16 the row
                *reinterpret_cast<u32x4*>(lds + stage + (i & 15) * kPitch + (((i >> 4) ^ (i & 15)) * 16)) = u32x4{0, 0, 0, 0};
            asm volatile("" ::: "memory");
#pragma unroll
            for (int s0 = 0; s0 < kKS; s0 += 4) {
#pragma unroll
                for (int s = s0; s < s0 + 4; ++s) wf[n][s] = *reinterpret_cast<const f16x8*>(frag[s % 4] + 256 * (s / 4));
#pragma unroll
                for (int s = s0; s < s0 + 4; ++s) asm volatile("" : "+a"(wf[n][s]));
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        });
        __syncthreads();  // (the stages lie where h goes)
    };

    // ---- this wavefront's quarter of the rows of h: load instruction j of part c
    unsigned h_src[kParts][kLoads], h_dst[kLoads];
    auto h_row = [&](int j) { return 4 * kRT * wave + (64 * j + lane) / (4 * Traits::kPartSteps); };
    auto h_piece = [&](int c, int j) { return 4 * Traits::kPartSteps * c + (64 * j + lane) % (4 * Traits::kPartSteps); };

    f32x4 bias_v[kTW];
    float c_state[kTW][kRT];
    unsigned h_out[kTW][kRT];  // byte offset of the word of h_t that a lane stores

    for (;; group = -1) {
        if (group < 0) {
            // ---- the next group of rows: the holder of the XCD's first ticket finds one that no XCD has
            if (threadIdx.x == 0) {
                int mine = groups;
                if (s_tile[0] == 0) {
#pragma unroll 1
                    for (int k = 0; k < groups; ++k)
                        if (__hip_atomic_load(claims + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0 && claim(k) == 0) {
                            mine = k;
                            break;
                        }
                    __hip_atomic_store(group_word, unsigned(served + 1) << 16 | unsigned(mine), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
#pragma unroll 1
                    for (int n = 0; n <= limit; ++n) {  // (given up: the workgroup leaves, whose slice the others of the next group miss)
                        const unsigned v = __hip_atomic_load(group_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if ((v >> 16) == unsigned(served + 1)) {
                            mine = int(v & 0xffffu);
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                s_word[0] = mine;
            }
            __syncthreads();
            group = __builtin_amdgcn_readfirstlane(s_word[0]);
            __syncthreads();
            if (group >= groups) return;
        }
        ++served;
        const int row0 = group * Traits::kRows;
        const int rows = min(B - row0, Traits::kRows);

        // every word of h that this workgroup will write holds ~0 until then (steps 0 .. T - 2: the last one is not read here)
        auto fill = [&](int slice) {
            constexpr int kPieces = Traits::kUnits / 8;
            const int p = threadIdx.x % kPieces, unit0 = slice * Traits::kUnits + 8 * p;
#pragma unroll 1
            for (int r = threadIdx.x / kPieces; r < Traits::kRows * (T - 1); r += Traits::kThreads / kPieces)
                if (r % Traits::kRows < rows && unit0 < H)
                    *reinterpret_cast<u32x4*>(h_all + (size_t(r / Traits::kRows) * B + row0 + r % Traits::kRows) * H + unit0) = u32x4{~0u, ~0u, ~0u, ~0u};
        };

#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int r = h_row(j);
#pragma unroll
            for (int c = 0; c < kParts; ++c) {
                const int p = h_piece(c, j);
                h_src[c][j] = r < rows && 8 * p < H ? unsigned(r * H + 8 * p) * 2u : detail::kBufferNone;
            }
            h_dst[j] = r * kPitch + ((h_piece(0, j) ^ (r & 15)) * 16);  // (part c: 64 kPartSteps bytes further; a multiple of 256)
        }

        // pre-activations of a step to LDS, 16 bytes per lane
        auto load_pre = [&](int t, int slice) __attribute__((always_inline)) {
            t = __builtin_amdgcn_readfirstlane(t);
            const float* base = detail::uniform(pre + (size_t(t) * B + row0) * (4 * size_t(H)) + slice * Traits::kUnits);
            const unsigned dst = lds0 + Traits::kPreOffset + (Traits::kPreBuffers == 2 ? (t & 1) * Traits::kPreBytes : 0) + wave * kRT * kTW * 1024;
#pragma unroll
            for (int j = 0; j < kRT * kTW; ++j) {
                const int i = (wave * kRT * kTW + j) * 64 + lane;
                const int row = i / (4 * kTW) % Traits::kRows, gate = i / (4 * kTW * Traits::kRows), quad = (i % (4 * kTW)) ^ Traits::pre_key(row);
                const int unit = slice * Traits::kUnits + 4 * quad < H ? 4 * quad : 0;
                detail::load_lds_16B_sbase(unsigned(min(row, rows - 1) * 4 * H + gate * H + unit) * 4u, base, dst + j * 1024);
            }
        };
        f32x4 pre_v[kTW][kRT];
        auto read_pre = [&](int t) __attribute__((always_inline)) {
            const unsigned char* src = lds + Traits::kPreOffset + (Traits::kPreBuffers == 2 ? (t & 1) * Traits::kPreBytes : 0);
#pragma unroll
            for (int n = 0; n < kTW; ++n)
#pragma unroll
                for (int r = 0; r < kRT; ++r)
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        pre_v[n][r][k] = *reinterpret_cast<const float*>(src + Traits::pre_slot(k, 16 * r + line, 4 * n + wave) * 16 + g * 4);
        };
        auto load_cell = [&](int slice, const float* c) __attribute__((always_inline)) {
            float c_raw[kTW][kRT];
            __half b_raw[kTW][4];
#pragma unroll
            for (int n = 0; n < kTW; ++n) {
                const int unit = min(unit_of(slice, n) + g, H - 1);  // (units and rows beyond the ends: anything, stored nowhere)
#pragma unroll
                for (int k = 0; k < 4; ++k) b_raw[n][k] = bias[k * H + unit];
#pragma unroll
                for (int r = 0; r < kRT; ++r) {
                    c_raw[n][r] = 0.f;
                    if (c) c_raw[n][r] = c[size_t(row0 + min(16 * r + line, rows - 1)) * H + unit];
                }
            }
#pragma unroll
            for (int n = 0; n < kTW; ++n) {
                const int unit = unit_of(slice, n) + g;
#pragma unroll
                for (int k = 0; k < 4; ++k) bias_v[n][k] = __half2float(b_raw[n][k]);
#pragma unroll
                for (int r = 0; r < kRT; ++r) {
                    h_out[n][r] = (g & 1) == 0 && unit < H && 16 * r + line < rows ? unsigned((16 * r + line) * H + unit) * 2u : detail::kBufferNone;
                    c_state[n][r] = c_raw[n][r];
                }
            }
        };
        auto store_cell = [&](int slice) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < kTW; ++n) {
                const int unit = unit_of(slice, n) + g;
#pragma unroll
                for (int r = 0; r < kRT; ++r)
                    if (unit < H && 16 * r + line < rows) c_out[size_t(row0 + 16 * r + line) * H + unit] = c_state[n][r];
            }
        };
        // One step of one slice. next_t: the step whose pre-activations are to be requested (or -1).
        auto step = [&](int t, int slice, int next_t) __attribute__((always_inline)) {
            const detail::buffer_t out = __builtin_amdgcn_make_buffer_rsrc(h_all + size_t(t) * B * H + size_t(row0) * H, 0, rows * H * 2, 0x00020000);
            const __half* h_prev = t == 0 ? h0 : h_all + size_t(t - 1) * B * H;
            f32x4 acc[kTW][kRT];
            if (h_prev) {
                const detail::buffer_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half*>(h_prev + size_t(row0) * H), 0, rows * H * 2, 0x00020000);
                unsigned char* const panel = lds + (t & 1) * Traits::kPanelBytes;
                u32x4 v[kParts][kLoads];
#pragma unroll
                for (int c = 0; c < kParts; ++c)
#pragma unroll
                    for (int j = 0; j < kLoads; ++j) v[c][j] = detail::buffer_fresh(b, h_src[c][j]);
                int tries = 0;
                static_for<kParts>([&](auto c_) __attribute__((always_inline)) {
                    constexpr int c = c_;
#pragma unroll 1
                    for (;;) {
                        unsigned top[2] = {0, 0};
#pragma unroll
                        for (int j = 0; j < kLoads; ++j) {
                            top[0] = max(top[0], max(v[c][j][0], v[c][j][1]));
                            top[1] = max(top[1], max(v[c][j][2], v[c][j][3]));
                        }
                        if (t == 0 || !__any(max(top[0], top[1]) == ~0u)) break;
                        if (tries >= limit) {
                            limit = -1;
                            break;
                        }
                        ++tries;
                        // some of it is not there yet: read once more (a count that the optimiser can follow becomes a copy of the loop each)
                        asm volatile("" : "+s"(tries)::"memory");
#pragma unroll
                        for (int j = 0; j < kLoads; ++j) v[c][j] = detail::buffer_fresh(b, h_src[c][j]);
                    }
#pragma unroll
                    for (int j = 0; j < kLoads; ++j) *reinterpret_cast<u32x4*>(panel + h_dst[j] + c * 64 * Traits::kPartSteps) = v[c][j];
                    detail::lds_barrier<63>();  // (every wavefront's loads of the pre-activations are older than those of h: landed too)
                    if constexpr (c == 0) read_pre(t);
                    constexpr int kGroup = kRT == 1 ? 4 : 2;  // steps whose fragments are read ahead
                    f16x8 f[2][kGroup][kRT];
                    auto read = [&](f16x8(&d)[kGroup][kRT], int s0) __attribute__((always_inline)) {
#pragma unroll
                        for (int s = 0; s < kGroup; ++s)
#pragma unroll
                            for (int r = 0; r < kRT; ++r)
                                d[s][r] = *reinterpret_cast<const f16x8*>(panel + (16 * r + line) * kPitch + (((4 * (s0 + s) + g) ^ line) * 16));
                    };
                    read(f[0], c * Traits::kPartSteps);
                    static_for<Traits::kPartSteps / kGroup>([&](auto i_) __attribute__((always_inline)) {
                        constexpr int i = i_, s0 = c * Traits::kPartSteps + i * kGroup;
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr (i + 1 < Traits::kPartSteps / kGroup) read(f[(i + 1) & 1], s0 + kGroup);
                        if constexpr (c + 1 == kParts && i == (Traits::kPartSteps / kGroup > 1 ? 1 : 0))
                            if (next_t >= 0) load_pre(next_t, slice);
#pragma unroll
                        for (int s = 0; s < kGroup; ++s)
#pragma unroll
                            for (int n = 0; n < kTW; ++n)
#pragma unroll
                                for (int r = 0; r < kRT; ++r) {
                                    if (s0 + s == 0) detail::mfma16_weights_in_agprs(acc[n][r], wf[n][0], f[i & 1][s][r], pre_v[n][r]);
                                    else detail::mfma16_weights_in_agprs(acc[n][r], wf[n][s0 + s], f[i & 1][s][r]);
                                }
                    });
                });
                // the compiler does not know the statements above are MFMAs: wait for the last results
                detail::mfma_results_wait();
#pragma unroll
                for (int n = 0; n < kTW; ++n)
#pragma unroll
                    for (int r = 0; r < kRT; ++r) asm volatile("" : "+v"(acc[n][r]));
            } else {
                detail::lds_barrier<0>();
                read_pre(t);
                // (one buffer: the next step's go where every wavefront has read this one's. Beside an h_prev the barrier of its
                // second part lies between the two)
                if constexpr (Traits::kPreBuffers == 1) detail::lds_barrier<63>();
                if (next_t >= 0) load_pre(next_t, slice);
#pragma unroll
                for (int n = 0; n < kTW; ++n)
#pragma unroll
                    for (int r = 0; r < kRT; ++r) acc[n][r] = pre_v[n][r];
            }
            if (__builtin_expect(limit < 0, 0)) {
#pragma unroll
                for (int n = 0; n < kTW; ++n)
#pragma unroll
                    for (int r = 0; r < kRT; ++r) c_state[n][r] = __builtin_nanf("");
            }
#pragma unroll
            for (int n = 0; n < kTW; ++n)
#pragma unroll
                for (int r = 0; r < kRT; ++r) {
                    float z[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) z[k] = acc[n][r][k] + bias_v[n][k];
                    const float cn = detail::sigmoid_fast(z[1]) * c_state[n][r] + detail::sigmoid_tanh(z[0], z[2]);
                    c_state[n][r] = cn;
                    const unsigned h = __half_as_ushort(__float2half(detail::sigmoid_tanh(z[3], cn)));
                    // lanes g and g ^ 1 hold neighbouring units of a row: the even ones store both
                    const auto pair = __builtin_amdgcn_permlane16_swap(h, h, false, false);
                    unsigned word = pair[0] | pair[1] << 16;
                    if (word == ~0u) word = 0xfffefffeu;  // two NaNs stay NaNs and are told from a word not yet written
                    __builtin_amdgcn_raw_buffer_store_b32(word, out, h_out[n][r], 0, 0);
                }
        };

        // ---- the steps of the slices held, mostly one. Step 0 needs no other workgroup; before step 1 everyone's words have to be
        // filled: from then on h itself says when it is there. A slice still without a workgroup `steal_ticks` later is taken over by
        // one that runs.
        int t = 0, i = 0;
        bool ahead = false;  // the pre-activations of this step have been requested by the one before
        for (;;) {
            const int slice = __builtin_amdgcn_readfirstlane(s_tile[i]);
            if (!ahead) {
                // (what was requested for a next step, before another slice came in between, may have the same place: landed first)
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
                __syncthreads();
                if (t == 0) fill(slice);
                load_pre(t, slice);
                load_cell(slice, t == 0 ? c0 : c_out);
            }
            if (slice != loaded) load_weights(slice);
            if (!ahead) {
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no wait for these is left to the steps
                if (t == 0) {
                    detail::lds_barrier<0>();  // everyone's words are filled
                    if (threadIdx.x == 0) __hip_atomic_fetch_add(ready, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            ahead = tiles == 1 && t + 1 < T;
            step(t, slice, ahead ? t + 1 : -1);
            if (t == 0 || tiles > 1 || t + 1 == T) store_cell(slice);
            if (++i < tiles) continue;
            i = 0;
            if (t == 0 && T > 1) {
                if (threadIdx.x == 0) {
                    const unsigned target = unsigned(peers) * unsigned(served);
                    const unsigned long long start = __builtin_amdgcn_s_memrealtime();
                    int stolen = -2;  // -1: all slices are marked; -2: given up
#pragma unroll 1
                    for (int n = 0;; ++n) {
                        if (__hip_atomic_load(ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= target) {
                            stolen = -1;
                            break;
                        }
                        if (__builtin_amdgcn_s_memrealtime() - start > (unsigned long long)steal_ticks &&
                            __hip_atomic_load(tickets, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < unsigned(peers)) {
                            const int k = int(__hip_atomic_fetch_add(tickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                            if (k < peers) {
                                stolen = k;
                                break;
                            }
                        }
                        if (n >= limit) break;
                        __builtin_amdgcn_s_sleep(1);
                    }
                    if (stolen >= 0) s_tile[tiles] = static_cast<unsigned char>(stolen);
                    s_word[0] = stolen;
                }
                __syncthreads();
                const int stolen = __builtin_amdgcn_readfirstlane(s_word[0]);
                __syncthreads();
                if (stolen == -2) limit = -1;
                if (stolen >= 0) {
                    i = tiles++;
                    ahead = false;
                    continue;
                }
            }
            if (++t == T) break;
        }
        __syncthreads();
    }
}

}  // namespace tiledcuda::kernels
