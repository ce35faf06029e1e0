// One time step of the fused LSTM layer for any batch, input and hidden size in multiples of 16, known at run time. Same
// contract as kernels/lstm_fwd.hpp: gates = concat(x_t, h_{t-1}) · Wᵀ + bias (W [4H, I + H], gate rows i, f, g, o),
// c_t = σ(f) c_{t-1} + σ(i) tanh(g), h_t = σ(o) tanh(c_t); f16 operands, f32 gates and cell state.
//
// What bounds a step is the path from the L2s into the CUs (64 bytes per clock and CU; 45 reached) and the launch: hence
//   * tiles of 4 to 16 hidden units x 16 to 64 batch rows, chosen by the launcher so that the workgroups fill the CUs once
//     and their rows (16 per unit tile, 16 per batch tile) are as few as possible;
//   * the 8 wavefronts of a workgroup split the columns of [x_t | h_{t-1}] in chunks of 64: a wavefront brings its chunks
//     to LDS in whole 128-byte lines, one or two ahead, in a ring of its own - no barrier before the sums are added. (The
//     same split with operands read straight from global memory as MFMA fragments ran at 16 bytes per clock: 16 lanes,
//     16 rows, 16 lines per quarter of a load.)
//   * a weight tile's 16 rows are 4 units x 4 gates, so that with v_mfma_f32_16x16x32_f16 a lane's accumulator holds the
//     four gates of one unit and batch row;
//   * the eight partial sums meet in LDS, where each thread collects consecutive units of one row: pre-activations, cell
//     state and outputs move in runs of 16 to 64 bytes.
// Measured per step in a graph, us, before -> now: B 80, I 336, H 656: 16.6 -> 4.5 (the kernel with fragments from global
// memory, lstm_ragged.hpp); 16, 1024, 1024: 36.8 -> 3.9; 256, 1024, 1024: 12.0 -> 9.7, its recurrent half only 8.5 -> 7.2
// (lstm_fwd.hpp); 64, 128, 128: 4.3 -> 2.8; 2.6 of each are the launch and the latency of a first load.
#pragma once

#include "config.hpp"
#include "hip_utils.hpp"
#include "kernels/flash_attn_fwd.hpp"  // detail::xcd_head_block
#include "kernels/lstm_fwd.hpp"        // detail::sigmoid_fast, tanh_fast

namespace tiledcuda::kernels {

/// kUT: 16-row tiles of weights (4 hidden units x 4 gates each) and kRT: 16-row tiles of the batch per workgroup.
template <const int kUT_, const int kRT_>
struct LstmDirectTraits {
    static constexpr int kUT = kUT_, kRT = kRT_;
    static constexpr int kWaves = 8, kThreads = kWaves * kWaveSize;
    static constexpr int kUnits = 4 * kUT, kRows = 16 * kRT;
    static constexpr int kBK = 64;                           // columns of a chunk: rows of 128 bytes
    static constexpr int kLoads = 2 * (kUT + kRT);           // 1 KiB direct-to-LDS instructions (8 rows) per chunk
    static constexpr int kRing = kUT + kRT <= 4 ? 2 : 1;     // chunks in flight per wavefront
    static constexpr int kWaveBytes = kRing * kLoads * 1024;
    static constexpr int kTiles = kUT * kRT;
    static constexpr int kLdsBytes = kWaves * kWaveBytes;
    static_assert(kTiles * 1024 <= kWaveBytes, "a wavefront's sums take the place of its chunks");
    static constexpr int kOutputs = kUnits * kRows;
    static constexpr int kPerThread = (kOutputs + kThreads - 1) / kThreads;
};

/// grid = ceil(H / kUnits) * ceil(B / kRows), block = 512, dynamic LDS = Traits::kLdsBytes. h_in / c_in may be null (zeros);
/// h_out must not alias h_in. B, I, H multiples of 16, 4H * (I + H) and B * max(I, H) below 2^31 (32-bit byte offsets).
/// kHoisted: pre_t [B, 4H] f32 holds x_t · W[:, :I]ᵀ, x_t is not read.
template <typename Traits, bool kHoisted>
__global__ void __launch_bounds__(Traits::kThreads)
    lstm_cell_direct(const __half* __restrict__ x_t, const __half* __restrict__ h_in, const __half* __restrict__ W,
                     const __half* __restrict__ bias, const float* c_in, float* c_out, __half* __restrict__ h_out, int B,
                     const float* __restrict__ pre_t, int I, int H) {
    constexpr int kUT = Traits::kUT, kRT = Traits::kRT, kWaves = Traits::kWaves, kRing = Traits::kRing, kBK = Traits::kBK;
    extern __shared__ __align__(1024) unsigned char lds[];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_id());
    const int line = lane & 15, group = lane >> 4;
    const int KK = I + H;

    int u_block, r_block;
    detail::xcd_head_block((B + Traits::kRows - 1) / Traits::kRows, (H + Traits::kUnits - 1) / Traits::kUnits, u_block, r_block);
    const int unit0 = u_block * Traits::kUnits, row0 = r_block * Traits::kRows;

    // ---- global -> LDS: instruction q of a chunk fills 8 rows of 128 bytes, those of the weights (row 16 u + 4 (unit % 4) +
    // gate) before those of the batch; physical 16-byte piece p of row r holds logical piece p ^ (r / 2) % 8
    const int lrow = lane >> 3;
    unsigned w_row[2 * kUT], a_row[2 * kRT];  // the lane's row in units of W's, x's or h's rows
    unsigned piece[2];                        // ... and piece, for even and odd instructions
#pragma unroll
    for (int q = 0; q < 2 * kUT; ++q) w_row[q] = (lrow & 3) * H + min(unit0 + 2 * q + (lrow >> 2), H - 1);
#pragma unroll
    for (int q = 0; q < 2 * kRT; ++q) a_row[q] = min(row0 + 8 * q + lrow, B - 1);
#pragma unroll
    for (int o = 0; o < 2; ++o) piece[o] = (lane & 7) ^ (4 * o + (lrow >> 1));
    // The columns in chunks of 64, those of x_t first; the wavefronts take them in turn. The last chunk of either part may
    // be partial: pieces beyond it are fetched from the row's first one and zeroed before the product.
    const int nx = kHoisted ? 0 : (I + kBK - 1) / kBK, nh = h_in ? (H + kBK - 1) / kBK : 0, total = nx + nh;
    const int n = (total - wave + kWaves - 1) / kWaves;
    unsigned char* const ring = lds + wave * Traits::kWaveBytes;
    const unsigned ring0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(ring));
    auto columns = [&](int c) { return c < nx ? min(I - kBK * c, kBK) : min(H - kBK * (c - nx), kBK); };
    auto issue = [&](int i) {
        const int c = wave + kWaves * i;
        const bool in_x = c < nx;
        const int k = in_x ? kBK * c : kBK * (c - nx);
        const __half* a_base = (in_x ? x_t : h_in) + k;
        const __half* w_base = W + (in_x ? 0 : I) + k;
        const unsigned a_pitch = 2u * (in_x ? I : H), valid = columns(c) / 8;
        const unsigned dst = ring0 + (i % kRing) * Traits::kLoads * 1024;
        unsigned off[2];
#pragma unroll
        for (int o = 0; o < 2; ++o) off[o] = piece[o] < valid ? 16 * piece[o] : 0;
#pragma unroll
        for (int q = 0; q < 2 * kUT; ++q) detail::load_lds_16B_sbase(w_row[q] * (2u * KK) + off[q & 1], w_base, dst + q * 1024);
#pragma unroll
        for (int q = 0; q < 2 * kRT; ++q)
            detail::load_lds_16B_sbase(a_row[q] * a_pitch + off[q & 1], a_base, dst + (2 * kUT + q) * 1024);
    };
#pragma unroll
    for (int i = 0; i < kRing; ++i)
        if (i < n) issue(i);

    // ---- operands of the cell update: thread t takes outputs t, t + 512, ... of the workgroup's [row][unit]
    float c_prev[Traits::kPerThread], pre_v[Traits::kPerThread][4];
    __half bias_v[Traits::kPerThread][4];
#pragma unroll
    for (int p = 0; p < Traits::kPerThread; ++p) {
        const int o = threadIdx.x + p * Traits::kThreads;
        const int unit = min(unit0 + o % Traits::kUnits, H - 1), row = min(row0 + o / Traits::kUnits, B - 1);
        c_prev[p] = c_in ? c_in[size_t(row) * H + unit] : 0.f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            bias_v[p][g] = bias[g * H + unit];
            if constexpr (kHoisted) pre_v[p][g] = pre_t[size_t(row) * 4 * H + g * H + unit];
        }
    }

    f32x4 acc[kUT][kRT];
#pragma unroll
    for (int u = 0; u < kUT; ++u)
#pragma unroll
        for (int r = 0; r < kRT; ++r) acc[u][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < n; ++i) {
        if (kRing == 2 && i + 1 < n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Traits::kLoads) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned char* src = ring + (i % kRing) * Traits::kLoads * 1024;
        f16x8 wf[2][kUT], af[2][kRT];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int off = line * 128 + (((4 * s + group) ^ (line >> 1)) * 16);
#pragma unroll
            for (int u = 0; u < kUT; ++u) wf[s][u] = *reinterpret_cast<const f16x8*>(src + u * 2048 + off);
#pragma unroll
            for (int r = 0; r < kRT; ++r) af[s][r] = *reinterpret_cast<const f16x8*>(src + (kUT + r) * 2048 + off);
        }
        if (i + kRing < n) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the fragments have left the slot about to be refilled
            issue(i + kRing);
        }
        const int cols = columns(wave + kWaves * i);
        if (cols < kBK) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (32 * s + 8 * group >= cols) {
#pragma unroll
                    for (int u = 0; u < kUT; ++u) wf[s][u] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                    for (int r = 0; r < kRT; ++r) af[s][r] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
                }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int u = 0; u < kUT; ++u)
#pragma unroll
                for (int r = 0; r < kRT; ++r)
                    acc[u][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[s][u], af[s][r], acc[u][r], 0, 0, 0);
    }

    // ---- add the eight wavefronts' sums through LDS. A lane's accumulator holds the four gates of (unit 4 u + lane / 16,
    // batch row 16 r + lane % 16); its 16 bytes go to slot 16 (lane / 16) + (lane % 16 + 4 (lane / 16) + u) % 16 of the
    // tile's KiB: a thread reads consecutive units of one row, which this spreads over the banks.
#pragma unroll
    for (int u = 0; u < kUT; ++u)
#pragma unroll
        for (int r = 0; r < kRT; ++r)
            *reinterpret_cast<f32x4*>(ring + ((u * kRT + r) * 64 + 16 * group + ((line + 4 * group + u) & 15)) * 16) = acc[u][r];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < Traits::kPerThread; ++p) {
        const int o = threadIdx.x + p * Traits::kThreads;
        const int uo = o % Traits::kUnits, ro = o / Traits::kUnits;
        const int unit = unit0 + uo, row = row0 + ro;
        if (o >= Traits::kOutputs || unit >= H || row >= B) continue;
        const int slot = 16 * (uo & 3) + (((ro & 15) + 4 * (uo & 3) + (uo >> 2)) & 15);
        f32x4 gate = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
            gate += *reinterpret_cast<const f32x4*>(lds + w * Traits::kWaveBytes + (((uo >> 2) * kRT + (ro >> 4)) * 64 + slot) * 16);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            gate[g] += __half2float(bias_v[p][g]);
            if constexpr (kHoisted) gate[g] += pre_v[p][g];
        }
        const float cn = detail::sigmoid_fast(gate[1]) * c_prev[p] + detail::sigmoid_fast(gate[0]) * detail::tanh_fast(gate[2]);
        c_out[size_t(row) * H + unit] = cn;
        h_out[size_t(row) * H + unit] = __float2half(detail::sigmoid_fast(gate[3]) * detail::tanh_fast(cn));
    }
}

}  // namespace tiledcuda::kernels
