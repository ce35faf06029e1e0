// Back-to-back GEMM D = f16(A·B)·C for gfx950 with long N and many rows: same contract as kernels/b2b_gemm_fwd.hpp
// (A [M, K] and D [M, P] row-major, B stored [N, K], C stored [P, N], K = P = 128; the reference's example runs N = 1024 and
// 2048, examples/cpp/02_fused_two_gemms/fused_gemm.cu:236-259).
//
// What bounds the kernel with 32 rows per workgroup is that every workgroup streams all of B and C through its CU: 512 N bytes
// for 32 rows. Here a workgroup takes 128 or 256 rows and the weights pass once for all of them:
//   * blocks of 64 columns of B and of C (16 KiB each) go through a ring of four in LDS, three in flight, one barrier per
//     block;
//   * a wavefront owns 32 rows outright: their A fragments stay in registers, and the first product's accumulators,
//     rounded to f16 (part of the specification of this operation), are the second product's operand without leaving the
//     lane: a lane holds n = 4 g .. + 3 of two adjacent 16-wide tiles, which are declared to be the 8 contraction slots of
//     lane group g; fragments of C are read in the same order (two 8-byte reads).
// What is left is the LDS: every wavefront reads the whole block, 32 KiB for 64 matrix instructions: 1.6 us per block with 8
// wavefronts, where LDS and matrix pipes need 0.85 each (requesting the fragments a product ahead changed nothing).
// Kernel with 32 rows per workgroup -> this one with 8 wavefronts, us: 65536 x 1024: 69.0 -> 35.0; 5 x 8128 x 2048: 82.5 -> 57.3;
// 16 x 2112 x 512: 27.3 -> 19.2; with 4 wavefronts 16 x 1600 x 1024: 33.6 -> 27.0. 16384 x 512 stays: 10.8 against 13.9.
#pragma once

#include "config.hpp"
#include "hip_utils.hpp"
#include "kernels/flash_attn_fwd.hpp"  // detail::xcd_head_block
#include "kernels/gemm_w128.hpp"       // detail::load_lds_16B_sbase

namespace tiledcuda::kernels {

/// kMT: 16-row tiles of a wavefront.
template <const int kWaves_, const int kMT_>
struct B2bStreamTraits {
    static constexpr int kK = 128, kP = 128, kBN = 64;
    static constexpr int kWaves = kWaves_, kThreads = kWaves * kWaveSize, kMT = kMT_;
    static constexpr int kTM = kWaves * kMT * 16;
    static constexpr int kStageBytes = 2 * kBN * kK * 2;  // B's rows of 256 bytes, then C's 128 rows of 128 bytes
    static constexpr int kStages = 4;
    static constexpr int kLoads = kStageBytes / 1024 / kWaves;  // per wavefront and stage, the first half of them B
    static constexpr int kLdsBytes = kStages * kStageBytes;     // 128 KiB; the output tile passes through it at the end
    static_assert(kWaves * 16 * kP * 4 <= kLdsBytes && kLoads % 2 == 0);
};

/// grid = ceil(M / kTM) * batch, block = T::kThreads, dynamic LDS = T::kLdsBytes. M % 16 == 0, N % 64 == 0, N >= 256,
/// N < 2^23 (32-bit byte offsets inside a block of C).
template <typename T, typename OutType>
__global__ void __launch_bounds__(T::kThreads)
    b2b_gemm_stream(const __half* __restrict__ A, const __half* __restrict__ B, const __half* __restrict__ C,
                    OutType* __restrict__ D, int M, int N, int batch) {
    constexpr int kK = T::kK, kP = T::kP, kMT = T::kMT, kStages = T::kStages, kHalf = T::kLoads / 2;
    extern __shared__ __align__(1024) unsigned char lds[];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_id());
    const int L = lane & 15, g = lane >> 4;
    int item, m_block;  // the workgroups of one batch item run on one XCD: they share its weights in the L2
    detail::xcd_head_block((M + T::kTM - 1) / T::kTM, batch, item, m_block);
    const int m0 = m_block * T::kTM + wave * 16 * kMT;  // (a wavefront beyond M works on the last row and stores nothing)
    const __half* Ab = A + size_t(item) * M * kK;
    const __half* Bb = B + size_t(item) * N * kK;
    const __half* Cb = C + size_t(item) * kP * N;

    f16x8 fa[kMT][kK / 32];
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
        for (int s = 0; s < kK / 32; ++s)
            fa[mt][s] = *reinterpret_cast<const f16x8*>(Ab + size_t(min(m0 + 16 * mt + L, M - 1)) * kK + 32 * s + 8 * g);

    // ---- global -> LDS. B: 4 rows of 256 bytes per instruction, physical 16-byte piece p of row r holds logical piece
    // p ^ r % 16; C: 8 rows of 128 bytes, piece p ^ (r / 2) % 8
    unsigned b_off[kHalf], c_off[kHalf];
#pragma unroll
    for (int j = 0; j < kHalf; ++j) {
        const int q = kHalf * wave + j, br = 4 * q + (lane >> 4), cr = 8 * q + (lane >> 3);
        b_off[j] = br * 256 + ((lane & 15) ^ (br & 15)) * 16;
        c_off[j] = unsigned(cr) * (2u * N) + ((lane & 7) ^ ((cr >> 1) & 7)) * 16;
    }
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds));
    auto issue = [&](int i) {
        const unsigned dst = lds0 + (i % kStages) * T::kStageBytes + kHalf * wave * 1024;
        const __half* b = Bb + size_t(i) * T::kBN * kK;
        const __half* c = Cb + size_t(i) * T::kBN;
#pragma unroll
        for (int j = 0; j < kHalf; ++j) detail::load_lds_16B_sbase(b_off[j], b, dst + j * 1024);
#pragma unroll
        for (int j = 0; j < kHalf; ++j) detail::load_lds_16B_sbase(c_off[j], c, dst + T::kStageBytes / 2 + j * 1024);
    };
    const int blocks = N / T::kBN;
#pragma unroll
    for (int i = 0; i < kStages - 1; ++i) issue(i);  // N >= 256: they exist

    f32x4 acc[kP / 16][kMT];
#pragma unroll
    for (int p = 0; p < kP / 16; ++p)
#pragma unroll
        for (int mt = 0; mt < kMT; ++mt) acc[p][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < blocks; ++i) {
        // this wavefront's share of block i has landed (the one or two behind it may be on their way), then everyone's; everyone
        // is done with block i - 1, whose slot the next loads go to
        const int behind = min(blocks - 1 - i, kStages - 2);
        if (behind == 2) detail::lds_barrier<2 * T::kLoads>();
        else if (behind == 1) detail::lds_barrier<T::kLoads>();
        else detail::lds_barrier<0>();
        if (i + kStages - 1 < blocks) issue(i + kStages - 1);
        const unsigned char* bs = lds + (i % kStages) * T::kStageBytes;
        const unsigned char* cs = bs + T::kStageBytes / 2;
#pragma unroll
        for (int h = 0; h < T::kBN / 32; ++h) {  // 32 columns of B: 32 contraction slots of the second product
            f32x4 s[2][kMT];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int mt = 0; mt < kMT; ++mt) s[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < kK / 32; ++k)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int n = 32 * h + 16 * t + L;
                    const f16x8 fb = *reinterpret_cast<const f16x8*>(bs + n * 256 + ((4 * k + g) ^ L) * 16);
#pragma unroll
                    for (int mt = 0; mt < kMT; ++mt) s[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb, fa[mt][k], s[t][mt], 0, 0, 0);
                }
            f16x8 fs[kMT];
#pragma unroll
            for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
                for (int e = 0; e < 8; ++e) fs[mt][e] = static_cast<_Float16>(s[e >> 2][mt][e & 3]);
#pragma unroll
            for (int p = 0; p < kP / 16; ++p) {
                const unsigned char* row = cs + (16 * p + L) * 128 + (g & 1) * 8;
                const f16x4 lo = *reinterpret_cast<const f16x4*>(row + ((4 * h + (g >> 1)) ^ (L >> 1)) * 16);
                const f16x4 hi = *reinterpret_cast<const f16x4*>(row + ((4 * h + 2 + (g >> 1)) ^ (L >> 1)) * 16);
                const f16x8 fc = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int mt = 0; mt < kMT; ++mt) acc[p][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fc, fs[mt], acc[p][mt], 0, 0, 0);
            }
        }
    }

    // ---- acc[p][mt][e] = D[m0 + 16 mt + L][16 p + 4 g + e]: 16 rows at a time through 8 KiB of LDS of the wavefront's own, out in
    // whole rows. Slots of four outputs are XOR-ed with twice the row (f16: pairs of slots stay pairs) or the row (f32).
    __syncthreads();  // everyone is done with the last block
    constexpr int kPitch = kP * sizeof(OutType), kSlot = 4 * sizeof(OutType), kPieces = kPitch / 16;
    unsigned char* stage = lds + wave * 16 * kP * 4;
    auto slot_of = [](int row, int slot) { return sizeof(OutType) == 2 ? slot ^ ((2 * row) & 31) : slot ^ row; };
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt) {
#pragma unroll
        for (int p = 0; p < kP / 16; ++p) {
            unsigned char* dst = stage + L * kPitch + slot_of(L, 4 * p + g) * kSlot;
            if constexpr (sizeof(OutType) == 2) {
                f16x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = static_cast<_Float16>(acc[p][mt][e]);
                *reinterpret_cast<f16x4*>(dst) = v;
            } else {
                *reinterpret_cast<f32x4*>(dst) = acc[p][mt];
            }
        }
        // (LDS operations of one wavefront execute in order: the reads see the writes above)
#pragma unroll
        for (int it = 0; it < 16 * kPieces / kWaveSize; ++it) {
            const int piece = it * kWaveSize + lane, row = piece / kPieces, c = piece % kPieces;
            const int slot = sizeof(OutType) == 2 ? 2 * c : c;
            const u32x4 v = *reinterpret_cast<const u32x4*>(stage + row * kPitch + slot_of(row, slot) * kSlot);
            if (m0 + 16 * mt + row < M)
                __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(D + (size_t(item) * M + m0 + 16 * mt + row) * kP + c * (16 / sizeof(OutType))));
        }
    }
}

}  // namespace tiledcuda::kernels
