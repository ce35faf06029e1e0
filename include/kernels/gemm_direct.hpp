// fp16 GEMM for gfx950 for products with few output tiles: C[M, N] = A[M, K] . B, A row-major, B column-major (stored [N, K]),
// f32 accumulate, C row-major f16 or f32; any M, N, K in multiples of 16. (The reference has compile-time shapes only:
// examples/cpp/01_gemm/01_gemm_global_reg/gemm.hpp:52-81.)
//
// What bounds such a product is how fast operands reach the CUs that work on it, and the launch: hence
//   * tiles of 16 to 64 columns x 16 to 64 rows of C, chosen by the launcher so that the workgroups fill the CUs once and
//     fetch as few rows of operands as possible;
//   * the 8 wavefronts of a workgroup split K in chunks of 64 (128-byte lines): each brings its own chunks to LDS and has
//     up to four of them in flight in a ring of its own, so nothing waits for a barrier before the partial sums are added;
//   * those meet in LDS, where each thread adds four consecutive outputs.
// Measured in a graph, us, before -> now (others, split-K ones among them -> this kernel): 128 x 64 x 256: 3.1 -> 2.3 (1 x 1 tiles
// of 16); 32 x 4096 x 4096: 18.1 -> 10.5 (1 x 2; 34 MB from memory take 6.5); 64 x 4096 x 4096: 18.9 -> 11.9 (2 x 2);
// 128 x 4096 x 4096: 20.3 -> 15.3 (2 x 4); 256 x 256 x 8192: 18.1 -> 8.9 (1 x 1); 512 x 1024 x 1024: 6.4 -> 5.1 (2 x 4). Loads of
// a full chip arrive at 70 to 100 KB per us and CU.
#pragma once

#include "config.hpp"
#include "hip_utils.hpp"
#include "kernels/flash_attn_fwd.hpp"  // detail::xcd_head_block
#include "kernels/gemm_w128.hpp"       // detail::load_lds_16B_sbase

namespace tiledcuda::kernels {

/// kUT: 16-column tiles of C (rows of the stored B) and kRT: 16-row tiles of C per workgroup.
template <const int kUT_, const int kRT_>
struct GemmDirectTraits {
    static constexpr int kUT = kUT_, kRT = kRT_;
    static constexpr int kBN = 16 * kUT, kBM = 16 * kRT;
    static constexpr int kWaves = 8, kThreads = kWaves * kWaveSize;
    static constexpr int kBK = 64;
    static constexpr int kLoads = 2 * (kUT + kRT);  // 1 KiB direct-to-LDS instructions (8 rows) per chunk
    static constexpr int kRing = kLoads >= 12 ? 1 : kLoads >= 8 ? 2 : kLoads == 6 ? 3 : 4;  // chunks in flight per wavefront
    static constexpr int kWaveBytes = kRing * kLoads * 1024;
    static constexpr int kLdsBytes = kWaves * kWaveBytes;
    static constexpr int kTiles = kUT * kRT;
    static constexpr int kQuads = kTiles * 64;      // outputs in groups of four
    static_assert(kTiles * 1024 <= kWaveBytes, "a wavefront's sums take the place of its chunks");
    static_assert(kLdsBytes <= kMaxLdsBytes);
};

/// grid = ceil(N / kBN) * ceil(M / kBM), block = 512, dynamic LDS = T::kLdsBytes. M, N, K multiples of 16, K < 2^24 (32-bit
/// byte offsets inside a tile's rows). kSide: B's stored rows are side_ldb < 2^24 elements apart (else K), and the first workgroup
/// sets zero_count device words at zero_words to zero on the side (for others these would cost up to 0.1 us of 2.4).
template <typename T, typename OutType, bool kSide = false>
__global__ void __launch_bounds__(T::kThreads)
    gemm_direct(const __half* __restrict__ A, const __half* __restrict__ Bt, OutType* __restrict__ C, int M, int N, int K, int side_ldb,
                unsigned int* __restrict__ zero_words, int zero_count) {
    const int ldb = kSide ? side_ldb : K;
    constexpr int kUT = T::kUT, kRT = T::kRT, kRing = T::kRing, kBK = T::kBK, kWaves = T::kWaves;
    extern __shared__ __align__(1024) unsigned char lds[];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_id());
    const int line = lane & 15, group = lane >> 4;
    if constexpr (kSide) {
        if (blockIdx.x == 0)
            for (int i = threadIdx.x; i < zero_count; i += T::kThreads) zero_words[i] = 0u;
    }

    // The blocks that share rows of the larger operand run on one XCD: these rows come to one L2 only. (With the row blocks of
    // one column block together whatever M and N: 4096 x 256 x 8192 41.4 us, 2048 x 256 x 8192 40.0, 8192 x 64 x 4096 21.1; in
    // this order 25.9, 18.8, 13.7.)
    const int m_blocks = (M + T::kBM - 1) / T::kBM, n_blocks = (N + T::kBN - 1) / T::kBN;
    const bool tall = M > N;
    int larger, smaller;
    detail::xcd_head_block(tall ? n_blocks : m_blocks, tall ? m_blocks : n_blocks, larger, smaller);
    const int n0 = (tall ? smaller : larger) * T::kBN, m0 = (tall ? larger : smaller) * T::kBM;
    const __half* const b_rows = Bt + size_t(n0) * ldb;
    const __half* const a_rows = A + size_t(m0) * K;

    // ---- global -> LDS: instruction q of a chunk fills 8 rows of 128 bytes, those of B before those of A (rows beyond the
    // matrix: its last one); physical 16-byte piece p of row r holds logical piece p ^ (r / 2) % 8
    const int lrow = lane >> 3;
    unsigned b_off[2 * kUT], a_off[2 * kRT];
#pragma unroll
    for (int q = 0; q < 2 * kUT; ++q) b_off[q] = min(8 * q + lrow, N - 1 - n0) * (2u * ldb);
#pragma unroll
    for (int q = 0; q < 2 * kRT; ++q) a_off[q] = min(8 * q + lrow, M - 1 - m0) * (2u * K);
    unsigned piece[2];  // for even and odd instructions
#pragma unroll
    for (int o = 0; o < 2; ++o) piece[o] = (lane & 7) ^ (4 * o + (lrow >> 1));
    // the wavefronts take the chunks in turn; pieces beyond a partial last one are fetched from the row's first piece of it and
    // zeroed before the product
    const int total = (K + kBK - 1) / kBK, n = (total - wave + kWaves - 1) / kWaves;
    unsigned char* const ring = lds + wave * T::kWaveBytes;
    const unsigned ring0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(ring));
    auto issue = [&](int i) {
        const int k = kBK * (wave + kWaves * i);
        const unsigned valid = min(K - k, kBK) / 8;
        const unsigned dst = ring0 + (i % kRing) * T::kLoads * 1024;
        unsigned off[2];
#pragma unroll
        for (int o = 0; o < 2; ++o) off[o] = piece[o] < valid ? 16 * piece[o] : 0;
#pragma unroll
        for (int q = 0; q < 2 * kUT; ++q) detail::load_lds_16B_sbase(b_off[q] + off[q & 1], b_rows + k, dst + q * 1024);
#pragma unroll
        for (int q = 0; q < 2 * kRT; ++q) detail::load_lds_16B_sbase(a_off[q] + off[q & 1], a_rows + k, dst + (2 * kUT + q) * 1024);
    };
#pragma unroll
    for (int i = 0; i < kRing; ++i)
        if (i < n) issue(i);

    f32x4 acc[kUT][kRT];
#pragma unroll
    for (int u = 0; u < kUT; ++u)
#pragma unroll
        for (int r = 0; r < kRT; ++r) acc[u][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < n; ++i) {
        // chunk i has landed; as many of the chunks behind it as were issued may still be on their way
        const int behind = min(n - 1 - i, kRing - 1);
        if (kRing >= 4 && behind >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kRing >= 4 ? 3 * T::kLoads : 0) : "memory");
        else if (kRing >= 3 && behind == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kRing >= 3 ? 2 * T::kLoads : 0) : "memory");
        else if (kRing >= 2 && behind == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kRing >= 2 ? T::kLoads : 0) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned char* src = ring + (i % kRing) * T::kLoads * 1024;
        f16x8 bf[2][kUT], af[2][kRT];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int off = line * 128 + (((4 * s + group) ^ (line >> 1)) * 16);
#pragma unroll
            for (int u = 0; u < kUT; ++u) bf[s][u] = *reinterpret_cast<const f16x8*>(src + u * 2048 + off);
#pragma unroll
            for (int r = 0; r < kRT; ++r) af[s][r] = *reinterpret_cast<const f16x8*>(src + (kUT + r) * 2048 + off);
        }
        if (i + kRing < n) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the fragments have left the slot about to be refilled
            issue(i + kRing);
        }
        const int cols = K - kBK * (wave + kWaves * i);
        if (cols < kBK) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (32 * s + 8 * group >= cols) {
#pragma unroll
                    for (int u = 0; u < kUT; ++u) bf[s][u] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                    for (int r = 0; r < kRT; ++r) af[s][r] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
                }
        }
        // a chunk's sum is added to the total as a whole: the error of the sums stays that of short chains (256 x 256 x 8192: 1.1e-7; 2.1e-7
        // with one chain per wavefront, as fast to within 2 %)
#pragma unroll
        for (int u = 0; u < kUT; ++u)
#pragma unroll
            for (int r = 0; r < kRT; ++r) {
                f32x4 part = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[0][u], af[0][r], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[1][u], af[1][r], part, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[u][r][e] += part[e];
            }
    }

    // ---- add the eight wavefronts' sums through LDS. A lane's accumulator holds columns 16 u + 4 (lane / 16) .. + 3 of row
    // 16 r + lane % 16; its 16 bytes go to slot 16 (lane / 16) + (lane % 16 + 4 (lane / 16) + u) % 16 of the tile's KiB: a
    // thread reads consecutive columns of one row, which this spreads over the banks.
#pragma unroll
    for (int u = 0; u < kUT; ++u)
#pragma unroll
        for (int r = 0; r < kRT; ++r)
            *reinterpret_cast<f32x4*>(ring + ((u * kRT + r) * 64 + 16 * group + ((line + 4 * group + u) & 15)) * 16) = acc[u][r];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < (T::kQuads + T::kThreads - 1) / T::kThreads; ++p) {
        const int o = threadIdx.x + p * T::kThreads;
        const int quad = o % (4 * kUT), m = o / (4 * kUT), g = quad & 3, u = quad >> 2;
        const int row = m0 + m, col = n0 + 4 * quad;
        if (o >= T::kQuads || row >= M || col >= N) continue;
        const int slot = (u * kRT + (m >> 4)) * 64 + 16 * g + (((m & 15) + 4 * g + u) & 15);
        f32x4 sum = *reinterpret_cast<const f32x4*>(lds + slot * 16);
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(lds + w * T::kWaveBytes + slot * 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += v[e];
        }
        OutType* dst = C + size_t(row) * N + col;
        if constexpr (sizeof(OutType) == 2) {
            f16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(sum[e]);
            *reinterpret_cast<f16x4*>(dst) = h;
        } else {
            *reinterpret_cast<f32x4*>(dst) = sum;
        }
    }
}

}  // namespace tiledcuda::kernels
