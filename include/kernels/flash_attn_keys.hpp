// FlashAttention-2 forward for launches with few query blocks, O = softmax(scale · Q·Kᵀ)·V, f16 in/out, f32 statistics:
// the wavefronts of a workgroup share one block of 64 (or 32) queries and split the keys, and several workgroups may split
// the keys once more (f32 partial outputs, added by flash_attention_combine). The other tuned kernels give a
// wavefront its own queries: 64 queries against 8192 keys are then two wavefronts' work on one CU, and a head of 576
// queries three workgroups'.
//
// Design (per workgroup: 4 wavefronts, one per SIMD at head size 128, two at 64; every wavefront owns all 64 (32) queries):
//   * a wavefront streams blocks of 32 keys (every fourth of its workgroup's) through a ring of its own, two K and two V
//     blocks: no barrier between the first and the last block;
//   * Sᵀ = K·Qᵀ and Oᵀ = Vᵀ·Pᵀ with v_mfma_f32_32x32x16_f16 as in flash_attn_fwd.hpp; the rows of the K tile are read with
//     bits 2 and 3 of the row exchanged, which makes the 8 scores a lane holds per k-step those of 8 consecutive keys -
//     a column-major V is then read from LDS 16 bytes per lane, a row-major one with the transposing read;
//   * the matrix instructions of a block's output and of the next block's scores are placed one by one, each followed by
//     its share of the exponentials, sums, maxima, fragment reads and of the requests for the blocks to come: the loads
//     of K run one block ahead of those of V, so that each has a whole block's time to land;
//   * the queries go through LDS once; the four outputs meet there as well (f32, each in the place of its own ring) and
//     are added with the weights of their maxima.
// What bounds it: with few workgroups the path that brings a block to LDS (64 bytes per clock and CU: 1024 clocks for the
// four wavefronts' 64 KiB per 32 keys, as long as the matrix instructions take; 0.67 us per block of 4 x 32 keys
// measured), with all CUs busy the L2s (1.05 us); queries and keys arriving, and the merge, cost 6 us per workgroup at
// head size 128, 4 us at 64.
// Where workgroups of 64 queries leave half of the chip idle they are of 32 (kQT = 1): one 32 x 32 tile of scores per block instead of
// two, half the fragments of Q, half the merge; 4.4 us for 64 x 64 of one head instead of 6.1, 0.5 per block instead of 0.7.
// Measured (us, before -> now): 32 heads x 64 queries x 8192 keys, head size 128: 174 -> 31 (the keys and values take 27 at
// the rate of a device copy); 8 x 2048^2 at 128: 50 -> 23; 1 x 2048^2: 49 -> 16; 64 x 256 of one head, column-major V: 12.0
// -> 7.6; 32 x 1024^2 at 64: 21.4 -> 15.2.
#pragma once

#include "config.hpp"
#include "hip_utils.hpp"
#include "kernels/flash_attn_fwd.hpp"  // detail::exchange32, exp2_raw
#include "kernels/flash_attn_w64.hpp"  // detail::mfma32_out_then_load
#include "kernels/gemm_pipelined.hpp"  // detail::load_lds_16B_sbase, wait_vmcnt

namespace tiledcuda::kernels {

template <const int kD_, const bool kVColMajor_, const int kQT_ = 2>
struct FlashKeysTraits {
    static constexpr int kD = kD_;
    static constexpr bool kVColMajor = kVColMajor_;
    static constexpr int kWaves = 4, kThreads = kWaves * kWaveSize;
    static constexpr int kQT = kQT_;          // 32-query tiles of a wavefront: two, or one where that leaves CUs idle
    static constexpr int kBM = 32 * kQT;      // queries of a workgroup (every wavefront works on all of them)
    static constexpr int kBN = 32;            // keys of a block: one wavefront's step
    static constexpr int kRowBytes = 2 * kD;
    static constexpr int kTileBytes = kBN * kRowBytes;        // one K or V block
    static constexpr int kLoads = kTileBytes / 1024;          // 1 KiB direct-to-LDS instructions per block
    // Per-lane offsets of these: at head size 64 an instruction fills 8 rows of 128 bytes and both swizzles repeat every 8
    // rows, so one offset serves all of them (256 registers per lane are just enough there)
    static constexpr int kOffsets = kD == 64 ? 1 : kLoads;
    static constexpr int kDSteps = kD / 16, kDTiles = kD / 32;
    static constexpr int kWaveBytes = 4 * kTileBytes;         // two K and two V slots
    static constexpr int kRingBytes = kWaves * kWaveBytes;
    static_assert(kBM * kD * 4 <= kWaveBytes, "a wavefront's f32 output takes the place of its own ring");
    static constexpr int kQOffset = kRingBytes;                          // the workgroup's queries
    static constexpr int kStatOffset = kQOffset + kBM * kRowBytes;       // (maximum, sum) per wavefront and query
    static constexpr int kFactorOffset = kStatOffset + kWaves * kBM * 8; // weight of each wavefront's output per query
    static constexpr int kLdsBytes = kFactorOffset + kWaves * kBM * 4;
    static constexpr int kGroupsPerCu = kD == 128 ? 1 : 2;
    static constexpr bool kAgprQ = kGroupsPerCu == 1;         // Q in AGPRs: 512 registers per lane (else 256, all VGPRs)
    static_assert(kD == 128 || (kD == 64 && !kVColMajor), "head size 64 or 128");
    static constexpr int kLoadsPerSlot = 2 * kLoads / (kQT * kDSteps);  // loads behind every matrix instruction of the scores
    static_assert(kLoadsPerSlot * kQT * kDSteps == 2 * kLoads && (kLoadsPerSlot == 1 || kLoadsPerSlot == 2));

    /// XOR on the 16-byte chunk index of K row `row` (rows of 256 or 128 bytes).
    HOST_DEVICE static constexpr int k_swz(int row) { return row & (kRowBytes / 16 - 1); }
    /// XOR on the 32-byte unit index of a row-major V row.
    HOST_DEVICE static constexpr int v_swz(int row) { return kRowBytes == 256 ? ((row & 3) << 1) : (row & 2); }
    /// XOR on the 16-byte chunk index of a column-major V row (64 bytes: the 32 keys of a block).
    HOST_DEVICE static constexpr int vc_swz(int row) { return (row >> 2) & 3; }
};

namespace detail {
/// d = a · b + c (kFirst) or d += a · b in VGPRs, then a direct-to-LDS load of 16 bytes per lane (see
/// mfma32_out_then_load). kAgprB: b in AGPRs (kernels that have the whole register file of a SIMD to themselves).
template <bool kFirst, bool kAgprB>
DEVICE void mfma32_score_then_load(f32x16& d, const f16x8& a, const f16x8& b, const f32x16& c, unsigned int voff,
                                   const void* sbase, unsigned int lds_addr) {
    if constexpr (kFirst && kAgprB)
        asm volatile("s_mov_b32 m0, %6\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %3\n\tglobal_load_lds_dwordx4 %4, %5"
                     : "=&v"(d) : "v"(a), "a"(b), "v"(c), "v"(voff), "s"(sbase), "s"(lds_addr) : "m0", "memory");
    else if constexpr (kFirst)
        asm volatile("s_mov_b32 m0, %6\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %3\n\tglobal_load_lds_dwordx4 %4, %5"
                     : "=&v"(d) : "v"(a), "v"(b), "v"(c), "v"(voff), "s"(sbase), "s"(lds_addr) : "m0", "memory");
    else if constexpr (kAgprB)
        asm volatile("s_mov_b32 m0, %5\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %3, %4"
                     : "+v"(d) : "v"(a), "a"(b), "v"(voff), "s"(sbase), "s"(lds_addr) : "m0", "memory");
    else
        asm volatile("s_mov_b32 m0, %5\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %3, %4"
                     : "+v"(d) : "v"(a), "v"(b), "v"(voff), "s"(sbase), "s"(lds_addr) : "m0", "memory");
}
}  // namespace detail

/// M % kBM == 0, N % 32 == 0, 1 <= splits <= N / 32, column-major V: N < 2^24 (32-bit offsets into a head's V).
/// block = 256, dynamic LDS = Traits::kLdsBytes, grid = batch * splits * (M / kBM).
/// part (null when splits == 1): f32 [splits][batch * M][kD] outputs relative to the split's own maximum, followed by
/// [splits][batch * M] pairs (maximum in the log2 domain, sum).
template <typename Traits>
__global__ void __launch_bounds__(Traits::kThreads, Traits::kGroupsPerCu)
    flash_attention_keys(const __half* __restrict__ Q, const __half* __restrict__ K, const __half* __restrict__ V,
                         __half* __restrict__ O, float* __restrict__ part, int batch, int M, int N, int splits, float scale) {
    constexpr int kD = Traits::kD, kQT = Traits::kQT, kRowBytes = Traits::kRowBytes;
    constexpr int kChunks = kRowBytes / 16;
    extern __shared__ __align__(1024) unsigned char lds[];

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_id());
    const int q32 = lane & 31, h = lane >> 5;

    const int q_blocks = M / Traits::kBM;
    int unit, q_block;
    detail::xcd_head_block(q_blocks, batch * splits, unit, q_block);
    const int head = unit / splits, split = unit - head * splits;
    const int m0 = q_block * Traits::kBM;
    const __half* Qh = Q + (size_t(head) * M + m0) * kD;
    const __half* Kh = K + size_t(head) * N * kD;
    const __half* Vh = V + size_t(head) * N * kD;

    // this wavefront's blocks of 32 keys: every fourth of the split's
    const int blocks = N / Traits::kBN;
    const int b_first = int((long)blocks * split / splits), b_end = int((long)blocks * (split + 1) / splits);
    const int nb = (b_end - b_first - wave + Traits::kWaves - 1) / Traits::kWaves;

    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)) + wave * Traits::kWaveBytes;
    unsigned char* const ring = lds + wave * Traits::kWaveBytes;
    auto k_slot = [](int s) { return s * Traits::kTileBytes; };
    auto v_slot = [](int s) { return (2 + s) * Traits::kTileBytes; };

    // ---- global -> LDS: per-lane byte offsets of a block's load instructions (the swizzles are applied here)
    unsigned k_off[Traits::kOffsets], v_off[Traits::kOffsets];
#pragma unroll
    for (int t = 0; t < Traits::kOffsets; ++t) {
        const int row = t * (64 / kChunks) + lane / kChunks, chk = lane % kChunks;
        k_off[t] = row * kRowBytes + (chk ^ Traits::k_swz(row)) * 16;
        if constexpr (Traits::kVColMajor) {
            const int d = t * 16 + lane / 4;
            v_off[t] = unsigned(d) * (2u * N) + ((lane % 4) ^ Traits::vc_swz(d)) * 16;
        } else {
            v_off[t] = row * kRowBytes + (chk ^ (Traits::v_swz(row) << 1)) * 16;
        }
    }
    auto load_off = [](const unsigned (&off)[Traits::kOffsets], int t) { return off[t % Traits::kOffsets]; };
    auto load_base = [](const __half* base, int t) { return Traits::kOffsets == 1 ? base + t * 512 : base; };
    auto issue_k = [&](int j) {
        const __half* base = Kh + size_t(b_first + wave + j * Traits::kWaves) * (Traits::kBN * kD);
#pragma unroll
        for (int t = 0; t < Traits::kLoads; ++t) detail::load_lds_16B_sbase(load_off(k_off, t), load_base(base, t), lds0 + k_slot(j & 1) + t * 1024);
    };
    auto issue_v = [&](int j) {
        const size_t key = size_t(b_first + wave + j * Traits::kWaves) * Traits::kBN;
        const __half* base = Vh + (Traits::kVColMajor ? key : key * kD);
#pragma unroll
        for (int t = 0; t < Traits::kLoads; ++t) detail::load_lds_16B_sbase(load_off(v_off, t), load_base(base, t), lds0 + v_slot(j & 1) + t * 1024);
    };

    f32x16 o_acc[kQT][Traits::kDTiles];
#pragma unroll
    for (int t = 0; t < kQT; ++t)
#pragma unroll
        for (int dt = 0; dt < Traits::kDTiles; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o_acc[t][dt][e] = 0.f;
    float m_run[kQT], l_run[kQT];
#pragma unroll
    for (int t = 0; t < kQT; ++t) m_run[t] = -INFINITY, l_run[t] = 0.f;

    // The queries go through LDS once (as fragments from global memory every wavefront would fetch all of them in pieces
    // of 32 bytes): a quarter per wavefront, requested first, in the swizzle of the keys.
    constexpr int kQLoads = Traits::kBM * kRowBytes / 1024 / Traits::kWaves;
#pragma unroll
    for (int t = 0; t < kQLoads; ++t) {
        const int row = (wave * kQLoads + t) * (64 / kChunks) + lane / kChunks;
        detail::load_lds_16B_sbase(row * kRowBytes + ((lane % kChunks) ^ Traits::k_swz(row)) * 16, Qh,
                                   static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)) + Traits::kQOffset + (wave * kQLoads + t) * 1024);
    }
    if (nb > 0) issue_k(0);
    if (nb > 1) issue_k(1);
    if (nb > 0) issue_v(0);
    if (nb > 1) detail::lds_barrier<3 * Traits::kLoads>();  // (each branch: this wavefront's queries have landed)
    else if (nb > 0) detail::lds_barrier<2 * Traits::kLoads>();
    else detail::lds_barrier<0>();

    if (nb > 0) {
        // B operand of Sᵀ = K Qᵀ: lane (q, h) holds Q[q][16 s + 8 h .. + 7], times scale * log2(e)
        f16x8 qf[kQT][Traits::kDSteps];
        const float c = scale * 1.4426950408889634f;
#pragma unroll
        for (int t = 0; t < kQT; ++t)
#pragma unroll
            for (int s = 0; s < Traits::kDSteps; ++s) {
                const f16x8 raw = *reinterpret_cast<const f16x8*>(lds + Traits::kQOffset + (32 * t + q32) * kRowBytes +
                                                                  (((2 * s + h) ^ Traits::k_swz(q32)) * 16));
#pragma unroll
                for (int e = 0; e < 8; ++e) qf[t][s][e] = static_cast<_Float16>(__builtin_fmaf(static_cast<float>(raw[e]), c, 0.f));
            }

        // A operand of Sᵀ: row i of the tile is key pi(i), pi exchanging bits 2 and 3: a lane's accumulators 8 s .. 8 s + 7
        // are then the scores of keys 16 s + 8 h .. + 7, the k order of the second product's operands
        const int krow = (q32 & ~12) | ((q32 & 4) << 1) | ((q32 & 8) >> 1);
        const unsigned char* k_addr = ring + krow * kRowBytes;
        const int k_chunk = h ^ Traits::k_swz(krow);
        // A operand of Oᵀ = Vᵀ Pᵀ
        const int g = lane >> 4, L = lane & 15;
        const int vrow = 8 * h + (L >> 2);                      // row-major: rows 16 s + 4 part + vrow through the transposing read
        const int vcol_b = (16 * (g & 1) + 4 * (L & 3)) * 2;
        const int vunit_swz = Traits::v_swz(vrow);

        auto k_frag = [&](int slot, int s) {
            return *reinterpret_cast<const f16x8*>(k_addr + k_slot(slot) + ((k_chunk ^ (2 * s)) * 16));
        };
        auto v_frag = [&](int slot, int dt, int s) {
            f16x8 vf;
            if constexpr (Traits::kVColMajor) {
                const int d = 32 * dt + q32;
                vf = *reinterpret_cast<const f16x8*>(ring + v_slot(slot) + d * 64 + (((2 * s + h) ^ Traits::vc_swz(d)) * 16));
            } else {
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int row = 16 * s + 4 * p + vrow;
                    const int byte_in_row = 64 * dt + vcol_b;
                    const int u = (byte_in_row >> 5) ^ vunit_swz;
                    using fp16x4 = __fp16 __attribute__((ext_vector_type(4)));
                    const fp16x4 v4 = __builtin_amdgcn_ds_read_tr16_b64_v4f16((fp16x4 __attribute__((address_space(3)))*)(
                        ring + v_slot(slot) + row * kRowBytes + u * 32 + (byte_in_row & 31)));
#pragma unroll
                    for (int e = 0; e < 4; ++e) vf[4 * p + e] = static_cast<_Float16>(v4[e]);
                }
            }
            return vf;
        };

#pragma unroll
        for (int t = 0; t < kQT; ++t)
#pragma unroll
            for (int sd = 0; sd < Traits::kDSteps; ++sd)
                if constexpr (Traits::kAgprQ) asm volatile("" : "+a"(qf[t][sd]));
                else asm volatile("" : "+v"(qf[t][sd]));

        f32x16 s_a[kQT], s_b[kQT];
        f32x16 m_init[kQT];  // -m_run in every element: what the accumulators of the scores start at

        // block 0: exact maximum
        if (nb > 1) detail::wait_vmcnt<2 * Traits::kLoads>();
        else detail::wait_vmcnt<Traits::kLoads>();
#pragma unroll
        for (int t = 0; t < kQT; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) s_a[t][e] = 0.f;
#pragma unroll
        for (int s = 0; s < Traits::kDSteps; ++s) {
            const f16x8 kf = k_frag(0, s);
#pragma unroll
            for (int t = 0; t < kQT; ++t) s_a[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[t][s], s_a[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < kQT; ++t) {
            float mx = s_a[t][0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s_a[t][e]);
            m_run[t] = fmaxf(mx, detail::exchange32(mx));
        }
        // Every score of block 0 may be -infinity (keys masked by an infinite feature; any of 4 * splits blocks of the sequence
        // is some wavefront's block 0): then the exact maximum of this wavefront's first block with another score, its keys
        // read once more, is where the query starts. A query without any starts at 0 and keeps a sum of 0.
        auto any_masked = [&]() {
            bool masked = false;
#pragma unroll
            for (int t = 0; t < kQT; ++t) masked = masked || m_run[t] == -INFINITY;
            return __any(masked);
        };
        if (__builtin_expect(any_masked(), 0)) {
            for (int j = 1; j < nb; ++j) {
                const __half* k_row = Kh + (size_t(b_first + wave + j * Traits::kWaves) * Traits::kBN + krow) * kD + 8 * h;
#pragma unroll
                for (int t = 0; t < kQT; ++t) {
                    f32x16 sc;
#pragma unroll
                    for (int e = 0; e < 16; ++e) sc[e] = 0.f;
#pragma unroll
                    for (int s = 0; s < Traits::kDSteps; ++s)
                        sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8*>(k_row + 16 * s), qf[t][s], sc, 0, 0, 0);
                    float mx = sc[0];
#pragma unroll
                    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, sc[e]);
                    mx = fmaxf(mx, detail::exchange32(mx));
                    if (m_run[t] == -INFINITY) m_run[t] = mx;
                }
                if (!any_masked()) break;
            }
#pragma unroll
            for (int t = 0; t < kQT; ++t)
                if (m_run[t] == -INFINITY) m_run[t] = 0.f;
        }
#pragma unroll
        for (int t = 0; t < kQT; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) s_a[t][e] -= m_run[t], m_init[t][e] = -m_run[t];

        constexpr float kLazy = 8.0f;  // a maximum moves only when a block exceeds it by 2^8 (p stays inside f16)
        // One block: the matrix instructions of the next block's scores (the first kQkSlots slots) and of this block's
        // output, each followed by its share of the exponentials, sums and maxima, in this order (sched_barrier).
        constexpr int kQkSlots = kQT * Traits::kDSteps, kPvHalf = kQT * Traits::kDTiles, kSlots = kQkSlots + 2 * kPvHalf;
        auto step = [&](int j, auto has_next, f32x16 (&s_cur)[kQT], f32x16 (&s_nxt)[kQT]) {
            constexpr bool kNext = decltype(has_next)::value;
            // K of block j + 1 (requested before V of block j) has landed; the reads of the slots about to be refilled are done
            if constexpr (kNext) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(Traits::kLoads) : "memory");
            // (the last block's keys are requested again where there is no block j + 2: every step then issues the same loads)
            const __half* k_base = Kh + size_t(b_first + wave + min(j + 2, nb - 1) * Traits::kWaves) * (Traits::kBN * kD);
            const size_t v_key = size_t(b_first + wave + (j + 1) * Traits::kWaves) * Traits::kBN;
            const __half* v_base = Vh + (Traits::kVColMajor ? v_key : v_key * kD);
            f16x8 kf[3], vf[3], pf[kQT][2];
            float mx[kQT];
            if constexpr (kNext) {
                kf[0] = k_frag((j + 1) & 1, 0);
                kf[1] = k_frag((j + 1) & 1, 1);
            }
            constexpr int kFirst = kNext ? 0 : kQkSlots;
            constexpr int kExps = 16 * kQT, kHalf = 8 * kQT;
            auto exp_slot = [](int n) constexpr {  // the slot that exponential n (of kExps) is computed in
                return n < kHalf ? n * (kQkSlots - 1) / kHalf : kQkSlots - 1 + (n - kHalf) * (kPvHalf - 1) / kHalf;
            };
            auto exps = [&](auto n_) {
                constexpr int n = n_, s = n / kHalf, t = (n / 2) % kQT, e = 8 * s + (n % kHalf) / (2 * kQT) * 2 + n % 2;
                const float p = detail::exp2_raw(s_cur[t][e]);
                l_run[t] += p;
                pf[t][s][e % 8] = static_cast<_Float16>(p);
            };
            if constexpr (!kNext) {
                detail::static_for<kExps>([&](auto n) { exps(n); });
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                vf[0] = v_frag(j & 1, 0, 0);
                vf[1] = v_frag(j & 1, 1, 0);
            }
            detail::static_for<kSlots - kFirst>([&](auto i_) {
                constexpr int i = i_ + kFirst;
                if constexpr (i < kQkSlots) {
                    constexpr int s = i / kQT, t = i % kQT;
                    if constexpr (t == 0 && s + 2 < Traits::kDSteps) kf[(s + 2) % 3] = k_frag((j + 1) & 1, s + 2);
                    // with K of block j + 2, then V of block j + 1 requested behind the instruction
                    constexpr int kPer = Traits::kLoadsPerSlot;
                    constexpr bool kOfK = i * kPer < Traits::kLoads;
                    constexpr int l = kOfK ? i * kPer : i * kPer - Traits::kLoads;
                    const unsigned off = load_off(kOfK ? k_off : v_off, l);
                    const unsigned dst = lds0 + (kOfK ? k_slot(j & 1) : v_slot((j + 1) & 1)) + l * 1024;
                    detail::mfma32_score_then_load<s == 0, Traits::kAgprQ>(s_nxt[t], kf[s % 3], qf[t][s], m_init[t], off,
                                                                           load_base(kOfK ? k_base : v_base, l), dst);
                    if constexpr (kPer == 2)
                        detail::load_lds_16B_sbase(load_off(kOfK ? k_off : v_off, l + 1), load_base(kOfK ? k_base : v_base, l + 1), dst + 1024);
                } else {
                    constexpr int f = (i - kQkSlots) / kQT, t = i % kQT, s = f / Traits::kDTiles, dt = f % Traits::kDTiles;
                    constexpr int fn = f + 2;
                    if constexpr (t == 0 && fn < 2 * Traits::kDTiles)
                        vf[fn % 3] = v_frag(j & 1, fn % Traits::kDTiles, fn / Traits::kDTiles);
                    o_acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[f % 3], pf[t][s], o_acc[t][dt], 0, 0, 0);
                }
                if constexpr (kNext) {
                    detail::static_for<kExps>([&](auto n) {
                        if constexpr (exp_slot(n) == i) exps(n);
                    });
                    if constexpr (i == kQkSlots - 3) {
                        // V of block j has landed: only this step's own loads, those of i + 1 slots, are younger
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((i + 1) * Traits::kLoadsPerSlot) : "memory");
                        vf[0] = v_frag(j & 1, 0, 0);
                        vf[1] = v_frag(j & 1, 1, 0);
                    }
                    constexpr int r = i - kQkSlots - 2;  // maxima of the next block's scores (written by instructions three slots back or more)
                    if constexpr (r >= 0) {
                        constexpr int kPer = (kExps + (kSlots - kQkSlots - 2) - 1) / (kSlots - kQkSlots - 2);
                        detail::static_for<kPer>([&](auto u) {
                            constexpr int n = r * kPer + u;
                            if constexpr (n < kExps) {
                                constexpr int t = n / 16, e = n % 16;
                                mx[t] = e == 0 ? s_nxt[t][0] : fmaxf(mx[t], s_nxt[t][e]);
                            }
                        });
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (kNext) {
                if (__any((kQT == 2 ? fmaxf(mx[0], mx[kQT - 1]) : mx[0]) > kLazy)) {
#pragma unroll
                    for (int t = 0; t < kQT; ++t) {
                        const float mxq = fmaxf(mx[t], detail::exchange32(mx[t]));
                        const float up = mxq > kLazy ? mxq : 0.f;
                        const float alpha = detail::exp2_raw(-up);
                        m_run[t] += up;
                        l_run[t] *= alpha;
#pragma unroll
                        for (int e = 0; e < 16; ++e) s_nxt[t][e] -= up, m_init[t][e] = -m_run[t];
#pragma unroll
                        for (int dt = 0; dt < Traits::kDTiles; ++dt)
#pragma unroll
                            for (int e = 0; e < 16; ++e) o_acc[t][dt][e] *= alpha;
                    }
                }
            }
        };
        int j = 0;
        for (; j + 2 < nb; j += 2) {
            step(j, std::true_type{}, s_a, s_b);
            step(j + 1, std::true_type{}, s_b, s_a);
        }
        if (j + 1 < nb) {
            step(j, std::true_type{}, s_a, s_b);
#pragma unroll
            for (int t = 0; t < kQT; ++t) s_a[t] = s_b[t];
            ++j;
        }
        step(j, std::false_type{}, s_a, s_b);
    }

    // ---- merge the four wavefronts' outputs: each leaves its sums as they are in the place of its own ring
    // ([query][d] f32, 16-byte slots XOR-ed with the query), then the weights of the four are worked out, then applied
    float2* stat = reinterpret_cast<float2*>(lds + Traits::kStatOffset);
    float* factor = reinterpret_cast<float*>(lds + Traits::kFactorOffset);
    const size_t rows = size_t(batch) * M, row0 = size_t(head) * M + m0;
#pragma unroll
    for (int t = 0; t < kQT; ++t) {
        const float l = l_run[t] + detail::exchange32(l_run[t]);
        // (a sum of 0: no key, or none but masked ones; its weight below is 0)
        if (h == 0) stat[wave * Traits::kBM + 32 * t + q32] = make_float2(l == 0.f ? -INFINITY : m_run[t], l);
        unsigned char* dst = ring + (32 * t + q32) * (kD * 4);
#pragma unroll
        for (int dt = 0; dt < Traits::kDTiles; ++dt)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const int slot = (8 * dt + 2 * qd + h) ^ (q32 & (kD / 4 - 1));
                *reinterpret_cast<f32x4*>(dst + slot * 16) = f32x4{o_acc[t][dt][4 * qd], o_acc[t][dt][4 * qd + 1], o_acc[t][dt][4 * qd + 2], o_acc[t][dt][4 * qd + 3]};
            }
    }
    detail::lds_barrier<0>();
    static_assert(Traits::kThreads % (Traits::kBM * Traits::kWaves) == 0 && (Traits::kBM * Traits::kWaves) % kWaveSize == 0);
    if (threadIdx.x < Traits::kBM * Traits::kWaves) {
        const int q = threadIdx.x / 4, w = threadIdx.x % 4;
        const float2 ml = stat[w * Traits::kBM + q];
        float mm = fmaxf(ml.x, __shfl_xor(ml.x, 1, 4));
        mm = fmaxf(mm, __shfl_xor(mm, 2, 4));
        float f = detail::exp2_raw(ml.x - (mm == -INFINITY ? 0.f : mm));
        float ll = ml.y * f;
        ll += __shfl_xor(ll, 1, 4);
        ll += __shfl_xor(ll, 2, 4);
        if (splits == 1) f /= ll;
        else if (w == 0) reinterpret_cast<float2*>(part + splits * rows * kD)[split * rows + row0 + q] = make_float2(mm, ll);
        factor[threadIdx.x] = f;
    }
    detail::lds_barrier<63>();
    constexpr int kSlots = kD / 4;
#pragma unroll
    for (int i = threadIdx.x; i < Traits::kBM * kSlots; i += Traits::kThreads) {
        const int q = i / kSlots, slot = i % kSlots;
        const f32x4 f = *reinterpret_cast<const f32x4*>(factor + 4 * q);
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < Traits::kWaves; ++w)
            sum += f[w] * *reinterpret_cast<const f32x4*>(lds + w * Traits::kWaveBytes + q * (kD * 4) + ((slot ^ (q & 31 & (kSlots - 1))) * 16));
        if (splits == 1) {
            f16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = static_cast<_Float16>(sum[e]);
            *reinterpret_cast<f16x4*>(O + (row0 + q) * kD + slot * 4) = o;
        } else {
            __builtin_nontemporal_store(sum, reinterpret_cast<f32x4*>(part + (split * rows + row0 + q) * kD + slot * 4));
        }
    }
}

/// O = the partial outputs of flash_attention_keys added with the weights of their maxima. One thread per 4 elements; all
/// of its loads are requested before the first is used (splits <= kMax).
template <int kD, int kMax>
__global__ void __launch_bounds__(256)
    flash_attention_combine(const float* __restrict__ part, __half* __restrict__ O, size_t rows, int splits) {
    constexpr int kSlots = kD / 4;
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    const size_t row = i / kSlots;
    const int slot = i % kSlots;
    if (row >= rows) return;
    const float2* stat = reinterpret_cast<const float2*>(part + splits * rows * kD);
    float2 ml[kMax];
    f32x4 v[kMax];
#pragma unroll
    for (int s = 0; s < kMax; ++s) ml[s] = stat[min(s, splits - 1) * rows + row];
#pragma unroll
    for (int s = 0; s < kMax; ++s)
        v[s] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(part + (min(s, splits - 1) * rows + row) * kD + slot * 4));
    float mm = ml[0].x;
#pragma unroll
    for (int s = 1; s < kMax; ++s) mm = fmaxf(mm, ml[s].x);
    if (mm == -INFINITY) mm = 0.f;
    float ll = 0.f;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < kMax; ++s) {
        const float f = s < splits ? detail::exp2_raw(ml[s].x - mm) : 0.f;
        ll += ml[s].y * f;
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += (s < splits ? v[s][e] : 0.f) * f;  // (a value may be infinite)
    }
    const float inv = 1.f / ll;
    f16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = static_cast<_Float16>(sum[e] * inv);
    *reinterpret_cast<f16x4*>(O + row * kD + slot * 4) = o;
}

}  // namespace tiledcuda::kernels
