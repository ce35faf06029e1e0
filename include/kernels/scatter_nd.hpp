// scatter_nd for gfx950: data[indices[i, 0], ..., indices[i, k-1], :] (=|+=) updates[i, :] for i in [0, n).
// The reference's kernel (src/kernels/scatter_nd.cu:25-55) runs one thread per index row that walks its whole
// slice with scalar atomicAdds; its host code passes the index buffer as the update source (:104-107), leaks the
// device stride array it allocates per call (:72-75) and its own test expects assignment, not accumulation
// (tests/python/test_scatter_nd.py:47-56). Here: the strides travel by value in the kernel arguments (no
// allocation), one lane per 16-byte piece of a slice (or per element when a slice is not a multiple of 16 bytes)
// so that a wavefront writes contiguous memory, and the mode is explicit: assign (what the reference's test
// checks; duplicate index rows then leave one of their updates, unspecified which) or atomic add (what the
// reference's kernel body does).
#pragma once

#include "config.hpp"
#include "hip_utils.hpp"

#include <cstdint>

namespace tiledcuda::kernels {

constexpr int kScatterMaxRank = 8;

struct ScatterNdShape {
    int64_t strides[kScatterMaxRank];  // element strides of the first k dimensions of `data`
    int64_t dims[kScatterMaxRank];     // their extents (indices are checked against them)
    int64_t n;                         // index rows
    int64_t slice;                     // elements per slice
    int k;                             // index components per row
};

enum class ScatterMode : int { kAssign = 0, kAdd = 1 };

namespace detail {
DEVICE void atomic_add_elem(float* p, float v) { atomicAdd(p, v); }
DEVICE void atomic_add_elem(__half* p, __half v) {
    // 16-bit atomic add through a compare-and-swap on the aligned 32-bit word that holds the element
    auto* word = reinterpret_cast<unsigned int*>(reinterpret_cast<uintptr_t>(p) & ~uintptr_t(3));
    const bool high = (reinterpret_cast<uintptr_t>(p) & 2) != 0;
    unsigned int old = *word, assumed;
    do {
        assumed = old;
        const unsigned short cur = high ? (assumed >> 16) : (assumed & 0xffffu);
        const __half sum = __float2half(__half2float(__ushort_as_half(cur)) + __half2float(v));
        const unsigned int repl = high ? ((assumed & 0xffffu) | (unsigned(__half_as_ushort(sum)) << 16))
                                       : ((assumed & 0xffff0000u) | __half_as_ushort(sum));
        old = atomicCAS(word, assumed, repl);
    } while (old != assumed);
}
using scatter_pair_t = _Float16 __attribute__((ext_vector_type(2)));
/// Both halves of a 4-byte aligned word in coarse-grained device memory.
DEVICE void atomic_add_pair(__half* p, scatter_pair_t v) {
    __builtin_amdgcn_global_atomic_fadd_v2f16((__attribute__((address_space(1))) scatter_pair_t*)(p), v);
}

/// Element offset of the slice that index row `row` names; false if a component lies outside its extent.
DEVICE bool scatter_base(const int64_t* indices, const ScatterNdShape& shape, int64_t row, int64_t& base) {
    const int64_t* idx = indices + row * shape.k;
    bool ok = true;
    base = 0;
#pragma unroll 4
    for (int c = 0; c < shape.k; ++c) {
        const int64_t v = idx[c];
        ok = ok && v >= 0 && v < shape.dims[c];
        base += v * shape.strides[c];
    }
    return ok;
}
}  // namespace detail

/// One lane per group of kVec elements of one slice. kVec * sizeof(T) is 16 (vector path, assign mode only,
/// slice % kVec == 0 and 16-byte aligned bases) or sizeof(T) (kVec = 1).
/// Rows with an index component outside its extent are skipped and counted in *bad_rows (if not null).
template <typename T, const int kVec, const ScatterMode kMode>
__global__ void __launch_bounds__(256)
    scatter_nd_kernel(T* __restrict__ data, const T* __restrict__ updates, const int64_t* __restrict__ indices,
                      const ScatterNdShape shape, unsigned int* __restrict__ bad_rows) {
    const int64_t groups_per_slice = shape.slice / kVec;
    const int64_t total = shape.n * groups_per_slice;
    for (int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < total; g += int64_t(gridDim.x) * blockDim.x) {
        const int64_t row = g / groups_per_slice;
        const int64_t off = (g - row * groups_per_slice) * kVec;
        int64_t base;
        if (!detail::scatter_base(indices, shape, row, base)) {
            if (bad_rows != nullptr && off == 0) atomicAdd(bad_rows, 1u);
            continue;
        }
        const T* src = updates + row * shape.slice + off;
        T* dst = data + base + off;
        if constexpr (kMode == ScatterMode::kAssign) {
            if constexpr (kVec == 1) {
                *dst = *src;
            } else {
                // streamed both ways: nothing here is touched twice, and lines left dirty in the L2s would be written
                // back after the last wavefront (65536 rows of 4 KiB: 103.5 -> 99.8 us, a plain device copy takes 99.2)
                __builtin_nontemporal_store(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src)),
                                            reinterpret_cast<u32x4*>(dst));
            }
        } else {
            static_assert(kMode == ScatterMode::kAssign || kVec == 1, "atomic add is per element");
            detail::atomic_add_elem(dst, *src);
        }
    }
}

/// Words a lane takes one after the other. One where slices start or stop inside a word: their compare-and-swap loops would
/// follow each other (4096 rows of 3: 7.4 us with two, 5.1 with one; 16384 of 513: 26.5, 26.3).
HOST_DEVICE constexpr int scatter_pair_pieces(bool whole) { return whole ? 2 : 1; }
/// Aligned 32-bit words of `data` that a slice of f16 touches; with whole = false it may start or end inside a word.
HOST_DEVICE int64_t scatter_pair_words(bool whole, int64_t slice) { return whole ? slice / 2 : slice / 2 + 1; }

/// f16 add: one lane per aligned 32-bit word of `data`, both elements added by one global_atomic_pk_add_f16 (each half rounded
/// to nearest even, subnormals kept: what the f32 addition and conversion of the compare-and-swap loop give); the ends of a
/// slice that start or stop inside a word by that loop. kWhole: there are none (even slices, `data` and `updates` 4-byte
/// aligned). A workgroup takes 512 (or 256) consecutive words of the updates, so that the 64-bit division by the words of a slice is
/// done once for all of them.
/// What bounds it: the L2s carry out about one 32-bit atomic per clock and channel (f32 addition: 8.4 M words in 31 us). In
/// the loop neighbouring lanes also contended for each word. 8192 rows of 1024 added into 32768: 300 -> 19 us, of
/// 1023: 281 -> 24, 32768 rows of 48 into 65536: 43 -> 9.7 us.
/// Rows with an index component outside its extent are skipped and counted in *bad_rows (if not null).
template <const bool kWhole>
__global__ void __launch_bounds__(256)
    scatter_nd_add_pairs(__half* __restrict__ data, const __half* __restrict__ updates, const int64_t* __restrict__ indices,
                         const ScatterNdShape shape, unsigned int* __restrict__ bad_rows) {
    using detail::scatter_pair_t;
    constexpr int kPieces = scatter_pair_pieces(kWhole), kBlock = 256 * kPieces;
    const int64_t words = scatter_pair_words(kWhole, shape.slice), total = shape.n * words;
    for (int64_t g0 = int64_t(blockIdx.x) * kBlock; g0 < total; g0 += int64_t(gridDim.x) * kBlock) {
        const int64_t row0 = g0 / words, rest0 = g0 - row0 * words;
        int64_t dst[kPieces];          // first element of the word
        int lo[kPieces], hi[kPieces];  // its elements that belong to the slice: [lo, hi)
        scatter_pair_t v[kPieces];
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
            const int local = threadIdx.x + 256 * p;
            lo[p] = hi[p] = 0;
            if (g0 + local >= total) continue;
            const int64_t rest = rest0 + local;
            // rest < words + 512: 32 bits, unless a slice has about 2^31 words, and then it lies in one slice or the next
            const int64_t more = words < (1ll << 31) ? int64_t(unsigned(rest) / unsigned(words)) : int64_t(rest >= words);
            const int64_t row = row0 + more, word = rest - more * words;
            int64_t base;
            if (!detail::scatter_base(indices, shape, row, base)) {
                if (bad_rows != nullptr && word == 0) atomicAdd(bad_rows, 1u);
                continue;
            }
            if constexpr (kWhole) {
                hi[p] = 2;
                dst[p] = base + 2 * word;
                v[p] = __builtin_nontemporal_load(reinterpret_cast<const scatter_pair_t*>(updates + row * shape.slice + 2 * word));
            } else {
                const int64_t e0 = 2 * word - (reinterpret_cast<uintptr_t>(data + base) & 2 ? 1 : 0);
                lo[p] = e0 < 0 ? 1 : 0;
                hi[p] = e0 + 1 < shape.slice ? 2 : e0 < shape.slice ? 1 : 0;
                dst[p] = base + e0;
                const auto* src = reinterpret_cast<const _Float16*>(updates + row * shape.slice + e0);
                v[p] = scatter_pair_t{0, 0};
                if (lo[p] == 0 && hi[p] > 0) v[p][0] = src[0];
                if (hi[p] == 2) v[p][1] = src[1];
            }
        }
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
            if (lo[p] >= hi[p]) continue;
            if (kWhole || hi[p] - lo[p] == 2) detail::atomic_add_pair(data + dst[p], v[p]);
            else detail::atomic_add_elem(data + dst[p] + lo[p], __half(v[p][lo[p]]));
        }
    }
}

}  // namespace tiledcuda::kernels
