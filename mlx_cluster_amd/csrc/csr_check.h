// CSR validation on the device, shared by the preparation kernels and the
// node2vec walk of few walks.
#pragma once

#include "walk_device.h"

namespace mlxc {

__device__ __forceinline__ int64_t wave_sum(int64_t x) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) x += __shfl_xor(x, off, kWave);
    return x;
}

__device__ __forceinline__ uint32_t wave_or(uint32_t x) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) x |= __shfl_xor(x, off, kWave);
    return x;
}

// CSR validation, accumulated per thread and reduced per block.  Rows are
// sorted iff every position i >= 1 with col[i] < col[i-1] starts a non-empty
// row, i.e. iff desc == start_desc.
struct CsrCheck {
    bool bad_rowptr = false;  // rowptr[0] != 0, rowptr[V] != E, or decreasing
    bool bad_col = false;     // a col value outside [0, V)
    int64_t desc = 0;
    int64_t start_desc = 0;

    // node-parallel part: thread gid of a grid of `stride` threads
    __device__ void nodes(const int64_t* rowptr, int64_t V, const int64_t* col, int64_t E,
                          int64_t gid, int64_t stride) {
        if (gid == 0 && (rowptr[0] != 0 || rowptr[V] != E)) bad_rowptr = true;
        for (int64_t v = gid; v < V; v += stride) {
            const int64_t rs = rowptr[v], re = rowptr[v + 1];
            if (re < rs) bad_rowptr = true;
            if (rs >= 1 && re > rs && re <= E && col[rs] < col[rs - 1]) ++start_desc;
        }
    }
    // edge-parallel part: entry i holding c
    __device__ void edge(const int64_t* col, int64_t V, int64_t i, int64_t c) {
        if (!node_ok(c, V)) bad_col = true;
        if (i >= 1 && c < col[i - 1]) ++desc;
    }
    // entries gid, gid + stride, ... in fours from a 16-byte aligned col, each
    // compared with the one before it
    __device__ void edges4(const int64_t* col, int64_t V, int64_t E, int64_t gid, int64_t stride) {
        typedef int64_t i64x2 __attribute__((ext_vector_type(2)));
        for (int64_t q = gid; 4 * q < E; q += stride) {
            const int64_t i = 4 * q;
            if (i + 4 <= E) {
                const i64x2 a = reinterpret_cast<const i64x2*>(col + i)[0];
                const i64x2 b = reinterpret_cast<const i64x2*>(col + i)[1];
                const int64_t before = i > 0 ? col[i - 1] : a.x;
                bad_col |= !node_ok(a.x, V) | !node_ok(a.y, V) | !node_ok(b.x, V) |
                           !node_ok(b.y, V);
                desc += (a.x < before) + (a.y < a.x) + (b.x < a.y) + (b.y < b.x);
            } else {
                for (int64_t k = i; k < E; ++k) edge(col, V, k, col[k]);
            }
        }
    }
    // The block's totals, in thread 0: the status bits, and the descents that
    // start no row (desc - start_desc, over all blocks zero exactly when the
    // rows are sorted).  Every thread of the block calls it.
    __device__ void totals(uint32_t rowptr_bit, uint32_t col_bit, uint32_t& bits, int64_t& diff) {
        __shared__ uint32_t block_bits[kBlock / kWave];
        __shared__ int64_t block_diff[kBlock / kWave];
        const uint32_t wave_bits =
            wave_or((bad_rowptr ? rowptr_bit : 0u) | (bad_col ? col_bit : 0u));
        const int64_t d = wave_sum(desc - start_desc);
        if (__lane_id() == 0) {
            block_bits[threadIdx.x / kWave] = wave_bits;
            block_diff[threadIdx.x / kWave] = d;
        }
        __syncthreads();
        bits = 0;
        diff = 0;
        if (threadIdx.x == 0) {
            for (int i = 0; i < kBlock / kWave; ++i) {
                bits |= block_bits[i];
                diff += block_diff[i];
            }
        }
    }
    // Adds the totals to the given words, one atomic each from thread 0.
    // (Atomics on one word serialize: three per wavefront, 49,000 per call,
    // took 0.3 ms of the 0.42 ms pass over configuration 3's 31 M entries.)
    __device__ void flush(unsigned long long* bits_word, uint32_t rowptr_bit, uint32_t col_bit,
                          unsigned long long* diff_word) {
        uint32_t bits;
        int64_t diff;
        totals(rowptr_bit, col_bit, bits, diff);
        if (bits) atomicOr(bits_word, static_cast<unsigned long long>(bits));
        if (diff) atomicAdd(diff_word, static_cast<unsigned long long>(diff));
    }
};

}  // namespace mlxc
