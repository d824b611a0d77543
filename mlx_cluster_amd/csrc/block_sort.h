// Sort of up to 16,384 keys of 32 bits by one block of 1,024 threads: a bitonic
// network over keys held in registers, 16 consecutive keys a thread.
//
// Why a network and not radix passes: at 16 keys a thread a network stage
// costs one VALU instruction a key inside a thread (a min or a max), two
// across lanes (a DPP move, then a median with a per-lane bound that makes it
// a min or a max) and LDS only where it crosses wavefronts, 105 stages for
// 16,384 keys, about 180 instructions a key.  A stable 8-bit radix pass costs
// about 64 a key (the wavefront match of the digit) and two trips through
// LDS, whatever the digits.  Being oblivious, the network takes the same time
// on skewed keys.
#pragma once

#include "walk_device.h"

namespace mlxc {

constexpr int kSortBlock = 1024;    // threads
constexpr int kSortItems = 16;      // keys per thread
constexpr int kSortItemBits = 4;
constexpr int kWaveKeyBits = 10;    // keys of a wavefront: 1,024

// min / max of two keys in one instruction each.
__device__ __forceinline__ void sort_pair(uint32_t& a, uint32_t& b) {
    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    a = lo;
    b = hi;
}

// The key of lane ^ M, M < 16 (DPP: inside a row of 16 lanes).
template <int M>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
    static_assert(M == 1 || M == 2 || M == 4 || M == 8, "one lane bit inside a row");
    const int v = static_cast<int>(x);
    if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);  // quad 1,0,3,2
    if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);  // quad 2,3,0,1
    if constexpr (M == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true); // rotate by 8
    // 4 = 7 ^ 3: a mirror of 8 lanes, then of each quad
    return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true), 0x1B, 0xf,
                                    0xf, true);
}

// The smaller of a and b where upper is 0, the larger where it is ~0: the
// median of the two and the bound.
__device__ __forceinline__ uint32_t keep_half(uint32_t a, uint32_t b, uint32_t upper) {
    uint32_t d;
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(upper));
    return d;
}

template <int M>
__device__ __forceinline__ void row_stage(uint32_t (&key)[kSortItems], int lane) {
    const uint32_t upper = lane & M ? ~0u : 0u;
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) key[r] = keep_half(key[r], lane_xor<M>(key[r]), upper);
}

// Lane bits 4 and 5: two keys a pair of lanes trade halves of their registers
// (v_permlane16_swap / v_permlane32_swap), so that each lane holds both keys of
// a comparison, and trade them back.
template <int M>
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
    static_assert(M == 16 || M == 32, "one lane bit across rows");
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 r;
    if constexpr (M == 16) r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    else r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
template <int M>
__device__ __forceinline__ void cross_row_stage(uint32_t (&key)[kSortItems]) {
#pragma unroll
    for (int r = 0; r < kSortItems; r += 2) {
        swap_halves<M>(key[r], key[r + 1]);
        sort_pair(key[r], key[r + 1]);
        swap_halves<M>(key[r], key[r + 1]);
    }
}

// Strides 2^(bits-1) .. 1 over the register index, ascending.
template <int kBits>
__device__ __forceinline__ void item_stages(uint32_t (&key)[kSortItems]) {
#pragma unroll
    for (int s = 1 << (kBits - 1); s > 0; s >>= 1) {
#pragma unroll
        for (int r = 0; r < kSortItems; ++r)
            if (!(r & s)) sort_pair(key[r], key[r | s]);
    }
}

// Flips every bit of the keys where m is ~0: an ascending network then sorts
// them descending.
__device__ __forceinline__ void flip_keys(uint32_t (&key)[kSortItems], uint32_t m) {
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) key[r] ^= m;
}

// Merge step k (blocks of 2^k keys) from stride 2^kTop down, where kTop is
// below a wavefront's 10 bits.
template <int kTop>
__device__ __forceinline__ void wave_stages(uint32_t (&key)[kSortItems], int lane) {
    if constexpr (kTop >= 9) cross_row_stage<32>(key);
    if constexpr (kTop >= 8) cross_row_stage<16>(key);
    if constexpr (kTop >= 7) row_stage<8>(key, lane);
    if constexpr (kTop >= 6) row_stage<4>(key, lane);
    if constexpr (kTop >= 5) row_stage<2>(key, lane);
    if constexpr (kTop >= 4) row_stage<1>(key, lane);
    item_stages<kSortItemBits>(key);
}

// Direction mask of merge step k >= 4: blocks of 2^k keys alternate, thread
// t's 16 keys all in one.
__device__ __forceinline__ uint32_t step_mask(int t, int k) {
    return (t >> (k - kSortItemBits)) & 1 ? ~0u : 0u;
}

template <int kStep>
__device__ __forceinline__ void wave_step(uint32_t (&key)[kSortItems], int t, int lane) {
    flip_keys(key, step_mask(t, kStep - 1) ^ step_mask(t, kStep));
    wave_stages<kStep - 1>(key, lane);
}

// LDS words of the sort: one key a slot, a pad every 16 so that a thread's 16
// consecutive keys and a wavefront's consecutive keys both spread over the banks.
constexpr int kSortLds = kSortBlock * (kSortItems + 1);
__device__ __forceinline__ int sort_slot(int i) { return i + i / kSortItems; }

// Sorts key i (i < n; thread t holds keys 16 t .. 16 t + 15, the ones from n on
// set to ~0 by the caller) ascending over the block.  Every thread calls it;
// contains barriers.  lds: kSortLds keys, free on entry and on return (after a
// barrier of the caller's).
__device__ inline void block_sort(uint32_t (&key)[kSortItems], int n, uint32_t* lds) {
    constexpr int kBits = 14;
    static_assert(kSortBlock * kSortItems == 1 << kBits, "16,384 keys");
    // The other layout: thread t holds keys (r << kLow) | t, so that the
    // strides 2^kLow and up lie inside a thread.
    constexpr int kLow = kBits - kSortItemBits;
    const int t = threadIdx.x, lane = t % kWave;
    // blocks of 2, 4, 8 keys: alternating directions known at compile time
#pragma unroll
    for (int k = 1; k < kSortItemBits; ++k) {
#pragma unroll
        for (int s = 1 << (k - 1); s > 0; s >>= 1) {
#pragma unroll
            for (int r = 0; r < kSortItems; ++r) {
                if (r & s) continue;
                if (r & (1 << k)) sort_pair(key[r | s], key[r]);
                else sort_pair(key[r], key[r | s]);
            }
        }
    }
    // A wavefront that holds only padding is sorted in either direction.
    const bool some = (t - lane) * kSortItems < n;
    if (some) {
        flip_keys(key, step_mask(t, 4));
        item_stages<kSortItemBits>(key);
        wave_step<5>(key, t, lane);
        wave_step<6>(key, t, lane);
        wave_step<7>(key, t, lane);
        wave_step<8>(key, t, lane);
        wave_step<9>(key, t, lane);
        wave_step<10>(key, t, lane);
        flip_keys(key, step_mask(t, 10));
    }
    // Blocks of more than a wavefront's keys, as far as n reaches: the strides
    // of 2^kLow and up in the other layout, the rest in this one.
    for (int k = kWaveKeyBits + 1; k <= kBits && n > (1 << (k - 1)); ++k) {
        // the last step's blocks all ascend
        flip_keys(key, step_mask(t, k));
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) lds[sort_slot(t * kSortItems + r)] = key[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) key[r] = lds[sort_slot((r << kLow) | t)];
#pragma unroll
        for (int s = kSortItems / 2; s > 0; s >>= 1) {
            if (((s << kLow) >> k) == 0) {  // stride below this step's blocks
#pragma unroll
                for (int r = 0; r < kSortItems; ++r)
                    if (!(r & s)) sort_pair(key[r], key[r | s]);
            }
        }
        // each thread wrote back only where it read
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) lds[sort_slot((r << kLow) | t)] = key[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) key[r] = lds[sort_slot(t * kSortItems + r)];
        __syncthreads();
        wave_stages<kLow - 1>(key, lane);
        flip_keys(key, step_mask(t, k));
    }
}

}  // namespace mlxc
