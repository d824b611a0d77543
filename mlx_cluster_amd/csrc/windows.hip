// Skip-gram context windows over walks: the consumer right after the walk in
// node2vec training.  Not part of the reference (it stops at the walks,
// /root/reference/random_walks/BiasedRandomWalk.cpp:96); the layout follows
// torch_geometric's Node2Vec.pos_sample / neg_sample:
//   W = walk_nodes - context_size + 1 windows per walk, window-major:
//   out[(j * N + n) * C + k] = walk[n][j + k],  j < W, k < C.
// Negative windows use the same layout over the walk
//   [start[n], u(n, 1), ..., u(n, L)],  u(n, l) = node drawn uniformly from
//   [0, num_nodes) by Philox4x32-10 (key = seed, counter = (n lo, n hi, l, 0),
//   word 0 x): u = (x * num_nodes) >> 32.
//
// One block serves a tile of walks for every window position j: the tile's
// walk rows are staged in LDS once (one coalesced read), and the stores of one
// j are one contiguous run of tile * C entries.
#include "walk_host.h"

namespace mlxc {

namespace {

constexpr int kWinTile = 64;  // walks per block (at most)
constexpr int kMaxContext = 32;
constexpr int kWinSlots = (kWinTile * kMaxContext + kBlock - 1) / kBlock;
constexpr int kLineBytes = 128;
constexpr size_t kTileLds = 64 * 1024;  // LDS bytes for the walk rows of a tile

// Walks past the tile whose windows the tile's last line of a window position
// can reach: the entries of a line but one, in whole walks.
__host__ __device__ __forceinline__ int halo_walks(int32_t ctx, size_t esz) {
    return static_cast<int>((kLineBytes / esz - 1 + ctx - 1) / ctx);
}

// Window stores are streamed past the caches: nothing here reads them again.
#ifndef MLXC_WIN_NT
#define MLXC_WIN_NT 1
#endif
template <typename T>
__device__ __forceinline__ void put(T* p, T v) {
#if MLXC_WIN_NT
    __builtin_nontemporal_store(v, p);
#else
    *p = v;
#endif
}

// Writes the tile's part of every window position j from its rows (LDS,
// walk_nodes entries each): the entries of its walks, with both ends moved up
// to the next line boundary when kHalo (the rows then include the halo_walks
// after the tile), so that every line is written by one block, whole, and
// every wavefront store covers whole lines.  Entry e of a position (walk
// e / ctx of the tile, offset e % ctx) is at output index
// (j * num_walks + n0) * ctx + e.
//
// Bound by the write stream.  Without the shift a wavefront's 512 bytes start
// at any 8-byte offset unless num_walks * ctx fills whole lines, and the
// non-temporal partial lines at its ends cost as much as whole ones:
// 1,000,003 walks of 21 nodes, ctx 10, int64 (0.96 GB): 300 -> 182 us a
// launch, 5.3 TB/s over both window kernels; 2^20 walks, whose runs fill whole
// lines as they are, keep their 205 us a launch.
template <typename T, bool kHalo>
__device__ __forceinline__ void emit_windows(const T* rw, int64_t tile, int64_t n0,
                                             int64_t num_walks, int32_t walk_nodes, int32_t ctx,
                                             T* __restrict__ out) {
    constexpr int kLine = kLineBytes / sizeof(T);
    const int entries = static_cast<int>(tile) * ctx;  // one window of every walk in the tile
    const int windows = walk_nodes - ctx + 1;
    if (!kHalo) {
        // this thread's entries of a window position: places in the rows
        int32_t src[kWinSlots];
#pragma unroll
        for (int i = 0; i < kWinSlots; ++i) {
            const int e = threadIdx.x + i * kBlock;
            src[i] = e < entries ? (e / ctx) * walk_nodes + e % ctx : -1;
        }
        for (int j = 0; j < windows; ++j) {
            T* const o = out + (static_cast<int64_t>(j) * num_walks + n0) * ctx;
#pragma unroll
            for (int i = 0; i < kWinSlots; ++i)
                if (src[i] >= 0) put(o + threadIdx.x + i * kBlock, rw[src[i] + j]);
        }
        return;
    }
    const bool first = n0 == 0, last = n0 + tile == num_walks;
    // entries of a position from the tile on, as far as the rows reach
    const int64_t left = num_walks - n0;
    const int rest = left < kWinTile + kLineBytes ? static_cast<int>(left) * ctx : INT32_MAX;
    // e / ctx as (e * inv) >> 16: exact while e * (ctx - 1) < 2^16, and
    // e < kWinTile * ctx + kLine (at ctx = 32: 2,080 * 31 = 64,480)
    static_assert((kWinTile * kMaxContext + kLineBytes / 4) * (kMaxContext - 1) < (1 << 16),
                  "the reciprocal is exact");
    const uint32_t inv = ((1u << 16) + ctx - 1) / ctx;
    for (int j = 0; j < windows; ++j) {
        T* const o = out + (static_cast<int64_t>(j) * num_walks + n0) * ctx;
        int lo = 0, hi = entries;
        const int at = static_cast<int>((reinterpret_cast<uintptr_t>(o) / sizeof(T)) % kLine);
        if (!first) lo = (kLine - at) % kLine;
        if (!last) hi += (kLine - (at + entries) % kLine) % kLine;
        if (hi > rest) hi = rest;  // the position ends there
        for (int e = lo + static_cast<int>(threadIdx.x); e < hi; e += kBlock) {
            const int w = static_cast<int>((static_cast<uint32_t>(e) * inv) >> 16);
            put(o + e, rw[w * walk_nodes + (e - w * ctx) + j]);
        }
    }
}

// Rows in LDS of a tile at n0: per_block walks (<= kWinTile), and the halo's
// when the launch has room for them, as far as there are walks.
__device__ __forceinline__ int staged_walks(int64_t n0, int64_t num_walks, int32_t per_block,
                                            int32_t halo) {
    const int64_t left = num_walks - n0;
    return left < per_block + halo ? static_cast<int>(left) : per_block + halo;
}

template <typename T, bool kHalo>
__global__ __launch_bounds__(kBlock) void context_windows_kernel(const T* __restrict__ walks,
                                                                 int64_t num_walks,
                                                                 int32_t walk_nodes, int32_t ctx,
                                                                 int32_t per_block, int32_t halo,
                                                                 T* __restrict__ out) {
    extern __shared__ unsigned char smem[];
    T* rw = reinterpret_cast<T*>(smem);
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * per_block;
    const int64_t tile = num_walks - n0 < per_block ? num_walks - n0 : per_block;
    const int cells = staged_walks(n0, num_walks, per_block, halo) * walk_nodes;
    const T* in = walks + n0 * walk_nodes;  // the tile's rows are contiguous
    for (int e = threadIdx.x; e < cells; e += kBlock) rw[e] = in[e];
    __syncthreads();
    emit_windows<T, kHalo>(rw, tile, n0, num_walks, walk_nodes, ctx, out);
}

__device__ __forceinline__ int64_t negative_node(int64_t n, int32_t l, int64_t num_nodes,
                                                 uint32_t k0, uint32_t k1) {
    uint32_t c0 = static_cast<uint32_t>(n), c1 = static_cast<uint32_t>(static_cast<uint64_t>(n) >> 32),
             c2 = static_cast<uint32_t>(l), c3 = 0;
    philox4x32_10(c0, c1, c2, c3, k0, k1);
    return static_cast<int64_t>((static_cast<uint64_t>(c0) * static_cast<uint64_t>(num_nodes)) >> 32);
}

template <typename T, bool kHalo>
__global__ __launch_bounds__(kBlock) void negative_windows_kernel(
    const int64_t* __restrict__ start, int64_t num_walks, int32_t walk_length, int32_t ctx,
    int64_t num_nodes, uint32_t k0, uint32_t k1, int32_t per_block, int32_t halo,
    T* __restrict__ out) {
    // the tile's walks [start, u_1..u_L] are generated once into LDS
    extern __shared__ unsigned char smem[];
    T* rw = reinterpret_cast<T*>(smem);
    const int walk_nodes = walk_length + 1;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * per_block;
    const int64_t tile = num_walks - n0 < per_block ? num_walks - n0 : per_block;
    const int cells = staged_walks(n0, num_walks, per_block, halo) * walk_nodes;
    for (int e = threadIdx.x; e < cells; e += kBlock) {
        const int w = e / walk_nodes, l = e % walk_nodes;
        const int64_t n = n0 + w;
        rw[e] = static_cast<T>(l == 0 ? start[n] : negative_node(n, l, num_nodes, k0, k1));
    }
    __syncthreads();
    emit_windows<T, kHalo>(rw, tile, n0, num_walks, walk_nodes, ctx, out);
}

}  // namespace

// Walks per block whose rows of walk_nodes entries fit kTileLds bytes.
int tile_walks(int32_t walk_nodes, size_t esz) {
    const size_t fit = kTileLds / (static_cast<size_t>(walk_nodes) * esz);
    return fit > static_cast<size_t>(kWinTile) ? kWinTile : static_cast<int>(fit);
}

namespace {

// Grid and LDS of a window launch.  The halo's rows join the tile's where it
// pays (lines_pay) and both fit kTileLds (int64, ctx 10: walks of up to 124
// nodes); other calls write their lines where the tiles happen to cut them.
struct WinLaunch {
    int per_block, halo;
    int64_t grid;
    size_t lds;
};

// Whether moving the tiles' ends to line boundaries is worth its halo and the
// walk that each entry of it has to find.  Not where every run fills whole
// lines as it is; not below two blocks or so a compute unit, where a block's
// own time counts; not where the caches put the partial lines together; and
// not for pairs, whose runs are short and whose halo is long.  Kernel us,
// tiles as they are / moved, int64 but where noted:
//   21 nodes, ctx 10:  30,011 walks (29 MB) 8.9 / 7.1, 60,013 (58 MB) 17.9 / 12.8,
//                      1,000,003 (960 MB) 294 / 181;  10,007 (10 MB) 6.5 / 6.4
//   81 nodes, ctx 10:  10,007 (58 MB, 157 blocks) 19.1 / 22.6, 30,011 int32 (86 MB) 33.8 / 24.5
//   31 nodes, ctx 16:  30,011 int32 (31 MB) 7.9 / 8.9, 60,013 int32 (61 MB) 14.9 / 13.6,
//                      10,007 (20 MB, whole lines) 7.8 / 8.9
//   30 nodes, ctx 3:   60,013 int32 (20 MB) 9.7 / 11.5, 100,003 int32 (34 MB) 14.9 / 15.4,
//                      200,003 int32 (67 MB) 32.0 / 25.9, 60,013 (40 MB) 13.2 / 11.3
//   11 nodes, ctx 2:   1,000,003 (160 MB) 44.8 / 47.4, int32 (80 MB) 33.8 / 43.8
bool lines_pay(const WinLaunch& w, int64_t num_walks, int32_t walk_nodes, int32_t ctx, size_t esz,
               const void* out) {
    const size_t run = static_cast<size_t>(ctx) * esz;  // bytes a walk and a window position
    if (static_cast<size_t>(num_walks) * run % kLineBytes == 0 &&
        static_cast<size_t>(w.per_block) * run % kLineBytes == 0 &&
        reinterpret_cast<uintptr_t>(out) % kLineBytes == 0)
        return false;
    if (ctx <= 2 || w.grid < 400) return false;
    const size_t bytes = static_cast<size_t>(walk_nodes - ctx + 1) * num_walks * run;
    return bytes >= (w.halo <= 7 && w.grid >= 768 ? size_t{24} << 20 : size_t{64} << 20);
}

WinLaunch win_launch(int64_t num_walks, int32_t walk_nodes, int32_t ctx, size_t esz,
                     const void* out) {
    WinLaunch w;
    w.per_block = tile_walks(walk_nodes, esz);
    w.halo = halo_walks(ctx, esz);
    const size_t row = static_cast<size_t>(walk_nodes) * esz;
    w.grid = w.per_block < 1 ? 0 : (num_walks + w.per_block - 1) / w.per_block;
    if ((w.per_block + w.halo) * row > kTileLds ||
        !lines_pay(w, num_walks, walk_nodes, ctx, esz, out))
        w.halo = 0;
    w.lds = (w.per_block + w.halo) * row;
    return w;
}

template <typename T>
void context_windows_typed(const WinLaunch& w, const void* walks, int64_t num_walks,
                           int32_t walk_nodes, int32_t ctx, void* out, hipStream_t stream) {
    auto* kernel = w.halo ? context_windows_kernel<T, true> : context_windows_kernel<T, false>;
    hipLaunchKernelGGL(kernel, dim3(w.grid), dim3(kBlock), w.lds, stream,
                       static_cast<const T*>(walks), num_walks, walk_nodes, ctx, w.per_block,
                       w.halo, static_cast<T*>(out));
}

template <typename T>
void negative_windows_typed(const WinLaunch& w, const int64_t* start, int64_t num_walks,
                            int32_t walk_length, int32_t ctx, int64_t num_nodes, uint64_t seed,
                            void* out, hipStream_t stream) {
    auto* kernel = w.halo ? negative_windows_kernel<T, true> : negative_windows_kernel<T, false>;
    hipLaunchKernelGGL(kernel, dim3(w.grid), dim3(kBlock), w.lds, stream, start, num_walks,
                       walk_length, ctx, num_nodes, static_cast<uint32_t>(seed),
                       static_cast<uint32_t>(seed >> 32), w.per_block, w.halo,
                       static_cast<T*>(out));
}

}  // namespace

int launch_context_windows(const void* walks, int64_t num_walks, int32_t walk_nodes, int32_t ctx,
                           int32_t elem_type, void* out, hipStream_t stream) {
    const bool narrow = elem_type == MLXC_OUT_INT32;
    const WinLaunch w = win_launch(num_walks, walk_nodes, ctx, narrow ? 4 : 8, out);
    if (w.per_block < 1) return fail(MLXC_ERR_INVALID_ARGUMENT, "walks too long for windows");
    if (narrow) context_windows_typed<int32_t>(w, walks, num_walks, walk_nodes, ctx, out, stream);
    else context_windows_typed<int64_t>(w, walks, num_walks, walk_nodes, ctx, out, stream);
    MLXC_HIP_TRY(hipGetLastError());
    return MLXC_OK;
}

int windows_max_nodes(int32_t elem_type) {
    return static_cast<int>(kTileLds / (elem_type == MLXC_OUT_INT32 ? 4 : 8));
}

int launch_negative_windows(const int64_t* start, int64_t num_walks, int32_t walk_length,
                            int32_t ctx, int64_t num_nodes, uint64_t seed, int32_t out_type,
                            void* out, hipStream_t stream) {
    const bool narrow = out_type == MLXC_OUT_INT32;
    const WinLaunch w = win_launch(num_walks, walk_length + 1, ctx, narrow ? 4 : 8, out);
    if (w.per_block < 1) return fail(MLXC_ERR_INVALID_ARGUMENT, "walk_length too large");
    if (narrow)
        negative_windows_typed<int32_t>(w, start, num_walks, walk_length, ctx, num_nodes, seed,
                                        out, stream);
    else
        negative_windows_typed<int64_t>(w, start, num_walks, walk_length, ctx, num_nodes, seed,
                                        out, stream);
    MLXC_HIP_TRY(hipGetLastError());
    return MLXC_OK;
}

}  // namespace mlxc
