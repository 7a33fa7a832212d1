// f32 matmul: C[m, n] = A[m, k] . B[k, n] (+ a row bias or a residual).
//
// Semantics are the reference's `matmul_with_addend` (src/kernels.rs:5518-5789,
// src/kernels.cu:1262-1306): optional transposes (A stored [k, m], B stored
// [n, k]), f32 accumulation, the addend added to the finished sum.
//
// Kernel families, chosen by shape:
//  - MFMA tiles. A workgroup owns a BM x BN tile of C and sums it as bf16
//    plane products (split_tile.hpp): each operand is read into registers
//    two or three stages ahead of its use, split there into three bf16 planes
//    and written to LDS once for all the waves that read it. Every operand
//    orientation, alignment and weight format gives the same bits. Ragged
//    edges repeat the last row or column, so edge tiles run the same loop.
//    Four configurations, picked by a time model: 256 x 256 tiles of 8 waves
//    (one per CU) for large products; 128 x 128 of 4 waves (two per CU) or of
//    8 waves (one per CU); 64 x 64 of 8 waves in two k groups. Tiles are
//    ordered so that consecutive tiles share a block row of A and each of the
//    8 XCDs (own L2) gets a contiguous band of tiles. When the tiles cannot
//    fill the device, k is split: over up to 8 workgroups per tile (split-k),
//    or in equal runs of (tile, k slice) units per workgroup (stream-K) when
//    the tiles divide the device badly; partial tiles go to a workspace and a
//    second launch adds them in k order (deterministic) with the addend.
//  - Few rows over a large B (few_rows.hpp): 9-32 rows stream B past A's
//    planes; up to 8 rows take B [n, k], or rows that are no whole vectors, as
//    it lies.
//  - m <= kGemvMaxRows (decode), or up to 32 rows of a small product with
//    k > 1024 in row blocks of 8: the work is reading B once (HBM-bound), so
//    each wave streams 256 columns of B (512 for compact bf16 weights on up
//    to 4 rows) with 16-byte loads over one k slice, keeping m x 4 partial
//    sums per lane; partial sums per k slice go to a workspace and a second
//    launch adds them in a fixed order (deterministic), four waves per 256
//    columns.
//  - 16-32 rows of a small product with k <= 1024: one launch of 32 x 32
//    MFMA tiles whose 16 waves split k and meet in LDS (small_mfma_kernel).
#include <type_traits>

#include <utility>

#include "common.hpp"

#include <mutex>
#include "internal.hpp"
#include "decode_merge.hpp"
#include "reduce.hpp"
#include "few_rows.hpp"
#include "split_tile.hpp"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kGemvMaxRows = 8;

// The epilogue of a finished sum v with its addend element a. Modes 1 (a bias
// row, indexed by column) and 2 (a full matrix) add it; mode 3, internal to
// the library (the up product of a gated matmul, its addend the gate
// product), gates the sum as the silu-mul kernel does: silu(a) * v, so the
// gated product equals the two matmuls and silu-mul bit for bit. Modes 2 and
// 3 index the addend as the output.
__device__ __forceinline__ float apply_addend(float v, float a, int mode) {
    return mode == 3 ? mhip::silu1(a) * v : v + a;
}
__device__ __forceinline__ float4 apply_addend(float4 v, float4 a, int mode) {
    return make_float4(apply_addend(v.x, a.x, mode), apply_addend(v.y, a.y, mode),
                       apply_addend(v.z, a.z, mode), apply_addend(v.w, a.w, mode));
}
// Largest product (m x k x n multiply-adds) that 16-32 rows run on the small
// MFMA tiles or the GEMV's row blocks rather than on the large MFMA tiles.
constexpr uint64_t kGemvSmallProduct = 1ull << 26;

// Split-k partial sums live in the context's workspace; stream order makes
// reuse by the next call safe. During mhip_matmul_f32_noalloc they live in
// the device's fixed scratch array instead, and a product that needs more
// than it holds is refused.
mhip_status workspace(mhip_ctx* ctx, size_t bytes, float** out) {
    if (ctx->fixed_scratch) {
        if (bytes > ctx->fixed_scratch_bytes)
            return mhip::fail(MHIP_SHAPE_UNSUPPORTED,
                              "matmul: this product needs " + std::to_string(bytes) +
                                  " bytes of scratch; the allocation-free matmul has " +
                                  std::to_string(ctx->fixed_scratch_bytes));
        *out = static_cast<float*>(ctx->fixed_scratch);
        return MHIP_OK;
    }
    void* p = nullptr;
    mhip_status st = mhip::workspace(ctx, bytes, &p);
    *out = static_cast<float*>(p);
    return st;
}

// ---------------------------------------------------------------------------
// MFMA tiles
// ---------------------------------------------------------------------------

using mhip::elem;
using mhip::load4;
using mhip::load4_nt;

// One tile configuration (mhip::SplitTile's parameters but the operands').
template <int BM_, int BN_, int WM_, int WN_, int KG_, int BK_, int BUFS_>
struct TileShape {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, KG = KG_, BK = BK_, BUFS = BUFS_;
    static constexpr int kWaves = (BM / WM) * (BN / WN) * KG;
    // Workgroups per CU a configuration is planned for: one of 8 waves
    // already gives each SIMD two.
    static constexpr uint64_t kPerCu = kWaves >= 8 ? 1 : 2;
    template <bool A_T, bool B_T, class BT>
    using Tile = mhip::SplitTile<BM, BN, WM, WN, KG, BK, A_T, B_T, BT, BUFS>;
};

// How a product's operands may be read: 16-byte (8-byte bf16) loads of rows
// along k, pairs of bf16 columns, and rows short enough for the 32-bit
// offsets of a tile's buffer loads.
struct Access {
    bool wide_a, wide_b, short_rows;
};
// Longest leading dimension (elements) whose 256-row slice of f32 stays under
// 2^31 bytes.
constexpr uint64_t kShortRows = 1ull << 21;
// Splits and stream-K runs are planned in slices of this much k.
constexpr uint64_t kSliceK = 32;

// Maps the linear workgroup id to a (tile_m, tile_n): each XCD (ids are
// dealt round-robin over 8) takes a contiguous band, and inside a band tiles
// go down groups of 8 tile rows so neighbours share A rows and B columns.
__device__ __forceinline__ void tile_coords(uint32_t tiles_m, uint32_t tiles_n, uint32_t* tm,
                                            uint32_t* tn) {
    const uint32_t total = tiles_m * tiles_n;
    uint32_t id = blockIdx.x;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    constexpr uint32_t kGroup = 8;
    const uint32_t per_group = kGroup * tiles_n;
    const uint32_t group = id / per_group;
    const uint32_t first_m = group * kGroup;
    const uint32_t rows_in_group = min(tiles_m - first_m, kGroup);
    const uint32_t in_group = id % per_group;
    *tm = first_m + in_group % rows_in_group;
    *tn = in_group / rows_in_group;
}

// One tile's product, C[m0 .., n0 ..] summed over k in [k_begin, k_end),
// written to out[(row - out_r0) * ldo + (col - out_c0)] for the rows < M and
// columns < N, plus the addend when addend_mode is not 0. LDS is free on entry
// and again on return.
template <class Shape, bool A_T, bool B_T, class BT>
__device__ __forceinline__ void gemm_tile(const float* __restrict__ A, const BT* __restrict__ B,
                                          uint64_t M, uint64_t K, uint64_t N, uint64_t m0,
                                          uint64_t n0, uint64_t k_begin, uint64_t k_end, Access access,
                                          char* lds, float* __restrict__ out, uint64_t out_r0,
                                          uint64_t out_c0, uint64_t ldo,
                                          const float* __restrict__ addend, int addend_mode) {
    using Tile = typename Shape::template Tile<A_T, B_T, BT>;
    Tile tile;
    typename Tile::Mask again;
    bool redo = true;
    if (K >= mhip::kSplitMinK) {
        redo = tile.sum(A, B, M, K, N, m0, n0, k_begin, k_end, access.wide_a, access.wide_b, access.short_rows, lds,
                        again);
    } else {
        tile.clear();
#pragma unroll
        for (int w = 0; w < Tile::kWords; ++w) again[w] = 0xFFFFFFFFu;
    }
    auto sum_again = [&]() {
        tile.sum_f32(A, B, M, K, N, m0, n0, k_begin, k_end, access.wide_a, access.wide_b, access.short_rows, lds);
    };
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int kg = wave / Tile::kTileWaves, wt = wave % Tile::kTileWaves;
    const int wm = wt / Tile::kWavesN, wn = wt % Tile::kWavesN;
    const int lrow = lane & 31, lk = lane >> 5;

    // Accumulator r of lane l holds C[8*(r/4) + 4*(l/32) + r%4][l%32] of its
    // 32x32 block; registers [R0, R1) are written, all of them or those whose
    // bit of `again` is not `flip`.
    auto store = [&](auto r0, auto r1, auto all, uint32_t flip) {
#pragma unroll
        for (int i = 0; i < Tile::kMI; ++i) {
#pragma unroll
            for (int j = 0; j < Tile::kNI; ++j) {
                const uint64_t col = n0 + wn * Shape::WN + j * 32 + lrow;
                if (col >= N) continue;
#pragma unroll
                for (int r = decltype(r0)::value; r < decltype(r1)::value; ++r) {
                    const uint64_t row = m0 + wm * Shape::WM + i * 32 + 8 * (r / 4) + 4 * lk + (r % 4);
                    const int bit = (i * Tile::kNI + j) * 16 + r;
                    if (!decltype(all)::value && (again[bit / 32] >> bit % 32 & 1u) == flip) continue;
                    if (row < M) {
                        float v = tile.acc[i][j][r];
                        if (addend_mode == 1) v = v + addend[col];
                        else if (addend_mode >= 2) v = apply_addend(v, addend[row * N + col], addend_mode);
                        // The 64-tile kernel writes C non-temporally: all its
                        // workgroups store at once, at the end (0.3-0.7 us of
                        // 21-28); for the larger tiles it was 0.5-0.9 % slower.
                        if constexpr (Shape::KG == 2)
                            __builtin_nontemporal_store(v, out + (row - out_r0) * ldo + (col - out_c0));
                        else
                            out[(row - out_r0) * ldo + (col - out_c0)] = v;
                    }
                }
            }
        }
    };
    using R0 = std::integral_constant<int, 0>;
    using R8 = std::integral_constant<int, 8>;
    using R16 = std::integral_constant<int, 16>;

    if constexpr (Shape::KG == 2) {
        if (redo) {
            mhip::f32x16 first[Tile::kMI][Tile::kNI];
#pragma unroll
            for (int i = 0; i < Tile::kMI; ++i)
#pragma unroll
                for (int j = 0; j < Tile::kNI; ++j) first[i][j] = tile.acc[i][j];
            sum_again();
#pragma unroll
            for (int i = 0; i < Tile::kMI; ++i)
#pragma unroll
                for (int j = 0; j < Tile::kNI; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int bit = (i * Tile::kNI + j) * 16 + r;
                        if (!(again[bit / 32] >> bit % 32 & 1u)) tile.acc[i][j][r] = first[i][j][r];
                    }
        }
        // Two k groups: each finishes half of every block's rows, group 0
        // registers 0-7 (rows 0-15 of a 32x32 block), group 1 registers
        // 8-15, handing the other half to its partner through LDS, so both
        // groups add and write. The sum is group 0's plus group 1's either way.
        constexpr int kHalf = Tile::kMI * Tile::kNI * 8 * 64;  // floats per wave and half
        float* const meet = reinterpret_cast<float*>(lds);
        float* const given = meet + (kg * Tile::kTileWaves + wt) * kHalf;
        const float* const taken = meet + ((1 - kg) * Tile::kTileWaves + wt) * kHalf;
        auto give = [&](auto base) {
#pragma unroll
            for (int i = 0; i < Tile::kMI; ++i)
#pragma unroll
                for (int j = 0; j < Tile::kNI; ++j)
#pragma unroll
                    for (int r = 0; r < 8; ++r)
                        given[((i * Tile::kNI + j) * 8 + r) * 64 + lane] = tile.acc[i][j][decltype(base)::value + r];
        };
        auto take = [&](auto base, auto first) {
#pragma unroll
            for (int i = 0; i < Tile::kMI; ++i)
#pragma unroll
                for (int j = 0; j < Tile::kNI; ++j)
#pragma unroll
                    for (int r = 0; r < 8; ++r) {
                        const float a = tile.acc[i][j][decltype(base)::value + r];
                        const float b = taken[((i * Tile::kNI + j) * 8 + r) * 64 + lane];
                        tile.acc[i][j][decltype(base)::value + r] = decltype(first)::value ? a + b : b + a;
                    }
        };
        if (kg == 0) give(R8{});
        else give(R0{});
        __syncthreads();
        if (kg == 0) take(R0{}, std::true_type{});
        else take(R8{}, std::false_type{});
        __syncthreads();  // LDS is free again
        if (kg == 0) store(R0{}, R8{}, std::true_type{}, 0);
        else store(R8{}, R16{}, std::true_type{}, 0);
    } else if (!redo) {
        store(R0{}, R16{}, std::true_type{}, 0);
    } else {
        // (The registers hold one set of sums: those that stay are written first.)
        store(R0{}, R16{}, std::false_type{}, 1);
        sum_again();
        store(R0{}, R16{}, std::false_type{}, 0);
    }
}

// One tile per workgroup. blockIdx.y is the k split: the workgroup sums k in
// [y * k_split, min(K, (y + 1) * k_split)) and, with more than one split,
// writes that partial product to C + y * M * N (no addend) for
// splitk_reduce_kernel.
template <class Shape, bool A_T, bool B_T, class BT>
__global__ __launch_bounds__(64 * Shape::kWaves, 2) void mfma_gemm_kernel(
    const float* __restrict__ A, const BT* __restrict__ B, float* __restrict__ C, uint64_t M,
    uint64_t K, uint64_t N, const float* __restrict__ addend, int addend_mode, uint64_t k_split,
    Access access) {
    extern __shared__ char lds[];
    constexpr int BM = Shape::BM, BN = Shape::BN;
    uint32_t tm, tn;
    tile_coords(static_cast<uint32_t>((M + BM - 1) / BM), static_cast<uint32_t>((N + BN - 1) / BN),
                &tm, &tn);
    const uint64_t k_begin = static_cast<uint64_t>(blockIdx.y) * k_split;
    const uint64_t k_end = min(K, k_begin + k_split);
    const bool split = gridDim.y > 1;
    float* out = split ? C + static_cast<uint64_t>(blockIdx.y) * M * N : C;
    gemm_tile<Shape, A_T, B_T, BT>(A, B, M, K, N, static_cast<uint64_t>(tm) * BM, static_cast<uint64_t>(tn) * BN,
                                   k_begin, k_end, access, lds, out, 0, 0, N, addend, split ? 0 : addend_mode);
}

// Stream-K: the (tile, k slice) units, tile-major (tile t = tm * tiles_n +
// tn, its slices in k order), are dealt in equal runs of `per` to the
// workgroups, so every CU does the same MFMA work however the tiles divide.
// Workgroup w covers units [w * per, (w + 1) * per); per <= slices per tile,
// so that run touches at most two tiles, and the part of the j-th one goes to
// slot 2w + j as a BM x BN tile for stream_reduce_kernel.
template <class Shape, bool A_T, bool B_T, class BT>
__global__ __launch_bounds__(64 * Shape::kWaves, 2) void mfma_gemm_stream_kernel(
    const float* __restrict__ A, const BT* __restrict__ B, float* __restrict__ slots, uint64_t M,
    uint64_t K, uint64_t N, uint64_t per, Access access) {
    extern __shared__ char lds[];
    constexpr int BM = Shape::BM, BN = Shape::BN;
    const uint64_t tiles_n = (N + BN - 1) / BN;
    const uint64_t kslices = (K + kSliceK - 1) / kSliceK;
    const uint64_t total = (M + BM - 1) / BM * tiles_n * kslices;
    const uint64_t u0 = static_cast<uint64_t>(blockIdx.x) * per;
    const uint64_t end = min(total, u0 + per);
    if (u0 >= end) return;
    // The run's first part and, when it crosses into the next tile, its
    // second (k from 0). Not in a loop: that spilled registers.
    auto part = [&](uint64_t t, uint64_t a, uint64_t b, uint64_t slot) {
        const uint64_t m0 = t / tiles_n * BM, n0 = t % tiles_n * BN;
        gemm_tile<Shape, A_T, B_T, BT>(A, B, M, K, N, m0, n0, a * kSliceK, min(K, b * kSliceK), access, lds,
                                       slots + slot * (BM * BN), m0, n0, BN, nullptr, 0);
    };
    const uint64_t t0 = u0 / kslices, a0 = u0 % kslices;
    const uint64_t b0 = min(kslices, a0 + (end - u0));
    part(t0, a0, b0, 2 * static_cast<uint64_t>(blockIdx.x));
    const uint64_t u1 = u0 + (b0 - a0);
    if (u1 < end) part(u1 / kslices, 0, min(kslices, end - u1), 2 * static_cast<uint64_t>(blockIdx.x) + 1);
}

// C = the stream-K slots covering each output's tile, added in k order (the
// workgroups' order), + addend: deterministic. Four consecutive outputs per
// thread; `vec` (N % 4 == 0, aligned C and addend): one dwordx4 each.
template <int BM, int BN>
__global__ __launch_bounds__(256) void stream_reduce_kernel(const float* __restrict__ slots,
                                                            float* __restrict__ C, uint64_t M,
                                                            uint64_t N, uint64_t kslices,
                                                            uint64_t per,
                                                            const float* __restrict__ addend,
                                                            int addend_mode, int vec) {
    const uint64_t total = M * N;
    const uint64_t i = (static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    const uint64_t tiles_n = (N + BN - 1) / BN;
    auto slot_of = [&](uint64_t row, uint64_t col, uint64_t* w_first, uint64_t* w_last) {
        const uint64_t t = row / BM * tiles_n + col / BN;
        *w_first = t * kslices / per;
        *w_last = ((t + 1) * kslices - 1) / per;
        return t * kslices;  // the tile's first unit
    };
    auto at = [&](uint64_t w, uint64_t first_unit, uint64_t row, uint64_t col) {
        const uint64_t seg = w * per < first_unit ? 1 : 0;
        return slots + (2 * w + seg) * (BM * BN) + (row % BM) * BN + col % BN;
    };
    if (vec && i + 3 < total) {
        const uint64_t row = i / N, col = i % N;  // four columns of one tile (BN % 4 == 0)
        uint64_t w0, w1;
        const uint64_t first = slot_of(row, col, &w0, &w1);
        float4 v = mhip::load_nt(reinterpret_cast<const float4*>(at(w0, first, row, col)));
        for (uint64_t w = w0 + 1; w <= w1; ++w) {
            const float4 p = mhip::load_nt(reinterpret_cast<const float4*>(at(w, first, row, col)));
            v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
        }
        if (addend_mode == 1) {
            const float4 b = *reinterpret_cast<const float4*>(addend + col);
            v.x = v.x + b.x; v.y = v.y + b.y; v.z = v.z + b.z; v.w = v.w + b.w;
        } else if (addend_mode >= 2) {
            v = apply_addend(v, *reinterpret_cast<const float4*>(addend + i), addend_mode);
        }
        *reinterpret_cast<float4*>(C + i) = v;
        return;
    }
    for (uint64_t e = i; e < i + 4 && e < total; ++e) {
        const uint64_t row = e / N, col = e % N;
        uint64_t w0, w1;
        const uint64_t first = slot_of(row, col, &w0, &w1);
        float v = *at(w0, first, row, col);
        for (uint64_t w = w0 + 1; w <= w1; ++w) v += *at(w, first, row, col);
        if (addend_mode == 1) v = v + addend[col];
        else if (addend_mode >= 2) v = apply_addend(v, addend[e], addend_mode);
        C[e] = v;
    }
}

// C = sum over splits s = 0, 1, ... of partial[s] (+ addend), added in split
// order: deterministic. Four consecutive outputs of one row per thread.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial,
                                                            float* __restrict__ C, uint64_t M,
                                                            uint64_t N, uint32_t splits,
                                                            const float* __restrict__ addend,
                                                            int addend_mode) {
    const uint64_t total = M * N;
    const uint64_t i = (static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    float4 v = mhip::load_nt(reinterpret_cast<const float4*>(partial + i));
    for (uint32_t s = 1; s < splits; ++s) {
        const float4 p = mhip::load_nt(reinterpret_cast<const float4*>(partial + s * total + i));
        v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
    }
    if (addend_mode == 1) {
        const float4 b = *reinterpret_cast<const float4*>(addend + i % N);
        v.x = v.x + b.x; v.y = v.y + b.y; v.z = v.z + b.z; v.w = v.w + b.w;
    } else if (addend_mode >= 2) {
        v = apply_addend(v, *reinterpret_cast<const float4*>(addend + i), addend_mode);
    }
    *reinterpret_cast<float4*>(C + i) = v;
}

// The same, one element per thread (rows that are not whole vectors), eight
// splits' loads in flight.
__global__ __launch_bounds__(256) void splitk_reduce_scalar_kernel(const float* __restrict__ partial,
                                                                   float* __restrict__ C, uint64_t M, uint64_t N,
                                                                   uint32_t splits, const float* __restrict__ addend,
                                                                   int addend_mode) {
    const uint64_t total = M * N;
    const uint64_t e = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= total) return;
    float v = partial[e];
    uint32_t s = 1;
    for (; s + 7 < splits; s += 8) {
        float p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = partial[(s + u) * total + e];
#pragma unroll
        for (int u = 0; u < 8; ++u) v += p[u];
    }
    for (; s < splits; ++s) v += partial[s * total + e];
    if (addend_mode == 1) v = v + addend[e % N];
    else if (addend_mode >= 2) v = apply_addend(v, addend[e], addend_mode);
    C[e] = v;
}

// The same for many splits of few outputs (row panels and ragged GEMVs of a
// long k): 16 waves of 64 V outputs each add a run of the splits in order, eight
// loads in flight, and the runs meet in LDS, in order. What bounds it: the
// chain of loads. 17 x 65536 x 256, 512 splits: the product 151 us with a
// thread per output running through all of them, 28 so.
constexpr int kDeepWaves = 16;
template <int V>
__global__ __launch_bounds__(64 * kDeepWaves) void splitk_reduce_deep_kernel(const float* __restrict__ partial,
                                                                             float* __restrict__ C, uint64_t M,
                                                                             uint64_t N, uint32_t splits,
                                                                             const float* __restrict__ addend,
                                                                             int addend_mode) {
    __shared__ float red[kDeepWaves][V][64];
    const uint64_t total = M * N;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t e = (static_cast<uint64_t>(blockIdx.x) * 64 + lane) * V;
    const uint32_t run = (splits + kDeepWaves - 1) / kDeepWaves;
    const uint32_t s0 = min(splits, wave * run), s1 = min(splits, s0 + run);
    float v[V];
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = 0.0f;
    if (e < total) {  // (V 4: whole vectors)
        constexpr int kU = 8;
        for (uint32_t s = s0; s < s1; s += kU) {
            float p[kU][V];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const float* const at = partial + min(s + u, s1 - 1) * total + e;
                if constexpr (V == 4) {
                    const float4 t = *reinterpret_cast<const float4*>(at);
                    p[u][0] = t.x; p[u][1] = t.y; p[u][2] = t.z; p[u][3] = t.w;
                } else {
                    p[u][0] = *at;
                }
            }
#pragma unroll
            for (int u = 0; u < kU; ++u)
#pragma unroll
                for (int i = 0; i < V; ++i)
                    if (s + u < s1) v[i] += p[u][i];
        }
    }
#pragma unroll
    for (int i = 0; i < V; ++i) red[wave][i][lane] = v[i];
    __syncthreads();
    if (wave != 0 || e >= total) return;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        float t = red[0][i][lane];
#pragma unroll
        for (int w = 1; w < kDeepWaves; ++w) t += red[w][i][lane];
        if (addend_mode == 1) t = t + addend[(e + i) % N];
        else if (addend_mode >= 2) t = apply_addend(t, addend[e + i], addend_mode);
        v[i] = t;
    }
    if constexpr (V == 4) *reinterpret_cast<float4*>(C + e) = make_float4(v[0], v[1], v[2], v[3]);
    else C[e] = v[0];
}

// Adds a product's partial results (splits of m x n at `partial`) into c.
mhip_status launch_splitk_reduce(mhip_ctx* ctx, const float* partial, float* c, uint64_t m, uint64_t n,
                                 uint64_t splits, const float* addend, int mode, const char* what) {
    // dwordx4: whole rows of 4 and 16-byte aligned output and addend.
    const bool vec = n % 4 == 0 && mhip::aligned16(c) && (mode == 0 || mhip::aligned16(addend));
    if (splits >= 64) {
        const uint64_t per = vec ? 256 : 64;
        mhip::launch(ctx, vec ? splitk_reduce_deep_kernel<4> : splitk_reduce_deep_kernel<1>,
                     dim3(static_cast<unsigned>((m * n + per - 1) / per)), dim3(64 * kDeepWaves), 0, partial, c, m, n,
                     static_cast<uint32_t>(splits), addend, mode);
    } else if (vec)
        mhip::launch(ctx, splitk_reduce_kernel, dim3(static_cast<unsigned>((m * n + 1023) / 1024)), dim3(256), 0,
                     partial, c, m, n, static_cast<uint32_t>(splits), addend, mode);
    else
        mhip::launch(ctx, splitk_reduce_scalar_kernel, dim3(static_cast<unsigned>((m * n + 255) / 256)), dim3(256), 0,
                     partial, c, m, n, static_cast<uint32_t>(splits), addend, mode);
    return mhip::check_launch(what);
}

// How many k splits fill the device best: minimises the number of rounds of
// `slots` resident workgroups per unit of full-k work, ceil(tiles * s /
// slots) / s, keeping each split at least 256 deep (and a multiple of bk).
uint64_t choose_splits(uint64_t tiles, uint64_t k, uint64_t slots, uint64_t bk,
                       uint64_t* k_split) {
    uint64_t best = 1;
    double best_cost = static_cast<double>((tiles + slots - 1) / slots);
    for (uint64_t s = 2; s <= 8; ++s) {
        if (k / s < 256) break;
        const double cost = static_cast<double>((tiles * s + slots - 1) / slots) / static_cast<double>(s);
        if (cost < best_cost * (1.0 - 1e-9)) {
            best = s;
            best_cost = cost;
        }
    }
    uint64_t per = (k + best - 1) / best;
    per = (per + bk - 1) / bk * bk;
    *k_split = per;
    return (k + per - 1) / per;
}

// How one tile configuration covers an m x k x n product on `slots`
// resident workgroups: k splits of whole tiles (split-k, one launch per
// round of tiles), or stream-K runs of `per` (tile, k slice) units when that
// gives every workgroup less work (tiles that do not divide the device).
struct GemmPlan {
    uint64_t tiles, kslices;
    uint64_t splits, k_split;  // split-k
    bool stream;
    uint64_t per, groups;      // stream-K: units per workgroup, workgroups
    uint64_t steps;            // k slices per workgroup along the critical path
    double partial_tiles;      // partial-result traffic, in whole products (m x n)
};

GemmPlan plan_gemm(uint64_t m, uint64_t k, uint64_t n, uint64_t bm, uint64_t bn, uint64_t bk,
                   uint64_t slots) {
    GemmPlan p{};
    p.tiles = ((m + bm - 1) / bm) * ((n + bn - 1) / bn);
    p.kslices = (k + bk - 1) / bk;
    p.splits = choose_splits(p.tiles, k, slots, bk, &p.k_split);
    const uint64_t rounds = (p.tiles * p.splits + slots - 1) / slots;
    p.steps = rounds * ((p.k_split + bk - 1) / bk);
    p.partial_tiles = p.splits > 1 ? static_cast<double>(p.splits) : 0.0;
    const uint64_t units = p.tiles * p.kslices;
    const uint64_t per = (units + slots - 1) / slots;
    // Stream-K when it cuts the critical path by over 10 %; its runs must
    // stay within two tiles (per <= kslices) and, as splits do, cover at
    // least 256 of k (8 slices of 32), or partial results outweigh them.
    if (p.tiles < slots && per <= p.kslices && per * bk >= 256 && per * 10 < p.steps * 9) {
        p.stream = true;
        p.per = per;
        p.groups = (units + per - 1) / per;
        p.steps = per;
        p.partial_tiles = static_cast<double>(p.groups + p.tiles) / static_cast<double>(p.tiles);
    }
    return p;
}

// Estimated seconds for a product m rows high and n wide on plan p of one tile configuration:
// the critical path's k slices at the configuration's measured rate (as a
// fraction of the f32 MFMA's peak, which the split products exceed), plus the
// partial results' traffic, plus a fixed cost per launch (a k split or
// stream-K adds the reduction's). Splits are planned for `plan_per_cu`
// workgroups per CU, which share its MFMA pipes; below two waves per SIMD the
// fraction scales with waves per SIMD / 2. Picks among the tile kernels.
// Rates, partial traffic (3-4 TB/s written and read) and launch cost are
// chosen against 2,100 timings of 304 shapes (m 16-4096, k 80-11008, n
// 1024-14336) with each configuration and split forced: the plans picked are
// 2.7 % faster on average than with the f32 MFMA kernels' constants, and up to
// 1.5 times (777 x 4096 x 11008 809 -> 540 us).
double gemm_seconds(const mhip_ctx* ctx, uint64_t m, uint64_t n, const GemmPlan& p, uint64_t bm,
                    uint64_t bn, uint64_t plan_per_cu, int waves, double efficiency, double traffic) {
    const uint64_t cus = ctx->compute_units ? ctx->compute_units : 256;
    const uint64_t slots = plan_per_cu * cus;
    const uint64_t wgs = p.stream ? p.groups : p.tiles * p.splits;
    const uint64_t resident =
        std::max<uint64_t>(1, std::min<uint64_t>(plan_per_cu, (std::min(wgs, slots) + cus - 1) / cus));
    const double per_simd = static_cast<double>(resident * waves) / 4.0;
    const double occupancy = std::min(1.0, per_simd / 2.0);
    const double cu_flops = 157.3e12 / 256.0;  // dense fp32 MFMA per CU per second
    const double slot_flops = cu_flops * efficiency * occupancy / static_cast<double>(resident);
    // A dependent launch costs about 4 us on this device even when it moves
    // little (start-up, the first memory latency, end-of-kernel cache work).
    constexpr double kLaunchSeconds = 4.0e-6;
    double t = static_cast<double>(p.steps) * 2.0 * bm * bn * kSliceK / slot_flops + kLaunchSeconds;
    if (p.partial_tiles > 0.0) t += (p.partial_tiles + 1.0) * m * n * 4.0 / traffic + kLaunchSeconds;
    return t;
}

template <class Shape, bool A_T, bool B_T, class BT>
mhip_status launch_mfma(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t m,
                        uint64_t k, uint64_t n, const float* addend, int mode, Access access) {
    using Tile = typename Shape::template Tile<A_T, B_T, BT>;
    constexpr int BM = Shape::BM, BN = Shape::BN;
    const uint64_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
    if (tiles >= (1ULL << 31)) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "matmul: too many tiles");
    const uint64_t slots = Shape::kPerCu * (ctx->compute_units ? ctx->compute_units : 256);
    const GemmPlan plan = plan_gemm(m, k, n, BM, BN, kSliceK, slots);
    const size_t lds = Tile::kLdsBytes;
    static bool configured = false;  // raise the dynamic-LDS cap above 64 KiB once
    if (!configured) {
        for (const void* f : {reinterpret_cast<const void*>(&mfma_gemm_kernel<Shape, A_T, B_T, BT>),
                              reinterpret_cast<const void*>(&mfma_gemm_stream_kernel<Shape, A_T, B_T, BT>)})
            (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        configured = true;
    }
    const uint64_t groups_out = (m * n + 1023) / 1024;
    if (groups_out >= (1ULL << 31)) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "matmul: output too large");
    // dwordx4 reduction: whole rows of 4 and 16-byte aligned output and addend.
    const int vec4 = n % 4 == 0 && mhip::aligned16(c) && (mode == 0 || mhip::aligned16(addend));

    if (plan.stream) {
        float* slot_mem = nullptr;
        mhip_status st = workspace(ctx, plan.groups * 2 * BM * BN * sizeof(float), &slot_mem);
        if (st != MHIP_OK) return st;
        mhip::launch(ctx, (mfma_gemm_stream_kernel<Shape, A_T, B_T, BT>), dim3(static_cast<unsigned>(plan.groups)),
                     dim3(Tile::kThreads), lds, a, b, slot_mem, m, k, n, plan.per, access);
        st = mhip::check_launch("matmul (MFMA stream-K)");
        if (st != MHIP_OK) return st;
        mhip::launch(ctx, (stream_reduce_kernel<BM, BN>), dim3(static_cast<unsigned>(groups_out)),
                     dim3(256), 0, slot_mem, c, m, n, plan.kslices, plan.per, addend, mode, vec4);
        return mhip::check_launch("matmul (stream-K reduction)");
    }

    float* target = c;
    if (plan.splits > 1) {
        mhip_status st = workspace(ctx, plan.splits * m * n * sizeof(float), &target);
        if (st != MHIP_OK) return st;
    }
    const dim3 grid(static_cast<unsigned>(tiles), static_cast<unsigned>(plan.splits));
    mhip::launch(ctx, (mfma_gemm_kernel<Shape, A_T, B_T, BT>), grid, dim3(Tile::kThreads), lds, a, b, target, m, k,
                 n, addend, mode, plan.k_split, access);
    mhip_status st = mhip::check_launch("matmul (MFMA tiles)");
    if (st != MHIP_OK || plan.splits == 1) return st;
    return launch_splitk_reduce(ctx, target, c, m, n, plan.splits, addend, mode, "matmul (split-k reduction)");
}

template <class Shape, class BT>
mhip_status launch_tiles(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t m, uint64_t k, uint64_t n,
                         bool ta, bool tb, const float* addend, int mode, Access access) {
    if (!ta && !tb) return launch_mfma<Shape, false, false, BT>(ctx, a, b, c, m, k, n, addend, mode, access);
    if (ta && !tb) return launch_mfma<Shape, true, false, BT>(ctx, a, b, c, m, k, n, addend, mode, access);
    if (!ta && tb) return launch_mfma<Shape, false, true, BT>(ctx, a, b, c, m, k, n, addend, mode, access);
    return launch_mfma<Shape, true, true, BT>(ctx, a, b, c, m, k, n, addend, mode, access);
}

// ---------------------------------------------------------------------------
// Decode GEMV: m <= kGemvMaxRows, B row-major [k][n] with n % 4 == 0.
// ---------------------------------------------------------------------------

constexpr int kGemvThreads = 256;
constexpr int kGemvCols = 256;  // columns per workgroup: 64 lanes x 4

// How a GEMV lane reads CPL consecutive columns of one row of B: f32 as one
// dwordx4, compact bf16 as 8 bytes (CPL 4) or one dwordx4 of 8 values (CPL
// 8), kept raw in registers until widened (exactly) at use.
template <class BT, int CPL>
struct GemvLoad;
template <>
struct GemvLoad<float, 4> {
    using Raw = float4;
    template <bool NT>
    static __device__ __forceinline__ Raw load(const float* p) {
        if constexpr (NT) return load4_nt(p);
        else return load4(p);
    }
    static __device__ __forceinline__ float4 part(const Raw& v, int) { return v; }
};
template <>
struct GemvLoad<uint16_t, 4> {
    using Raw = uint2;
    template <bool NT>
    static __device__ __forceinline__ Raw load(const uint16_t* p) {
        if constexpr (NT) {
            const mhip::u32x2 t = __builtin_nontemporal_load(reinterpret_cast<const mhip::u32x2*>(p));
            return make_uint2(t.x, t.y);
        } else {
            return *reinterpret_cast<const uint2*>(p);
        }
    }
    static __device__ __forceinline__ float4 part(const Raw& v, int) { return mhip::widen(v); }
};
template <>
struct GemvLoad<uint16_t, 8> {
    using Raw = uint4;
    template <bool NT>
    static __device__ __forceinline__ Raw load(const uint16_t* p) {
        if constexpr (NT) return mhip::load_nt(reinterpret_cast<const uint4*>(p));
        else return *reinterpret_cast<const uint4*>(p);
    }
    static __device__ __forceinline__ float4 part(const Raw& v, int h) {
        return mhip::widen(h ? make_uint2(v.z, v.w) : make_uint2(v.x, v.y));
    }
};

// One workgroup's share of a decode GEMV: column group `cg` (64 * CPL
// columns, CPL per lane) and k slice `slice`. Its 4 waves split the slice's
// rows and meet in LDS. Each column's sum runs over the same k in the same
// order whatever CPL is, so CPL changes loads, not results.
// `direct`: write C (+ addend) itself (the only slice); otherwise write the
// slice's partial sums for the reduction. STREAM: read B non-temporally (a
// matrix larger than an XCD's L2, read once per call); a small B is read
// through the caches, where it stays between calls. (A template parameter:
// a run-time choice inside the load loop doubled the registers.)
// The GEMV's input as stored: row r of A [rows, K].
struct StoredRows {
    const float* __restrict__ a;
    uint64_t k;
    __device__ __forceinline__ float operator()(int r, uint64_t kk) const { return a[r * k + kk]; }
};

// `A(r, k)` gives the input's row r at k (StoredRows, or a row normalised in
// the launch). `prologue()` runs on every thread after the first batch of B
// rows is in flight (a normalised input's scale; its latency hides under
// theirs), before any A is read.
struct NoPrologue {
    __device__ __forceinline__ void operator()() const {}
};
template <int ROWS, class BT, bool STREAM, int CPL, class AF, class PRO = NoPrologue>
__device__ __forceinline__ void gemv_partial_body(
    const AF& A, const PRO& prologue, const BT* __restrict__ B, float* __restrict__ partial,
    float* __restrict__ C, uint64_t K, uint64_t N, uint64_t k_per_slice, uint32_t cg,
    uint32_t slice, bool direct, const float* __restrict__ addend, int addend_mode) {
    constexpr int H = CPL / 4;  // float4 groups per lane
    using L = GemvLoad<BT, CPL>;
    __shared__ float4 red[4][ROWS][H][64];
    const int lane = threadIdx.x & 63;
    // (A scalar: the stored rows' elements are then scalar loads.)
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const uint64_t col = static_cast<uint64_t>(cg) * (64 * CPL) + lane * CPL;
    const bool live = col < N;  // N % CPL == 0: a live lane's columns are all in range
    const uint64_t k_begin = static_cast<uint64_t>(slice) * k_per_slice;
    const uint64_t k_end = min(K, k_begin + k_per_slice);
    float4 acc[ROWS][H];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int h = 0; h < H; ++h) acc[r][h] = make_float4(0.f, 0.f, 0.f, 0.f);
    auto fma_row = [&](const typename L::Raw& raw, uint64_t k) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const float4 b = L::part(raw, h);
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const float a = A(r, k);
                acc[r][h].x = __builtin_fmaf(a, b.x, acc[r][h].x);
                acc[r][h].y = __builtin_fmaf(a, b.y, acc[r][h].y);
                acc[r][h].z = __builtin_fmaf(a, b.z, acc[r][h].z);
                acc[r][h].w = __builtin_fmaf(a, b.w, acc[r][h].w);
            }
        }
    };
    // B rows in flight per lane: 256 bytes for compact weights read 8
    // columns at a time and for blocks of 8 rows of a small matrix (measured:
    // bf16 1x4096x11008 22.1 -> 18.3 us, the C1 block 80 -> 61 us), 128 bytes
    // otherwise (256 was no faster for the f32 decode GEMVs, and for 8 rows of
    // a large one its registers cost the waves that hide the latency: with A's
    // elements as scalar loads, 8x4096x32000 184 -> 92 us, compact 158 -> 82).
    constexpr int kU = (CPL == 8 || (ROWS >= 8 && !STREAM) ? 256 : 128) / sizeof(typename L::Raw);
    // Slices are multiples of 32 rows, 8 a wave: where a batch is longer, the
    // rows past whole batches go in one of 8, not one by one (compact down and
    // gate/up streams of a decoder step end in such 8, its K and V slices are
    // nothing else: the step 113 -> 107 us).
    constexpr int kTail = kU > 8 ? 8 : kU;
    uint64_t kk = k_begin + wave;
    typename L::Raw first[kU];
    const bool first_batch = live && kk + 4 * (kU - 1) < k_end;
    const bool first_tail = kTail < kU && live && !first_batch && kk + 4 * (kTail - 1) < k_end;
    if (first_batch) {
#pragma unroll
        for (int u = 0; u < kU; ++u) first[u] = L::template load<STREAM>(B + (kk + 4 * u) * N + col);
    } else if (first_tail) {
#pragma unroll
        for (int u = 0; u < kTail; ++u) first[u] = L::template load<STREAM>(B + (kk + 4 * u) * N + col);
    }
    prologue();
    if (live) {
        if (first_batch) {
#pragma unroll
            for (int u = 0; u < kU; ++u) fma_row(first[u], kk + 4 * u);
            kk += 4 * kU;
        } else if (first_tail) {
#pragma unroll
            for (int u = 0; u < kTail; ++u) fma_row(first[u], kk + 4 * u);
            kk += 4 * kTail;
        }
        for (; kk + 4 * (kU - 1) < k_end; kk += 4 * kU) {
            typename L::Raw bv[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) bv[u] = L::template load<STREAM>(B + (kk + 4 * u) * N + col);
#pragma unroll
            for (int u = 0; u < kU; ++u) fma_row(bv[u], kk + 4 * u);
        }
        if constexpr (kTail < kU) {
            for (; kk + 4 * (kTail - 1) < k_end; kk += 4 * kTail) {
                typename L::Raw bv[kTail];
#pragma unroll
                for (int u = 0; u < kTail; ++u) bv[u] = L::template load<STREAM>(B + (kk + 4 * u) * N + col);
#pragma unroll
                for (int u = 0; u < kTail; ++u) fma_row(bv[u], kk + 4 * u);
            }
        }
        for (; kk < k_end; kk += 4) fma_row(L::template load<STREAM>(B + kk * N + col), kk);
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int h = 0; h < H; ++h) red[wave][r][h][lane] = acc[r][h];
    __syncthreads();
    if (wave != 0 || !live) return;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const uint64_t c = col + 4 * h;
            float4 v = red[0][r][h][lane];
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                const float4 o = red[w][r][h][lane];
                v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
            }
            if (direct) {
                if (addend_mode == 1) {
                    const float4 b4 = *reinterpret_cast<const float4*>(addend + c);
                    v.x = v.x + b4.x; v.y = v.y + b4.y; v.z = v.z + b4.z; v.w = v.w + b4.w;
                } else if (addend_mode >= 2) {
                    v = apply_addend(v, *reinterpret_cast<const float4*>(addend + r * N + c), addend_mode);
                }
                *reinterpret_cast<float4*>(C + r * N + c) = v;
            } else {
                *reinterpret_cast<float4*>(partial + (static_cast<uint64_t>(slice) * ROWS + r) * N + c) = v;
            }
        }
    }
}

// blockIdx.z is a block of ROWS rows of A and C: each is an independent
// ROWS-row GEMV with its own partial sums (B is shared through L2).
template <int ROWS, class BT, bool STREAM, int CPL>
__global__ __launch_bounds__(kGemvThreads) void gemv_partial_kernel(
    const float* __restrict__ A, const BT* __restrict__ B, float* __restrict__ partial,
    float* __restrict__ C, uint64_t K, uint64_t N, uint64_t k_per_slice, uint32_t slices,
    const float* __restrict__ addend, int addend_mode) {
    const uint64_t rb = blockIdx.z;
    A += rb * ROWS * K;
    C += rb * ROWS * N;
    if (partial) partial += rb * slices * ROWS * N;
    if (addend_mode >= 2) addend += rb * ROWS * N;
    gemv_partial_body<ROWS, BT, STREAM, CPL>(StoredRows{A, K}, NoPrologue{}, B, partial, C, K, N, k_per_slice,
                                             blockIdx.x, blockIdx.y, slices == 1, addend, addend_mode);
}

// A one-row decode GEMV whose input row is attention's output, merged here
// from its key-chunk records (mhip::merge_decode_chunks, the merge kernel's
// order) instead of by a merge launch: each workgroup merges its k slice,
// which lies within one head of D = 4 * D4 columns, into LDS once its first
// weight rows are in flight.
template <class BT, bool STREAM, int CPL, int D4>
__global__ __launch_bounds__(kGemvThreads) void gemv_partial_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, uint64_t chunks,
    const BT* __restrict__ B, float* __restrict__ partial, uint64_t K, uint64_t N,
    uint64_t k_per_slice, uint32_t slices) {
    static_assert(kGemvThreads == 256, "the merge takes 256 threads");
    constexpr int D = 4 * D4;
    __shared__ float sa[D];
    const uint32_t slice = blockIdx.y;
    const uint64_t k0 = static_cast<uint64_t>(slice) * k_per_slice;
    const uint64_t head = k0 / D;
    const int q0 = static_cast<int>(k0 % D) / 4;
    const int nq = static_cast<int>(min(K, k0 + k_per_slice) - k0) / 4;
    auto merge = [&]() {
        const float4 v = mhip::merge_decode_chunks<D4>(part_ml + 2 * head * chunks,
                                                       part_o + head * chunks * D, chunks, q0, nq);
        if (static_cast<int>(threadIdx.x) >= q0 && static_cast<int>(threadIdx.x) < q0 + nq)
            *reinterpret_cast<float4*>(sa + 4 * (threadIdx.x - q0)) = v;
        __syncthreads();
    };
    auto merged = [&](int, uint64_t k) { return sa[k - k0]; };
    gemv_partial_body<1, BT, STREAM, CPL>(merged, merge, B, partial, nullptr, K, N, k_per_slice,
                                          blockIdx.x, slice, slices == 1, nullptr, 0);
}

// Sums of the slices' partial sums of 256 columns, for NSEG matrices of the
// same shape at once: wave w adds a fixed quarter of the slices, each row in
// slice order, then wave 0 adds the quarters in order -- the same order on
// every run. Loads go out in batches of 16 float4 (every segment's rows of
// 16 / (ROWS * NSEG) slices) before any is added, so a quarter costs
// ceil(slices / 4 / batch) memory round trips for all segments together,
// not one per slice, row or segment. The results are valid in wave 0 only;
// every thread of the workgroup must call it (it synchronises), and a second
// call must come after a __syncthreads().
template <int ROWS, int NSEG = 1>
__device__ __forceinline__ void gemv_reduce_sum(const float* const (&partial)[NSEG], uint64_t N,
                                                uint32_t slices, uint64_t col, bool live,
                                                float4 (&out)[NSEG][ROWS]) {
    __shared__ float4 red[4][ROWS][64];
    constexpr int kBatch = ROWS * NSEG >= 16 ? 1 : 16 / (ROWS * NSEG);  // slices per batch
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t quarter = (slices + 3) / 4;
    const uint32_t s_begin = min(slices, wave * quarter), s_end = min(slices, s_begin + quarter);
    float4 v[NSEG][ROWS];
#pragma unroll
    for (int q = 0; q < NSEG; ++q)
#pragma unroll
        for (int r = 0; r < ROWS; ++r) v[q][r] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (live) {
        for (uint32_t s = s_begin; s < s_end; s += kBatch) {
            float4 p[NSEG][kBatch][ROWS];
#pragma unroll
            for (int q = 0; q < NSEG; ++q)
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
#pragma unroll
                    for (int r = 0; r < ROWS; ++r)
                        if (s + u < s_end)
                            p[q][u][r] = *reinterpret_cast<const float4*>(
                                partial[q] + ((s + u) * static_cast<uint64_t>(ROWS) + r) * N + col);
#pragma unroll
            for (int q = 0; q < NSEG; ++q)
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
#pragma unroll
                    for (int r = 0; r < ROWS; ++r)
                        if (s + u < s_end) {
                            v[q][r].x += p[q][u][r].x; v[q][r].y += p[q][u][r].y;
                            v[q][r].z += p[q][u][r].z; v[q][r].w += p[q][u][r].w;
                        }
        }
    }
#pragma unroll
    for (int q = 0; q < NSEG; ++q) {
        if (q > 0) __syncthreads();  // wave 0 has read the previous segment's quarters
#pragma unroll
        for (int r = 0; r < ROWS; ++r) red[wave][r][lane] = v[q][r];
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                float4 t = red[0][r][lane];
#pragma unroll
                for (int w = 1; w < 4; ++w) {
                    const float4 o = red[w][r][lane];
                    t.x += o.x; t.y += o.y; t.z += o.z; t.w += o.w;
                }
                out[q][r] = t;
            }
        }
    }
}

// C = the slices' partial sums (+ addend).
// chunk_ss (one row): also the RMSNorm chunk sum of squares of the 256
// columns written (mhip::chunk_sumsq), at chunk_ss[column group].
template <int ROWS>
__global__ __launch_bounds__(kGemvThreads) void gemv_reduce_kernel(
    const float* __restrict__ partial, float* __restrict__ C, uint64_t N, uint32_t slices,
    const float* __restrict__ addend, int addend_mode, float* __restrict__ chunk_ss) {
    const uint64_t rb = blockIdx.z;  // row block, as in gemv_partial_kernel
    partial += rb * slices * ROWS * N;
    C += rb * ROWS * N;
    if (addend_mode >= 2) addend += rb * ROWS * N;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t col = static_cast<uint64_t>(blockIdx.x) * kGemvCols + lane * 4;
    const bool live = col < N;
    // The addend goes out with the partial sums (one memory round trip).
    float4 add[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        add[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (wave == 0 && live && addend_mode != 0)
            add[r] = *reinterpret_cast<const float4*>(addend + (addend_mode >= 2 ? r * N : 0) + col);
    }
    float4 v[1][ROWS];
    gemv_reduce_sum<ROWS>({partial}, N, slices, col, live, v);
    if (wave != 0) return;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        float4& o = v[0][r];
        if (!live) {
            o = make_float4(0.f, 0.f, 0.f, 0.f);
            continue;
        }
        if (addend_mode == 3) {
            o = apply_addend(o, add[r], 3);
        } else if (addend_mode != 0) {
            o.x = o.x + add[r].x; o.y = o.y + add[r].y; o.z = o.z + add[r].z; o.w = o.w + add[r].w;
        }
        *reinterpret_cast<float4*>(C + r * N + col) = o;
    }
    if constexpr (ROWS == 1) {
        if (chunk_ss) {
            const float cs = mhip::chunk_sumsq(v[0][0]);  // dead lanes hold zeros
            if (lane == 0) chunk_ss[blockIdx.x] = cs;
        }
    }
}

// ---------------------------------------------------------------------------
// Sets of decode GEMVs over one input, with fused epilogues
// ---------------------------------------------------------------------------

struct GemvSeg {
    const void* b;  // f32, or bf16 bits (the set's element type)
    float* partial;
    float* out;
    const uint64_t* out_advance;  // captured step: rows of `out` move by the replay offset
    uint64_t n;
    uint64_t k_per_slice;
    uint32_t col_groups, slices;
    uint32_t first_block;  // this segment's first workgroup in the partial launch
    uint32_t first_group;  // ... and in the reduction launch
};

struct GemvSet {
    GemvSeg seg[3];
    int count;
};

// Rotation of one projection's rows: interleaved pairs, head_width and
// dimension multiples of 4 (the vector RoPE kernel's case).
struct RopeEpi {
    const float* table;  // [half] frequencies then [half] amplitudes
    uint64_t head_width, dimension, half, offset;
    float scale;
    const uint64_t* advance;  // captured step: replay offset added to `offset`
};

// Segment `i` of the set with constant indices, so the fields stay in the
// kernel argument segment.
__device__ __forceinline__ GemvSeg pick(const GemvSet& set, int i) {
    if (i == 0) return set.seg[0];
    if (i == 1) return set.seg[1];
    return set.seg[2];
}

// A set's single input row normalised by RMSNorm inside the partial launch
// (the decode block's FFN RMSNorm): a[k] = src[k] * inv * gain[k], with inv
// from the row's chunk sums of squares (mhip::chunk_sumsq, written by the
// launch that produced the row) added in order -- the RMSNorm kernel's bits,
// for a prologue of `chunks` scalar reads instead of the whole row.
struct NormIn {
    const float* src;
    const float* chunk_ss;
    const float* gain;
    float eps;
    uint32_t chunks;
};

// Longest k slice a normalised input can have (its LDS staging).
constexpr uint64_t kNormSliceMax = 4096;

// NORM: 0, rows of A as stored; 1, the single row norm.src normalised.
template <int ROWS, class BT, bool STREAM, int CPL, int NORM>
__global__ __launch_bounds__(kGemvThreads) void gemv_set_partial_kernel(const float* __restrict__ A,
                                                                        uint64_t K, GemvSet set,
                                                                        NormIn norm) {
    const uint32_t b = blockIdx.x;
    const int i = (set.count > 2 && b >= set.seg[2].first_block) ? 2
                  : (set.count > 1 && b >= set.seg[1].first_block) ? 1 : 0;
    const GemvSeg s = pick(set, i);
    const uint32_t local = b - s.first_block;
    const uint64_t rb = blockIdx.y;  // row block of ROWS rows
    const BT* B = static_cast<const BT*>(s.b);
    float* partial = s.partial + rb * s.slices * ROWS * s.n;
    const uint32_t cg = local % s.col_groups, slice = local / s.col_groups;
    if constexpr (NORM == 0) {
        gemv_partial_body<ROWS, BT, STREAM, CPL>(StoredRows{A + rb * ROWS * K, K}, NoPrologue{}, B,
                                                 partial, nullptr, K, s.n, s.k_per_slice, cg, slice,
                                                 false, nullptr, 0);
    } else {
        static_assert(ROWS == 1, "a normalised input is one row");
        // The workgroup's k slice of the normalised row, staged in LDS once.
        __shared__ float sa[kNormSliceMax];
        const uint64_t k0 = static_cast<uint64_t>(slice) * s.k_per_slice;
        const uint64_t len = min(K, k0 + s.k_per_slice) - k0;
        auto scale = [&]() {
            float ss = 0.0f;
            for (uint32_t c = 0; c < norm.chunks; ++c) ss = ss + norm.chunk_ss[c];
            const float inv = mhip::inv_rms(ss, K, norm.eps);
            for (uint64_t j = threadIdx.x; j < len; j += kGemvThreads) {
                const float y = norm.src[k0 + j] * inv;
                sa[j] = norm.gain ? y * norm.gain[k0 + j] : y;
            }
            __syncthreads();
        };
        auto normed = [&](int, uint64_t k) { return sa[k - k0]; };
        gemv_partial_body<1, BT, STREAM, CPL>(normed, scale, B, partial, nullptr, K, s.n,
                                              s.k_per_slice, cg, slice, false, nullptr, 0);
    }
}

// The RoPE factors of one lane's 4 columns (two pairs): read before the
// reduction's partial sums are awaited, so they cost no round trip of their own.
struct RopeCoef {
    float f0, a0, f1, a1;  // frequency and amplitude of the two pairs
    uint64_t offset;
    bool on;               // the columns lie in the rotated dimensions
};

__device__ __forceinline__ RopeCoef rope_coef(const RopeEpi& e, uint64_t col) {
    RopeCoef c{};
    const uint64_t j = col % e.head_width;
    c.on = j < e.dimension;
    if (c.on) {
        const uint64_t p = j / 2;
        c.f0 = e.table[p];
        c.a0 = e.table[e.half + p];
        c.f1 = e.table[p + 1];
        c.a1 = e.table[e.half + p + 1];
    }
    c.offset = e.offset + (e.advance ? *e.advance : 0);
    return c;
}

__device__ __forceinline__ float4 rope_vec(const RopeCoef& c, float scale, uint64_t row, float4 v) {
    if (!c.on) return v;
    const float position = mhip::rope_position(c.offset, row, scale);
    float c0, s0, c1, s1;
    mhip::rope_freq_cs(position, c.f0, c.a0, &c0, &s0);
    mhip::rope_freq_cs(position, c.f1, c.a1, &c1, &s1);
    float4 r;
    mhip::rope_rotate(v.x, v.y, c0, s0, &r.x, &r.y);
    mhip::rope_rotate(v.z, v.w, c1, s1, &r.z, &r.w);
    return r;
}

template <int ROWS>
__global__ __launch_bounds__(kGemvThreads) void gemv_set_reduce_kernel(GemvSet set, int epilogue,
                                                                       RopeEpi rope_q,
                                                                       RopeEpi rope_k) {
    const uint32_t b = blockIdx.x;
    const int i = (set.count > 2 && b >= set.seg[2].first_group) ? 2
                  : (set.count > 1 && b >= set.seg[1].first_group) ? 1 : 0;
    const GemvSeg s = pick(set, i);
    const uint64_t rb = blockIdx.y;  // row block, as in gemv_set_partial_kernel
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t col = static_cast<uint64_t>(b - s.first_group) * kGemvCols + lane * 4;
    const bool live = col < s.n;
    float* out = s.out + rb * ROWS * s.n;
    if (epilogue == mhip::kGemvSiluMul) {
        // Gate (segment 0) and up (segment 1, the same columns) summed together.
        const GemvSeg u = pick(set, 1);
        const uint64_t advance = (wave == 0 && s.out_advance) ? *s.out_advance : 0;
        float4 v[2][ROWS];
        gemv_reduce_sum<ROWS, 2>({s.partial + rb * s.slices * ROWS * s.n,
                                  u.partial + rb * u.slices * ROWS * u.n},
                                 s.n, s.slices, col, live, v);
        if (wave != 0 || !live) return;
        out += advance * s.n;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            float4 o;
            o.x = mhip::silu1(v[0][r].x) * v[1][r].x;
            o.y = mhip::silu1(v[0][r].y) * v[1][r].y;
            o.z = mhip::silu1(v[0][r].z) * v[1][r].z;
            o.w = mhip::silu1(v[0][r].w) * v[1][r].w;
            *reinterpret_cast<float4*>(out + r * s.n + col) = o;
        }
        return;
    }
    const bool rotate = epilogue == mhip::kGemvRopeQK && i < 2;
    RopeCoef coef{};
    uint64_t advance = 0;
    if (wave == 0 && live) {
        if (rotate) coef = rope_coef(i == 0 ? rope_q : rope_k, col);
        if (s.out_advance) advance = *s.out_advance;
    }
    float4 v[1][ROWS];
    gemv_reduce_sum<ROWS>({s.partial + rb * s.slices * ROWS * s.n}, s.n, s.slices, col, live, v);
    if (wave != 0 || !live) return;
    out += advance * s.n;
    const float scale = i == 0 ? rope_q.scale : rope_k.scale;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        float4 o = v[0][r];
        if (rotate) o = rope_vec(coef, scale, rb * ROWS + r, o);
        *reinterpret_cast<float4*>(out + r * s.n + col) = o;
    }
}

// Whether a GEMV reads its matrix non-temporally: one larger than an XCD's
// 4 MB L2 is streamed; a smaller one is kept in the caches across calls
// (the small blocks' weights), which saves a trip to HBM per launch.
bool gemv_streams_b(uint64_t bytes) { return bytes > (4ull << 20); }

// Split-k shape of a decode GEMV: about four workgroups per CU, each slice a
// multiple of 32 rows (four waves x eight rows in flight); one slice when
// the column groups alone fill the device.
void gemv_slicing(const mhip_ctx* ctx, uint64_t k, uint64_t n, uint64_t* slices_out,
                  uint64_t* k_per_slice_out) {
    const uint64_t col_groups = (n + kGemvCols - 1) / kGemvCols;
    const uint64_t target_blocks = static_cast<uint64_t>(ctx->compute_units ? ctx->compute_units : 256) * 4;
    uint64_t slices = (target_blocks + col_groups - 1) / col_groups;
    uint64_t k_per_slice = ((k + slices - 1) / slices + 31) / 32 * 32;
    if (k_per_slice < 32) k_per_slice = 32;
    slices = (k + k_per_slice - 1) / k_per_slice;
    if (slices <= 1) {
        slices = 1;
        k_per_slice = k;
    }
    *slices_out = slices;
    *k_per_slice_out = k_per_slice;
}

// Compact weights on up to 4 rows read 8 columns per lane (16-byte loads)
// when every row of B starts 16-byte aligned; otherwise 4.
template <int ROWS, class BT>
constexpr bool kGemvWideable = sizeof(BT) == 2 && ROWS <= 4;

template <int ROWS, class BT, int CPL>
void launch_gemv_partial(mhip_ctx* ctx, dim3 grid, bool stream, const float* a, const BT* b,
                         float* partial, float* c, uint64_t k, uint64_t n, uint64_t k_per_slice,
                         uint64_t slices, const float* addend, int mode) {
    if (stream)
        mhip::launch(ctx, (gemv_partial_kernel<ROWS, BT, true, CPL>), grid, dim3(kGemvThreads), 0, a,
                     b, partial, c, k, n, k_per_slice, static_cast<uint32_t>(slices), addend, mode);
    else
        mhip::launch(ctx, (gemv_partial_kernel<ROWS, BT, false, CPL>), grid, dim3(kGemvThreads), 0,
                     a, b, partial, c, k, n, k_per_slice, static_cast<uint32_t>(slices), addend,
                     mode);
}

// chunk_ss (one row, split k): the output's RMSNorm chunk sums too.
template <int ROWS, class BT>
mhip_status launch_gemv(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t k,
                        uint64_t n, const float* addend, int mode, uint64_t row_blocks = 1,
                        float* chunk_ss = nullptr) {
    const uint64_t col_groups = (n + kGemvCols - 1) / kGemvCols;  // of the reduction
    uint64_t slices, k_per_slice;
    gemv_slicing(ctx, k, n, &slices, &k_per_slice);
    float* partial = nullptr;
    if (slices > 1) {
        mhip_status st = workspace(ctx, row_blocks * slices * ROWS * n * sizeof(float), &partial);
        if (st != MHIP_OK) return st;
    }
    const bool stream = gemv_streams_b(k * n * sizeof(BT));
    bool wide = false;
    if constexpr (kGemvWideable<ROWS, BT>) wide = n % 8 == 0 && mhip::aligned16(b);
    const uint64_t part_groups = wide ? (n + 511) / 512 : col_groups;
    const dim3 grid(static_cast<unsigned>(part_groups), static_cast<unsigned>(slices),
                    static_cast<unsigned>(row_blocks));
    if constexpr (kGemvWideable<ROWS, BT>) {
        if (wide)
            launch_gemv_partial<ROWS, BT, 8>(ctx, grid, stream, a, b, partial, c, k, n, k_per_slice,
                                             slices, addend, mode);
        else
            launch_gemv_partial<ROWS, BT, 4>(ctx, grid, stream, a, b, partial, c, k, n, k_per_slice,
                                             slices, addend, mode);
    } else {
        launch_gemv_partial<ROWS, BT, 4>(ctx, grid, stream, a, b, partial, c, k, n, k_per_slice,
                                         slices, addend, mode);
    }
    mhip_status st = mhip::check_launch("matmul (decode partial sums)");
    if (st != MHIP_OK || slices == 1) return st;
    mhip::launch(ctx, gemv_reduce_kernel<ROWS>,
                 dim3(static_cast<unsigned>(col_groups), 1, static_cast<unsigned>(row_blocks)),
                 dim3(kGemvThreads), 0, partial, c, n, static_cast<uint32_t>(slices), addend, mode,
                 chunk_ss);
    return mhip::check_launch("matmul (decode reduction)");
}

template <int ROWS, class BT, int CPL, int NORM>
void launch_gemv_set_partial_n(mhip_ctx* ctx, dim3 grid, bool stream, const float* a, uint64_t k,
                               const GemvSet& set, const NormIn& norm) {
    if (stream)
        mhip::launch(ctx, (gemv_set_partial_kernel<ROWS, BT, true, CPL, NORM>), grid,
                     dim3(kGemvThreads), 0, a, k, set, norm);
    else
        mhip::launch(ctx, (gemv_set_partial_kernel<ROWS, BT, false, CPL, NORM>), grid,
                     dim3(kGemvThreads), 0, a, k, set, norm);
}

// `norm_mode` (NORM of gemv_set_partial_kernel) is nonzero only for one row.
template <int ROWS, class BT, int CPL>
void launch_gemv_set_partial(mhip_ctx* ctx, dim3 grid, bool stream, const float* a, uint64_t k,
                             const GemvSet& set, int norm_mode, const NormIn& norm) {
    if constexpr (ROWS == 1) {
        if (norm_mode == 1) return launch_gemv_set_partial_n<1, BT, CPL, 1>(ctx, grid, stream, a, k, set, norm);
    }
    launch_gemv_set_partial_n<ROWS, BT, CPL, 0>(ctx, grid, stream, a, k, set, norm);
}

// `wide`: the set's segments were planned with 8 columns per lane.
template <int ROWS, class BT>
mhip_status launch_gemv_set(mhip_ctx* ctx, const float* a, uint64_t k, GemvSet set, int epilogue,
                            const RopeEpi& rq, const RopeEpi& rk, uint32_t reduce_groups,
                            bool stream, bool wide, int norm_mode, const NormIn& norm,
                            uint32_t row_blocks = 1) {
    uint32_t blocks = 0;
    for (int i = 0; i < set.count; ++i) blocks += set.seg[i].col_groups * set.seg[i].slices;
    const dim3 grid(blocks, row_blocks);
    if constexpr (kGemvWideable<ROWS, BT>) {
        if (wide) launch_gemv_set_partial<ROWS, BT, 8>(ctx, grid, stream, a, k, set, norm_mode, norm);
        else launch_gemv_set_partial<ROWS, BT, 4>(ctx, grid, stream, a, k, set, norm_mode, norm);
    } else {
        if (wide) return MHIP_LAYOUT_UNSUPPORTED;
        launch_gemv_set_partial<ROWS, BT, 4>(ctx, grid, stream, a, k, set, norm_mode, norm);
    }
    mhip_status st = mhip::check_launch("decode projections (partial sums)");
    if (st != MHIP_OK) return st;
    mhip::launch(ctx, gemv_set_reduce_kernel<ROWS>, dim3(reduce_groups, row_blocks),
                 dim3(kGemvThreads), 0, set, epilogue, rq, rk);
    return mhip::check_launch("decode projections (reduction)");
}

template <class BT>
mhip_status dispatch_gemv(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t m,
                          uint64_t k, uint64_t n, const float* addend, int mode) {
    switch (m) {
        case 1: return launch_gemv<1, BT>(ctx, a, b, c, k, n, addend, mode);
        case 2: return launch_gemv<2, BT>(ctx, a, b, c, k, n, addend, mode);
        case 3: return launch_gemv<3, BT>(ctx, a, b, c, k, n, addend, mode);
        case 4: return launch_gemv<4, BT>(ctx, a, b, c, k, n, addend, mode);
        case 5: return launch_gemv<5, BT>(ctx, a, b, c, k, n, addend, mode);
        case 6: return launch_gemv<6, BT>(ctx, a, b, c, k, n, addend, mode);
        case 7: return launch_gemv<7, BT>(ctx, a, b, c, k, n, addend, mode);
        default: return launch_gemv<8, BT>(ctx, a, b, c, k, n, addend, mode);
    }
}

// Small products of 16-32 rows in one launch (no partial sums, no reduction
// launch): a workgroup of kSmallWaves waves owns a 32 x 32 tile of C. Wave w
// takes k range [w * kq, (w + 1) * kq) (kq a multiple of 8; the last ranges
// short or empty) and sums it with v_mfma_f32_32x32x2_f32 in the k order
// 8g + 4h + e of the MFMA tiles: lane half h feeds A[row][g + 4h + e] from one
// 16-byte load and B[g + 4h + e][col]. Loads go out two k groups at a time.
// The waves' partial tiles meet in LDS and wave r adds register row r over
// the waves in wave order. Each output's sum depends only on its own row and
// column, so any row subset of a product taking this path gives the same
// bits, and a set of products (the GEMV sets' epilogues) the bits of each.
constexpr int kSmallWaves = 16;
constexpr uint64_t kSmallMaxK = 1024;
static_assert(kSmallWaves == 16, "one register row of the 32 x 32 tile per wave");

// The tile's sums at (small_row(row0), col0 + lane % 32) for the calling
// wave, of A times each of the T matrices B[t] (same shape; T = 2 for a
// gate/up pair shares A's loads and issues both matrices' loads together).
// Every thread of the workgroup calls it (it synchronises).
template <class BT, int T>
__device__ __forceinline__ void small_tiles(const float* __restrict__ A,
                                            const BT* const (&B)[T], uint64_t M, uint64_t K,
                                            uint64_t N, uint64_t kq, uint64_t row0, uint64_t col0,
                                            float (*red)[16][64], float (&out)[T]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    const uint64_t kb = wave * kq, ke = min(K, kb + kq);
    const uint64_t arow = row0 + l32, bcol = col0 + l32;
    const bool arow_ok = arow < M, bcol_ok = bcol < N;
    const float* ap = A + arow * K;
    v16f acc[T];
#pragma unroll
    for (int m = 0; m < T; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = 0.0f;
    constexpr int kBatch = 2;  // k groups of 8 per batch of loads
    for (uint64_t g0 = kb; g0 < ke; g0 += 8 * kBatch) {
        float4 a4[kBatch];
        float bv[T][kBatch][4];
#pragma unroll
        for (int t = 0; t < kBatch; ++t) {
            const uint64_t kk = g0 + 8 * t + 4 * h;  // K % 4 == 0: all four or none
            a4[t] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (arow_ok && kk < ke) a4[t] = *reinterpret_cast<const float4*>(ap + kk);
#pragma unroll
            for (int m = 0; m < T; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    bv[m][t][e] = (bcol_ok && kk + e < ke) ? elem(B[m] + (kk + e) * N + bcol) : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < T; ++m)
#pragma unroll
            for (int t = 0; t < kBatch; ++t) {
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a4[t].x, bv[m][t][0], acc[m], 0, 0, 0);
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a4[t].y, bv[m][t][1], acc[m], 0, 0, 0);
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a4[t].z, bv[m][t][2], acc[m], 0, 0, 0);
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a4[t].w, bv[m][t][3], acc[m], 0, 0, 0);
            }
    }
#pragma unroll
    for (int m = 0; m < T; ++m) {
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave][r][lane] = acc[m][r];
        __syncthreads();
        float v = red[0][wave][lane];
#pragma unroll
        for (int w = 1; w < kSmallWaves; ++w) v += red[w][wave][lane];
        out[m] = v;
        __syncthreads();  // `red` is written again
    }
}

template <class BT>
__device__ __forceinline__ float small_tile(const float* __restrict__ A, const BT* __restrict__ B,
                                            uint64_t M, uint64_t K, uint64_t N, uint64_t kq,
                                            uint64_t row0, uint64_t col0,
                                            float (*red)[16][64]) {
    const BT* const bs[1] = {B};
    float v[1];
    small_tiles<BT, 1>(A, bs, M, K, N, kq, row0, col0, red, v);
    return v[0];
}

// Register row r = wave of the tile holds row row0 + 8 (r / 4) + 4h + r % 4.
__device__ __forceinline__ uint64_t small_row(uint64_t row0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    return row0 + 8 * (wave / 4) + 4 * (lane >> 5) + (wave % 4);
}

template <class BT>
__global__ __launch_bounds__(64 * kSmallWaves) void small_mfma_kernel(
    const float* __restrict__ A, const BT* __restrict__ B, float* __restrict__ C, uint64_t M,
    uint64_t K, uint64_t N, uint64_t kq, const float* __restrict__ addend, int addend_mode) {
    __shared__ float red[kSmallWaves][16][64];
    const uint64_t col0 = static_cast<uint64_t>(blockIdx.x) * 32;
    const uint64_t row0 = static_cast<uint64_t>(blockIdx.y) * 32;
    float v = small_tile<BT>(A, B, M, K, N, kq, row0, col0, red);
    const uint64_t row = small_row(row0), col = col0 + (threadIdx.x & 31);
    if (row >= M || col >= N) return;
    if (addend_mode == 1) v = v + addend[col];
    else if (addend_mode >= 2) v = apply_addend(v, addend[row * N + col], addend_mode);
    C[row * N + col] = v;
}

// A GEMV set (gemv_set_f32) of 16-32 rows on the small tiles: workgroup x
// takes a 32-column tile of one target (targets' tiles in order); with the
// silu-mul epilogue the workgroup sums the gate and up tiles of the same
// columns together and stores silu(gate) * up; with the RoPE epilogue targets 0
// and 1 rotate each interleaved pair (columns 2i, 2i + 1, in lanes l, l ^ 1)
// with the factors of the vector RoPE kernel. Each target's sums are those of
// small_mfma_kernel for it alone.
struct SmallSeg {
    const void* b;
    float* out;
    const uint64_t* out_advance;  // captured step: rows of `out` move by the replay offset
    uint64_t n;
    uint32_t first_tile;
};

struct SmallSet {
    SmallSeg seg[3];
    int count;
};

__device__ __forceinline__ SmallSeg pick(const SmallSet& set, int i) {
    if (i == 0) return set.seg[0];
    if (i == 1) return set.seg[1];
    return set.seg[2];
}

template <class BT>
__global__ __launch_bounds__(64 * kSmallWaves) void small_mfma_set_kernel(
    const float* __restrict__ A, uint64_t M, uint64_t K, uint64_t kq, SmallSet set, int epilogue,
    RopeEpi rope_q, RopeEpi rope_k) {
    __shared__ float red[kSmallWaves][16][64];
    const uint32_t b = blockIdx.x;
    const int i = (set.count > 2 && b >= set.seg[2].first_tile) ? 2
                  : (set.count > 1 && b >= set.seg[1].first_tile) ? 1 : 0;
    const SmallSeg s = pick(set, i);
    const int l32 = threadIdx.x & 31;
    const uint64_t col0 = static_cast<uint64_t>(b - s.first_tile) * 32;
    const uint64_t row0 = static_cast<uint64_t>(blockIdx.y) * 32;
    const uint64_t row = small_row(row0), col = col0 + l32;
    float v;
    if (epilogue == mhip::kGemvSiluMul) {
        // Gate (segment 0) and up (segment 1, the same columns) summed together.
        const BT* const bs[2] = {static_cast<const BT*>(s.b), static_cast<const BT*>(set.seg[1].b)};
        float gu[2];
        small_tiles<BT, 2>(A, bs, M, K, s.n, kq, row0, col0, red, gu);
        v = mhip::silu1(gu[0]) * gu[1];
    } else {
        v = small_tile<BT>(A, static_cast<const BT*>(s.b), M, K, s.n, kq, row0, col0, red);
    }
    if (epilogue == mhip::kGemvRopeQK && i < 2) {
        const float other = __shfl_xor(v, 1, 64);  // the pair's other column
        const RopeEpi& e = i == 0 ? rope_q : rope_k;
        const uint64_t j = col % e.head_width;
        if (j < e.dimension) {
            const uint64_t p = j / 2;
            const float position =
                mhip::rope_position(e.offset + (e.advance ? *e.advance : 0), row, e.scale);
            float c, sn;
            mhip::rope_freq_cs(position, e.table[p], e.table[e.half + p], &c, &sn);
            const bool even = (l32 & 1) == 0;
            float re, ro;
            mhip::rope_rotate(even ? v : other, even ? other : v, c, sn, &re, &ro);
            v = even ? re : ro;
        }
    }
    if (row >= M || col >= s.n) return;
    float* out = s.out + (s.out_advance ? *s.out_advance : 0) * s.n;
    out[row * s.n + col] = v;
}

// Whether a product of a few rows takes small_mfma_kernel: A's 16-byte loads
// need k % 4 == 0 and an aligned base; past kSmallMaxK the waves' 4-byte B
// loads make it slower than the row-blocked GEMV.
bool small_mfma_fits(uint64_t k, bool a_aligned) {
    return k % 4 == 0 && k <= kSmallMaxK && a_aligned;
}

template <class BT>
mhip_status launch_small_mfma(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t m,
                              uint64_t k, uint64_t n, const float* addend, int mode) {
    const uint64_t kq = (k + 8 * kSmallWaves - 1) / (8 * kSmallWaves) * 8;
    const dim3 grid(static_cast<unsigned>((n + 31) / 32), static_cast<unsigned>((m + 31) / 32));
    mhip::launch(ctx, small_mfma_kernel<BT>, grid, dim3(64 * kSmallWaves), 0, a, b, c, m, k, n, kq,
                 addend, mode);
    return mhip::check_launch("matmul (small MFMA tiles)");
}

template <class BT>
mhip_status launch_small_set(mhip_ctx* ctx, const float* a, uint64_t rows, uint64_t k,
                             const SmallSet& set, uint64_t tiles, int epilogue, const RopeEpi& rq,
                             const RopeEpi& rk) {
    const uint64_t kq = (k + 8 * kSmallWaves - 1) / (8 * kSmallWaves) * 8;
    const dim3 grid(static_cast<unsigned>(tiles), static_cast<unsigned>((rows + 31) / 32));
    mhip::launch(ctx, small_mfma_set_kernel<BT>, grid, dim3(64 * kSmallWaves), 0, a, rows, k, kq,
                 set, epilogue, rq, rk);
    return mhip::check_launch("GEMV set (small MFMA tiles)");
}

// The epilogue of one finished sum at (row, col) (apply_addend).
struct AddendEpilogue {
    const float* addend;
    uint64_t n;
    int mode;
    __device__ __forceinline__ float operator()(float v, uint64_t row, uint64_t col) const {
        if (mode == 1) return v + addend[col];
        if (mode >= 2) return apply_addend(v, addend[row * n + col], mode);
        return v;
    }
};

// The k slices of a product on panel_kernel: as many as two workgroups per CU
// (one round of them) allow, at least 128 k each. (The same for compact
// weights, whose sums are then the f32 weights' bits.)
void panel_slicing(const mhip_ctx* ctx, uint64_t k, uint64_t n, uint64_t* slices, uint64_t* k_slice) {
    const uint64_t groups = (n + mhip::kPanelCols<float> - 1) / mhip::kPanelCols<float>;
    const uint64_t room = (ctx->compute_units ? ctx->compute_units : 256) * 2 / groups;
    const uint64_t s = std::max<uint64_t>(1, std::min(room, k / 128));
    *k_slice = ((k + s - 1) / s + 15) / 16 * 16;
    *slices = (k + *k_slice - 1) / *k_slice;
}

template <class BT>
mhip_status launch_panel(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t m, uint64_t k, uint64_t n,
                         const float* addend, int mode) {
    constexpr uint64_t kCols = mhip::kPanelCols<BT>;
    uint64_t slices, k_slice;
    panel_slicing(ctx, k, n, &slices, &k_slice);
    float* target = c;
    if (slices > 1) {
        mhip_status st = workspace(ctx, slices * m * n * sizeof(float), &target);
        if (st != MHIP_OK) return st;
    }
    static bool configured = false;  // raise the dynamic-LDS cap above 64 KiB once
    if (!configured) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mhip::panel_kernel<BT, AddendEpilogue>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, mhip::kPanelLdsBytes<BT>);
        configured = true;
    }
    mhip::launch(ctx, (mhip::panel_kernel<BT, AddendEpilogue>),
                 dim3(static_cast<unsigned>((n + kCols - 1) / kCols), static_cast<unsigned>(slices)),
                 dim3(64 * mhip::kPanelWaves), mhip::kPanelLdsBytes<BT>, a, b, target, m, k, n, k_slice,
                 AddendEpilogue{addend, n, mode});
    mhip_status st = mhip::check_launch("matmul (row panel)");
    if (st != MHIP_OK || slices == 1) return st;
    return launch_splitk_reduce(ctx, target, c, m, n, slices, addend, mode, "matmul (row panel reduction)");
}

// gemv_slicing, but one slice where the second launch costs more than a wave's
// few rows of B one after the other (8 x 64 x 33 5.3 us in two slices, 4.4 in one).
void ragged_slicing(const mhip_ctx* ctx, uint64_t k, uint64_t n, uint64_t* slices, uint64_t* k_per_slice) {
    if (k > 64) return gemv_slicing(ctx, k, n, slices, k_per_slice);
    *slices = 1;
    *k_per_slice = k;
}

template <class BT, int ROWS>
mhip_status launch_ragged_gemv(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t k, uint64_t n,
                               const float* addend, int mode) {
    uint64_t slices, k_per_slice;
    ragged_slicing(ctx, k, n, &slices, &k_per_slice);
    float* target = c;
    if (slices > 1) {
        mhip_status st = workspace(ctx, slices * ROWS * n * sizeof(float), &target);
        if (st != MHIP_OK) return st;
    }
    mhip::launch(ctx, (mhip::ragged_gemv_kernel<ROWS, BT, AddendEpilogue>),
                 dim3(static_cast<unsigned>((n + 255) / 256), static_cast<unsigned>(slices)), dim3(256), 0, a, b,
                 target, k, n, k_per_slice, AddendEpilogue{addend, n, mode});
    mhip_status st = mhip::check_launch("matmul (decode partial sums, ragged rows)");
    if (st != MHIP_OK || slices == 1) return st;
    return launch_splitk_reduce(ctx, target, c, ROWS, n, slices, addend, mode, "matmul (decode reduction)");
}

template <class BT>
mhip_status dispatch_ragged_gemv(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t m, uint64_t k,
                                 uint64_t n, const float* addend, int mode) {
    switch (m) {
        case 1: return launch_ragged_gemv<BT, 1>(ctx, a, b, c, k, n, addend, mode);
        case 2: return launch_ragged_gemv<BT, 2>(ctx, a, b, c, k, n, addend, mode);
        case 3: return launch_ragged_gemv<BT, 3>(ctx, a, b, c, k, n, addend, mode);
        case 4: return launch_ragged_gemv<BT, 4>(ctx, a, b, c, k, n, addend, mode);
        case 5: return launch_ragged_gemv<BT, 5>(ctx, a, b, c, k, n, addend, mode);
        case 6: return launch_ragged_gemv<BT, 6>(ctx, a, b, c, k, n, addend, mode);
        case 7: return launch_ragged_gemv<BT, 7>(ctx, a, b, c, k, n, addend, mode);
        default: return launch_ragged_gemv<BT, 8>(ctx, a, b, c, k, n, addend, mode);
    }
}

// Rows of B per wave: 4 where that leaves every CU eight waves, fewer for
// short outputs and for more rows of A (their registers).
template <int ROWS, class BT>
mhip_status launch_dot(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t k, uint64_t n,
                       const float* addend, int mode) {
    const uint64_t waves = static_cast<uint64_t>(ctx->compute_units ? ctx->compute_units : 256) * 8;
    const AddendEpilogue epilogue{addend, n, mode};
    auto go = [&](auto cols) {
        constexpr int kCols = decltype(cols)::value;
        mhip::launch(ctx, (mhip::dot_kernel<ROWS, kCols, BT, AddendEpilogue>),
                     dim3(static_cast<unsigned>((n + 4 * kCols - 1) / (4 * kCols))), dim3(256), 0, a, b, c, k, n,
                     epilogue);
        return mhip::check_launch("matmul (row dots)");
    };
    if (ROWS <= 4 && n >= 4 * waves) return go(std::integral_constant<int, ROWS <= 4 ? 4 : 2>{});
    if (n >= 2 * waves) return go(std::integral_constant<int, 2>{});
    return go(std::integral_constant<int, 1>{});
}

template <class BT>
mhip_status dispatch_dot(mhip_ctx* ctx, const float* a, const BT* b, float* c, uint64_t m, uint64_t k, uint64_t n,
                         const float* addend, int mode) {
    switch (m) {
        case 1: return launch_dot<1, BT>(ctx, a, b, c, k, n, addend, mode);
        case 2: return launch_dot<2, BT>(ctx, a, b, c, k, n, addend, mode);
        case 3: return launch_dot<3, BT>(ctx, a, b, c, k, n, addend, mode);
        case 4: return launch_dot<4, BT>(ctx, a, b, c, k, n, addend, mode);
        case 5: return launch_dot<5, BT>(ctx, a, b, c, k, n, addend, mode);
        case 6: return launch_dot<6, BT>(ctx, a, b, c, k, n, addend, mode);
        case 7: return launch_dot<7, BT>(ctx, a, b, c, k, n, addend, mode);
        default: return launch_dot<8, BT>(ctx, a, b, c, k, n, addend, mode);
    }
}

// Zero-inner-dimension product: C = 0 (+ addend).
__global__ void fill_addend_kernel(float* C, uint64_t M, uint64_t N, const float* addend,
                                   int mode) {
    const uint64_t idx = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= M * N) return;
    float v = 0.0f;
    if (mode == 1) v = v + addend[idx % N];
    else if (mode >= 2) v = apply_addend(v, addend[idx], mode);
    C[idx] = v;
}

// The shared body of the f32 and compact-weight matmuls: B as f32 or as bf16
// bit patterns; everything else (A, C, the addend, the arithmetic) is f32.
// The tile configurations, picked per shape by the time model. What bounds
// them, and TFLOP/s at 4096^3 and 2048^3 (f32 MFMA kernels before: 146, 134 us
// at 2048^3):
//  - kBig: 256 x 256 tiles, 8 waves of 64 x 128: 218-231 TFLOP/s, 595-630 us
//    at 4096^3 by the inputs (938 before), 400 with compact weights. The card's
//    power limit bounds it: MFMAs are busy 68 % of the cycles at 1.85 GHz, and a
//    loop of nothing but these MFMAs runs at 1.79 GHz. Three buffers and the barrier
//    that leaves the next stage's reads in flight took 1.17 M cycles to 1.05 M
//    and 606 us to 591.
//  - kSmall: 128 x 128 tiles, 4 waves of 64 x 64, two workgroups per CU: 190;
//  - kMid: 128 x 128 tiles, 8 waves of 32 x 64: 167-185, 103-120 us at 2048^3,
//    bound by issue: 5.9 VALU instructions (the split) per MFMA, of which
//    about 4 hide behind it, and 96 bytes of LDS reads per cycle;
//  - kTiny: 64 x 64 tiles, 8 waves of 32 x 32 in two k groups: 93-130; products
//    of about one such tile per CU (1024^3: 256 tiles), which then need no k
//    split and no second launch. Bound by the split's VALU, 13 instructions per
//    MFMA, and by its waits: 23.0 us at 1024^3 where the f32 MFMA took 21.0.
enum class TileChoice { kBig, kSmall, kMid, kTiny };

using BigShape = TileShape<256, 256, 64, 128, 1, 16, 3>;
using SmallShape = TileShape<128, 128, 64, 64, 1, 16, 2>;
using MidShape = TileShape<128, 128, 32, 64, 1, 32, 2>;
using TinyShape = TileShape<64, 64, 32, 32, 2, 32, 2>;

// One configuration on one product: its estimated time and the bytes of its
// partial sums.
struct TileOption {
    TileChoice choice;
    double seconds;
    uint64_t bytes;
};

// The fastest option by `efficiency` (of kBig, kSmall, kMid, kTiny), of those
// whose partial sums take at most `limit` bytes; on equal times the one the
// comparisons name.
TileOption fastest_tiles(const mhip_ctx* ctx, uint64_t m, uint64_t k, uint64_t n, const double (&efficiency)[4],
                         double traffic, uint64_t limit) {
    auto option = [&](auto shape, TileChoice choice) {
        using Shape = decltype(shape);
        const uint64_t slots = Shape::kPerCu * (ctx->compute_units ? ctx->compute_units : 256);
        const GemmPlan p = plan_gemm(m, k, n, Shape::BM, Shape::BN, kSliceK, slots);
        const uint64_t bytes = (p.stream       ? p.groups * 2 * Shape::BM * Shape::BN
                                : p.splits > 1 ? p.splits * m * n
                                               : 0) * sizeof(float);
        double t = gemm_seconds(ctx, m, n, p, Shape::BM, Shape::BN, Shape::kPerCu, Shape::kWaves,
                                efficiency[static_cast<int>(choice)], traffic);
        if (bytes > limit) t = INFINITY;
        return TileOption{choice, t, bytes};
    };
    const TileOption big = option(BigShape{}, TileChoice::kBig), small = option(SmallShape{}, TileChoice::kSmall),
                     mid = option(MidShape{}, TileChoice::kMid), tiny = option(TinyShape{}, TileChoice::kTiny);
    if (tiny.seconds < big.seconds && tiny.seconds < small.seconds && tiny.seconds < mid.seconds) return tiny;
    if (big.seconds < small.seconds && big.seconds <= mid.seconds) return big;
    if (mid.seconds < small.seconds) return mid;
    return small;
}

// Which products the entry points with limited scratch take was settled by the
// plans of the f32 MFMA kernels, whose fractions of the peak kF32 is.
// mhip_matmul_f32_noalloc, which gives mhip_matmul_f32's bits, refuses partial
// sums beyond its array: a product whose plan was within it stays within, by
// the fastest option that does (one product in 500 over m 9-16384, k and n
// 1-65536). A capture refuses those beyond the context's workspace: for a
// product whose plan was within it the workspace grows (mhip::CaptureGrowth).
constexpr double kSplit[4] = {1.40, 1.30, 1.20, 0.76}, kF32[4] = {0.88, 0.82, 0.83, 0.65};

bool within_before(const mhip_ctx* ctx, uint64_t m, uint64_t k, uint64_t n, uint64_t limit) {
    return fastest_tiles(ctx, m, k, n, kF32, 5.0e12, UINT64_MAX).bytes <= limit;
}

TileChoice choose_tiles(const mhip_ctx* ctx, uint64_t m, uint64_t k, uint64_t n) {
    TileOption best = fastest_tiles(ctx, m, k, n, kSplit, 4.0e12, UINT64_MAX);
    if (best.bytes > MHIP_NOALLOC_SCRATCH_BYTES && within_before(ctx, m, k, n, MHIP_NOALLOC_SCRATCH_BYTES))
        best = fastest_tiles(ctx, m, k, n, kSplit, 4.0e12, MHIP_NOALLOC_SCRATCH_BYTES);
    return best.choice;
}

// Few-row products by shape (few_rows.hpp), after the vector GEMV: up to 8
// rows over a B stored [k, n] whose rows (or base) are no whole vectors; up to
// 8 rows over a B stored [n, k]; 9-32 rows over a B stored [k, n]. Against
// the 64 x 64 tiles, f32, k 4096, us: 8 ragged rows x 32001 101 (237 on the
// tiles), 8 row dots x 32000 173 (188); the panel 32 x 11008 53 (74), while
// 9-32 rows over [n, k] stay on the tiles (16 x 32000 184; a panel whose lanes
// read along k, 230).
bool ragged_gemv_fits(uint64_t m, uint64_t n, bool ta, bool tb) {
    return m <= kGemvMaxRows && !ta && !tb && m * n < (1ULL << 31);
}
// A wave's lanes run along k: a short k leaves them idle before many outputs'
// butterflies (8 x 32 x 11008 9.1 us, tiles 4.8; 8 x 128 x 11008 9.4 and 7.9; 8
// x 128 x 4096 5.2 and 6.1), and where a few hundred columns give each CU hardly
// a wave, a very long k is a chain of its loads (8 x 65536 x 256 149, tiles 75;
// 3 x 65536 x 256 109 and 74). Both sides measured over m 1-8, k 32-65536, n
// 32-32000.
bool dot_fits(uint64_t m, uint64_t k, uint64_t n, bool ta, bool tb, bool b_aligned) {
    const bool lanes = m == 1 || k >= 256 || m * n <= std::max<uint64_t>(512 * k, 24576);
    const bool chain = k > (m <= 4 && n >= 128 ? 32768 : n >= 128 ? 16384 : m <= 4 ? UINT64_MAX : 32768);
    return m <= kGemvMaxRows && !ta && tb && k % 8 == 0 && b_aligned && n < (1ULL << 31) && lanes &&
           !(chain && n < 1024);
}
// (Pairs of a compact B's columns; 32-bit offsets over 16 rows of B.)
bool panel_fits(uint64_t m, uint64_t n, bool ta, bool tb) {
    return m > kGemvMaxRows && m <= mhip::kPanelRows && !ta && !tb && n % 2 == 0 && n < (1ULL << 24);
}

// Which kernel path a product takes (the decode GEMV rules of matmul_impl,
// then the tile choice); `b_aligned`: B's base allows its vector loads.
mhip_matmul_plan plan_matmul(const mhip_ctx* ctx, uint64_t m, uint64_t k, uint64_t n, bool ta,
                             bool tb, bool b_aligned) {
    mhip_matmul_plan out{};
    if (m <= kGemvMaxRows && !ta && !tb && n % 4 == 0 && b_aligned) {
        uint64_t slices, per;
        gemv_slicing(ctx, k, n, &slices, &per);
        out.path = MHIP_MATMUL_PATH_GEMV;
        out.splits = static_cast<uint32_t>(slices);
        return out;
    }
    if (m <= 4 * kGemvMaxRows && m % kGemvMaxRows == 0 && m * k * n <= kGemvSmallProduct && !ta &&
        !tb && n % 4 == 0 && b_aligned) {
        if (small_mfma_fits(k, true)) {
            out.path = MHIP_MATMUL_PATH_SMALL_TILES;
            out.tile_m = out.tile_n = 32;
            out.waves = kSmallWaves;
            out.splits = 1;
            return out;
        }
        uint64_t slices, per;
        gemv_slicing(ctx, k, n, &slices, &per);
        out.path = MHIP_MATMUL_PATH_GEMV_ROW_BLOCKS;
        out.splits = static_cast<uint32_t>(slices);
        return out;
    }
    if (ragged_gemv_fits(m, n, ta, tb)) {
        uint64_t slices, per;
        ragged_slicing(ctx, k, n, &slices, &per);
        out.path = MHIP_MATMUL_PATH_GEMV_RAGGED;
        out.splits = static_cast<uint32_t>(slices);
        return out;
    }
    if (dot_fits(m, k, n, ta, tb, b_aligned)) {
        out.path = MHIP_MATMUL_PATH_ROW_DOTS;
        out.splits = 1;
        return out;
    }
    if (panel_fits(m, n, ta, tb)) {
        uint64_t slices, per;
        panel_slicing(ctx, k, n, &slices, &per);
        out.path = MHIP_MATMUL_PATH_ROW_PANEL;
        out.tile_m = mhip::kPanelRows;
        out.tile_n = mhip::kPanelCols<float>;
        out.waves = mhip::kPanelWaves;
        out.splits = static_cast<uint32_t>(slices);
        return out;
    }
    out.path = MHIP_MATMUL_PATH_TILES;
    uint64_t bm = 128, waves = SmallShape::kWaves, per_cu = SmallShape::kPerCu;
    switch (choose_tiles(ctx, m, k, n)) {
        case TileChoice::kBig: bm = 256; waves = BigShape::kWaves; per_cu = BigShape::kPerCu; break;
        case TileChoice::kMid: waves = MidShape::kWaves; per_cu = MidShape::kPerCu; break;
        case TileChoice::kTiny: bm = 64; waves = TinyShape::kWaves; per_cu = TinyShape::kPerCu; break;
        case TileChoice::kSmall: break;
    }
    const GemmPlan p = plan_gemm(m, k, n, bm, bm, 32, per_cu * (ctx->compute_units ? ctx->compute_units : 256));
    out.tile_m = out.tile_n = static_cast<uint32_t>(bm);
    out.waves = static_cast<uint32_t>(waves);
    out.splits = p.stream ? 1u : static_cast<uint32_t>(p.splits);
    out.stream_k = p.stream ? 1u : 0u;
    return out;
}

template <class BT>
mhip_status matmul_impl(mhip_ctx* ctx, const float* a, const BT* b, float* out, uint64_t m,
                        uint64_t k, uint64_t n, int transpose_a, int transpose_b,
                        const float* addend, int addend_mode, bool gated = false) {
    MHIP_REQUIRE_CTX(ctx);
    if (gated ? addend_mode != 3 : (addend_mode < 0 || addend_mode > 2))
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "matmul addend mode must be 0, 1 or 2");
    if (addend_mode != 0 && !addend)
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "matmul addend is null");
    if (m == 0 || n == 0) return MHIP_OK;
    if (!a || !b || !out) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "matmul: null buffer");
    if (k == 0) {
        mhip::launch(ctx, fill_addend_kernel, dim3(static_cast<unsigned>((m * n + 255) / 256)),
                     dim3(256), 0, out, m, n, addend, addend_mode);
        return mhip::check_launch("matmul (empty inner dimension)");
    }
    // One row of A lies the same either way.
    const bool ta = transpose_a != 0 && m != 1, tb = transpose_b != 0;
    // B's vector accesses (dwordx4 of f32, or 8 bytes of bf16) need rows of a
    // multiple of 4 elements and an aligned base.
    const uintptr_t b_align = sizeof(BT) == 4 ? 15u : 7u;
    const bool b_aligned = (reinterpret_cast<uintptr_t>(b) & b_align) == 0;
    // (A row of A stored [k, 1] took the tiles before.)
    auto taken_before = [&] { return ctx->capturing && within_before(ctx, m, k, n, ctx->workspace_bytes); };
    if (m <= kGemvMaxRows && !ta && !tb && n % 4 == 0 && b_aligned) {
        const mhip::CaptureGrowth growth(ctx, transpose_a != 0 && taken_before());
        return dispatch_gemv<BT>(ctx, a, b, out, m, k, n, addend, addend_mode);
    }
    // A few rows of a small product (up to 32 rows in blocks of 8, at most
    // 2^26 multiply-adds): one launch of small_mfma_kernel up to k = 1024,
    // else the GEMV's two short launches; both beat MFMA tiles that would be
    // three quarters padding and walk k serially.
    if (m <= 4 * kGemvMaxRows && m % kGemvMaxRows == 0 && m * k * n <= kGemvSmallProduct && !ta && !tb &&
        n % 4 == 0 && b_aligned) {
        if (small_mfma_fits(k, mhip::aligned16(a)))
            return launch_small_mfma<BT>(ctx, a, b, out, m, k, n, addend, addend_mode);
        return launch_gemv<kGemvMaxRows, BT>(ctx, a, b, out, k, n, addend, addend_mode, m / kGemvMaxRows);
    }
    const mhip::CaptureGrowth growth(ctx, taken_before());
    if (ragged_gemv_fits(m, n, ta, tb))
        return dispatch_ragged_gemv<BT>(ctx, a, b, out, m, k, n, addend, addend_mode);
    if (dot_fits(m, k, n, ta, tb, mhip::aligned16(b)) && mhip::aligned16(a))
        return dispatch_dot<BT>(ctx, a, b, out, m, k, n, addend, addend_mode);
    if (panel_fits(m, n, ta, tb) && reinterpret_cast<uintptr_t>(b) % 4 == 0)
        return launch_panel<BT>(ctx, a, b, out, m, k, n, addend, addend_mode);
    const uint64_t lda = ta ? m : k, ldb = tb ? k : n;
    // A stored [m, k] and B stored [n, k] read 4 elements along k at a time,
    // a compact B stored [k, n] two columns, where rows and base allow it.
    const uint64_t b_pack = sizeof(BT) == 2 && !tb ? 2 : 4;
    const Access access{
        .wide_a = lda % 4 == 0 && mhip::aligned16(a),
        .wide_b = ldb % b_pack == 0 && reinterpret_cast<uintptr_t>(b) % (b_pack * sizeof(BT)) == 0,
        .short_rows = lda <= kShortRows && ldb <= kShortRows};
    switch (choose_tiles(ctx, m, k, n)) {
        case TileChoice::kTiny:
            return launch_tiles<TinyShape, BT>(ctx, a, b, out, m, k, n, ta, tb, addend, addend_mode, access);
        case TileChoice::kBig:
            return launch_tiles<BigShape, BT>(ctx, a, b, out, m, k, n, ta, tb, addend, addend_mode, access);
        case TileChoice::kMid:
            return launch_tiles<MidShape, BT>(ctx, a, b, out, m, k, n, ta, tb, addend, addend_mode, access);
        case TileChoice::kSmall:
            break;
    }
    return launch_tiles<SmallShape, BT>(ctx, a, b, out, m, k, n, ta, tb, addend, addend_mode, access);
}

}  // namespace

extern "C" mhip_status mhip_matmul_plan_f32(mhip_ctx* ctx, uint64_t m, uint64_t k, uint64_t n,
                                            int transpose_a, int transpose_b,
                                            mhip_matmul_plan* plan) {
    MHIP_REQUIRE_CTX(ctx);
    if (!plan) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "matmul plan: null output");
    *plan = plan_matmul(ctx, m, k, n, transpose_a != 0 && m != 1, transpose_b != 0, true);
    return MHIP_OK;
}

// The up product of a gated matmul (src/executor.rs:1484-1494): out =
// silu(gate) * (a . b), gate the [m, n] gate product, through the matmul's
// own kernels with the gate as an epilogue (addend mode 3), so it equals the
// product followed by silu-mul bit for bit, with no [m, n] temporary for the
// up product and no separate silu-mul launch.
mhip_status mhip::matmul_gated_f32(mhip_ctx* ctx, const float* a, const void* b, bool bf16,
                                   float* out, uint64_t m, uint64_t k, uint64_t n,
                                   bool transpose_a, bool transpose_b, const float* gate) {
    if (bf16)
        return matmul_impl<uint16_t>(ctx, a, static_cast<const uint16_t*>(b), out, m, k, n,
                                     transpose_a, transpose_b, gate, 3, true);
    return matmul_impl<float>(ctx, a, static_cast<const float*>(b), out, m, k, n, transpose_a,
                              transpose_b, gate, 3, true);
}

extern "C" mhip_status mhip_matmul_f32(mhip_ctx* ctx, const float* a, const float* b, float* out,
                                       uint64_t m, uint64_t k, uint64_t n, int transpose_a,
                                       int transpose_b, const float* addend, int addend_mode) {
    return matmul_impl<float>(ctx, a, b, out, m, k, n, transpose_a, transpose_b, addend, addend_mode);
}

// ---------------------------------------------------------------------------
// Allocation-free matmul: the partial sums in a fixed device array
// ---------------------------------------------------------------------------

// The scratch of mhip_matmul_f32_noalloc (split-k, stream-K and GEMV partial
// sums). Each GPU the library runs on holds its own copy until the process
// ends. On the host this name is a stand-in, not a device address: host code
// only ever uses the address hipGetSymbolAddress gives for a device.
static __device__ __align__(256) float scratch[MHIP_NOALLOC_SCRATCH_BYTES / sizeof(float)];

namespace {

constexpr int kScratchDevices = 64;
std::mutex scratch_mutex;
float* scratch_address[kScratchDevices] = {};

}  // namespace

// The device address of `scratch` on the context's device: looked up once
// per device, with that device current, when the first context on it is
// created (or, if that failed, on the entry point's next call there).
mhip_status mhip::noalloc_scratch(mhip_ctx* ctx, float** out) {
    if (ctx->device < 0 || ctx->device >= kScratchDevices)
        return mhip::fail(MHIP_DEVICE_UNAVAILABLE, "allocation-free matmul: device ordinal out of range");
    std::lock_guard<std::mutex> lock(scratch_mutex);
    float*& address = scratch_address[ctx->device];
    if (!address) {
        // The caller's current device is put back afterwards.
        int previous = -1;
        hipError_t err = hipGetDevice(&previous);
        if (err == hipSuccess) err = hipSetDevice(ctx->device);
        void* p = nullptr;
        if (err == hipSuccess) err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (previous >= 0 && previous != ctx->device) (void)hipSetDevice(previous);
        if (err != hipSuccess) return mhip::from_hip(err, "locating the allocation-free matmul's scratch");
        address = static_cast<float*>(p);
    }
    if (out) *out = address;
    return MHIP_OK;
}

namespace {

// Points the context's matmul scratch at the fixed array for one call.
struct FixedScratch {
    mhip_ctx* ctx;
    FixedScratch(mhip_ctx* c, float* p) : ctx(c) {
        ctx->fixed_scratch = p;
        ctx->fixed_scratch_bytes = MHIP_NOALLOC_SCRATCH_BYTES;
    }
    ~FixedScratch() {
        ctx->fixed_scratch = nullptr;
        ctx->fixed_scratch_bytes = 0;
    }
};

}  // namespace

extern "C" mhip_status mhip_matmul_f32_noalloc(mhip_ctx* ctx, const float* a, const float* b,
                                               float* out, uint64_t m, uint64_t k, uint64_t n,
                                               int transpose_a, int transpose_b,
                                               const float* addend, int addend_mode) {
    MHIP_REQUIRE_CTX(ctx);
    float* p = nullptr;
    mhip_status st = mhip::noalloc_scratch(ctx, &p);
    if (st != MHIP_OK) return st;
    FixedScratch use(ctx, p);
    return matmul_impl<float>(ctx, a, b, out, m, k, n, transpose_a, transpose_b, addend, addend_mode);
}

extern "C" mhip_status mhip_matmul_bf16w_f32(mhip_ctx* ctx, const float* a, const uint16_t* b,
                                             float* out, uint64_t m, uint64_t k, uint64_t n,
                                             int transpose_a, int transpose_b, const float* addend,
                                             int addend_mode) {
    return matmul_impl<uint16_t>(ctx, a, b, out, m, k, n, transpose_a, transpose_b, addend,
                                 addend_mode);
}

namespace {

template <class BT>
mhip_status dispatch_gemv_set(mhip_ctx* ctx, const float* a, uint64_t rows, uint64_t k,
                              const GemvSet& set, int epilogue, const RopeEpi& rq,
                              const RopeEpi& rk, uint32_t g, bool stream, bool wide, int norm_mode,
                              const NormIn& norm) {
    switch (rows) {
        case 1: return launch_gemv_set<1, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, norm_mode, norm);
        case 2: return launch_gemv_set<2, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, 0, norm);
        case 3: return launch_gemv_set<3, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, 0, norm);
        case 4: return launch_gemv_set<4, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, 0, norm);
        case 5: return launch_gemv_set<5, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, 0, norm);
        case 6: return launch_gemv_set<6, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, 0, norm);
        case 7: return launch_gemv_set<7, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, 0, norm);
        default:
            return launch_gemv_set<8, BT>(ctx, a, k, set, epilogue, rq, rk, g, stream, wide, 0, norm,
                                          static_cast<uint32_t>(rows / kGemvMaxRows));
    }
}

}  // namespace

namespace mhip {

mhip_status gemv_chunks_f32(mhip_ctx* ctx, const float* a, const void* b, float* out, uint64_t k,
                            uint64_t n, const float* addend, int addend_mode, bool bf16_weights,
                            float* chunk_ss) {
    MHIP_REQUIRE_CTX(ctx);
    // The one-row GEMV path of mhip_matmul_f32 with a split k (the chunk
    // sums come from its reduction launch).
    const uintptr_t b_align = bf16_weights ? 7u : 15u;
    if (!a || !b || !out || !chunk_ss || k == 0 || n % 4 != 0 || !aligned16(out) ||
        (reinterpret_cast<uintptr_t>(b) & b_align) != 0 || (addend_mode != 0 && !addend) ||
        addend_mode < 0 || addend_mode > 2)
        return MHIP_LAYOUT_UNSUPPORTED;
    uint64_t slices, k_per_slice;
    gemv_slicing(ctx, k, n, &slices, &k_per_slice);
    if (slices < 2) return MHIP_LAYOUT_UNSUPPORTED;
    return bf16_weights
               ? launch_gemv<1, uint16_t>(ctx, a, static_cast<const uint16_t*>(b), out, k, n, addend,
                                          addend_mode, 1, chunk_ss)
               : launch_gemv<1, float>(ctx, a, static_cast<const float*>(b), out, k, n, addend,
                                       addend_mode, 1, chunk_ss);
}

size_t gemv_merge_bytes(mhip_ctx* ctx, uint64_t heads, uint64_t d, uint64_t n, const void* b,
                        const float* out, bool bf16_weights) {
    const uintptr_t b_align = bf16_weights ? 7u : 15u;
    if (!ctx || !b || !out || !aligned16(out) || (reinterpret_cast<uintptr_t>(b) & b_align) != 0 ||
        heads == 0 || n == 0 || n % 4 != 0 || (d != 32 && d != 64 && d != 128 && d != 256))
        return 0;
    uint64_t slices, k_per_slice;
    gemv_slicing(ctx, heads * d, n, &slices, &k_per_slice);
    if (slices < 2 || k_per_slice > d || d % k_per_slice != 0) return 0;
    return (slices * n * sizeof(float) + 255) / 256 * 256;
}

namespace {

template <class BT, int CPL, int D4>
void launch_merge_partial(mhip_ctx* ctx, dim3 grid, bool stream, const DecodeChunks& r,
                          const BT* b, float* partial, uint64_t k, uint64_t n, uint64_t k_per_slice,
                          uint64_t slices) {
    if (stream)
        mhip::launch(ctx, (gemv_partial_merge_kernel<BT, true, CPL, D4>), grid, dim3(kGemvThreads),
                     0, r.part_o, r.part_ml, r.chunks, b, partial, k, n, k_per_slice,
                     static_cast<uint32_t>(slices));
    else
        mhip::launch(ctx, (gemv_partial_merge_kernel<BT, false, CPL, D4>), grid, dim3(kGemvThreads),
                     0, r.part_o, r.part_ml, r.chunks, b, partial, k, n, k_per_slice,
                     static_cast<uint32_t>(slices));
}

template <class BT, int CPL>
void launch_merge_partial_d(mhip_ctx* ctx, dim3 grid, bool stream, const DecodeChunks& r,
                            const BT* b, float* partial, uint64_t k, uint64_t n,
                            uint64_t k_per_slice, uint64_t slices) {
    switch (r.d) {
        case 32: return launch_merge_partial<BT, CPL, 8>(ctx, grid, stream, r, b, partial, k, n, k_per_slice, slices);
        case 64: return launch_merge_partial<BT, CPL, 16>(ctx, grid, stream, r, b, partial, k, n, k_per_slice, slices);
        case 128: return launch_merge_partial<BT, CPL, 32>(ctx, grid, stream, r, b, partial, k, n, k_per_slice, slices);
        default: return launch_merge_partial<BT, CPL, 64>(ctx, grid, stream, r, b, partial, k, n, k_per_slice, slices);
    }
}

// launch_gemv<1, BT>'s launches (same slicing, column groups, loads and
// reduction) with the merge kernel's partial launch.
template <class BT>
mhip_status launch_gemv_merge(mhip_ctx* ctx, const DecodeChunks& r, const BT* b, float* c,
                              uint64_t n, const float* addend, int mode, float* chunk_ss) {
    const uint64_t k = r.heads * r.d;
    const uint64_t col_groups = (n + kGemvCols - 1) / kGemvCols;
    uint64_t slices, k_per_slice;
    gemv_slicing(ctx, k, n, &slices, &k_per_slice);
    float* partial = r.extra;
    const bool stream = gemv_streams_b(k * n * sizeof(BT));
    bool wide = false;
    if constexpr (kGemvWideable<1, BT>) wide = n % 8 == 0 && mhip::aligned16(b);
    const uint64_t part_groups = wide ? (n + 511) / 512 : col_groups;
    const dim3 grid(static_cast<unsigned>(part_groups), static_cast<unsigned>(slices), 1);
    if constexpr (kGemvWideable<1, BT>) {
        if (wide)
            launch_merge_partial_d<BT, 8>(ctx, grid, stream, r, b, partial, k, n, k_per_slice, slices);
        else
            launch_merge_partial_d<BT, 4>(ctx, grid, stream, r, b, partial, k, n, k_per_slice, slices);
    } else {
        launch_merge_partial_d<BT, 4>(ctx, grid, stream, r, b, partial, k, n, k_per_slice, slices);
    }
    mhip_status st = mhip::check_launch("attention merge + output projection (partial sums)");
    if (st != MHIP_OK) return st;
    mhip::launch(ctx, gemv_reduce_kernel<1>, dim3(static_cast<unsigned>(col_groups), 1, 1),
                 dim3(kGemvThreads), 0, partial, c, n, static_cast<uint32_t>(slices), addend, mode,
                 chunk_ss);
    return mhip::check_launch("attention merge + output projection (reduction)");
}

}  // namespace

mhip_status gemv_merge_f32(mhip_ctx* ctx, const DecodeChunks& records, const void* b, float* out,
                           uint64_t n, const float* addend, int addend_mode, bool bf16_weights,
                           float* chunk_ss) {
    MHIP_REQUIRE_CTX(ctx);
    const size_t need = gemv_merge_bytes(ctx, records.heads, records.d, n, b, out, bf16_weights);
    if (need == 0 || records.extra_bytes < need || !records.extra || !records.part_o ||
        !records.part_ml || records.chunks == 0 || !chunk_ss || !aligned16(records.extra) ||
        (addend_mode != 0 && !addend) || addend_mode < 0 || addend_mode > 2)
        return MHIP_LAYOUT_UNSUPPORTED;
    return bf16_weights ? launch_gemv_merge<uint16_t>(ctx, records, static_cast<const uint16_t*>(b),
                                                      out, n, addend, addend_mode, chunk_ss)
                        : launch_gemv_merge<float>(ctx, records, static_cast<const float*>(b), out,
                                                   n, addend, addend_mode, chunk_ss);
}

mhip_status gemv_set_f32(mhip_ctx* ctx, const float* a, uint64_t rows, uint64_t k,
                         const GemvTarget* targets, int count, int epilogue,
                         const mhip_rope_params* rope, bool bf16_weights, const RowNorm* row_norm) {
    MHIP_REQUIRE_CTX(ctx);
    if (!targets || count < 1 || count > 3 || rows == 0 || k == 0) return MHIP_LAYOUT_UNSUPPORTED;
    if (!row_norm && !a) return MHIP_LAYOUT_UNSUPPORTED;
    NormIn norm{};
    int norm_mode = 0;
    if (row_norm) {
        // One row that the RMSNorm kernel would normalise with its vector
        // kernel (k % 4 == 0, at most 16384 floats, 16-byte aligned), so that
        // the chunk sums carry its order.
        const RowNorm& rn = *row_norm;
        int g = 0, vpt = 0;
        if (rows != 1 || k % 4 != 0 || !rn.src || !rn.chunk_ss || !(rn.eps > 0.0f) ||
            !aligned16(rn.src) || (rn.gain && !aligned16(rn.gain)) || !rms_layout(k / 4, &g, &vpt))
            return MHIP_LAYOUT_UNSUPPORTED;
        norm.src = rn.src;
        norm.chunk_ss = rn.chunk_ss;
        norm.gain = rn.gain;
        norm.eps = rn.eps;
        norm.chunks = static_cast<uint32_t>((k / 4 + 63) / 64);
        norm_mode = 1;
    }
    // Up to 8 rows, or up to 32 in blocks of 8 when every product is small
    // (as for the row-blocked matmul).
    if (rows > kGemvMaxRows) {
        if (rows > 4 * kGemvMaxRows || rows % kGemvMaxRows != 0) return MHIP_LAYOUT_UNSUPPORTED;
        for (int i = 0; i < count; ++i)
            if (rows * k * targets[i].n > kGemvSmallProduct) return MHIP_LAYOUT_UNSUPPORTED;
    }
    if (epilogue == kGemvSiluMul && (count != 2 || targets[0].n != targets[1].n))
        return MHIP_LAYOUT_UNSUPPORTED;
    if (epilogue == kGemvRopeQK && (count < 2 || !rope)) return MHIP_LAYOUT_UNSUPPORTED;
    GemvSet set{};
    set.count = count;
    bool stream = false;
    // Compact weights on up to 4 rows: 8 columns per lane when every matrix
    // allows 16-byte loads (as launch_gemv decides for one).
    bool wide = bf16_weights && rows <= 4;
    for (int i = 0; i < count; ++i)
        if (targets[i].n % 8 != 0 || !aligned16(targets[i].b)) wide = false;
    uint64_t floats = 0, blocks = 0, groups = 0;
    uint64_t offsets[3];
    for (int i = 0; i < count; ++i) {
        const GemvTarget& t = targets[i];
        const bool needs_out = !(epilogue == kGemvSiluMul && i == 1);
        const uintptr_t b_align = bf16_weights ? 7u : 15u;
        if (!t.b || t.n == 0 || t.n % 4 != 0 || (reinterpret_cast<uintptr_t>(t.b) & b_align) != 0 ||
            (needs_out && (!t.out || !aligned16(t.out))))
            return MHIP_LAYOUT_UNSUPPORTED;
        GemvSeg& g = set.seg[i];
        uint64_t slices, k_per_slice;
        gemv_slicing(ctx, k, t.n, &slices, &k_per_slice);
        g.b = t.b;
        g.out = t.out;
        g.out_advance = t.row_advances
                            ? advance_ptr(ctx, MHIP_ADVANCE_ROW_OFFSET, t.row_advance_limit)
                            : nullptr;
        g.n = t.n;
        g.k_per_slice = k_per_slice;
        g.col_groups = static_cast<uint32_t>((t.n + (wide ? 511 : 255)) / (wide ? 512 : 256));
        g.slices = static_cast<uint32_t>(slices);
        // The set streams its matrices when any of them is large.
        if (gemv_streams_b(k * t.n * (bf16_weights ? 2 : 4))) stream = true;
        g.first_block = static_cast<uint32_t>(blocks);
        g.first_group = static_cast<uint32_t>(groups);
        offsets[i] = floats;
        floats += (slices * rows * t.n + 63) / 64 * 64;
        blocks += g.col_groups * slices;
        // The reduction always takes 256 columns per workgroup.
        if (!(epilogue == kGemvSiluMul && i == 1)) groups += (t.n + kGemvCols - 1) / kGemvCols;
    }
    if (blocks >= (1ULL << 31)) return MHIP_LAYOUT_UNSUPPORTED;
    if (norm_mode)
        for (int i = 0; i < count; ++i)
            if (set.seg[i].k_per_slice > kNormSliceMax) return MHIP_LAYOUT_UNSUPPORTED;
    RopeEpi rq{}, rk{};
    if (epilogue == kGemvRopeQK) {
        for (int i = 0; i < 2; ++i) {
            const mhip_rope_params& p = rope[i];
            if (p.head_count == 0 || targets[i].n % p.head_count != 0) return MHIP_LAYOUT_UNSUPPORTED;
            const uint64_t hw = targets[i].n / p.head_count;
            if (p.half_split || p.dimension == 0 || p.dimension % 4 != 0 || p.dimension > hw ||
                hw % 4 != 0 || !(p.base > 0.0f) || !std::isfinite(p.base) || !(p.scale > 0.0f) ||
                !std::isfinite(p.scale) || (p.banded_factor > 0.0f && p.yarn_factor > 0.0f))
                return MHIP_LAYOUT_UNSUPPORTED;
            mhip_rope_params q = p;
            if (q.rotated_pairs > q.dimension / 2) q.rotated_pairs = q.dimension / 2;
            const float* table = nullptr;
            mhip_status st = rope_device_table(ctx, q, &table);
            if (st != MHIP_OK) return st;
            RopeEpi& e = i == 0 ? rq : rk;
            e.table = table;
            e.head_width = hw;
            e.dimension = q.dimension;
            e.half = q.dimension / 2;
            e.offset = q.position_offset;
            e.scale = q.scale;
            e.advance = advance_ptr(ctx, MHIP_ADVANCE_POSITION_OFFSET, UINT64_MAX);
        }
    }
    // 16-32 rows whose products take small_mfma_kernel as separate matmuls
    // take its set form (the same sums), in one launch.
    if (rows > kGemvMaxRows && norm_mode == 0 && small_mfma_fits(k, aligned16(a))) {
        SmallSet ss{};
        ss.count = count;
        uint64_t tiles = 0;
        for (int i = 0; i < count; ++i) {
            SmallSeg& g = ss.seg[i];
            g.b = targets[i].b;
            g.out = targets[i].out;
            g.out_advance = set.seg[i].out_advance;
            g.n = targets[i].n;
            if (epilogue == kGemvSiluMul && i == 1) {
                g.first_tile = UINT32_MAX;  // summed with the gate's tiles
                continue;
            }
            g.first_tile = static_cast<uint32_t>(tiles);
            tiles += (targets[i].n + 31) / 32;
        }
        return bf16_weights ? launch_small_set<uint16_t>(ctx, a, rows, k, ss, tiles, epilogue, rq, rk)
                            : launch_small_set<float>(ctx, a, rows, k, ss, tiles, epilogue, rq, rk);
    }
    void* scratch = nullptr;
    mhip_status st = workspace(ctx, floats * sizeof(float), &scratch);
    if (st != MHIP_OK) return st;
    float* partial = static_cast<float*>(scratch);
    for (int i = 0; i < count; ++i) set.seg[i].partial = partial + offsets[i];
    const uint32_t g = static_cast<uint32_t>(groups);
    return bf16_weights ? dispatch_gemv_set<uint16_t>(ctx, a, rows, k, set, epilogue, rq, rk, g, stream,
                                                      wide, norm_mode, norm)
                        : dispatch_gemv_set<float>(ctx, a, rows, k, set, epilogue, rq, rk, g, stream,
                                                   wide, norm_mode, norm);
}

}  // namespace mhip
