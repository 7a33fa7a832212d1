// Products of a few rows whose time is the reading of B once.
//
//  - ragged_gemv_kernel: up to 8 rows, B stored [k, n] with rows that are not
//    whole 16-byte vectors.
//  - panel_kernel: 9-32 rows, B stored [k, n]. Every wave streams its own 32
//    columns (64 of a compact B) of a k slice straight into the MFMA's operand
//    layout, 64 k ahead, splits them in registers and multiplies them with A's
//    planes, which the workgroup keeps in LDS; nothing waits between the waves
//    but the change of A's chunk.
//  - dot_kernel: up to 8 rows, B stored [n, k] (a tied output head). Lanes run
//    along k, a wave takes several rows of B at a time.
#pragma once

#include "split_tile.hpp"

namespace mhip {

// ---------------------------------------------------------------------------
// 9-32 rows, B [k, n]
// ---------------------------------------------------------------------------

constexpr int kPanelRows = 32;
constexpr int kPanelWaves = 8;
// k of A in LDS at a time: its planes take 72 KB, two workgroups per CU, or 48
// KB with a compact B, whose second column block leaves no registers for the
// 24 that 384 k are fetched into (they spilled: 12 x 4096 x 32000 54 -> 59 us).
template <class BT>
constexpr int kPanelK = sizeof(BT) == 2 ? 256 : 384;
template <class BT>
constexpr int kPanelLdsBytes = 3 * kPanelRows * kPanelK<BT> * 2;
constexpr int kPanelDepth = 4;  // steps of 16 k that a wave reads ahead
// Column blocks of 32 a wave takes: two of a compact B, read in pairs of columns.
template <class BT>
constexpr int kPanelBlocks = sizeof(BT) == 2 ? 2 : 1;
template <class BT>
constexpr int kPanelCols = kPanelWaves * 32 * kPanelBlocks<BT>;

// A k slice's sums of 32 rows by kPanelCols columns: blockIdx.x the columns,
// blockIdx.y the slice [y * k_slice, ...), k_slice a multiple of 16. Writes C
// itself (one slice, with the addend) or the slice's partial product at
// C + y * M * N. n is even and B 4-byte aligned.
//
// What bounds it: the bytes in flight, so the waves a CU holds (two workgroups
// at 128 registers). The 64 x 64 tiles that these products took before keep 8
// KB of B in flight per workgroup; here each of 16 waves per CU keeps 8 KB.
// 24 x 4096 x 11008: f32 MFMA tiles 149 us, split tiles 74, this 43 (37 at 5.2
// TB/s and the slices' sum); compact 27.
template <class BT, class Addend>
__global__ __launch_bounds__(64 * kPanelWaves, 4) void panel_kernel(
    const float* __restrict__ A, const BT* __restrict__ B, float* __restrict__ C, uint64_t M, uint64_t K,
    uint64_t N, uint64_t k_slice, Addend epilogue) {
    constexpr bool kBf16 = sizeof(BT) == 2;
    constexpr int kBlocks = kPanelBlocks<BT>;
    constexpr int kPlanes = kBf16 ? 1 : 3;
    constexpr int kChunkBytes = kPanelRows * 16, kPlaneBytes = kPanelK<BT> / 8 * kChunkBytes;
    constexpr int kStream = 2;  // non-temporal
    static_assert(3 * kPlaneBytes == kPanelLdsBytes<BT>, "the launch's LDS");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ int redo, any_tiny;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int l32 = lane & 31, h = lane >> 5;
    const uint32_t n = static_cast<uint32_t>(N);  // the launch checks n < 2^24
    const uint32_t col0 = (blockIdx.x * kPanelWaves + wave) * 32 * kBlocks;
    const uint64_t k_begin = static_cast<uint64_t>(blockIdx.y) * k_slice;
    const uint64_t k_end = min(K, k_begin + k_slice);
    const uint32_t steps = static_cast<uint32_t>((k_end - k_begin + 15) / 16);
    // Columns past the edge repeat the last one (the last pair).
    const uint32_t col = min(col0 + l32 * kBlocks, n - kBlocks);

    // Step t of B: word i is k 16 t + 8 h + i, by buffer loads whose range ends
    // with the matrix (k past its end reads as zero; a slice that ends before
    // it is whole steps). Steps past the slice repeat its last. The row goes
    // into the vector offset: the range check takes a scalar offset off the
    // range instead, which wraps where that row starts past the end.
    const uint32_t voff = (8 * h * n + col) * static_cast<uint32_t>(sizeof(BT));
    auto load = [&](uint32_t t, uint32_t (&r)[8]) {
        const uint64_t k0 = k_begin + min(t, steps - 1) * 16;
        const uint64_t left = (K - k0) * N * sizeof(BT);
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<BT*>(B + k0 * N), 0, static_cast<int>(static_cast<uint32_t>(left < 0xFFFFFFFFu ? left : 0xFFFFFFFFu)),
            0x00020000);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t row = i * n * static_cast<uint32_t>(sizeof(BT));
            r[i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff + row, 0, kStream);
        }
    };

    // The element of column block j in a word of B.
    auto word = [](uint32_t r, int j) {
        return !kBf16 ? __uint_as_float(r) : j == 0 ? bf16_lo(r) : bf16_hi(r);
    };

    f32x16 acc[kBlocks];
    auto clear = [&]() {
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[b][r] = 0.0f;
    };
    uint32_t tiny = 0xFFFFFFFFu;
    // A's chunk: 8 threads to a row and 32 k, zeros past the slice. Its loads
    // are 16 bytes where A allows them; a k past the slice reads its first.
    constexpr int kUnits = kPanelRows * kPanelK<BT> / 4 / (64 * kPanelWaves);
    const bool wide = K % 4 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0;
    const int row_a = threadIdx.x / 8 % kPanelRows;
    const uint32_t kk0 = threadIdx.x % 8 * 4 + threadIdx.x / (8 * kPanelRows) * 32;  // + 64 a unit
    static_assert(64 * kPanelWaves == 16 * kPanelRows, "a unit is 64 k of every row");
    const uint32_t len = static_cast<uint32_t>(k_end - k_begin);
    const float* const a_row = A + (static_cast<uint64_t>(row_a) < M ? row_a : M - 1) * K + k_begin;
    auto fetch = [&](uint32_t c0, float4 (&x)[kUnits]) {
#pragma unroll
        for (int q = 0; q < kUnits; ++q) {
            const uint32_t k = c0 * 16 + kk0 + 64 * q;
            if (c0 * 16 + 64 * q >= len) break;  // (short slices: no step reads the unit)
            if (wide) {  // (the slice ends on whole fours, too)
                x[q] = *reinterpret_cast<const float4*>(a_row + (k < len ? k : 0));
            } else {
                x[q].x = a_row[k < len ? k : 0];
                x[q].y = a_row[k + 1 < len ? k + 1 : 0];
                x[q].z = a_row[k + 2 < len ? k + 2 : 0];
                x[q].w = a_row[k + 3 < len ? k + 3 : 0];
            }
        }
    };
    auto put = [&](uint32_t c0, const float4 (&x)[kUnits]) {
        uint32_t tiny_a = 0xFFFFFFFFu;
#pragma unroll
        for (int q = 0; q < kUnits; ++q) {
            const uint32_t k = c0 * 16 + kk0 + 64 * q, kk = kk0 + 64 * q;
            if (c0 * 16 + 64 * q >= len) break;
            const float y[4] = {k < len ? x[q].x : 0.0f, k + 1 < len ? x[q].y : 0.0f,
                                k + 2 < len ? x[q].z : 0.0f, k + 3 < len ? x[q].w : 0.0f};
            uint32_t lo[3], hi[3];
            split_pair(y[0], y[1], lo);
            split_pair(y[2], y[3], hi);
            tiny_a = split_min(split_min(tiny_a, y[0], y[1]), y[2], y[3]);
            char* at = lds + kk / 8 * kChunkBytes + row_a * 16 + kk % 8 * 2;
#pragma unroll
            for (int p3 = 0; p3 < 3; ++p3) *reinterpret_cast<u32x2*>(at + p3 * kPlaneBytes) = u32x2{lo[p3], hi[p3]};
        }
        if (tiny_a < kSplitTiny) redo = any_tiny = 1;
    };
    uint32_t raw[kPanelDepth][8];
    if (threadIdx.x == 0) redo = K < kSplitMinK, any_tiny = 0;
    // A's first chunk ahead of an f32 B: loads come back in order, so behind
    // B's it would wait for all of them (as the next chunks do). With 384 k a
    // chunk 24 x 4096 x 11008 44.8 -> 42.9 us, 32 x 11008 x 4096 51 -> 48.
    if constexpr (!kBf16) {
        float4 x[kUnits];
        fetch(0, x);
#pragma unroll
        for (int d = 0; d < kPanelDepth; ++d) load(d, raw[d]);
        __syncthreads();
        put(0, x);
        __syncthreads();
    } else {
#pragma unroll
        for (int d = 0; d < kPanelDepth; ++d) load(d, raw[d]);
    }
    clear();
    constexpr uint32_t kChunkSteps = kPanelK<BT> / 16;
    for (uint32_t c0 = 0; c0 < steps; c0 += kChunkSteps) {
        if (kBf16 || c0) {
            float4 x[kUnits];
            if constexpr (kBf16) __syncthreads();
            fetch(c0, x);
            if constexpr (!kBf16) __syncthreads();
            put(c0, x);
            __syncthreads();
        }
        const uint32_t c_end = min(steps, c0 + kChunkSteps);
        for (uint32_t t0 = c0; t0 < c_end; t0 += kPanelDepth) {
#pragma unroll
            for (int d = 0; d < kPanelDepth; ++d) {
                const uint32_t t = t0 + d;
                if (t >= c_end) break;
                uint32_t(&r)[8] = raw[d];
                u32x4 b[kBlocks][kPlanes];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (kBf16) {
                        b[0][0][i] = __builtin_amdgcn_perm(r[2 * i + 1], r[2 * i], 0x05040100u);
                        b[kBlocks - 1][0][i] = __builtin_amdgcn_perm(r[2 * i + 1], r[2 * i], 0x07060302u);
#pragma unroll
                        for (int e = 0; e < 2; ++e)
                            tiny = split_min(tiny, bf16_lo(r[2 * i + e]), bf16_hi(r[2 * i + e]));
                    } else {
                        uint32_t p[3];
                        const float x0 = __uint_as_float(r[2 * i]), x1 = __uint_as_float(r[2 * i + 1]);
                        split_pair(x0, x1, p);
                        tiny = split_min(tiny, x0, x1);
#pragma unroll
                        for (int q = 0; q < 3; ++q) b[0][q][i] = p[q];
                    }
                }
                load(t + kPanelDepth, r);
                bf16x8 a[3];
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    a[q] = *reinterpret_cast<const bf16x8*>(lds + q * kPlaneBytes +
                                                            (2 * static_cast<int>(t - c0) + h) * kChunkBytes + l32 * 16);
                auto mul = [&](int p, int q) {
#pragma unroll
                    for (int j = 0; j < kBlocks; ++j)
                        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p], __builtin_bit_cast(bf16x8, b[j][q]),
                                                                         acc[j], 0, 0, 0);
                };
                // The order of SplitTile::stage.
                if constexpr (!kBf16) mul(0, 2);
                mul(2, 0);
                if constexpr (!kBf16) {
                    mul(1, 1);
                    mul(0, 1);
                }
                mul(1, 0);
                mul(0, 0);
            }
        }
    }

    // Sums outside the split (split_tile.hpp), entry by entry, in waves that
    // have any: again with the f32 MFMA, straight from memory. 24 x 4096 x 11008
    // with a value below 2^-100 in 64 of A 72 us, 43 with none.
    float probe = 0.0f;
#pragma unroll
    for (int j = 0; j < kBlocks; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(acc[j][r], 0.0f, probe);
    if (probe != 0.0f) redo = 1;
    if (tiny < kSplitTiny) redo = any_tiny = 1;
    __syncthreads();
    if (redo) {
        // The extents of the slice's 32 rows (in LDS, whose planes are done
        // with) and of the lane's columns.
        float2 col_line[kBlocks];
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) col_line[j] = make_float2(0.f, 0.f);
        uint32_t* const least_a = reinterpret_cast<uint32_t*>(lds);
        uint32_t* const big_a = least_a + kPanelRows;
        const float count = static_cast<float>(len);
        if (any_tiny) {
            if (threadIdx.x < kPanelRows) least_a[threadIdx.x] = 0xFFFFFFFFu, big_a[threadIdx.x] = 0;
            __syncthreads();
            constexpr int kRowThreads = 64 * kPanelWaves / kPanelRows;
            const int row = threadIdx.x / kRowThreads;
            const float* const x = A + (static_cast<uint64_t>(row) < M ? row : M - 1) * K + k_begin;
            uint32_t least = 0xFFFFFFFFu, big = 0;
            for (uint32_t k = threadIdx.x % kRowThreads; k < len; k += kRowThreads) {
                least = split_min(least, x[k], 0.0f);
                big = split_max(big, x[k], 0.0f);
            }
            atomicMin(least_a + row, least);
            atomicMax(big_a + row, big);
            uint32_t least_b[kBlocks], big_b[kBlocks];
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) least_b[j] = 0xFFFFFFFFu, big_b[j] = 0;
            for (uint32_t t = 0; t < steps; t += kPanelDepth) {
#pragma unroll
                for (int d = 0; d < kPanelDepth; ++d) load(t + d, raw[d]);
#pragma unroll
                for (int d = 0; d < kPanelDepth; ++d)
#pragma unroll
                    for (int i = 0; i < 8; ++i)
#pragma unroll
                        for (int j = 0; j < kBlocks; ++j) {
                            const float y = word(raw[d][i], j);
                            least_b[j] = split_min(least_b[j], y, 0.0f);
                            big_b[j] = split_max(big_b[j], y, 0.0f);
                        }
            }
#pragma unroll
            for (int j = 0; j < kBlocks; ++j)
                col_line[j] = split_line(min(least_b[j], __shfl_xor(least_b[j], 32, 64)),
                                         max(big_b[j], __shfl_xor(big_b[j], 32, 64)));
            __syncthreads();
        }
        uint32_t again = 0, zero = 0;
        auto line_of = [&](int row) {
            return any_tiny ? split_line(least_a[row], big_a[row]) : make_float2(0.f, 0.f);
        };
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float2 row_line = line_of(8 * (r / 4) + 4 * h + r % 4);
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) {
                const bool is = split_lost(acc[j][r], split_loss(row_line, col_line[j], count));
                again |= (is ? 1u : 0u) << (j * 16 + r);
                zero |= (is && acc[j][r] == 0.0f ? 1u : 0u) << (j * 16 + r);
            }
        }
        for (uint64_t lanes; (lanes = __builtin_amdgcn_ballot_w64(zero != 0)) != 0;) {
            const int l = __builtin_ctzll(lanes);
            const int bit = __builtin_ctz(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(zero), l)));
            const int r = bit % 16, row = 8 * (r / 4) + 4 * (l >> 5) + r % 4;
            const float2 row_line = line_of(row);
            float2 line = col_line[0];
            if (bit / 16) line = col_line[kBlocks - 1];
            line = make_float2(__shfl(line.x, l, 64), __shfl(line.y, l, 64));
            const float* const x = A + (static_cast<uint64_t>(row) < M ? row : M - 1) * K;
            const BT* const y = B + min(col0 + (l & 31) * kBlocks, n - kBlocks) + bit / 16;
            const bool kept = split_cancelled(row_line, line, split_loss(row_line, line, count), k_begin, k_end,
                                              [&](uint64_t k) { return x[k]; }, [&](uint64_t k) { return elem(y + k * N); });
            if (lane == l) {
                zero &= zero - 1;
                if (kept) again &= ~(1u << bit);
            }
        }
        if (K < kSplitMinK) again = 0xFFFFFFFFu;
        if (__builtin_amdgcn_ballot_w64(again != 0)) {
            f32x16 first[kBlocks];
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) first[j] = acc[j];
            clear();
            const float* const x = A + (static_cast<uint64_t>(l32) < M ? l32 : M - 1) * K + k_begin;
            for (uint32_t t = 0; t < steps; t += 2) {
                // (A half of the wave sums k 8 h + i of a step, as it holds B.)
                load(t, raw[0]);
                load(t + 1, raw[1]);
#pragma unroll
                for (int d = 0; d < 2; ++d)
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t k = (t + d) * 16 + 8 * h + i;
                        const float xa = k < len ? x[k] : 0.0f;
#pragma unroll
                        for (int j = 0; j < kBlocks; ++j)
                            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                xa, k < len ? word(raw[d][i], j) : 0.0f, acc[j], 0, 0, 0);
                    }
            }
#pragma unroll
            for (int j = 0; j < kBlocks; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (!(again >> (j * 16 + r) & 1u)) acc[j][r] = first[j][r];
        }
    }

    const bool split = gridDim.y > 1;
    float* out = split ? C + static_cast<uint64_t>(blockIdx.y) * M * N : C;
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
        const uint32_t c = col0 + l32 * kBlocks + j;
        if (c >= n) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t row = 8 * (r / 4) + 4 * h + r % 4;
            if (row < M) out[row * N + c] = split ? acc[j][r] : epilogue(acc[j][r], row, c);
        }
    }
}

// ---------------------------------------------------------------------------
// Up to 8 rows, B [k, n] of any width and alignment
// ---------------------------------------------------------------------------

// The decode GEMV's split (256 columns and a k slice per workgroup, the
// slice's rows dealt to 4 waves that meet in LDS) for rows of B that 16-byte
// loads cannot read: lane l takes columns l, 64 + l, 128 + l, 192 + l of the
// 256, whole 256-byte runs per load. Such products ran on the 64 x 64 tiles
// before: 1 x 4096 x 32001 291 us, 8 rows 302; now 93 and 101 us (5.2-5.6 TB/s).
// The wave number is a scalar, so that A's elements are scalar loads: as vector
// loads, one per row and k, they bounded 8 rows at 182 us.
template <int ROWS, class BT, class Addend>
__global__ __launch_bounds__(256) void ragged_gemv_kernel(const float* __restrict__ A, const BT* __restrict__ B,
                                                          float* __restrict__ C, uint64_t K, uint64_t N,
                                                          uint64_t k_per_slice, Addend epilogue) {
    __shared__ float red[4][ROWS][4][64];
    const int lane = threadIdx.x & 63;
    // (A scalar: A's elements are then scalar loads.)
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const uint64_t col0 = static_cast<uint64_t>(blockIdx.x) * 256 + lane;
    const uint64_t k_begin = static_cast<uint64_t>(blockIdx.y) * k_per_slice;
    const uint64_t k_end = min(K, k_begin + k_per_slice);
    uint64_t col[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) col[j] = min(col0 + 64 * j, N - 1);
    float acc[ROWS][4];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[r][j] = 0.0f;
    auto add = [&](const BT (&b)[4], uint64_t k) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float a = A[r * K + k];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[r][j] = __builtin_fmaf(a, elem(&b[j]), acc[r][j]);
        }
    };
    constexpr int kU = 8;  // rows of B in flight: 128 bytes per lane
    uint64_t k = k_begin + wave;
    for (; k + 4 * (kU - 1) < k_end; k += 4 * kU) {
        BT b[kU][4];
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) b[u][j] = __builtin_nontemporal_load(B + (k + 4 * u) * N + col[j]);
#pragma unroll
        for (int u = 0; u < kU; ++u) add(b[u], k + 4 * u);
    }
    for (; k < k_end; k += 4) {
        BT b[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = B[k * N + col[j]];
        add(b, k);
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j) red[wave][r][j][lane] = acc[r][j];
    __syncthreads();
    // Wave j adds column block j over the waves, in order.
    const uint64_t c = col0 + 64 * wave;
    if (c >= N) return;
    const bool split = gridDim.y > 1;
    float* out = split ? C + static_cast<uint64_t>(blockIdx.y) * ROWS * N : C;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        float v = red[0][r][wave][lane];
#pragma unroll
        for (int w = 1; w < 4; ++w) v += red[w][r][wave][lane];
        out[r * N + c] = split ? v : epilogue(v, r, c);
    }
}

// ---------------------------------------------------------------------------
// Up to 8 rows, B [n, k]
// ---------------------------------------------------------------------------

// C[r, n] = sum_k A[r, k] B[n, k] for ROWS rows of A: a wave takes COLS rows
// of B, lane l the k of [512 i + 8 l, + 8), its sums met by a butterfly. k is
// a multiple of 8 and the rows are 16-byte aligned. The f32 and the compact B
// sum in the same order.
//
// What bounds it: HBM for few rows, A's reads from L1 towards 8 (a wave reads
// all of A for COLS rows of B). One row on the 64 x 64 tiles, 63 of 64 rows of
// MFMA work for padding, read a 32000 x 4096 head in 370 us (f32 MFMA) and 188
// (split); here 1 row 104 us (5.0 TB/s), 4 rows 115, 8 rows 173.
template <int ROWS, int COLS, class BT, class Addend>
__global__ __launch_bounds__(256) void dot_kernel(const float* __restrict__ A, const BT* __restrict__ B,
                                                  float* __restrict__ C, uint64_t K, uint64_t N,
                                                  Addend epilogue) {
    constexpr bool kBf16 = sizeof(BT) == 2;
    constexpr int kVecs = kBf16 ? 1 : 2;  // 16-byte loads per 8 elements
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const uint64_t n0 = (static_cast<uint64_t>(blockIdx.x) * 4 + wave) * COLS;
    if (n0 >= N) return;
    const BT* rows[COLS];
#pragma unroll
    for (int c = 0; c < COLS; ++c) rows[c] = B + min(n0 + c, N - 1) * K;
    float acc[ROWS][COLS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c) acc[r][c] = 0.0f;
    auto load = [&](uint64_t k, uint4 (&v)[COLS][kVecs]) {
#pragma unroll
        for (int c = 0; c < COLS; ++c)
#pragma unroll
            for (int q = 0; q < kVecs; ++q) {
                v[c][q] = make_uint4(0, 0, 0, 0);
                if (k < K) v[c][q] = load_nt(reinterpret_cast<const uint4*>(rows[c] + k) + q);
            }
    };
    uint4 next[COLS][kVecs];
    load(8 * lane, next);
    for (uint64_t k0 = 0; k0 < K; k0 += 512) {
        const uint64_t k = k0 + 8 * lane;
        uint4 cur[COLS][kVecs];
#pragma unroll
        for (int c = 0; c < COLS; ++c)
#pragma unroll
            for (int q = 0; q < kVecs; ++q) cur[c][q] = next[c][q];
        if (k0 + 512 < K) load(k + 512, next);
        float x[ROWS][8];
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                if (k < K) v = *reinterpret_cast<const float4*>(A + r * K + k + 4 * q);
                x[r][4 * q] = v.x; x[r][4 * q + 1] = v.y; x[r][4 * q + 2] = v.z; x[r][4 * q + 3] = v.w;
            }
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            float b[8];
            if constexpr (kBf16) {
                const uint32_t w[4] = {cur[c][0].x, cur[c][0].y, cur[c][0].z, cur[c][0].w};
#pragma unroll
                for (int e = 0; e < 8; ++e) b[e] = e & 1 ? bf16_hi(w[e / 2]) : bf16_lo(w[e / 2]);
            } else {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    b[4 * q] = __uint_as_float(cur[c][q].x); b[4 * q + 1] = __uint_as_float(cur[c][q].y);
                    b[4 * q + 2] = __uint_as_float(cur[c][q].z); b[4 * q + 3] = __uint_as_float(cur[c][q].w);
                }
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[r][c] = __builtin_fmaf(x[r][e], b[e], acc[r][c]);
        }
    }
    float mine = 0.0f;  // lane r * COLS + c: output (r, n0 + c)
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            float v = acc[r][c];
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
            if (lane == r * COLS + c) mine = v;
        }
    const int r = lane / COLS;
    const uint64_t c = n0 + lane % COLS;
    if (lane < ROWS * COLS && c < N) C[r * N + c] = epilogue(mine, r, c);
}

}  // namespace mhip
