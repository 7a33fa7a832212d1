// One C tile of an f32 product on the bf16 matrix cores.
//
// gfx950's f32 MFMA sustains about 150 TFLOP/s on this card and its bf16 MFMA
// 1,850-2,000 (32x32x16 and 16x16x32 register loops on 256 CUs), so an f32
// product costs less as six bf16 products. Every f32 operand x is split
// exactly into three bf16 planes, x = x1 + x2 + x3, each the nearest bf16 of
// what is left (8 significant bits a plane, 24 in all). Of the nine plane
// products the six of at least 2^-18 of x y are summed, smallest first, in
// the f32 accumulators:
//     a1 b3 + a3 b1 + a2 b2 + a1 b2 + a2 b1 + a1 b1;
// the other three add up to at most 1.01 x 2^-24 of |x y| (|x2| <= 2^-8 |x|, |x3|
// <= 2^-17 |x|; 2^-27.5 as the rms over mantissas), the largest rounding of one
// product. An accumulator is rounded 6 times per 16 k rather than about 16, so
// from k 3 on sums come out closer to the exact product than with the f32 MFMA
// on every distribution measured (kSplitMinK has the shorter ones): 2-norm errors against f64 of 32 x 32 tiles, f32 MFMA and split,
// N(0,1) x N(0,0.02): K 64 1.45e-7 and 1.10e-7, 256 2.9e-7 and 2.4e-7, 4096
// 1.15e-6 and 0.99e-6, 16384 2.3e-6 and 2.1e-6; U(0,1): K 4096 8.4e-7 and
// 5.3e-7; log-normal: 1.1e-6 and 6.1e-7. A compact bf16 B is its own single
// plane: three products (a3 b1 + a2 b1 + a1 b1), whose sums equal those of
// the six with zero planes bit for bit.
//
// The split holds for zeros and 2^-100 <= |x| < the largest f32 that rounds
// to a finite bf16; any other value that enters a sum costs it terms that the
// f32 MFMA keeps. An entry whose sum may have lost any is summed again with
// it, decided per entry from its own row of A and column of B, so that no
// other row or column moves its bits:
//  - a sum that is not finite (an infinity, a NaN or a value beyond turns the
//    planes' sums into NaN; a sum may overflow);
//  - a sum that a nonzero |x| < 2^-100 in its row or column may matter to.
//    Such a value's planes are off by less than 2^-124 (planes below 2^-126
//    may be flushed), its k products by 2^-124 k max|y| of the other operand's
//    column or row. Sums of at least 2^26 times that keep theirs.
#pragma once

#include "common.hpp"

namespace mhip {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Two f32 as packed bf16 (round to nearest even), x0 in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float x0, float x1) {
    const f32x2 v = {x0, x1};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float bf16_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t u) { return __uint_as_float(u & 0xFFFF0000u); }

// The planes of two f32 values, packed: p[0], p[1], p[2] are x1, x2, x3.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t (&p)[3]) {
    p[0] = pack_bf16(x0, x1);
    const float r0 = x0 - bf16_lo(p[0]), r1 = x1 - bf16_hi(p[0]);
    p[1] = pack_bf16(r0, r1);
    // What is left has at most 8 significant bits: its upper half is it.
    const float s0 = r0 - bf16_lo(p[1]), s1 = r1 - bf16_hi(p[1]);
    p[2] = __builtin_amdgcn_perm(__float_as_uint(s1), __float_as_uint(s0), 0x07060302u);
}

// Smallest magnitude seen: 2 |x| - 1 as an integer, so that a zero is the
// largest value there is. A minimum below kSplitTiny is a nonzero |x| < 2^-100.
constexpr uint32_t kSplitTiny = 2u * ((127u - 100u) << 23) - 1u;
__device__ __forceinline__ uint32_t split_min(uint32_t m, float x0, float x1) {
    const uint32_t t0 = (__float_as_uint(x0) << 1) - 1u, t1 = (__float_as_uint(x1) << 1) - 1u;
    return min(m, min(t0, t1));
}

// Largest magnitude seen, as 2 |x|.
__device__ __forceinline__ uint32_t split_max(uint32_t m, float x0, float x1) {
    return max(m, max(__float_as_uint(x0) << 1, __float_as_uint(x1) << 1));
}
// A row or column from its extents (least: split_min's, big: split_max's):
// whether it holds a nonzero below 2^-100 (1 or 0), and its largest magnitude.
__device__ __forceinline__ float2 split_line(uint32_t least, uint32_t big) {
    return make_float2(least < kSplitTiny ? 1.0f : 0.0f, __uint_as_float(big >> 1));
}
// What such values may cost the sum of k products of a row and a column, times
// 2^26. (0 times an infinite extent is NaN, taken for none: the sum is not
// finite then.)
__device__ __forceinline__ float split_loss(float2 row, float2 col, float k) {
    return fmaxf(row.x * col.y, col.x * row.y) * (k * 0x1p-98f);
}
__device__ __forceinline__ bool split_lost(float sum, float loss) {
    return !(fabsf(sum) < INFINITY) || fabsf(sum) < loss;
}
// Sums of so few products take the f32 MFMA outright: a product's six planes
// are rounded into the accumulator one by one, up to 2.3 u of it (u = 2^-24)
// where a single f32 product is rounded once. 2-norm errors of 256 x 256
// products, f32 MFMA and split, N(0,1): k 1 2.5e-8 and 3.5e-8, 2 3.2e-8 and
// 3.4e-8, 3 3.6e-8 and 3.3e-8, 16 7.3e-8 and 3.4e-8.
constexpr uint64_t kSplitMinK = 3;

// A sum of exactly 0 where 0 < loss: one in some 2^24 sums cancels to that, and
// has lost nothing if the magnitudes of its terms add up to the loss. The whole
// wave asks for one entry; x(k) and y(k) are its row and column.
template <class X, class Y>
__device__ __forceinline__ bool split_cancelled(float2 row, float2 col, float loss, uint64_t k_begin, uint64_t k_end,
                                                X x, Y y) {
    // No terms can add up to the loss of values that small.
    if ((row.x != 0.0f && row.y < 0x1p-98f) || (col.x != 0.0f && col.y < 0x1p-98f)) return false;
    const int lane = threadIdx.x & 63;
    float mine = 0.0f;
    for (uint64_t k0 = k_begin; k0 < k_end; k0 += 64) {
        const uint64_t k = k0 + lane;
        if (k < k_end) mine += fabsf(x(k) * y(k));
        if (__builtin_amdgcn_ballot_w64(mine >= loss)) return true;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mine += __shfl_xor(mine, off, 64);
    return mine >= loss;
}

// Workgroup barrier that publishes LDS writes without waiting for the global
// loads in flight (__syncthreads waits for every counter), nor for the last
// READS LDS reads of the wave: those were issued after its last LDS write
// (lds_order keeps them there), and LDS operations complete in order.
template <int READS>
__device__ __forceinline__ void lds_barrier() {
    static_assert(READS < 16, "the LDS counter has 4 bits");
    __asm__ volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(READS) : "memory");
}
// LDS accesses before it stay before it, and those after it after.
__device__ __forceinline__ void lds_order() { __asm__ volatile("" ::: "memory"); }

// One operand's share of a tile: ROWS rows along m or n by BK of k per stage,
// read from memory by every thread of the workgroup (E elements each), split
// and written to LDS. KMAJOR: rows along k in memory (A stored [k, m], B stored
// [k, n]): a thread takes UK consecutive k of COLS columns, lanes along the
// columns; otherwise (A [m, k], B [n, k]) a thread takes 4 consecutive k of
// E / 4 rows, BK / 4 lanes to a row.
//
// LDS holds, per plane, chunks of 8 k: [chunk][row] 16-byte slots, which is
// the MFMA's operand as one 16-byte read per lane, 16 rows in 256 consecutive
// bytes. The chunks are kPad apart so that the 8-byte writes of neighbouring
// chunks fall on different banks.
template <class T, bool KMAJOR, int ROWS, int BK, int THREADS>
struct SplitOperand {
    static constexpr bool kBf16 = std::is_same<T, uint16_t>::value;
    static constexpr int kPlanes = kBf16 ? 1 : 3;
    static constexpr int kElems = ROWS * BK / THREADS;  // per thread and stage
    static constexpr int kChunks = BK / 8;
    static constexpr int kPad = BK == 32 ? 64 : 128;     // bytes
    static constexpr int kChunkBytes = ROWS * 16 + kPad;
    static constexpr int kPlaneBytes = kChunks * kChunkBytes;
    static constexpr int kStageBytes = kPlanes * kPlaneBytes;
    static constexpr int kCols = KMAJOR && kBf16 && kElems >= 8 ? 2 : 1;
    static constexpr int kUK = KMAJOR ? kElems / kCols : 4;
    static constexpr int kUnits = KMAJOR ? 1 : kElems / 4;
    static_assert(!KMAJOR || kUK == 4 || kUK == 8, "a k-major unit is 4 or 8 k");
    static_assert(!KMAJOR || ROWS / kCols % 64 == 0, "a wave's k-major units share their k");
    static_assert(KMAJOR || THREADS % (BK / 4) == 0, "lanes cover whole rows");

    const T* g;        // the tile's first row (row-major) or column (k-major), at k 0
    uint64_t ld;
    uint64_t limit;    // rows (or columns) of the operand from the tile's first one
    bool wide;         // row-major: 16-byte (8-byte bf16) loads; k-major bf16: column pairs
    int kgroup;        // k-major: this wave's group of kUK k
    uint32_t voff[kUnits];
    uint32_t raw[KMAJOR ? kUK : kUnits * (kBf16 ? 2 : 4)];  // k-major bf16: column pairs

    __device__ __forceinline__ void init(const T* base, uint64_t lead, uint64_t first, uint64_t total,
                                         bool can_wide) {
        g = KMAJOR ? base + first : base + first * lead;
        ld = lead;
        limit = total - first;
        wide = can_wide;
        const int t = threadIdx.x;
        if constexpr (KMAJOR) {
            constexpr int kGroup = ROWS / kCols;
            kgroup = __builtin_amdgcn_readfirstlane(t / kGroup);
            // Columns past the edge repeat the last one (the last pair, of an
            // even number of columns): their products are not stored.
            const uint64_t c = static_cast<uint64_t>(t % kGroup) * kCols;
            const uint64_t last = limit - (kCols == 2 && wide ? 2 : 1);
            voff[0] = static_cast<uint32_t>(min(c, last) * sizeof(T));
        } else {
            kgroup = 0;
#pragma unroll
            for (int u = 0; u < kUnits; ++u) {
                const uint64_t r = (t + u * THREADS) / (BK / 4);
                voff[u] = static_cast<uint32_t>((min(r, limit - 1) * ld + (t % (BK / 4)) * 4) * sizeof(T));
            }
        }
    }

    // Unit u's loads of the whole stage at k0.
    __device__ __forceinline__ void load(uint64_t k0, int u) {
        const T* p = KMAJOR ? g + k0 * ld : g + k0;
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), 0, -1, 0x00020000);
        if constexpr (KMAJOR) {
#pragma unroll
            for (int i = 0; i < kUK; ++i) {
                const uint32_t soff = static_cast<uint32_t>((kgroup * kUK + i) * ld * sizeof(T));
                if constexpr (!kBf16) {
                    raw[i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff[0], soff, 0);
                } else if constexpr (kCols == 1) {
                    raw[i] = __builtin_amdgcn_raw_buffer_load_b16(rsrc, voff[0], soff, 0);
                } else if (wide) {
                    raw[i] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff[0], soff, 0);
                } else {
                    const uint32_t next = voff[0] / 2 + 1 < limit ? 2 : 0;
                    const uint32_t lo = __builtin_amdgcn_raw_buffer_load_b16(rsrc, voff[0], soff, 0);
                    const uint32_t hi = __builtin_amdgcn_raw_buffer_load_b16(rsrc, voff[0] + next, soff, 0);
                    raw[i] = (lo & 0xFFFFu) | hi << 16;
                }
            }
        } else if constexpr (!kBf16) {
            if (wide) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff[u], 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) raw[4 * u + e] = v[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    raw[4 * u + e] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff[u] + 4 * e, 0, 0);
            }
        } else {
            if (wide) {
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff[u], 0, 0);
                raw[2 * u] = v[0];
                raw[2 * u + 1] = v[1];
            } else {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t lo = __builtin_amdgcn_raw_buffer_load_b16(rsrc, voff[u] + 4 * e, 0, 0);
                    const uint32_t hi = __builtin_amdgcn_raw_buffer_load_b16(rsrc, voff[u] + 4 * e + 2, 0, 0);
                    raw[2 * u + e] = (lo & 0xFFFFu) | hi << 16;
                }
            }
        }
    }

    // The same for a stage that ends at k_end inside it (zeros beyond), or of
    // an operand whose rows are too long for 32-bit offsets.
    __device__ __forceinline__ void load_edge(uint64_t k0, uint64_t k_end, int u) {
        const int t = threadIdx.x;
        auto at = [&](uint64_t row, uint64_t k) -> uint32_t {
            row = min(row, limit - 1);
            if (k >= k_end) return 0;
            const T v = KMAJOR ? g[k * ld + row] : g[row * ld + k];
            return __builtin_bit_cast(typename std::conditional<kBf16, uint16_t, uint32_t>::type, v);
        };
        if constexpr (KMAJOR) {
            constexpr int kGroup = ROWS / kCols;
            const uint64_t c = static_cast<uint64_t>(t % kGroup) * kCols;
#pragma unroll
            for (int i = 0; i < kUK; ++i) {
                const uint64_t k = k0 + kgroup * kUK + i;
                raw[i] = at(c, k);
                if constexpr (kCols == 2) raw[i] |= at(c + 1, k) << 16;
            }
        } else {
            const uint64_t r = (t + u * THREADS) / (BK / 4);
            const uint64_t k = k0 + (t % (BK / 4)) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (!kBf16) raw[4 * u + e] = at(r, k + e);
                else if (e % 2 == 0) raw[2 * u + e / 2] = at(r, k + e) | at(r, k + e + 1) << 16;
            }
        }
    }

    // f32 element i of unit u: k-major, k i of column c; else k i of the row.
    __device__ __forceinline__ float value(int u, int i, int c = 0) const {
        if constexpr (!kBf16) return __uint_as_float(raw[KMAJOR ? i : 4 * u + i]);
        else if constexpr (KMAJOR) return c == 0 ? bf16_lo(raw[i]) : bf16_hi(raw[i]);
        else return (i & 1) ? bf16_hi(raw[2 * u + i / 2]) : bf16_lo(raw[2 * u + i / 2]);
    }

    // The extents (split_min, split_max) of the tile's rows (columns) over k in
    // [k_begin, k_end), into arrays in LDS: several stages' loads at a time, as
    // the loop waits for nothing else.
    template <int kAhead>
    __device__ __forceinline__ void extents(uint64_t k_begin, uint64_t k_end, bool short_rows, uint32_t* least,
                                            uint32_t* big) {
        constexpr int kLines = KMAJOR ? kCols : kUnits;  // column i of a k-major thread, else unit i's row
        uint32_t lo[kLines], hi[kLines];
#pragma unroll
        for (int i = 0; i < kLines; ++i) lo[i] = 0xFFFFFFFFu, hi[i] = 0;
        auto gather = [&](const SplitOperand& o) {
#pragma unroll
            for (int u = 0; u < kUnits; ++u)
#pragma unroll
                for (int c = 0; c < kCols; ++c)
#pragma unroll
                    for (int i = 0; i < kUK; i += 2) {
                        const float x0 = o.value(u, i, c), x1 = o.value(u, i + 1, c);
                        lo[u + c] = split_min(lo[u + c], x0, x1);
                        hi[u + c] = split_max(hi[u + c], x0, x1);
                    }
        };
        uint64_t k0 = k_begin;
        for (; short_rows && k0 + kAhead * BK <= k_end; k0 += kAhead * BK) {
            SplitOperand ahead[kAhead];
#pragma unroll
            for (int d = 0; d < kAhead; ++d) {
                ahead[d] = *this;
#pragma unroll
                for (int u = 0; u < kUnits; ++u) ahead[d].load(k0 + d * BK, u);
            }
#pragma unroll
            for (int d = 0; d < kAhead; ++d) gather(ahead[d]);
        }
        for (; k0 < k_end; k0 += BK) {
#pragma unroll
            for (int u = 0; u < kUnits; ++u) load_edge(k0, k_end, u);
            gather(*this);
        }
#pragma unroll
        for (int i = 0; i < kLines; ++i) {
            const int t = threadIdx.x;
            const int row = KMAJOR ? t % (ROWS / kCols) * kCols + i : (t + i * THREADS) / (BK / 4);
            atomicMin(least + row, lo[i]);
            atomicMax(big + row, hi[i]);
        }
    }

    // Splits unit u and writes its planes to the stage at `lds`.
    __device__ __forceinline__ void store(char* lds, int u, uint32_t& tiny) const {
        const int t = threadIdx.x;
        constexpr int kWords = kUK / 2;
#pragma unroll
        for (int c = 0; c < kCols; ++c) {
            uint32_t w[3][kWords];
#pragma unroll
            for (int i = 0; i < kWords; ++i) {
                const float x0 = value(u, 2 * i, c), x1 = value(u, 2 * i + 1, c);
                tiny = split_min(tiny, x0, x1);
                if constexpr (kBf16) {
                    if constexpr (!KMAJOR) w[0][i] = raw[2 * u + i];
                    else if constexpr (kCols == 1)
                        w[0][i] = __builtin_amdgcn_perm(raw[2 * i + 1], raw[2 * i], 0x05040100u);
                    else
                        w[0][i] = __builtin_amdgcn_perm(raw[2 * i + 1], raw[2 * i], c == 0 ? 0x05040100u : 0x07060302u);
                } else {
                    uint32_t p[3];
                    split_pair(x0, x1, p);
                    w[0][i] = p[0];
                    w[1][i] = p[1];
                    w[2][i] = p[2];
                }
            }
            int row, k;
            if constexpr (KMAJOR) {
                row = t % (ROWS / kCols) * kCols + c;
                k = kgroup * kUK;
            } else {
                row = (t + u * THREADS) / (BK / 4);
                k = t % (BK / 4) * 4;
            }
            char* at = lds + k / 8 * kChunkBytes + row * 16 + k % 8 * 2;
#pragma unroll
            for (int p = 0; p < kPlanes; ++p) {
                if constexpr (kWords == 4)
                    *reinterpret_cast<u32x4*>(at + p * kPlaneBytes) = u32x4{w[p][0], w[p][1], w[p][2], w[p][3]};
                else
                    *reinterpret_cast<u32x2*>(at + p * kPlaneBytes) = u32x2{w[p][0], w[p][1]};
            }
        }
    }

    // Unit u as f32 into [BK][ROWS + 4] (the f32 sum; 4 floats of padding put
    // a row-major wave's 4 k by 16 rows on distinct banks).
    static constexpr int kF32Bytes = BK * (ROWS + 4) * 4;
    __device__ __forceinline__ void store_f32(float* lds, int u) const {
        const int t = threadIdx.x;
#pragma unroll
        for (int c = 0; c < kCols; ++c)
#pragma unroll
            for (int i = 0; i < kUK; ++i) {
                if constexpr (KMAJOR)
                    lds[(kgroup * kUK + i) * (ROWS + 4) + t % (ROWS / kCols) * kCols + c] = value(u, i, c);
                else
                    lds[(t % (BK / 4) * 4 + i) * (ROWS + 4) + (t + u * THREADS) / (BK / 4)] = value(u, i);
            }
    }

    static __device__ __forceinline__ bf16x8 fragment(const char* lds, int plane, int chunk, int row) {
        return *reinterpret_cast<const bf16x8*>(lds + plane * kPlaneBytes + chunk * kChunkBytes + row * 16);
    }
};

// A BM x BN tile by waves of WM x WN, in stages of BK (16 or 32) of k,
// triple-buffered in LDS. KG 2: two groups of waves each take one half of
// every stage's k and meet in LDS at the end.
template <int BM, int BN, int WM, int WN, int KG, int BK, bool A_T, bool B_T, class BT, int BUFS = 3>
struct SplitTile {
    static constexpr int kWavesN = BN / WN;
    static constexpr int kTileWaves = (BM / WM) * kWavesN;
    static constexpr int kWaves = kTileWaves * KG;
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int kMI = WM / 32, kNI = WN / 32;
    using OpA = SplitOperand<float, A_T, BM, BK, kThreads>;
    using OpB = SplitOperand<BT, !B_T, BN, BK, kThreads>;
    static constexpr int kStageBytes = OpA::kStageBytes + OpB::kStageBytes;
    // One being summed, one complete (its first operands are read before the
    // barrier that ends the stage), one being written.
    static constexpr int kBufs = BUFS;
    static constexpr int kMeetBytes = KG == 2 ? kWaves * kMI * kNI * 8 * 64 * 4 : 0;
    static constexpr int cmax(int a, int b) { return a > b ? a : b; }
    static constexpr int kLdsBytes =
        cmax(kBufs * kStageBytes, cmax(cmax(OpA::kF32Bytes + OpB::kF32Bytes, (BM + BN) * 16), kMeetBytes));
    static_assert(kLdsBytes <= 160 * 1024, "a workgroup's LDS");
    static_assert(KG == 1 || BK == 32, "each k group takes one 16 of a stage");

    f32x16 acc[kMI][kNI];

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < kMI; ++i)
#pragma unroll
            for (int j = 0; j < kNI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    }

    // The operands of one step (16 of k): this wave's A blocks and its first
    // column block of B.
    static constexpr int kSteps = BK / 16 / KG;  // per stage and wave
    static constexpr int kHooks = kSteps * kNI;
    struct Operands {
        bf16x8 a[kMI][3], b[OpB::kPlanes];
    };
    struct Lane {
        int kg, row_a, row_b, h;
    };
    static __device__ __forceinline__ int chunk_of(const Lane& at, int step) {
        return 2 * (KG == 2 ? at.kg : step) + at.h;
    }
    static __device__ __forceinline__ void read_a(Operands& o, const char* la, const Lane& at, int step, int p) {
#pragma unroll
        for (int i = 0; i < kMI; ++i) o.a[i][p] = OpA::fragment(la, p, chunk_of(at, step), at.row_a + i * 32);
    }
    static __device__ __forceinline__ void read_b(bf16x8 (&b)[OpB::kPlanes], const char* la, const Lane& at, int step,
                                                  int j) {
#pragma unroll
        for (int p = 0; p < OpB::kPlanes; ++p)
            b[p] = OpB::fragment(la + OpA::kStageBytes, p, chunk_of(at, step), at.row_b + j * 32);
    }

    // One stage's MFMAs from the buffer `cur`, its first step's operands in
    // `o`; AHEAD leaves the first step's operands of the stage in `next` there,
    // read after the last hook. hook(q) runs before each of the kHooks column
    // blocks. Each column block's operands are read a block ahead, and a
    // step's A planes as soon as the step before has no more use for them.
    static constexpr int kAheadReads = kMI * 3 + OpB::kPlanes;
    template <bool AHEAD, class Hook>
    __device__ __forceinline__ void stage(const char* cur, const char* next, const Lane& at, Operands& o, Hook hook) {
        constexpr bool kSix = OpB::kPlanes == 3;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const bool final = s + 1 == kSteps;
            const char* const ahead = final ? next : cur;
            const int ahead_step = final ? 0 : s + 1;
#pragma unroll
            for (int j = 0; j < kNI; ++j) {
                const bool last = j + 1 == kNI && (AHEAD || !final);
                bf16x8 b[OpB::kPlanes];
                hook(s * kNI + j);
                if (j + 1 == kNI && final) lds_order();
                if (j + 1 < kNI) read_b(b, cur, at, s, j + 1);
                else if (last) read_b(b, ahead, at, ahead_step, 0);
                auto mul = [&](int p, int q) {
#pragma unroll
                    for (int i = 0; i < kMI; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(o.a[i][p], o.b[q], acc[i][j], 0, 0, 0);
                };
                if constexpr (kSix) mul(0, 2);
                mul(2, 0);
                if (last) read_a(o, ahead, at, ahead_step, 2);
                if constexpr (kSix) {
                    mul(1, 1);
                    mul(0, 1);
                }
                mul(1, 0);
                if (last) read_a(o, ahead, at, ahead_step, 1);
                mul(0, 0);
                if (last) read_a(o, ahead, at, ahead_step, 0);
#pragma unroll
                for (int p = 0; p < OpB::kPlanes; ++p) o.b[p] = b[p];
            }
        }
    }

    // C[m0 .., n0 ..] summed over k in [k_begin, k_end) into acc (per k
    // group) by the split's products; whether some of the sums in the workgroup
    // are to be summed again (`again`: lost()). LDS is free on entry and on return.
    __device__ __forceinline__ bool sum(const float* __restrict__ A, const BT* __restrict__ B, uint64_t M,
                                        uint64_t K, uint64_t N, uint64_t m0, uint64_t n0, uint64_t k_begin,
                                        uint64_t k_end, bool wide_a, bool wide_b, bool short_rows, char* lds,
                                        uint32_t (&again)[(kMI * kNI * 16 + 31) / 32]) {
        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
        const int kg = wave / kTileWaves, wt = wave % kTileWaves;
        const int wm = wt / kWavesN, wn = wt % kWavesN;
        OpA oa;
        OpB ob;
        oa.init(A, A_T ? M : K, m0, M, wide_a);
        ob.init(B, B_T ? K : N, n0, N, wide_b);
        clear();
        uint32_t tiny = 0xFFFFFFFFu;
        auto load = [&](uint64_t k0) {
#pragma unroll
            for (int u = 0; u < OpA::kUnits; ++u) oa.load(k0, u);
#pragma unroll
            for (int u = 0; u < OpB::kUnits; ++u) ob.load(k0, u);
        };
        auto load_edge = [&](uint64_t k0) {
#pragma unroll
            for (int u = 0; u < OpA::kUnits; ++u) oa.load_edge(k0, k_end, u);
#pragma unroll
            for (int u = 0; u < OpB::kUnits; ++u) ob.load_edge(k0, k_end, u);
        };
        auto store = [&](char* to) {
#pragma unroll
            for (int u = 0; u < OpA::kUnits; ++u) oa.store(to, u, tiny);
#pragma unroll
            for (int u = 0; u < OpB::kUnits; ++u) ob.store(to + OpA::kStageBytes, u, tiny);
        };
        const Lane at{kg, wm * WM + (lane & 31), wn * WN + (lane & 31), lane >> 5};
        Operands o;
        auto read_first = [&](const char* from) {
#pragma unroll
            for (int p = 0; p < 3; ++p) read_a(o, from, at, 0, p);
            read_b(o.b, from, at, 0, 0);
        };
        const uint64_t whole = short_rows ? (k_end - k_begin) / BK : 0;
        if (whole > 0) {
            // While stage s is summed, stage s + 2, loaded into registers a
            // stage ago, is split into the third buffer and stage s + 3 is
            // loaded. Past the end the last stage is read again, unused:
            // nothing in the loop is conditional.
            auto k_of = [&](uint64_t s) { return k_begin + min(s, whole - 1) * BK; };
            load(k_of(0));
            store(lds);
            load(k_of(1));
            if constexpr (BUFS == 3) {
                store(lds + kStageBytes);
                load(k_of(2));
            }
            lds_barrier<0>();
            if constexpr (BUFS == 3) read_first(lds);
            int cur = 0, next = kStageBytes, third = 2 * kStageBytes;
            for (uint64_t s = 0; s < whole; ++s) {
                const uint64_t k_next = k_of(s + BUFS);
                char* const to = lds + (BUFS == 3 ? third : next);
                if constexpr (BUFS == 2) read_first(lds + cur);
                // The units are spread over the column blocks.
                constexpr int kAll = OpA::kUnits + OpB::kUnits;
                auto unit = [&](int u) {
                    if (u < OpA::kUnits) {
                        oa.store(to, u, tiny);
                        oa.load(k_next, u);
                    } else {
                        ob.store(to + OpA::kStageBytes, u - OpA::kUnits, tiny);
                        ob.load(k_next, u - OpA::kUnits);
                    }
                };
                stage<BUFS == 3>(lds + cur, lds + next, at, o, [&](int q) {
#pragma unroll
                    for (int u = 0; u < kAll; ++u)
                        if (u * kHooks / kAll == q) unit(u);
                });
                lds_barrier<BUFS == 3 ? kAheadReads : 0>();
                const int freed = cur;
                cur = next;
                if constexpr (BUFS == 3) {
                    next = third;
                    third = freed;
                } else {
                    next = freed;
                }
            }
        }
        for (uint64_t k0 = k_begin + whole * BK; k0 < k_end; k0 += BK) {
            load_edge(k0);
            store(lds);
            lds_barrier<0>();
            read_first(lds);
            stage<false>(lds, lds, at, o, [](int) {});
            lds_barrier<0>();
        }

        // A sum that is not finite times 0 is a NaN.
        float probe = 0.0f;
#pragma unroll
        for (int i = 0; i < kMI; ++i)
#pragma unroll
            for (int j = 0; j < kNI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(acc[i][j][r], 0.0f, probe);
        if (!__syncthreads_or(tiny < kSplitTiny || probe != 0.0f)) return false;
        const bool any_tiny = __syncthreads_or(tiny < kSplitTiny);
        return lost(A, B, M, K, N, m0, n0, k_begin, k_end, wide_a, wide_b, short_rows, any_tiny, lds, again);
    }

    // The sums to be summed again, bit (i * kNI + j) * 16 + r of `again` for
    // register r of block (i, j); whether the workgroup has any. With values
    // below 2^-100 about (any_tiny) the extents of the tile's rows and columns
    // are read first. 4096^3 with one such value in 64 of A: 802 us, 688 with
    // none (1773 when such tiles were summed again, 985 on f32 MFMA kernels);
    // with every value of A at 1e-35, whose sums need it, 1875.
    static constexpr int kExtentsAhead = kMI * kNI >= 8 ? 2 : 4;  // (registers)
    static constexpr int kWords = (kMI * kNI * 16 + 31) / 32;
    using Mask = uint32_t[kWords];
    __device__ __forceinline__ bool lost(const float* __restrict__ A, const BT* __restrict__ B, uint64_t M,
                                         uint64_t K, uint64_t N, uint64_t m0, uint64_t n0, uint64_t k_begin,
                                         uint64_t k_end, bool wide_a, bool wide_b, bool short_rows, bool any_tiny,
                                         char* lds, Mask& again) {
        uint32_t* const least_a = reinterpret_cast<uint32_t*>(lds);
        uint32_t* const big_a = least_a + BM;
        uint32_t* const least_b = big_a + BM;
        uint32_t* const big_b = least_b + BN;
        float2* const lines = reinterpret_cast<float2*>(big_b + BN);
        if (any_tiny) {
            for (int i = threadIdx.x; i < BM; i += kThreads) least_a[i] = 0xFFFFFFFFu, big_a[i] = 0;
            for (int i = threadIdx.x; i < BN; i += kThreads) least_b[i] = 0xFFFFFFFFu, big_b[i] = 0;
            __syncthreads();
            OpA oa;
            oa.init(A, A_T ? M : K, m0, M, wide_a);
            oa.template extents<kExtentsAhead>(k_begin, k_end, short_rows, least_a, big_a);
            OpB ob;
            ob.init(B, B_T ? K : N, n0, N, wide_b);
            ob.template extents<kExtentsAhead>(k_begin, k_end, short_rows, least_b, big_b);
            __syncthreads();
            for (int i = threadIdx.x; i < BM; i += kThreads) lines[i] = split_line(least_a[i], big_a[i]);
            for (int i = threadIdx.x; i < BN; i += kThreads) lines[BM + i] = split_line(least_b[i], big_b[i]);
            __syncthreads();
        }
        const int lane = threadIdx.x & 63;
        const int wt = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)) % kTileWaves;
        const int row0 = wt / kWavesN * WM + 4 * (lane >> 5), col0 = wt % kWavesN * WN + (lane & 31);
        const float count = static_cast<float>(k_end - k_begin);
        float2 col[kNI];
#pragma unroll
        for (int j = 0; j < kNI; ++j) col[j] = any_tiny ? lines[BM + col0 + j * 32] : make_float2(0.f, 0.f);
        Mask zero;
#pragma unroll
        for (int w = 0; w < kWords; ++w) again[w] = zero[w] = 0;
#pragma unroll
        for (int i = 0; i < kMI; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float2 row = any_tiny ? lines[row0 + i * 32 + 8 * (r / 4) + r % 4] : make_float2(0.f, 0.f);
#pragma unroll
                for (int j = 0; j < kNI; ++j) {
                    const int bit = (i * kNI + j) * 16 + r;
                    const float sum = acc[i][j][r];
                    const bool is = split_lost(sum, split_loss(row, col[j], count));
                    again[bit / 32] |= (is ? 1u : 0u) << bit % 32;
                    zero[bit / 32] |= (is && sum == 0.0f ? 1u : 0u) << bit % 32;
                }
                // (All of the rows and comparisons at once spill.)
#pragma unroll
                for (int w = 0; w < kWords; ++w)
                    __asm__ volatile("" : "+v"(again[w]), "+v"(zero[w]) : : "memory");
            }
        // The zeros one at a time, lane by lane.
#pragma unroll
        for (int w = 0; w < kWords; ++w)
            for (uint64_t lanes; (lanes = __builtin_amdgcn_ballot_w64(zero[w] != 0)) != 0;) {
                const int l = __builtin_ctzll(lanes);
                const uint32_t mask = __builtin_amdgcn_readlane(static_cast<int>(zero[w]), l);
                const int bit = w * 32 + __builtin_ctz(mask), r = bit % 16;
                const int row = wt / kWavesN * WM + bit / 16 / kNI * 32 + 8 * (r / 4) + 4 * (l >> 5) + r % 4;
                const int column = wt % kWavesN * WN + bit / 16 % kNI * 32 + (l & 31);
                const float2 row_line = lines[row], col_line = lines[BM + column];
                const uint64_t m = min(m0 + row, M - 1), n = min(n0 + column, N - 1);
                const bool kept = split_cancelled(
                    row_line, col_line, split_loss(row_line, col_line, count), k_begin, k_end,
                    [&](uint64_t k) { return A_T ? A[k * M + m] : A[m * K + k]; },
                    [&](uint64_t k) { return elem(B + (B_T ? n * K + k : k * N + n)); });
                if (lane == l) {
                    zero[w] &= zero[w] - 1;
                    if (kept) again[w] &= ~(1u << bit % 32);
                }
            }
        uint32_t any = 0;
#pragma unroll
        for (int w = 0; w < kWords; ++w) any |= again[w];
        return __syncthreads_or(any != 0);  // (LDS is free again)
    }

    // The same sums with the f32 MFMA.
    __device__ __forceinline__ void sum_f32(const float* __restrict__ A, const BT* __restrict__ B, uint64_t M,
                                            uint64_t K, uint64_t N, uint64_t m0, uint64_t n0, uint64_t k_begin,
                                            uint64_t k_end, bool wide_a, bool wide_b, bool short_rows, char* lds) {
        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
        const int kg = wave / kTileWaves, wt = wave % kTileWaves;
        const int wm = wt / kWavesN, wn = wt % kWavesN;
        OpA oa;
        OpB ob;
        oa.init(A, A_T ? M : K, m0, M, wide_a);
        ob.init(B, B_T ? K : N, n0, N, wide_b);
        clear();
        float* const fa = reinterpret_cast<float*>(lds);
        float* const fb = reinterpret_cast<float*>(lds + OpA::kF32Bytes);
        const int l32 = lane & 31, h = lane >> 5;
        // A stage's loads are in flight while the one before is summed, where
        // the registers allow it.
        constexpr bool kAhead = kMI * kNI < 8;
        auto load = [&](uint64_t k0) {
            if (short_rows && k0 + BK <= k_end) {
#pragma unroll
                for (int u = 0; u < OpA::kUnits; ++u) oa.load(k0, u);
#pragma unroll
                for (int u = 0; u < OpB::kUnits; ++u) ob.load(k0, u);
            } else {
#pragma unroll
                for (int u = 0; u < OpA::kUnits; ++u) oa.load_edge(k0, k_end, u);
#pragma unroll
                for (int u = 0; u < OpB::kUnits; ++u) ob.load_edge(k0, k_end, u);
            }
        };
        if (kAhead) load(k_begin);
        for (uint64_t k0 = k_begin; k0 < k_end; k0 += BK) {
            if (!kAhead) load(k0);
#pragma unroll
            for (int u = 0; u < OpA::kUnits; ++u) oa.store_f32(fa, u);
#pragma unroll
            for (int u = 0; u < OpB::kUnits; ++u) ob.store_f32(fb, u);
            lds_barrier<0>();
            if (kAhead && k0 + BK < k_end) load(k0 + BK);
#pragma unroll 1
            for (int s = 0; s < BK / KG; s += 2) {
                const int k = kg * (BK / KG) + s + h;
                float af[kMI], bf[kNI];
#pragma unroll
                for (int i = 0; i < kMI; ++i) af[i] = fa[k * (BM + 4) + wm * WM + i * 32 + l32];
#pragma unroll
                for (int j = 0; j < kNI; ++j) bf[j] = fb[k * (BN + 4) + wn * WN + j * 32 + l32];
#pragma unroll
                for (int i = 0; i < kMI; ++i)
#pragma unroll
                    for (int j = 0; j < kNI; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i], bf[j], acc[i][j], 0, 0, 0);
            }
            lds_barrier<0>();
        }
    }
};

}  // namespace mhip
