// Scaled dot-product attention with causal / sliding-window masks and grouped
// KV heads.
//
// Semantics are the reference's `attention_valued` (src/kernels.rs:6505-6884)
// defined by its three-pass kernel (src/kernels.cu:1868-1959): q [seq, H*d],
// k [kv_rows, Hkv*d], v [kv_rows, Hkv*vd]; kv_seq = key_count (<= kv_rows);
// query i sits at position qpos = (kv_seq - seq) + i and admits keys
// [lo, hi): hi = causal ? qpos + 1 : kv_seq, lo = qpos - (window - 1) when a
// window is set; weights are softmax(q.k * scale) over the admitted keys and
// the output row is their weighted mean of V rows (zeros if none). The
// reference has no batch dimension; here `batch` calls with fixed strides run
// in one launch and equal that many separate calls.
//
// Three kernels:
//  - prefill (head dims 32, 64, 80, 96, 112 and 128): flash attention on the
//    bf16 matrix cores with every operand split into three bf16 planes. A
//    workgroup takes 256 queries of one (batch, head), eight waves of 32 (four
//    for short prompts of head dims 32 and 64), and
//    walks the admitted keys in 32-key tiles. Each wave computes S^T = K . Q^T
//    (Q^T lives in registers, pre-scaled by scale * log2 e), so every lane
//    owns one query column and 16 of the tile's keys: the online-softmax
//    max/sum need one exchange with lane l ^ 32. The accumulator registers
//    are then exactly the B operand of O^T = V^T . P^T, so the output stays
//    per-lane too. V is scaled down by a power of two above the sum of the
//    weights, so the running output never overflows (the reference's 1e38
//    known answer, src/tests_conformance.rs:2215-2312). Outputs that operands
//    outside the split matter to are summed again with the f32 MFMA.
//  - decode (one query row, head dim 4, 8, 16, ..., 256): split-KV. A
//    workgroup takes one (batch, KV head, key chunk) and the query heads
//    that share that KV head (up to 8; a larger group is split into slices
//    of 8, each reading the chunk), issues every K and V load of the chunk at once
//    (non-temporal dwordx4), keeps scores and probabilities in registers, and
//    writes the chunk's normalised output, max and weight sum; a second
//    kernel merges the chunks in a fixed order (deterministic).
//  - a generic kernel (any other shape): one wave per (query, head), online
//    softmax over 64-key chunks.
#include "common.hpp"
#include "decode_merge.hpp"
#include "internal.hpp"
#include "split_tile.hpp"

#include <algorithm>
#include <cmath>

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr float kLog2e = 1.4426950408889634f;

struct AttnArgs {
    const float* q;
    const float* k;
    const float* v;
    float* out;
    uint64_t seq, kv_seq, heads, kv_heads, d, vd;
    uint64_t offset;       // kv_seq - seq
    int causal;
    int64_t window;        // -1: none
    float qscale;          // scale * log2(e), applied to q
    uint64_t q_bs, k_bs, v_bs, o_bs;  // batch strides (floats)
    const uint64_t* advance;  // captured step: replay offset added to the key count
};

// A captured step's replay offset moves the key count, and with it the
// queries' positions (src/kernels.rs:1425-1435).
__device__ __forceinline__ void apply_advance(AttnArgs& a) {
    if (a.advance) {
        const uint64_t d = *a.advance;
        a.kv_seq += d;
        a.offset += d;
    }
}

// Admitted key range of the query at position qpos (src/kernels.cu:1909-1920).
__device__ __forceinline__ void key_range(const AttnArgs& a, uint64_t qpos, uint64_t* lo,
                                          uint64_t* hi) {
    uint64_t upper = a.causal ? qpos + 1 : a.kv_seq;
    if (upper > a.kv_seq) upper = a.kv_seq;
    uint64_t lower = 0;
    if (a.window >= 0) {
        const uint64_t w = static_cast<uint64_t>(a.window);
        const uint64_t back = w > 0 ? w - 1 : 0;
        lower = qpos > back ? qpos - back : 0;
        if (lower > upper) lower = upper;
    }
    *lo = lower;
    *hi = upper;
}

// ---------------------------------------------------------------------------
// Prefill: flash attention on split bf16 planes
// ---------------------------------------------------------------------------

// A head dimension of 16 n; the value columns go in blocks of 32 (the last one
// partly past the row, its columns zero and never stored).
//
// Four waves, two workgroups per CU, for up to 128 queries of a head dimension
// of up to 64 (above, K's, V's and Q's planes fill more than half of the LDS)
// where eight would take a second round of workgroups, half of their waves
// without a query: 8 x 20 queries over 2000 keys, 8 heads of 64 on 2, 63 us with
// eight, 44 with four; 8 x 128 over 1000, 32 on 8, 119 and 87. In one round four
// take 3-7 % longer for 64-128 queries, and less for up to 32, one wave's (32 of
// 4 heads 6.3 and 6.0). Either way the same chunks and the same bits.
template <int D, int WAVES = 8>
struct PrefillCfg {
    static_assert(D % 16 == 0 && D <= 128, "whole MFMA steps, and the registers of 128");
    static_assert(WAVES == 8 || (WAVES == 4 && D <= 64), "one or two waves split a chunk of V");
    static constexpr int kWaves = WAVES;
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int kBQ = 32 * kWaves;    // queries per workgroup
    static constexpr int kBKV = 32;            // keys per tile
    static constexpr int kSteps = D / 16;      // of the scores' sum
    static constexpr int kVB = (D + 31) / 32;  // blocks of value columns
    // K planes: [plane][8 of d][key] 16-byte slots, the chunks 16 bytes apart
    // in the banks (a row's 8-byte writes go down the chunks). V planes: [plane]
    // [chunk][column], a chunk the 8 keys of one half of the wave in one step.
    static constexpr int kKChunk = kBKV * 16 + 16;
    static constexpr int kKPlane = D / 8 * kKChunk;
    static constexpr int kVChunk = kVB * 32 * 16;
    static constexpr int kVPlane = 4 * kVChunk;
    // From 112 Q's third plane does not fit the registers: it stays in LDS.
    static constexpr bool kQLds = D > 96;
    static constexpr int kQBytes = kQLds ? kWaves * kSteps * 1024 : 0;
    static constexpr int kLdsBytes = 3 * (kKPlane + kVPlane) + kQBytes;
    // The f32 sum's tiles.
    static constexpr int kLdF = D + 4;
    static_assert(2 * kBKV * kLdF * 4 <= kLdsBytes, "its f32 tiles fit");
    static constexpr int kKUnits = (kBKV * D / 4 + kThreads - 1) / kThreads;
};

// A wave's queries recomputed over their admitted keys only, on the VALU,
// after its tile loop: taken when an edge tile of the wave held a non-finite
// V value. In an edge tile a key one query of the wave masks can be one
// another admits; it enters the P . V MFMA at weight 0 for the first, and a
// non-finite V there turns that 0 into NaN, where the reference never reads
// the key (src/kernels.cu:1909-1920). Here each query visits only [lo, hi)
// (within the workgroup's key chunk), one key at a time: the score from this
// lane's half of Q^T (scaled to the log2 domain) and the other half's
// in lane l ^ 32, an online softmax, and this lane's outputs
// (register r of block vb: column vb*32 + 8*(r/4) + 4*half + r%4), so an
// admitted inf or NaN gives what the reference's sum gives and a masked one
// nothing. Slow (each query reads its keys from memory), and only for inputs
// with non-finite values next to a mask edge; the tile loop's accumulators
// are dead here, which keeps the kernel within its registers.
template <int D>
__device__ __forceinline__ void recompute_admitted(const float* qhalf, float qscale, const float* K,
                                                   uint64_t k_ld, const float* V, uint64_t v_ld,
                                                   uint64_t lo, uint64_t hi, int half,
                                                   v16f (&o)[PrefillCfg<D>::kVB], float* m_out,
                                                   float* l_out) {
    constexpr int kVB = PrefillCfg<D>::kVB;
#pragma unroll
    for (int vb = 0; vb < kVB; ++vb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[vb][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    for (uint64_t j = lo; j < hi; ++j) {
        const float* krow = K + j * k_ld + half * (D / 2);
        float part = 0.0f;
        for (int t = 0; t < D / 2; t += 4) {
            const float4 k4 = *reinterpret_cast<const float4*>(krow + t);
            const float4 q4 = *reinterpret_cast<const float4*>(qhalf + t);
            part += q4.x * qscale * k4.x + q4.y * qscale * k4.y + q4.z * qscale * k4.z + q4.w * qscale * k4.w;
        }
        const float s = part + __shfl_xor(part, 32, 64);
        const float m_new = fmaxf(m, s);
        const float m_use = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_use);
        const float w = __builtin_amdgcn_exp2f(s - m_use);
        l = l * alpha + w;
        const float* vrow = V + j * v_ld;
#pragma unroll
        for (int vb = 0; vb < kVB; ++vb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = vb * 32 + 8 * g + 4 * half;
                if (D % 32 != 0 && c >= D) continue;
                const float4 v4 = *reinterpret_cast<const float4*>(vrow + c);
                o[vb][4 * g] = o[vb][4 * g] * alpha + w * v4.x;
                o[vb][4 * g + 1] = o[vb][4 * g + 1] * alpha + w * v4.y;
                o[vb][4 * g + 2] = o[vb][4 * g + 2] * alpha + w * v4.z;
                o[vb][4 * g + 3] = o[vb][4 * g + 3] * alpha + w * v4.w;
            }
        m = m_new;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int vb = 0; vb < kVB; ++vb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[vb][r] *= inv;
    *m_out = m;
    *l_out = l;
}

// Short prefills, whose query tiles alone would leave most of the device
// idle, split the key range: chunk c of nchunks covers key tiles [c *
// chunk_tiles, (c + 1) * chunk_tiles) counted from key 0, and writes, per
// query, the chunk's normalised output, running max (log2 domain) and weight
// sum for attn_prefill_combine_kernel. The split depends on one sequence's
// shape only, so a batch still equals its separate calls.
struct PrefillSplit {
    uint32_t nchunks;      // 1: no split, the kernel writes the output itself
    uint32_t chunk_tiles;
    uint32_t qtiles, pairs, group;  // query tiles; (batch, head) pairs; query heads of a KV head
    float* part_o;         // [batch * seq][heads][nchunks][VD]
    float* part_ml;        // [batch * seq][heads][nchunks][2]
};

// What a thread works on: its workgroup's operands and key tiles, its wave's
// and its lane's key ranges. Keys count from the workgroup's first tile (32-bit:
// the caller keeps key counts below 2^31).
struct PrefillPlace {
    const float *qrow, *K, *V;
    float* out;            // the query's output row, or its chunk record's
    float* ml;             // the chunk record's max and sum (nullptr: none)
    uint64_t tile_begin;
    int i_begin, i_end;    // tiles
    bool q_live;
    int lo, hi;            // keys the lane's query admits
    int any_lo, any_hi;    // keys any query of the wave admits
    int all_lo, all_hi;    // keys every query of the wave admits
};

// Heaviest (latest) query tiles first over the whole grid: under a causal
// mask they see the most keys. Block ids are dealt round-robin to the 8
// XCDs, so consecutive ids take the same query tile of different (batch,
// head) pairs: every XCD gets an equal share of each weight class and runs
// it heaviest first (ids of one head's query tiles, dealt to XCDs by
// query tile, left XCDs with 2.4x the work of others).
//
// Block and key counts are below 2^31, so all of it is 32-bit, mostly scalar,
// and a division that a call does not need (one query tile, one sequence, no
// shared KV heads) is skipped: a prompt of 32 waits for each in turn.
template <int D, int WAVES>
__device__ __forceinline__ PrefillPlace prefill_place(const AttnArgs& a, const PrefillSplit& sp, uint32_t block,
                                                      int thread) {
    using Cfg = PrefillCfg<D, WAVES>;
    const int lane = thread & 63, wave = __builtin_amdgcn_readfirstlane(thread >> 6);
    const uint32_t heads = static_cast<uint32_t>(a.heads);
    uint32_t bh = block, chunk = 0, qt = sp.qtiles - 1;
    if (sp.nchunks > 1) {
        bh = block / sp.nchunks;
        chunk = block - bh * sp.nchunks;
    }
    if (sp.qtiles > 1) {
        const uint32_t back = bh / sp.pairs;
        bh -= back * sp.pairs;
        qt -= back;
    }
    const uint32_t b = sp.pairs == heads ? 0 : bh / heads;
    const uint32_t head = bh - b * heads;
    const uint32_t kvh = sp.group == 1 ? head : head / sp.group;
    PrefillPlace w{};
    w.K = a.k + b * a.k_bs + static_cast<uint64_t>(kvh) * D;
    w.V = a.v + b * a.v_bs + static_cast<uint64_t>(kvh) * D;
    const int seq = static_cast<int>(a.seq), q_first = static_cast<int>(qt * Cfg::kBQ);
    const int w_first = q_first + wave * 32, q = w_first + (lane & 31);
    const uint64_t at = static_cast<uint64_t>(q) * (a.heads * D) + static_cast<uint64_t>(head) * D;
    w.qrow = a.q + b * a.q_bs + at;
    w.out = a.out + b * a.o_bs + at;
    if (sp.nchunks > 1) {
        const uint64_t rec = ((b * a.seq + q) * a.heads + head) * sp.nchunks + chunk;
        w.out = sp.part_o + rec * D;
        w.ml = sp.part_ml + 2 * rec;
    }
    w.q_live = q < seq;

    const int kv_seq = static_cast<int>(a.kv_seq), offset = static_cast<int>(a.offset);
    const int back = a.window < 0 ? kv_seq : static_cast<int>(a.window < kv_seq ? a.window : kv_seq) - 1;
    auto first = [&](int i) { return max(offset + i - max(back, 0), 0); };
    auto past = [&](int i) { return a.causal ? offset + i + 1 : kv_seq; };
    const int tile_begin = first(q_first) / Cfg::kBKV * Cfg::kBKV;
    const int ntiles = (past(min(seq, q_first + Cfg::kBQ) - 1) - tile_begin + Cfg::kBKV - 1) / Cfg::kBKV;
    w.tile_begin = tile_begin;
    // All of the ntiles from tile_begin, or the part inside the key chunk.
    w.i_end = ntiles;
    if (sp.nchunks > 1) {
        const int c0 = static_cast<int>(chunk * sp.chunk_tiles) - tile_begin / Cfg::kBKV;
        w.i_begin = min(max(c0, 0), ntiles);
        w.i_end = min(max(c0 + static_cast<int>(sp.chunk_tiles), 0), ntiles);
    }
    if (w.q_live) {
        w.lo = first(q) - tile_begin;
        w.hi = past(q) - tile_begin;
    }
    if (w_first < seq) {
        const int w_last = min(seq, w_first + 32) - 1;
        w.any_lo = first(w_first) - tile_begin;
        w.all_hi = past(w_first) - tile_begin;
        w.all_lo = first(w_last) - tile_begin;
        w.any_hi = past(w_last) - tile_begin;
    }
    return w;
}

// The keys [rel_lo, rel_hi) of a tile of 32, a bit each.
__device__ __forceinline__ uint32_t tile_keys(int rel_lo, int rel_hi) {
    const int lo = min(max(rel_lo, 0), 32), hi = min(max(rel_hi, 0), 32);
    return static_cast<uint32_t>(((1ull << hi) - 1ull) & ~((1ull << lo) - 1ull));
}

// One tile's masked scores: s[r] is key k0 + 8 (r / 4) + 4 half + r % 4 of the
// lane's query, -inf where it is not admitted (rel_lo, rel_hi: its admitted
// keys from the tile's first).
__device__ __forceinline__ void mask_scores(v16f& s, int rel_lo, int rel_hi, int half) {
    const uint32_t mine = tile_keys(rel_lo, rel_hi) >> (4 * half);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int key = 8 * (r / 4) + (r % 4);
        s[r] = (mine >> key) & 1u ? s[r] : -INFINITY;
    }
}

// The online softmax over one tile: s becomes the tile's weights 2^(s - m),
// and the sums so far are to be scaled by the result. The reference m moves
// only to a maximum more than 8 above it (weights reach 2^8), so that after the
// first tiles the result is 1 for every query and nothing is scaled. Every
// lane runs it (the MFMAs need the whole wave); a query with no admitted key
// yet keeps m = -inf, l = 0.
__device__ __forceinline__ float softmax_tile(v16f& s, float& m, float& l) {
    float tile_max = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) tile_max = fmaxf(tile_max, s[r]);
    tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, 64));
    const float m_new = tile_max > m + 8.0f ? tile_max : m;
    const float alpha = m_new == m ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
    const float base = m_new == -INFINITY ? 0.0f : m_new;
    float psum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        s[r] = __builtin_amdgcn_exp2f(s[r] - base);
        psum += s[r];
    }
    l = l * alpha + (psum + __shfl_xor(psum, 32, 64));
    m = m_new;
    return alpha;
}

// The same with s the tile's probabilities over the sum so far: the output so
// far, scaled by the result, stays a convex combination of V rows.
__device__ __forceinline__ float softmax_tile_mean(v16f& s, float& m, float& l) {
    const float m_old = m, l_old = l;
    const float alpha = softmax_tile(s, m, l);
    const float inv = l > 0.0f ? __builtin_amdgcn_rcpf(l) : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= inv;
    // A tile that adds nothing for this query leaves its output as it was.
    return (l == l_old && m == m_old) || l == 0.0f ? 1.0f : (l_old * alpha) * inv;
}

// The workgroup's tiles [i_begin, i_end) with the f32 MFMA, for the waves
// (`again`) with outputs that the bf16 split does not hold: values that are not
// finite, scores' operands above 2^60, outputs that scaled values below 2^-100
// matter to. Q is read
// from memory, K and V tiles lie in LDS; a key that one query masks and another
// admits enters P . V at weight 0, so a wave that met a V value that is not
// finite in an edge tile sums its queries' admitted keys again on the VALU
// (recompute_admitted).
template <int D, int WAVES>
__device__ __forceinline__ void prefill_f32(const AttnArgs& a, const PrefillPlace& w, int thread, bool again,
                                            float* lds, v16f (&o)[PrefillCfg<D>::kVB], float& m, float& l) {
    using Cfg = PrefillCfg<D, WAVES>;
    const int lane = thread & 63, l32 = lane & 31, half = lane >> 5;
    const uint64_t kv_ld = a.kv_heads * D;
    const float* const qhalf = w.qrow + half * (D / 2);
    m = -INFINITY;
    l = 0.0f;
#pragma unroll
    for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[vb][r] = 0.0f;
    float* const sk = lds;
    float* const sv = lds + Cfg::kBKV * Cfg::kLdF;
    bool redo = false;
    for (int i = w.i_begin; i < w.i_end; ++i) {
        const uint64_t k0 = w.tile_begin + static_cast<uint64_t>(i) * Cfg::kBKV;
        for (int f = thread; f < Cfg::kBKV * D / 4; f += Cfg::kThreads) {
            const int row = f / (D / 4), c = f % (D / 4) * 4;
            const uint64_t key = min(k0 + row, a.kv_seq - 1);
            *reinterpret_cast<float4*>(sk + row * Cfg::kLdF + c) = *reinterpret_cast<const float4*>(w.K + key * kv_ld + c);
            *reinterpret_cast<float4*>(sv + row * Cfg::kLdF + c) = *reinterpret_cast<const float4*>(w.V + key * kv_ld + c);
        }
        __syncthreads();
        const int rel = i * Cfg::kBKV;
        if (again && rel < w.any_hi && rel + Cfg::kBKV > w.any_lo) {
            const bool masked = !(rel >= w.all_lo && rel + Cfg::kBKV <= w.all_hi);
            if (masked) {
                uint32_t nonfinite = 0;
                for (int f = lane; f < Cfg::kBKV * D; f += 64) {
                    const float v = sv[f / D * Cfg::kLdF + f % D];
                    nonfinite |= (((__float_as_uint(v) >> 23) & 0xFFu) + 1u) >> 8;
                }
                redo |= __builtin_amdgcn_ballot_w64(nonfinite != 0) != 0;
            }
            v16f s;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll 1
            for (int t = 0; t < D / 2; t += 4) {
                float4 v4 = make_float4(0.f, 0.f, 0.f, 0.f);
                if (w.q_live) v4 = *reinterpret_cast<const float4*>(qhalf + t);
                const float q4[4] = {v4.x * a.qscale, v4.y * a.qscale, v4.z * a.qscale, v4.w * a.qscale};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(sk[l32 * Cfg::kLdF + half * (D / 2) + t + e], q4[e], s, 0, 0, 0);
            }
            if (masked) mask_scores(s, w.lo - rel, w.hi - rel, half);
            const float keep = softmax_tile_mean(s, m, l);
#pragma unroll
            for (int vb = 0; vb < Cfg::kVB; ++vb) {
                const int c = vb * 32 + l32;
#pragma unroll
                for (int r = 0; r < 16; ++r) o[vb][r] *= keep;
#pragma unroll
                for (int t = 0; t < 16; ++t) {
                    const int key = 8 * (t / 4) + 4 * half + (t % 4);
                    const float v = D % 32 == 0 || c < D ? sv[key * Cfg::kLdF + c] : 0.0f;
                    o[vb] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, s[t], o[vb], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    if (redo) {
        const int lo = max(w.lo, w.i_begin * Cfg::kBKV), hi = min(w.hi, w.i_end * Cfg::kBKV);
        recompute_admitted<D>(w.q_live ? qhalf : w.K, a.qscale, w.K, kv_ld, w.V, kv_ld,
                              w.tile_begin + lo, w.tile_begin + max(lo, hi), half, o, &m, &l);
    }
    if (!w.ml && l == 0.0f) {  // every admitted score at -inf
#pragma unroll
        for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[vb][r] = NAN;
    }
}

// The range of operands as they are split (2 |x| as an integer, see kSplitTiny).
struct SplitRange {
    uint32_t big = 0, least = 0xFFFFFFFFu;
    __device__ __forceinline__ void top(float x0, float x1) {
        big = max(big, max(__float_as_uint(x0) << 1, __float_as_uint(x1) << 1));
    }
    __device__ __forceinline__ void bottom(float x0, float x1) { least = mhip::split_min(least, x0, x1); }
};
constexpr uint32_t kScoreTop = 2u * ((127u + 60u) << 23);   // 2^60
constexpr uint32_t kValueTop = 2u * (254u << 23);           // (a scaled one is below 2^127 or not finite)

// Whether a lane's query admits a key, among its workgroup's, with a K beyond
// the scores' range. Its two lanes look at a half of each row. (Slow, as
// recompute_admitted is: only where a tile held such a key.)
template <int D>
__device__ __forceinline__ bool admits_far_key(const PrefillPlace& w, uint64_t kv_ld, int half) {
    const int lo = max(w.lo, w.i_begin * 32), hi = min(w.hi, w.i_end * 32);
    uint32_t big = 0;
    for (int j = lo; j < hi; ++j) {
        const float* const row = w.K + (w.tile_begin + j) * kv_ld + half * (D / 2);
        for (int t = 0; t < D / 2; ++t) big = max(big, __float_as_uint(row[t]) << 1);
    }
    const uint64_t far = __builtin_amdgcn_ballot_w64(big > kScoreTop);
    return (far | far >> 32) >> (threadIdx.x & 31) & 1;
}

// Flash attention of 256 queries of one (batch, head), eight waves of 32, on
// the bf16 matrix cores: Q, K and V split exactly into three bf16 planes
// (split_tile.hpp) and the probabilities too, six plane products a product.
// Per tile of 32 keys a wave needs 96 MFMAs of 32 cycles (D 128) where the f32
// MFMA needed 128 of 64.
//
// Q^T's planes live in registers, K's and V's in LDS, split once for the eight
// waves. K is split row by row; V so that a lane's 8 keys of a step are the
// ones whose scores the same half of the wave holds, so the probabilities feed
// P . V from the registers they are computed in. Two barriers per tile: scores
// and softmax while V is split into its buffer, then P . V while the next
// tile's K is; both are loaded a tile ahead.
//
// Against the f32 MFMA kernel (four waves, 128 queries), causal, us: 4
// sequences of 2048, 32 heads of 128, 1127 before and 727 now; one of 509 60
// and 42; 1024 keys, 16 heads of 64 53 and 38. (Batches of few queries of 128
// wait for a second round of workgroups: 8 of 20 over 2000, 8 heads on 2, 72 and
// 89, 6 of 7 over 420 31 and 40.) Head dims 32, 80,
// 96 and 112 ran on the generic kernel: 1024 keys, 32 heads of 80 5435 and 79.
// Bound by the chain within a wave (scores, softmax, the split of the
// probabilities, P . V) with two waves per SIMD to hide it: the registers of
// Q's planes and the output allow no third.
template <int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_prefill_kernel(AttnArgs a, PrefillSplit sp) {
    apply_advance(a);
    using Cfg = PrefillCfg<D, WAVES>;
    using mhip::bf16x8;
    using mhip::u32x2;
    using mhip::u32x4;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    char* const lk = lds;
    char* const lv = lds + 3 * Cfg::kKPlane;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    char* const lq = lv + 3 * Cfg::kVPlane + wave * Cfg::kSteps * 1024 + lane * 16;
    const int l32 = lane & 31, half = lane >> 5;

    const PrefillPlace w = prefill_place<D, WAVES>(a, sp, blockIdx.x, threadIdx.x);
    const float *const K = w.K, *const V = w.V, *const qrow = w.qrow;
    const uint64_t kv_ld = a.kv_heads * D, tile_begin = w.tile_begin;
    const int i_begin = w.i_begin, i_end = w.i_end;
    float m = -INFINITY, l = 0.0f;
    v16f o[Cfg::kVB];
#pragma unroll
    for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[vb][r] = 0.0f;
    // A tile's loads: K, 4 of d of one key per unit; V, 8 keys of one column
    // (the chunk of a pair of waves). Buffer loads whose range ends with the
    // last key: keys past it read as zeros, which the mask takes out. The key
    // goes into the vector offset: the range check takes a scalar offset off
    // the range instead, which wraps where that key lies past the end.
    u32x4 kr[Cfg::kKUnits];
    uint32_t vr[8];
    const int v_chunk = WAVES == 8 ? wave >> 1 : wave;  // step v_chunk / 2, half v_chunk % 2
    const int v_col = WAVES == 8 ? (wave & 1) * 64 + lane : lane;
    const bool v_on = v_col < Cfg::kVB * 32;
    const bool v_in = v_col < D;
    const uint32_t ld_bytes = static_cast<uint32_t>(kv_ld * sizeof(float));  // the launch checks 32 rows < 2^31
    uint32_t k_off[Cfg::kKUnits];
#pragma unroll
    for (int u = 0; u < Cfg::kKUnits; ++u) {
        const int f = min(static_cast<int>(threadIdx.x) + u * Cfg::kThreads, Cfg::kBKV * D / 4 - 1);
        k_off[u] = f / (D / 4) * ld_bytes + f % (D / 4) * 16;
    }
    const uint32_t v_off = min(v_col, D - 1) * 4;
    auto tile_rsrc = [&](const float* base, int i) {
        const uint64_t k0 = tile_begin + static_cast<uint64_t>(i) * Cfg::kBKV;
        const uint64_t bytes = ((a.kv_seq - 1 - k0) * kv_ld + D) * sizeof(float);
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(base + k0 * kv_ld), 0,
            static_cast<int>(static_cast<uint32_t>(bytes < 0xFFFFFFFFu ? bytes : 0xFFFFFFFFu)), 0x00020000);
    };
    auto load_k = [&](int i) {
        const __amdgpu_buffer_rsrc_t rsrc = tile_rsrc(K, i);
#pragma unroll
        for (int u = 0; u < Cfg::kKUnits; ++u) kr[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, k_off[u], 0, 0);
    };
    auto load_v = [&](int i) {
        const __amdgpu_buffer_rsrc_t rsrc = tile_rsrc(V, i);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            vr[e] = __builtin_amdgcn_raw_buffer_load_b32(
                rsrc, v_off + (16 * (v_chunk >> 1) + 4 * (v_chunk & 1) + (e / 4) * 8 + e % 4) * ld_bytes, 0, 0);
    };
    if (i_end > i_begin) {
        load_k(i_begin);
        load_v(i_begin);
    }
    SplitRange query;
    // What a tile (by parity) holds outside the split; the value columns with a
    // nonzero below 2^-100 (scaled).
    constexpr uint32_t kFarKey = 1, kBadValue = 2, kTinyValue = 4;
    __shared__ uint32_t outside[2];
    __shared__ uint8_t tiny_values[Cfg::kVB * 32];
    if (threadIdx.x < 2) outside[threadIdx.x] = 0;
    if (threadIdx.x < Cfg::kVB * 32) tiny_values[threadIdx.x] = 0;

    // Q^T's planes, pre-scaled: step t, k = 16 t + 8 half + i of the query.
    constexpr int kQRegs = Cfg::kQLds ? 2 : 3;
    u32x4 qp[Cfg::kSteps][kQRegs];
#pragma unroll
    for (int t = 0; t < Cfg::kSteps; ++t) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            float4 v4 = make_float4(0.f, 0.f, 0.f, 0.f);
            if (w.q_live) v4 = *reinterpret_cast<const float4*>(qrow + 16 * t + 8 * half + e);
            x[e] = v4.x * a.qscale; x[e + 1] = v4.y * a.qscale; x[e + 2] = v4.z * a.qscale; x[e + 3] = v4.w * a.qscale;
        }
        u32x4 third;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t p[3];
            mhip::split_pair(x[2 * e], x[2 * e + 1], p);
            query.top(x[2 * e], x[2 * e + 1]);
            qp[t][0][e] = p[0];
            qp[t][1][e] = p[1];
            third[e] = p[2];
        }
        if constexpr (Cfg::kQLds) *reinterpret_cast<u32x4*>(lq + t * 1024) = third;
        else qp[t][kQRegs - 1] = third;
    }
    // The wave's queries outside the split (decided here, or their values would
    // be kept until the end), and what it met in its tiles.
    const uint64_t far_q = __builtin_amdgcn_ballot_w64(query.big > kScoreTop);
    uint32_t met = 0;

    auto store_k = [&](int i) {
        SplitRange score;
#pragma unroll
        for (int u = 0; u < Cfg::kKUnits; ++u) {
            const int f = threadIdx.x + u * Cfg::kThreads;
            if (Cfg::kKUnits * Cfg::kThreads != Cfg::kBKV * D / 4 && f >= Cfg::kBKV * D / 4) continue;
            const int row = f / (D / 4), c = f % (D / 4);
            uint32_t p0[3], p1[3];
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = __uint_as_float(kr[u][e]);
            mhip::split_pair(x[0], x[1], p0);
            mhip::split_pair(x[2], x[3], p1);
            score.top(x[0], x[1]);
            score.top(x[2], x[3]);
            char* at = lk + c / 2 * Cfg::kKChunk + row * 16 + c % 2 * 8;
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(at + p * Cfg::kKPlane) = u32x2{p0[p], p1[p]};
        }
        if (score.big > kScoreTop) atomicOr(&outside[i & 1], kFarKey);
    };
    // V is scaled by a power of two that keeps any sum of 2^8 kv_seq weighted
    // rows finite, and the output by its inverse.
    const int v_shift = 9 + 64 - __builtin_clzll(a.kv_seq);
    const float v_scale = v_in ? __uint_as_float(static_cast<uint32_t>(127 - v_shift) << 23) : 0.0f;
    const uint32_t v_tiny = mhip::kSplitTiny + (static_cast<uint32_t>(v_shift) << 24);  // unscaled
    auto store_v = [&](int i) {
        if (!v_on) return;
        SplitRange value;
        u32x4 p[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float y0 = __uint_as_float(vr[2 * e]), y1 = __uint_as_float(vr[2 * e + 1]);
            const float x0 = y0 * v_scale, x1 = y1 * v_scale;
            uint32_t q[3];
            mhip::split_pair(x0, x1, q);
            value.top(x0, x1);
            value.bottom(y0, y1);
            p[0][e] = q[0];
            p[1][e] = q[1];
            p[2][e] = q[2];
        }
        char* at = lv + v_chunk * Cfg::kVChunk + v_col * 16;
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(at + q * Cfg::kVPlane) = p[q];
        if (value.big > kValueTop || value.least < v_tiny) {
            atomicOr(&outside[i & 1], (value.big > kValueTop ? kBadValue : 0) | (value.least < v_tiny ? kTinyValue : 0));
            if (value.least < v_tiny) tiny_values[v_col] = 1;
        }
    };
    auto mfma = [](bf16x8 x, bf16x8 y, v16f c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0); };
    auto as_bf16 = [](u32x4 v) { return __builtin_bit_cast(bf16x8, v); };

    __syncthreads();
    if (i_end > i_begin) {
        store_k(i_begin);
        if (i_begin + 1 < i_end) load_k(i_begin + 1);
        mhip::lds_barrier<0>();
        for (int i = i_begin; i < i_end; ++i) {
            const int rel = i * Cfg::kBKV;  // the tile's first key, from tile_begin
            const bool mine = rel < w.any_hi && rel + Cfg::kBKV > w.any_lo;
            auto next_v = [&]() {
                store_v(i);
                if (i + 1 < i_end) load_v(i + 1);
            };
            auto next_k = [&]() {
                if (i + 1 < i_end) store_k(i + 1);
                if (i + 2 < i_end) load_k(i + 2);
            };
            // (Read last in the tile before, set next after this tile's barrier.)
            if (threadIdx.x == 0) outside[(i + 1) & 1] = 0;
            v16f s;
            u32x4 pp[2][3];  // the probabilities' planes: step, plane
            float alpha = 1.0f;
            if (mine) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
                for (int t = 0; t < Cfg::kSteps; ++t) {
                    if (t == Cfg::kSteps / 2) next_v();
                    bf16x8 kf[3];
#pragma unroll
                    for (int p = 0; p < 3; ++p)
                        kf[p] = *reinterpret_cast<const bf16x8*>(lk + p * Cfg::kKPlane + (2 * t + half) * Cfg::kKChunk + l32 * 16);
                    u32x4 q3;
                    if constexpr (Cfg::kQLds) q3 = *reinterpret_cast<const u32x4*>(lq + t * 1024);
                    else q3 = qp[t][kQRegs - 1];
                    s = mfma(kf[0], as_bf16(q3), s);
                    s = mfma(kf[2], as_bf16(qp[t][0]), s);
                    s = mfma(kf[1], as_bf16(qp[t][1]), s);
                    s = mfma(kf[0], as_bf16(qp[t][1]), s);
                    s = mfma(kf[1], as_bf16(qp[t][0]), s);
                    s = mfma(kf[0], as_bf16(qp[t][0]), s);
                }
                // A tile every query of the wave admits whole needs no mask.
                if (!(rel >= w.all_lo && rel + Cfg::kBKV <= w.all_hi)) mask_scores(s, w.lo - rel, w.hi - rel, half);
                alpha = softmax_tile(s, m, l);
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        uint32_t p[3];
                        mhip::split_pair(s[8 * t + 2 * e], s[8 * t + 2 * e + 1], p);
                        pp[t][0][e] = p[0];
                        pp[t][1][e] = p[1];
                        pp[t][2][e] = p[2];
                    }
            } else {
                next_v();
            }
            mhip::lds_barrier<0>();
            if (mine) {
                met |= outside[i & 1];
                if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
                    for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[vb][r] *= alpha;
                }
#pragma unroll
                for (int vb = 0; vb < Cfg::kVB; ++vb) {
                    if (vb == Cfg::kVB / 2) next_k();
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        bf16x8 vf[3];
#pragma unroll
                        for (int p = 0; p < 3; ++p)
                            vf[p] = *reinterpret_cast<const bf16x8*>(lv + p * Cfg::kVPlane + (2 * t + half) * Cfg::kVChunk +
                                                                     (vb * 32 + l32) * 16);
                        o[vb] = mfma(vf[0], as_bf16(pp[t][2]), o[vb]);
                        o[vb] = mfma(vf[2], as_bf16(pp[t][0]), o[vb]);
                        o[vb] = mfma(vf[1], as_bf16(pp[t][1]), o[vb]);
                        o[vb] = mfma(vf[0], as_bf16(pp[t][1]), o[vb]);
                        o[vb] = mfma(vf[1], as_bf16(pp[t][0]), o[vb]);
                        o[vb] = mfma(vf[0], as_bf16(pp[t][0]), o[vb]);
                    }
                }
            } else {
                next_k();
            }
            mhip::lds_barrier<0>();
        }
    }
    // (No weight: a record's zeros, or, every admitted score at -inf, NaN.)
    const float inv = l > 0.0f ? 1.0f / l * __uint_as_float(static_cast<uint32_t>(127 + v_shift) << 23)
                               : sp.nchunks > 1 ? 0.0f : NAN;
#pragma unroll
    for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[vb][r] *= inv;
    // The thread's place once more from the kernel's arguments where the
    // registers are short, so that none of it is kept through the loop.
    uint32_t block = blockIdx.x;
    int thread = threadIdx.x;
    if constexpr (D > 64) __asm__ volatile("" : "+s"(block), "+v"(thread));
    const PrefillPlace end = prefill_place<D, WAVES>(a, sp, block, thread);
    // Register r of block vb holds O[q][vb*32 + 8*(r/4) + 4*half + r%4].
    const int first = 4 * (thread >> 5 & 1);
    auto store = [&]() {
        if (!end.q_live) return;
        if (end.ml && first == 0) *reinterpret_cast<float2*>(end.ml) = make_float2(m, l);
#pragma unroll
        for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = vb * 32 + 8 * g + first;
                if (D % 32 != 0 && c >= D) continue;
                *reinterpret_cast<float4*>(end.out + c) =
                    make_float4(o[vb][4 * g], o[vb][4 * g + 1], o[vb][4 * g + 2], o[vb][4 * g + 3]);
            }
    };
    // What is to be summed again: a query whose own row or keys lie outside the
    // split or whose wave met a value that is not finite, and an output so small
    // that its column's tiny values (planes off by less than 2^-124 of the
    // scaled mean) can have cost it a rounding.
    uint32_t redo[2] = {0, 0};
    bool again = false;
    met = __builtin_amdgcn_readfirstlane(met);
    bool some = met != 0 || far_q != 0;
    if (some) {
        again = (far_q | far_q >> 32) >> l32 & 1 || (met & kBadValue);
        if (met & kFarKey) again |= admits_far_key<D>(end, kv_ld, half);
        if (met & kTinyValue) {
            const float least = __uint_as_float(static_cast<uint32_t>(127 + v_shift - 98) << 23);
#pragma unroll
            for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int c = vb * 32 + 8 * (r / 4) + first + r % 4;
                    if (tiny_values[c] && fabsf(o[vb][r]) < least) redo[vb / 2] |= 1u << (vb % 2 * 16 + r);
                }
        }
        if (again) redo[0] = redo[1] = 0xFFFFFFFFu;
        if (!end.q_live) redo[0] = redo[1] = 0;
        some = __builtin_amdgcn_ballot_w64((redo[0] | redo[1]) != 0) != 0;
    }
    auto store_some = [&](uint32_t flip) {
        if (!end.q_live) return;
        if (end.ml && first == 0 && again == (flip == 0)) *reinterpret_cast<float2*>(end.ml) = make_float2(m, l);
#pragma unroll
        for (int vb = 0; vb < Cfg::kVB; ++vb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int c = vb * 32 + 8 * (r / 4) + first + r % 4;
                if (D % 32 != 0 && c >= D) continue;
                if ((redo[vb / 2] >> (vb % 2 * 16 + r) & 1u) != flip) end.out[c] = o[vb][r];
            }
    };
    if (!some) store();
    else store_some(1);
    if (__syncthreads_or(some)) {
        prefill_f32<D, WAVES>(a, end, thread, some, reinterpret_cast<float*>(lds), o, m, l);
        if (some) store_some(0);
    }
}

// Chunk records of split attention live in the context's workspace.
mhip_status attention_workspace(mhip_ctx* ctx, size_t bytes, float** out) {
    void* p = nullptr;
    mhip_status st = mhip::workspace(ctx, bytes, &p);
    *out = static_cast<float*>(p);
    return st;
}

// Merges a split prefill's chunk records per (query row, head): out = sum_c
// w_c o_c with w_c = l_c 2^(m_c - M) / sum_c' l_c' 2^(m_c' - M), in chunk
// order; a chunk without weight (no admitted key, or every score at -inf) has
// l_c = 0. VD / 4 threads per (row, head), one float4 of the output each.
template <int VD>
__global__ __launch_bounds__(256) void attn_prefill_combine_kernel(AttnArgs a, uint64_t rows,
                                                                   PrefillSplit sp) {
    constexpr int kLanes = VD / 4;
    constexpr int kItems = 256 / kLanes;
    const uint64_t item = static_cast<uint64_t>(blockIdx.x) * kItems + threadIdx.x / kLanes;
    const int t = threadIdx.x % kLanes;
    if (item >= rows * a.heads || threadIdx.x >= kItems * kLanes) return;
    const uint64_t row = item / a.heads, head = item % a.heads;
    const uint64_t b = row / a.seq, q = row % a.seq;
    const float* ml = sp.part_ml + 2 * item * sp.nchunks;
    const float* po = sp.part_o + item * sp.nchunks * VD + 4 * t;
    float M = -INFINITY;
    for (uint32_t c = 0; c < sp.nchunks; ++c) M = fmaxf(M, ml[2 * c]);
    float total = 0.0f;
    for (uint32_t c = 0; c < sp.nchunks; ++c)
        if (ml[2 * c + 1] != 0.0f) total += ml[2 * c + 1] * exp2f(ml[2 * c] - M);
    // Every query admits a key: no weight at all is every score at -inf, whose
    // weights are NaN as those of a NaN or +inf score are.
    float4 acc = make_float4(NAN, NAN, NAN, NAN);
    if (total > 0.0f) {
        acc = make_float4(0.f, 0.f, 0.f, 0.f);
        const float inv_total = 1.0f / total;
        for (uint32_t c = 0; c < sp.nchunks; ++c) {
            const float l = ml[2 * c + 1];
            if (l == 0.0f) continue;
            const float w = l * exp2f(ml[2 * c] - M) * inv_total;
            const float4 o = *reinterpret_cast<const float4*>(po + c * VD);
            acc.x += w * o.x; acc.y += w * o.y; acc.z += w * o.z; acc.w += w * o.w;
        }
    }
    *reinterpret_cast<float4*>(a.out + b * a.o_bs + q * (a.heads * VD) + head * VD + 4 * t) = acc;
}

// Key chunks for a prefill whose query tiles (per sequence) do not give every
// CU its workgroup: enough chunks of at least 4 key tiles to do so, at most 16.
void prefill_split(const mhip_ctx* ctx, const AttnArgs& a, bool replayable, uint64_t qtiles, uint64_t kbkv,
                   uint32_t* nchunks, uint32_t* chunk_tiles) {
    *nchunks = 1;
    *chunk_tiles = 0;
    // A replayed key count may pass the captured one: chunks sized here from
    // the captured count would leave the later keys to no workgroup. The call
    // outside a capture sums the same way, so that a replay gives its bits.
    if (replayable) return;
    const uint64_t slots = ctx->compute_units ? ctx->compute_units : 256;
    const uint64_t per_sequence = a.heads * qtiles;
    const uint64_t kv_tiles = (a.kv_seq + kbkv - 1) / kbkv;
    if (per_sequence >= slots || kv_tiles < 8) return;
    uint64_t n = std::min<uint64_t>((slots + per_sequence - 1) / per_sequence, kv_tiles / 4);
    n = std::min<uint64_t>(n, 16);
    if (n < 2) return;
    const uint64_t per = (kv_tiles + n - 1) / n;
    *chunk_tiles = static_cast<uint32_t>(per);
    *nchunks = static_cast<uint32_t>((kv_tiles + per - 1) / per);
}

template <int D, int WAVES = 8>
mhip_status launch_prefill(mhip_ctx* ctx, const AttnArgs& a, uint64_t batch, bool replayable) {
    using Cfg = PrefillCfg<D, WAVES>;
    const uint64_t qtiles = (a.seq + Cfg::kBQ - 1) / Cfg::kBQ;
    PrefillSplit sp{};
    prefill_split(ctx, a, replayable, qtiles, Cfg::kBKV, &sp.nchunks, &sp.chunk_tiles);
    // (The other head dimensions ran on the generic kernel, without chunks.)
    const mhip::CaptureGrowth growth(ctx, D != 64 && D != 128);
    const uint64_t blocks = batch * a.heads * qtiles * sp.nchunks;
    if constexpr (D <= 64 && WAVES == 8)
        if (a.seq <= 32 || (a.seq <= PrefillCfg<D, 4>::kBQ && blocks > (ctx->compute_units ? ctx->compute_units : 256)))
            return launch_prefill<D, 4>(ctx, a, batch, replayable);
    if (blocks >= (1ULL << 31)) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "attention: too many query tiles");
    sp.qtiles = static_cast<uint32_t>(qtiles);
    sp.pairs = static_cast<uint32_t>(batch * a.heads);
    sp.group = static_cast<uint32_t>(a.heads / a.kv_heads);
    const uint64_t rows = batch * a.seq;
    if (sp.nchunks > 1) {
        const uint64_t records = rows * a.heads * sp.nchunks;
        float* part = nullptr;
        mhip_status st = attention_workspace(ctx, records * (D + 2) * sizeof(float), &part);
        if (st != MHIP_OK) return st;
        sp.part_o = part;
        sp.part_ml = part + records * D;
    }
    const size_t lds = Cfg::kLdsBytes;
    static bool configured = false;
    if (!configured) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_prefill_kernel<D, WAVES>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        configured = true;
    }
    mhip::launch(ctx, (attn_prefill_kernel<D, WAVES>), dim3(static_cast<unsigned>(blocks)), dim3(Cfg::kThreads),
                 lds, a, sp);
    mhip_status st = mhip::check_launch("attention (MFMA prefill)");
    if (st != MHIP_OK || sp.nchunks == 1) return st;
    const uint64_t items = rows * a.heads;
    constexpr uint64_t kItems = 256 / (D / 4);
    mhip::launch(ctx, (attn_prefill_combine_kernel<D>),
                 dim3(static_cast<unsigned>((items + kItems - 1) / kItems)), dim3(256), 0, a, rows,
                 sp);
    return mhip::check_launch("attention (prefill chunk merge)");
}

// ---------------------------------------------------------------------------
// Decode: split-KV over key chunks, all query heads of a KV head together
// ---------------------------------------------------------------------------

constexpr int kMaxGroup = 8;  // query heads per workgroup; larger groups take several

// Keys per chunk for head dim 4*D4: kDecodeSteps(D4) steps of 256/D4 keys
// (D4 lanes hold one key row, 64/D4 keys per wave, four waves). At D >= 16
// a chunk is 32 KB of K plus 32 KB of V.
// Calls whose default chunks give every CU 16 workgroups or more (many
// batch rows or heads, long caches) take twice the steps: half the
// workgroups and records (B8 KV 4096, 32 heads on 32 KV heads: 175 -> 171 us;
// on 8 57 -> 54 with twice the steps and 59 with more waves resident instead).
__host__ __device__ constexpr int decode_steps(int d4) { return d4 >= 4 ? 8 : 2 * d4; }
__host__ __device__ constexpr int decode_chunk(int d4, int steps) { return steps * 256 / d4; }
__host__ __device__ constexpr int decode_chunk(int d4) { return decode_chunk(d4, decode_steps(d4)); }

constexpr int log2_of(int n) { return n <= 1 ? 0 : 1 + log2_of(n / 2); }

// A lane exchange of the VALU: quad_perm xor 1 and 2, row_half_mirror (l ^ 7),
// row_mirror (l ^ 15), row_ror 4 and 8.
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}

// Lanes whose bit MASK (16 or 32) is clear get a of both sides, the others b.
template <int MASK>
__device__ __forceinline__ float swap_sum(float a, float b) {
    const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
    const auto r = MASK == 32 ? __builtin_amdgcn_permlane32_swap(ua, ub, false, false)
                              : __builtin_amdgcn_permlane16_swap(ua, ub, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// a summed over the lane and its partner in bit MASK where that bit is clear, b
// where it is set. (The partner in bits 4 and 8 is the mirrored lane, which
// differs in the lower bits too: they are summed over after it.)
template <int MASK>
__device__ __forceinline__ float deal(float a, float b, int lane) {
    if constexpr (MASK >= 16) {
        return swap_sum<MASK>(a, b);
    } else {
        constexpr int kCtrl = MASK == 8 ? 0x140 : MASK == 4 ? 0x141 : MASK == 2 ? 0x4E : 0xB1;
        const bool upper = lane & MASK;
        return (upper ? b : a) + dpp<kCtrl>(upper ? a : b);
    }
}

// Sums x[0, NV) over the 2 MASK lanes of a group and deals the sums out: each
// step halves the values a lane holds, its bit MASK choosing the half, until
// one is left, which the further steps sum in every lane. NV values take NV - 1
// exchanges and the remaining steps, where a butterfly a value takes NV log2.
template <int MASK, int NV, int N>
__device__ __forceinline__ void sum_dealt(float (&x)[N], int lane) {
    if constexpr (MASK >= 1) {
#pragma unroll
        for (int i = 0; i < (NV + 1) / 2; ++i) x[i] = deal<MASK>(x[i], NV > 1 ? x[i + NV / 2] : x[i], lane);
        sum_dealt<MASK / 2, (NV + 1) / 2>(x, lane);
    }
}

// The power of two p with l p in [0.5, 1), for a normal l > 0.
__device__ __forceinline__ float half_over(float l) { return __uint_as_float((253u - (__float_as_uint(l) >> 23)) << 23); }

// Its inverse.
__device__ __forceinline__ float twice_under(float l) { return __uint_as_float(((__float_as_uint(l) >> 23) + 1u) << 23); }

// One workgroup per (batch, KV head, key chunk). Every thread issues all of
// its K and V loads before any arithmetic (2 * kSteps dwordx4 in flight).
// A wave's scores are summed and dealt out over the lanes (sum_dealt), so that
// each of them is exponentiated once, and its probabilities return to the
// lanes of their keys through LDS. A wave keeps its own maximum and weight
// sum; the four meet at the end. Writes, per query head of the group, the
// chunk's output normalised by its own weight sum, plus the chunk max (log2
// domain) and weight sum.
//
// With five exchanges a head and key and every lane exponentiating every
// score, grouped heads were bound by those, not by memory. One query over 4096
// keys, 8 sequences, head dimension 128, us before and now: 32 heads on 8 KV
// heads 68 and 54, on 4 68 and 40, on 32 175 and 172 (6.25 TB/s); 8192 keys of
// one sequence, 32 on 8, 28 and 21; 16 heads of 64 on 2 25 and 17.
template <int D4, int GT, int STEPS>
__global__ __launch_bounds__(256) void attn_decode_partial_kernel(
    AttnArgs a, uint64_t key_base, uint64_t chunks, float* __restrict__ part_o,
    float* __restrict__ part_ml) {
    constexpr int kLPK = D4;              // lanes per key
    constexpr int kKPS = 64 / kLPK;       // keys per wave step
    constexpr int kKPW = 4 * kKPS;        // keys per workgroup step
    constexpr int kSteps = STEPS;
    constexpr int D = 4 * D4;
    // A wave's scores: N per lane, of which it ends with kLeft: those of kHeads
    // heads and kKeys steps from value number `first`; 2^kCopies lanes hold the
    // same ones.
    constexpr int N = GT * kSteps;
    constexpr int kDealt = log2_of(N < kLPK ? N : kLPK);
    constexpr int kLeft = N >> kDealt, kCopies = log2_of(kLPK) - kDealt;
    constexpr int kKeys = kLeft < kSteps ? kLeft : kSteps, kHeads = kLeft / kKeys;
    constexpr int kRow = N + 4;  // (rows of a wave's subgroups in different banks)
    __shared__ float4 sq[GT][D4];
    __shared__ float4 red[4][GT][D4];
    __shared__ float4 sp[4][kKPS][kRow / 4];
    __shared__ float wm[4][GT], wl[4][GT];

    // (batch, KV head) varies fastest: workgroups in flight together read
    // whole K/V rows (all heads of the same keys) rather than one head's
    // 4*D-byte slice of many rows. A group of more than GT query heads is
    // taken GT heads at a time (head slice hs), each slice reading the chunk.
    const int group_all = static_cast<int>(a.heads / a.kv_heads);
    const int slices = (group_all + GT - 1) / GT;
    const uint64_t units = gridDim.x / chunks;
    const uint64_t c_idx = blockIdx.x / units;
    const uint64_t unit = blockIdx.x % units;
    const uint64_t pairs = units / static_cast<uint64_t>(slices);
    const int hs = static_cast<int>(unit / pairs);
    const uint64_t bkv = unit % pairs;
    const uint64_t kvh = bkv % a.kv_heads, b = bkv / a.kv_heads;
    const int group = min(GT, group_all - hs * GT);
    const uint64_t head0 = kvh * static_cast<uint64_t>(group_all) + static_cast<uint64_t>(hs) * GT;
    // The chunk's keys: [key_base + c * chunk, + chunk) inside the admitted
    // range of the query (at position offset; a replay may move it).
    apply_advance(a);
    uint64_t key_lo, key_hi;
    key_range(a, a.offset, &key_lo, &key_hi);
    const uint64_t c_base = key_base + c_idx * static_cast<uint64_t>(kSteps * kKPW);
    const uint64_t c_lo = max(c_base, key_lo);
    const uint64_t c_hi = min(c_base + static_cast<uint64_t>(kSteps * kKPW), key_hi);
    const int n = c_lo < c_hi ? static_cast<int>(c_hi - c_lo) : 0;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane / kLPK, sl = lane % kLPK;
    const uint64_t k_ld = a.kv_heads * D;
    const float* K = a.k + b * a.k_bs + kvh * D + 4 * sl;
    const float* V = a.v + b * a.v_bs + kvh * D + 4 * sl;

    float4 kr[kSteps], vr[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
        const int j = u * kKPW + wave * kKPS + sub;
        kr[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        vr[u] = kr[u];
        if (j < n) {
            kr[u] = mhip::load_nt(reinterpret_cast<const float4*>(K + (c_lo + j) * k_ld));
            vr[u] = mhip::load_nt(reinterpret_cast<const float4*>(V + (c_lo + j) * k_ld));
        }
    }
    const float* Qb = a.q + b * a.q_bs + head0 * D;
    for (int i = threadIdx.x; i < GT * D4; i += 256) {
        float4 q4 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < group * D4) q4 = *reinterpret_cast<const float4*>(Qb + 4 * static_cast<uint64_t>(i));
        q4.x *= a.qscale; q4.y *= a.qscale; q4.z *= a.qscale; q4.w *= a.qscale;
        sq[i / D4][i % D4] = q4;
    }
    __syncthreads();

    // Scores (log2 domain), the first step of the dealing as they come.
    float s[N];
    auto dot = [&](const float4& k4, const float4& q4) {
        return k4.x * q4.x + k4.y * q4.y + k4.z * q4.z + k4.w * q4.w;
    };
    if constexpr (kLPK == 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) s[i] = dot(kr[i % kSteps], sq[i / kSteps][0]);
    } else {
#pragma unroll
        for (int g = 0; g < (GT + 1) / 2; ++g) {
            const float4 q4 = sq[g][sl], other = sq[GT > 1 ? g + GT / 2 : g][sl];
#pragma unroll
            for (int u = 0; u < (GT > 1 ? kSteps : kSteps / 2); ++u)
                s[g * kSteps + u] = deal<kLPK / 2>(dot(kr[u], q4), dot(kr[GT > 1 ? u : u + kSteps / 2], other), lane);
        }
        sum_dealt<kLPK / 4, N / 2>(s, lane);
    }
    const int first = (sl >> kCopies) * kLeft;

    // The wave's maximum, probabilities and weight sum per head (heads past the
    // group among them, unused).
#pragma unroll
    for (int g = 0; g < kHeads; ++g) {
        float* const x = s + g * kKeys;
        float mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < kKeys; ++u) {
            const int j = (first % kSteps + u) * kKPW + wave * kKPS + sub;
            x[u] = j < n ? x[u] : -INFINITY;
            mx = fmaxf(mx, x[u]);
        }
        // Over the lanes that hold the head's other steps, then other keys.
#pragma unroll
        for (int off = 1 << kCopies; off < kSteps / kKeys << kCopies; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
#pragma unroll
        for (int off = kLPK; off < 64; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        float l = 0.0f;
#pragma unroll
        for (int u = 0; u < kKeys; ++u) {
            x[u] = x[u] == -INFINITY ? 0.0f : exp2f(x[u] - mx);
            l += x[u];
        }
#pragma unroll
        for (int off = 1 << kCopies; off < kSteps / kKeys << kCopies; off <<= 1) l += __shfl_xor(l, off, 64);
#pragma unroll
        for (int off = kLPK; off < 64; off <<= 1) l += __shfl_xor(l, off, 64);
        const float scale = l > 0.0f ? half_over(l) : 0.0f;
#pragma unroll
        for (int u = 0; u < kKeys; ++u) x[u] *= scale;
        if (sub == 0 && (sl & ((1 << kCopies) - 1)) == 0 && first % kSteps == 0) {
            wm[wave][first / kSteps + g] = mx;
            wl[wave][first / kSteps + g] = l;
        }
    }
    if constexpr (kLPK > 1) {
        float* const row = reinterpret_cast<float*>(sp[wave][sub]);
        if ((sl & ((1 << kCopies) - 1)) == 0)
#pragma unroll
            for (int i = 0; i < kLeft; ++i) row[first + i] = s[i];
        // The wave's own rows: its LDS operations are in order.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // V rows weighted by the probabilities over a power of two above their sum:
    // no partial sum overflows, and none of the weights is rounded again. The keys' lanes sum as
    // above, and lane group `sub` of the first kParts stores its part of a float4.
    constexpr int kParts = kKPS < 4 ? kKPS : 4;
#pragma unroll
    for (int g = 0; g < GT; ++g) {
        if (g >= group) break;
        float p[kSteps];
        if constexpr (kLPK > 1) {
#pragma unroll
            for (int u = 0; u < kSteps; u += 4) {
                const float4 p4 = sp[wave][sub][(g * kSteps + u) / 4];
                p[u] = p4.x; p[u + 1] = p4.y; p[u + 2] = p4.z; p[u + 3] = p4.w;
            }
        } else {
#pragma unroll
            for (int u = 0; u < kSteps; ++u) p[u] = s[g * kSteps + u];
        }
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            acc[0] += p[u] * vr[u].x;
            acc[1] += p[u] * vr[u].y;
            acc[2] += p[u] * vr[u].z;
            acc[3] += p[u] * vr[u].w;
        }
        // Bit 32 of the lane chooses components 2 and 3, bit 16 the odd one.
        if constexpr (kLPK <= 32) {
            acc[0] = swap_sum<32>(acc[0], acc[2]);
            acc[1] = swap_sum<32>(acc[1], acc[3]);
        }
        if constexpr (kLPK <= 16) acc[0] = swap_sum<16>(acc[0], acc[1]);
        if constexpr (kLPK <= 8) acc[0] += dpp<0x128>(acc[0]);
        if constexpr (kLPK <= 4) acc[0] += dpp<0x124>(acc[0]);
        if constexpr (kLPK <= 2) acc[0] += dpp<0x4E>(acc[0]);
        if constexpr (kLPK <= 1) acc[0] += dpp<0xB1>(acc[0]);
        float* const out = reinterpret_cast<float*>(&red[wave][g][sl]);
        if constexpr (kParts == 1) {
            red[wave][g][sl] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        } else if constexpr (kParts == 2) {
            *reinterpret_cast<float2*>(out + 2 * sub) = make_float2(acc[0], acc[1]);
        } else {
            if (lane % 16 < kLPK) out[lane / 32 * 2 + lane / 16 % 2] = acc[0];
        }
    }
    __syncthreads();

    // The four waves by their weights; a NaN among the scores is one in l.
    const uint64_t bh0 = b * a.heads + head0;
    for (int i = threadIdx.x; i < group * D4; i += 256) {
        const int g = i / D4, t = i % D4;
        const float m = fmaxf(fmaxf(wm[0][g], wm[1][g]), fmaxf(wm[2][g], wm[3][g]));
        float e[4], f[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            e[w] = wm[w][g] == -INFINITY ? 0.0f : exp2f(wm[w][g] - m);
            f[w] = wm[w][g] == -INFINITY ? wl[w][g] : wl[w][g] * e[w];
        }
        const float l = (f[0] + f[1]) + (f[2] + f[3]);
        // (Their weights over a power of two above the sum of them, the rest of
        // the division last.)
        const float scale = l > 0.0f ? half_over(l) : 0.0f;
        const float rest = l > 0.0f ? 1.0f / (l * scale) : 0.0f;
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float4 r = red[w][g][t];
            const float share = wl[w][g] > 0.0f ? e[w] * twice_under(wl[w][g]) * scale : 0.0f;
            o.x += share * r.x; o.y += share * r.y; o.z += share * r.z; o.w += share * r.w;
        }
        o.x *= rest; o.y *= rest; o.z *= rest; o.w *= rest;
        const uint64_t rec = (bh0 + g) * chunks + c_idx;
        *reinterpret_cast<float4*>(part_o + rec * D + 4 * t) = o;
        if (t == 0) *reinterpret_cast<float2*>(part_ml + 2 * rec) = make_float2(m, l);
    }
}

// Merges the chunk records of one (batch, head) (mhip::merge_decode_chunks,
// whose fixed order every run repeats) and writes its output row.
template <int D4>
__global__ __launch_bounds__(256) void attn_decode_combine_kernel(
    AttnArgs a, uint64_t chunks, const float* __restrict__ part_o,
    const float* __restrict__ part_ml) {
    constexpr int D = 4 * D4;
    const uint64_t bh = blockIdx.x;
    const uint64_t head = bh % a.heads, b = bh / a.heads;
    const float4 v = mhip::merge_decode_chunks<D4>(part_ml + 2 * bh * chunks, part_o + bh * chunks * D,
                                                   chunks, 0, D4);
    if (threadIdx.x < D4)
        *reinterpret_cast<float4*>(a.out + b * a.o_bs + head * D + 4 * threadIdx.x) = v;
}

// Keys [lo, hi) in chunks of STEPS steps. `keep`: leave the chunk records
// for the caller's merge (no combine launch) and reserve `keep->extra_bytes`
// more of the workspace for it.
template <int D4, int GT, int STEPS>
mhip_status launch_decode_chunks(mhip_ctx* ctx, const AttnArgs& a, uint64_t batch, uint64_t kv_rows,
                                 bool bounded, mhip::DecodeChunks* keep, uint64_t lo, uint64_t hi) {
    constexpr int D = 4 * D4;
    constexpr uint64_t kChunk = decode_chunk(D4, STEPS);
    uint64_t chunks = (hi - lo + kChunk - 1) / kChunk;
    if (chunks == 0) chunks = 1;
    const uint64_t slices = (a.heads / a.kv_heads + GT - 1) / GT;
    const uint64_t units = batch * a.kv_heads * slices;
    if (units * chunks >= (1ULL << 31))
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "attention decode: too many key chunks");
    const uint64_t records = batch * a.heads * chunks;
    // A call bounded by a key count sizes the scratch for every row of K/V
    // (at the shorter chunks, the most records), so a step captured later at
    // the same shape never needs to grow it.
    constexpr uint64_t kShortChunk = decode_chunk(D4);
    const uint64_t reserve = bounded ? batch * a.heads * std::max<uint64_t>(1, (kv_rows + kShortChunk - 1) / kShortChunk)
                                     : records;
    float* part = nullptr;
    const uint64_t record_floats = (std::max(records, reserve) * (D + 2) + 63) / 64 * 64;
    const size_t extra = keep ? keep->extra_bytes : 0;
    mhip_status st = attention_workspace(ctx, record_floats * sizeof(float) + extra, &part);
    if (st != MHIP_OK) return st;
    float* part_o = part;
    float* part_ml = part + records * D;
    mhip::launch(ctx, (attn_decode_partial_kernel<D4, GT, STEPS>),
                 dim3(static_cast<unsigned>(units * chunks)), dim3(256), 0, a, lo, chunks, part_o,
                 part_ml);
    st = mhip::check_launch("attention (decode chunks)");
    if (st != MHIP_OK) return st;
    if (keep) {
        keep->part_o = part_o;
        keep->part_ml = part_ml;
        keep->chunks = chunks;
        keep->extra = part + record_floats;
        return MHIP_OK;
    }
    mhip::launch(ctx, attn_decode_combine_kernel<D4>, dim3(static_cast<unsigned>(batch * a.heads)),
                 dim3(256), 0, a, chunks, part_o, part_ml);
    return mhip::check_launch("attention (decode combine)");
}

template <int D4, int GT>
mhip_status launch_decode_group(mhip_ctx* ctx, const AttnArgs& a, uint64_t batch,
                                uint64_t kv_rows, bool bounded, mhip::DecodeChunks* keep) {
    // The one query (seq == 1) sits at position kv_seq - 1 in every batch
    // row and head, so the admitted key range is the same for all of them.
    // A captured call whose key count advances covers every row of K/V; its
    // workgroups find their keys from the replayed count.
    uint64_t lo = 0, hi = kv_rows;
    if (!a.advance) {
        uint64_t upper = a.causal ? a.offset + 1 : a.kv_seq;
        if (upper > a.kv_seq) upper = a.kv_seq;
        uint64_t lower = 0;
        if (a.window >= 0) {
            const uint64_t w = static_cast<uint64_t>(a.window);
            const uint64_t back = w > 0 ? w - 1 : 0;
            lower = a.offset > back ? a.offset - back : 0;
            if (lower > upper) lower = upper;
        }
        lo = lower;
        hi = upper;
    }
    constexpr int kSteps = decode_steps(D4);
    if constexpr (D4 >= 4 && GT <= 4) {
        // The choice follows the capacity for a bounded call, so its eager
        // run and a capture of it take the same chunks.
        const uint64_t span = bounded ? kv_rows : hi - lo;
        const uint64_t slices = (a.heads / a.kv_heads + GT - 1) / GT;
        const uint64_t wgs = batch * a.kv_heads * slices * ((span + decode_chunk(D4) - 1) / decode_chunk(D4));
        const uint64_t cus = ctx->compute_units ? ctx->compute_units : 256;
        if (wgs >= 16 * cus)
            return launch_decode_chunks<D4, GT, 2 * kSteps>(ctx, a, batch, kv_rows, bounded, keep, lo, hi);
    }
    return launch_decode_chunks<D4, GT, kSteps>(ctx, a, batch, kv_rows, bounded, keep, lo, hi);
}

template <int D4>
mhip_status launch_decode(mhip_ctx* ctx, const AttnArgs& a, uint64_t batch, uint64_t kv_rows,
                          bool bounded, mhip::DecodeChunks* keep = nullptr) {
    const uint64_t group = a.heads / a.kv_heads;
    if (group == 1) return launch_decode_group<D4, 1>(ctx, a, batch, kv_rows, bounded, keep);
    if (group == 2) return launch_decode_group<D4, 2>(ctx, a, batch, kv_rows, bounded, keep);
    if (group <= 4) return launch_decode_group<D4, 4>(ctx, a, batch, kv_rows, bounded, keep);
    return launch_decode_group<D4, kMaxGroup>(ctx, a, batch, kv_rows, bounded, keep);
}

// ---------------------------------------------------------------------------
// Generic: one wave per (batch, query, head)
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void attn_generic_kernel(AttnArgs a, uint64_t total) {
    apply_advance(a);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t item = static_cast<uint64_t>(blockIdx.x) * 4 + wave;
    if (item >= total) return;
    const uint64_t head = item % a.heads;
    const uint64_t qi = (item / a.heads) % a.seq;
    const uint64_t b = item / (a.heads * a.seq);
    const uint64_t kvh = head / (a.heads / a.kv_heads);
    const float* qrow = a.q + b * a.q_bs + qi * a.heads * a.d + head * a.d;
    const float* K = a.k + b * a.k_bs + kvh * a.d;
    const float* V = a.v + b * a.v_bs + kvh * a.vd;
    const uint64_t k_ld = a.kv_heads * a.d, v_ld = a.kv_heads * a.vd;
    float* orow = a.out + b * a.o_bs + qi * a.heads * a.vd + head * a.vd;
    uint64_t lo, hi;
    key_range(a, a.offset + qi, &lo, &hi);
    constexpr int kMaxCols = 4;  // value columns per lane: vd <= 256
    float acc[kMaxCols] = {0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.0f;
    for (uint64_t k0 = lo; k0 < hi; k0 += 64) {
        const uint64_t key = k0 + lane;
        float s = -INFINITY;
        if (key < hi) {
            float dot = 0.0f;
            for (uint64_t t = 0; t < a.d; ++t) dot += qrow[t] * K[key * k_ld + t];
            s = dot * a.qscale;
        }
        float mx = s;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        const float m_new = fmaxf(m, mx);
        const float p = exp2f(s - m_new);
        float sum = p;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
        const float alpha = exp2f(m - m_new);
        const float l_new = l * alpha + sum;
        const float inv = 1.0f / l_new;
        const float keep = l * alpha * inv;
        const float p_hat = p * inv;
        const int nk = static_cast<int>(min<uint64_t>(64, hi - k0));
#pragma unroll
        for (int c = 0; c < kMaxCols; ++c) acc[c] *= keep;
        for (int j = 0; j < nk; ++j) {
            const float pj = __shfl(p_hat, j, 64);
#pragma unroll
            for (int c = 0; c < kMaxCols; ++c) {
                const uint64_t col = lane + 64 * c;
                if (col < a.vd) acc[c] += pj * V[(k0 + j) * v_ld + col];
            }
        }
        m = m_new;
        l = l_new;
    }
    for (int c = 0; c < kMaxCols; ++c) {
        const uint64_t col = lane + 64 * c;
        if (col < a.vd) orow[col] = acc[c];
    }
}

}  // namespace

namespace {

// The checks and kernel arguments of mhip_attention_f32; *empty when there
// is no query row (nothing to do).
mhip_status prepare_attention(mhip_ctx* ctx, const float* q, const float* k, const float* v,
                              float* out, const mhip_attention_params* p, AttnArgs* args,
                              uint64_t* batch_out, bool* empty) {
    *empty = false;
    if (!p) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "attention: null params");
    const uint64_t H = p->head_count, Hkv = p->kv_head_count, d = p->head_dimension;
    const uint64_t vd = p->value_dimension ? p->value_dimension : d;
    if (H == 0 || d == 0 || Hkv == 0 || vd == 0)
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED,
                          "head_count, kv_head_count, and head_dimension must all be positive");
    if (H % Hkv != 0)
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED,
                          "head_count " + std::to_string(H) +
                              " must be an exact multiple of kv_head_count " + std::to_string(Hkv));
    if (p->window_size == 0)
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED,
                          "window_size must be positive; a zero window admits no keys");
    if (p->window_size > 0 && !p->causal)
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "window_size is only defined for causal attention");
    if (p->kv_seq_len > p->kv_rows)
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED,
                          "key_count " + std::to_string(p->kv_seq_len) + " exceeds the " +
                              std::to_string(p->kv_rows) + " rows of K/V");
    if (p->seq_len > p->kv_seq_len)
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED,
                          "q sequence length " + std::to_string(p->seq_len) +
                              " cannot exceed k/v sequence length " + std::to_string(p->kv_seq_len));
    if (!(p->scale <= 0.0f) && !std::isfinite(p->scale))
        return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "attention scale must be finite and positive");
    const uint64_t batch = p->batch ? p->batch : 1;
    *batch_out = batch;
    if (p->seq_len == 0) {
        *empty = true;
        return MHIP_OK;
    }
    if (!q || !k || !v || !out) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "attention: null buffer");

    AttnArgs& a = *args;
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.seq = p->seq_len;
    a.kv_seq = p->kv_seq_len;
    a.heads = H;
    a.kv_heads = Hkv;
    a.d = d;
    a.vd = vd;
    a.offset = p->kv_seq_len - p->seq_len;
    a.causal = p->causal ? 1 : 0;
    a.window = p->window_size > 0 ? p->window_size : -1;
    const float scale = p->scale > 0.0f ? p->scale : 1.0f / std::sqrt(static_cast<float>(d));
    a.qscale = scale * kLog2e;
    // A captured call bounded by an explicit key count advances it with the
    // replay offset (one query row; several rows replay only at offset 0).
    a.advance = nullptr;
    if (p->bounded_key_count) {
        if (p->seq_len == 1)
            a.advance = mhip::advance_ptr(ctx, MHIP_ADVANCE_KEY_COUNT, p->kv_rows - p->kv_seq_len);
        else
            (void)mhip::advance_ptr(ctx, MHIP_ADVANCE_KEY_COUNT, 0);
    }
    a.q_bs = p->q_batch_stride ? p->q_batch_stride : p->seq_len * H * d;
    a.k_bs = p->kv_batch_stride ? p->kv_batch_stride : p->kv_rows * Hkv * d;
    a.v_bs = p->v_batch_stride ? p->v_batch_stride : p->kv_rows * Hkv * vd;
    a.o_bs = p->out_batch_stride ? p->out_batch_stride : p->seq_len * H * vd;
    return MHIP_OK;
}

bool decode_aligned(const AttnArgs& a) {
    return mhip::aligned16(a.q) && mhip::aligned16(a.k) && mhip::aligned16(a.v) &&
           mhip::aligned16(a.out) && a.q_bs % 4 == 0 && a.k_bs % 4 == 0 && a.v_bs % 4 == 0 &&
           a.o_bs % 4 == 0;
}

}  // namespace

namespace mhip {

mhip_status attention_decode_chunks_f32(mhip_ctx* ctx, const float* q, const float* k,
                                        const float* v, const mhip_attention_params* p,
                                        DecodeChunks* out) {
    MHIP_REQUIRE_CTX(ctx);
    if (!out || !p || p->seq_len != 1 || (p->batch && p->batch != 1)) return MHIP_LAYOUT_UNSUPPORTED;
    AttnArgs a;
    uint64_t batch = 1;
    bool empty = false;
    // No output row is written: the records' consumer merges them. Any
    // aligned address stands in for the output in the checks.
    mhip_status st = prepare_attention(ctx, q, k, v, const_cast<float*>(q), p, &a, &batch, &empty);
    if (st != MHIP_OK) return st;
    const uint64_t d = a.d;
    if (empty || !decode_aligned(a) || a.vd != d || d % 4 != 0 || d > 256 || p->kv_seq_len == 0)
        return MHIP_LAYOUT_UNSUPPORTED;
    out->heads = a.heads;
    out->d = d;
    const bool bounded = p->bounded_key_count != 0;
    switch (d / 4) {
        case 1: return launch_decode<1>(ctx, a, 1, p->kv_rows, bounded, out);
        case 2: return launch_decode<2>(ctx, a, 1, p->kv_rows, bounded, out);
        case 4: return launch_decode<4>(ctx, a, 1, p->kv_rows, bounded, out);
        case 8: return launch_decode<8>(ctx, a, 1, p->kv_rows, bounded, out);
        case 16: return launch_decode<16>(ctx, a, 1, p->kv_rows, bounded, out);
        case 32: return launch_decode<32>(ctx, a, 1, p->kv_rows, bounded, out);
        case 64: return launch_decode<64>(ctx, a, 1, p->kv_rows, bounded, out);
        default: return MHIP_LAYOUT_UNSUPPORTED;
    }
}

}  // namespace mhip

extern "C" mhip_status mhip_attention_f32(mhip_ctx* ctx, const float* q, const float* k,
                                          const float* v, float* out,
                                          const mhip_attention_params* p) {
    MHIP_REQUIRE_CTX(ctx);
    AttnArgs a;
    uint64_t batch = 1;
    bool empty = false;
    mhip_status pst = prepare_attention(ctx, q, k, v, out, p, &a, &batch, &empty);
    if (pst != MHIP_OK || empty) return pst;
    const uint64_t H = a.heads, d = a.d, vd = a.vd;

    const bool aligned = decode_aligned(a);
    if (aligned && p->seq_len == 1 && vd == d && d % 4 == 0 && d <= 256 && p->kv_seq_len > 0) {
        mhip_status st = MHIP_CAPTURE_UNSUPPORTED;
        switch (d / 4) {
            case 1: st = launch_decode<1>(ctx, a, batch, p->kv_rows, p->bounded_key_count != 0); break;
            case 2: st = launch_decode<2>(ctx, a, batch, p->kv_rows, p->bounded_key_count != 0); break;
            case 4: st = launch_decode<4>(ctx, a, batch, p->kv_rows, p->bounded_key_count != 0); break;
            case 8: st = launch_decode<8>(ctx, a, batch, p->kv_rows, p->bounded_key_count != 0); break;
            case 16: st = launch_decode<16>(ctx, a, batch, p->kv_rows, p->bounded_key_count != 0); break;
            case 32: st = launch_decode<32>(ctx, a, batch, p->kv_rows, p->bounded_key_count != 0); break;
            case 64: st = launch_decode<64>(ctx, a, batch, p->kv_rows, p->bounded_key_count != 0); break;
            default: break;
        }
        if (st != MHIP_CAPTURE_UNSUPPORTED) return st;  // else: no decode kernel for this d
    }
    // The MFMA kernel's key arithmetic is 32-bit, and so are its byte
    // offsets within a 32-row K or V tile.
    const bool small_keys = p->kv_rows < (1ULL << 31) - 512 && a.kv_heads * std::max(d, vd) < (1ULL << 24);
    if (aligned && small_keys && vd == d && a.kv_seq > 0) {
        const bool replayable = p->seq_len == 1 && p->bounded_key_count != 0;
        switch (d) {
            case 32: return launch_prefill<32>(ctx, a, batch, replayable);
            case 64: return launch_prefill<64>(ctx, a, batch, replayable);
            case 80: return launch_prefill<80>(ctx, a, batch, replayable);
            case 96: return launch_prefill<96>(ctx, a, batch, replayable);
            case 112: return launch_prefill<112>(ctx, a, batch, replayable);
            case 128: return launch_prefill<128>(ctx, a, batch, replayable);
            default: break;
        }
    }
    if (vd > 256) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "attention value dimension above 256");
    const uint64_t total = batch * p->seq_len * H;
    if (total / 4 >= (1ULL << 31)) return mhip::fail(MHIP_SHAPE_UNSUPPORTED, "attention: too many rows");
    mhip::launch(ctx, attn_generic_kernel, dim3(static_cast<unsigned>((total + 3) / 4)), dim3(256),
                 0, a, total);
    return mhip::check_launch("attention (generic)");
}
