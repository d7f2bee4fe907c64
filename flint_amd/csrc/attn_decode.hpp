// The paged attention kernels' launch arguments and the decode workgroup's
// body, shared by attention.hip (attn_mfma and the kernels that mix decode
// items with prefill blocks) and attn_spread.hip.
#pragma once

#include "codec.hpp"
#include "layout.hpp"
#include "lds_dma.hpp"
#include "pool.hpp"
#include "query_plan.hpp"
#include "rope.hpp"

namespace thb {

constexpr float kTau = 8.0f;          // lazy-rescale threshold (log2 units)
constexpr float kFloor = -1.0e30f;    // initial running max (finite on purpose)
constexpr uint32_t kMaxPartPages = 1024;
// Longest part_len in pages: its partitions, up to part_len + part_len / 64
// rounded up to the alignment, fit kMaxPartPages pages.
constexpr uint32_t kMaxPartLenPages = kMaxPartPages - kMaxPartPages / 64;

// Raw buffer resources (decode tile loads): word 3 of a gfx9 descriptor
// with a 32-bit data format (untyped loads need a nonzero one), the
// non-temporal cache-policy bit of a buffer load, and an offset that is out
// of range of every resource the kernels build (loads there return zeros).
constexpr int kBufferFlags = 0x00020000;
constexpr int kBufferNt = 2;
constexpr uint32_t kBufferOob = 0xFFFFFFF0u;
constexpr uint32_t kMaxParts = 512;   // partitions of one group the merge kernel takes
constexpr uint32_t kMergeWords = 8;   // merge record: r0, R, h0, H, n_parts, item0, 0, 0
// Work-item records carry their group's (or block's) words and the
// partition index, so a workgroup finds its work in one dependent load.
constexpr uint32_t kItemWords = kGroupWords + 1;
// A device plan's record may hold some of an item's waves (attn_pick): their
// first in bits 23:16 of the partition word, their count above (0: all).
constexpr uint32_t kRecRun = 16, kRecRuns = 24;
constexpr uint32_t kNoItem = 0xFFFFFFFFu;  // the empty second half of a prefill pair
constexpr uint32_t kBItemWords = kBlockWords + 1;

// Waves per workgroup and tiles in flight per wave of each head_dim
// template: up to head_dim 256, 8 waves (2 per SIMD, 256 registers each),
// with two tiles in flight up to 128 and one at 256 (the query, output and
// load registers grow with head_dim; at 256 the second wave per SIMD hides
// more than a second tile, 1.5% on Gemma-2 layers, and a second tile with
// the query halves in LDS measured 2% slower); at 512, 4 waves with one
// tile and the query halves in LDS.
#ifndef THB_ATTN_WAVES
#define THB_ATTN_WAVES 8
#endif
#ifndef THB_ATTN_RING
#define THB_ATTN_RING 2
#endif
#ifndef THB_ATTN_WAVES_256
#define THB_ATTN_WAVES_256 8
#endif
#ifndef THB_ATTN_RING_256
#define THB_ATTN_RING_256 1
#endif
constexpr int waves_for(int hd) { return hd >= 512 ? 4 : THB_ATTN_WAVES; }
constexpr int ring_for(int hd) { return hd >= 512 ? 1 : hd >= 256 ? THB_ATTN_RING_256 : THB_ATTN_RING; }
// Decode workgroups: head_dim 256 has its own wave count (fewer waves hold
// more tiles in flight each).
constexpr int decode_waves(int hd) { return hd == 256 ? THB_ATTN_WAVES_256 : waves_for(hd); }
// Tiles in the LDS ring of a spread launch's waves (32 KiB at head_dim 64, 64
// above: two workgroups per CU), and tiles computed at a time.
constexpr int spread_ring(int hd) { return hd <= 128 ? 8 : 4; }
constexpr int spread_step(int hd) { return hd <= 128 ? 2 : 1; }
// Decode keeps the query's high and low halves in LDS (one copy for the
// workgroup's waves, which share the query group) instead of registers.
constexpr bool q_in_lds(int hd) { return hd >= 512; }

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct AttnArgs {
    const void* q;
    void* y;
    const uint32_t* groups;
    const uint32_t* items;   // decode work items: group words + partition (kItemWords each)
    const uint32_t* ranges;  // [m][2]: lo, hi
    const uint32_t* bitems;  // prefill work items: block words + partition (kBItemWords each)
    // attn_prefill_wide: pairs of prefill work items one workgroup runs in
    // turn (first, second or kNoItem), 2 words each
    const uint32_t* bpairs;
    const uint32_t* order;   // attn_mixed: launch order of decode items and prefill pairs (bit 31)
    // attn_list: the device plan's header (entries, claim counter, done counter)
    uint32_t* list;
    const uint32_t* merge_groups;  // attn_merge: the groups that span several partitions
    const uint32_t* table;
    uint16_t* k;
    uint16_t* v;
    const void* k_src;  // fused append: new K/V rows [m, n_kvh, hd] (null: none)
    const void* v_src;
    uint32_t src_dtype;
    float* part_o;   // [n_items][n_kvh][16][hd_t]
    float* part_ml;  // [n_items][n_kvh][16][2]
    // Arrival counters of the decode groups of several partitions, one per
    // (first item, KV head), zero between launches; null: attn_merge combines
    // every group's partitions after the launch.
    uint32_t* merge_cnt;
    uint64_t plane;  // 16-bit elements per head plane
    uint32_t max_pages, page_shift, q_heads, nq_per_kv, head_dim, part_len, n_kvh;
    uint32_t pages;  // pages of the pool
    float qscale;  // scale * log2(e), or scale / softcap
    float cap2;    // softcap * log2(e), 0 = no soft-cap
    // attn_prefill_wide: the query carries qpre = the sign of qscale (an exact
    // multiply), and qpost = |qscale| scales its products inside the
    // exponent's fma.  (Splitting q * qscale into f16 halves instead measured
    // ~100x larger errors against an exact softmax, 2.6e-5 vs 3e-7.)
    float qpre, qpost;
    uint32_t q_dt, y_dt;       // THB_DT_* of the query (and gate) and of the output
    uint32_t q_stride;         // elements from one query head to the next
    const void* gate;          // sigmoid gate of the output (q_dt), or null
    uint32_t gate_stride;      // elements from one gate head to the next
    // full = 1 selects the kernels with the extensions of thb_attn_io (query
    // stride, gate, bf16 query/output, rope) and the logit soft-cap; the
    // others take f32/f16 q and y only and are the lean path of the common
    // call.
    uint32_t full;
    // Rotary position embedding (FULL kernels): the query is normalised and
    // rotated as it is loaded, the fused append rotates the key.
    uint32_t rope_on;
    const uint32_t* meta;  // row meta of the call's rows (positions)
    RopeDev qrope, krope;
};

// Decode items one wave per workgroup (attn_spread.hip; head_dim 64, 128 or
// 256 exactly, pages of at least 16 tokens).
void launch_spread(uint32_t hd, bool f16, dim3 grid, const AttnArgs& a, hipStream_t s);
void launch_pick(uint32_t hd, bool f16, dim3 grid, const AttnArgs& a, hipStream_t s);

namespace {

// Loads 8 query elements of dims [d0, d0 + 8) as f32: f32 or f16, and
// bf16 in the FULL kernels.
template <bool FULL>
__device__ inline void load_q8(const AttnArgs& a, uint64_t qbase, uint32_t d0, float (&x)[8]) {
    if (a.q_dt == THB_DT_F16) {
        const f16x8 w = *reinterpret_cast<const f16x8*>(static_cast<const _Float16*>(a.q) + qbase + d0);
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = static_cast<float>(w[e]);
    } else if (FULL && a.q_dt == THB_DT_BF16) {
        const uint4 w = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.q) + qbase + d0);
        const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            x[2 * e] = __uint_as_float(ws[e] << 16);
            x[2 * e + 1] = __uint_as_float(ws[e] & 0xffff0000u);
        }
    } else {
        const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(a.q) + qbase + d0);
        const f32x4 u0 = p[0], u1 = p[1];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            x[e] = u0[e];
            x[4 + e] = u1[e];
        }
    }
}

// The lane's KS chunks of 8 query elements as f32 (load_q8 for every k-step):
// every load is issued before the first conversion, from the query's first
// element where a chunk is out of range (then zeroed), so the KS round trips
// overlap instead of each waiting behind a branch.
template <int KS, bool FULL>
__device__ inline void load_q_all(const AttnArgs& a, bool con, uint64_t qbase, uint32_t a4, float (&x)[KS][8]) {
    const uint32_t hd = a.head_dim;
    bool ok[KS];
    uint64_t off[KS];
#pragma unroll
    for (int j = 0; j < KS; j++) {
        const uint32_t d0 = 32u * j + 8u * a4;
        ok[j] = con && d0 < hd;
        off[j] = ok[j] ? qbase + d0 : 0u;
    }
    if (a.q_dt == THB_DT_F16) {
        f16x8 w[KS];
#pragma unroll
        for (int j = 0; j < KS; j++) w[j] = *reinterpret_cast<const f16x8*>(static_cast<const _Float16*>(a.q) + off[j]);
#pragma unroll
        for (int j = 0; j < KS; j++)
#pragma unroll
            for (int e = 0; e < 8; e++) x[j][e] = ok[j] ? static_cast<float>(w[j][e]) : 0.0f;
    } else if (FULL && a.q_dt == THB_DT_BF16) {
        uint4 w[KS];
#pragma unroll
        for (int j = 0; j < KS; j++) w[j] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.q) + off[j]);
#pragma unroll
        for (int j = 0; j < KS; j++) {
            const uint32_t ws[4] = {w[j].x, w[j].y, w[j].z, w[j].w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[j][2 * e] = ok[j] ? __uint_as_float(ws[e] << 16) : 0.0f;
                x[j][2 * e + 1] = ok[j] ? __uint_as_float(ws[e] & 0xffff0000u) : 0.0f;
            }
        }
    } else {
        f32x4 u[KS][2];
#pragma unroll
        for (int j = 0; j < KS; j++) {
            const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(a.q) + off[j]);
            u[j][0] = p[0];
            u[j][1] = p[1];
        }
#pragma unroll
        for (int j = 0; j < KS; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[j][e] = ok[j] ? u[j][0][e] : 0.0f;
                x[j][4 + e] = ok[j] ? u[j][1][e] : 0.0f;
            }
    }
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float tanh_approx(float x) {
    // tanh(x) = 1 - 2 / (exp(2x) + 1); saturates cleanly at +-1.
    const float e = fast_exp2(x * 2.8853900817779268f);  // 2 * log2(e)
    return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
}
// tanh(x * c2 / (2 log2 e)) for a scale c2 folded into the exponent.
__device__ __forceinline__ float tanh_scaled(float x, float c2) {
    const float e = fast_exp2(x * c2);
    return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
}

// Max / sum over the four lanes c, c+16, c+32, c+48 (one MFMA column).
__device__ __forceinline__ float col_max(float x) {
    x = fmaxf(x, __shfl_xor(x, 16));
    return fmaxf(x, __shfl_xor(x, 32));
}
__device__ __forceinline__ float col_sum(float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}

// Operand types of one KV encoding.
template <bool F16>
struct Ops;

template <>
struct Ops<true> {
    typedef f16x8 in8;
    typedef f16x4 in4;
    // hi + lo split of an f32 (hi = RNE(x), lo = RNE(x - hi)).
    __device__ static void split(float x, _Float16& h, _Float16& l) {
        h = static_cast<_Float16>(x);
        l = static_cast<_Float16>(x - static_cast<float>(h));
    }
    __device__ static f32x4 qk(const u32x4& k, const in8& q, f32x4 acc) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(in8, k), q, acc, 0, 0, 0);
    }
    __device__ static f32x4 pv(const u32x2& v, const in4& p, f32x4 acc) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(in4, v), p, acc, 0, 0, 0);
    }
    // PV over 32 tokens: 8 tokens of one dimension (A) against 8 probabilities
    // of one column (B).
    __device__ static f32x4 pv32(const u32x4& v, const in8& p, f32x4 acc) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(in8, v), p, acc, 0, 0, 0);
    }
    __device__ static void split4(const float* p, in4& h, in4& l) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            _Float16 a, b;
            split(p[e], a, b);
            h[e] = a;
            l[e] = b;
        }
    }
    __device__ static void split8(const float* x, in8& h, in8& l) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            _Float16 a, b;
            split(x[e], a, b);
            h[e] = a;
            l[e] = b;
        }
    }
    // The same split (both halves rounded to nearest even), two elements per
    // conversion: three vector instructions per element.
    __device__ static void split8_fast(const float* x, in8& h, in8& l) {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const f16x2 hh = __builtin_convertvector((f32x2{x[e], x[e + 1]}), f16x2);
            const f16x2 ll = __builtin_convertvector(
                (f32x2{x[e] - static_cast<float>(hh[0]), x[e + 1] - static_cast<float>(hh[1])}), f16x2);
            h[e] = hh[0];
            h[e + 1] = hh[1];
            l[e] = ll[0];
            l[e + 1] = ll[1];
        }
    }
};

template <>
struct Ops<false> {
    typedef bf16x8 in8;
    typedef i16x4 in4;
    __device__ static void split(float x, __bf16& h, __bf16& l) {
        h = static_cast<__bf16>(x);
        l = static_cast<__bf16>(x - static_cast<float>(h));
    }
    __device__ static f32x4 qk(const u32x4& k, const in8& q, f32x4 acc) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(in8, k), q, acc, 0, 0, 0);
    }
    __device__ static f32x4 pv(const u32x2& v, const in4& p, f32x4 acc) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(in4, v), p, acc, 0, 0, 0);
    }
    __device__ static f32x4 pv32(const u32x4& v, const in8& p, f32x4 acc) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(in8, v), p, acc, 0, 0, 0);
    }
    __device__ static void split4(const float* p, in4& h, in4& l) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            __bf16 a, b;
            split(p[e], a, b);
            h[e] = __builtin_bit_cast(short, a);
            l[e] = __builtin_bit_cast(short, b);
        }
    }
    __device__ static void split8(const float* x, in8& h, in8& l) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            __bf16 a, b;
            split(x[e], a, b);
            h[e] = a;
            l[e] = b;
        }
    }
    __device__ static void split8_fast(const float* x, in8& h, in8& l) { split8(x, h, l); }
};

// One scalar of the sigmoid gate (same type as the query).
__device__ inline float gate_at(const AttnArgs& a, uint64_t i) {
    if (a.q_dt == THB_DT_F16) return static_cast<float>(static_cast<const _Float16*>(a.gate)[i]);
    if (a.q_dt == THB_DT_BF16) return __uint_as_float(static_cast<uint32_t>(static_cast<const uint16_t*>(a.gate)[i]) << 16);
    return static_cast<const float*>(a.gate)[i];
}

// f32 -> bf16 bits, round to nearest even (NaN stays NaN).
__device__ inline uint16_t f32_to_bf16_rne(float x) {
    const uint32_t b = __float_as_uint(x);
    if ((b & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((b >> 16) | 0x40u);
    return static_cast<uint16_t>((b + 0x7fffu + ((b >> 16) & 1u)) >> 16);
}

// Writes n (1 or 4) output values of (row, head) at dims [d, d + n): y =
// o / l, times the sigmoid gate 1 / (1 + exp(-g)) when there is one
// (sigmoid_mul.wgsl), in the output type.  The gate and bf16 outputs exist
// in the FULL kernels only.
template <int N, bool FULL>
__device__ inline void store_y(const AttnArgs& a, uint32_t row, uint32_t head, uint32_t d, const float (&v)[N]) {
    float yv[N];
#pragma unroll
    for (int e = 0; e < N; e++) yv[e] = v[e];
    if (FULL && a.gate) {
        const uint64_t gi = (static_cast<uint64_t>(row) * a.q_heads + head) * a.gate_stride + d;
#pragma unroll
        for (int e = 0; e < N; e++) yv[e] = yv[e] / (1.0f + __expf(-gate_at(a, gi + e)));
    }
    const uint64_t yi = (static_cast<uint64_t>(row) * a.q_heads + head) * a.head_dim + d;
    if constexpr (N == 4) {
        if (a.y_dt == THB_DT_F32) {
            *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + yi) = f32x4{yv[0], yv[1], yv[2], yv[3]};
        } else if (!FULL || a.y_dt == THB_DT_F16) {
            f16x4 h;
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = static_cast<_Float16>(yv[e]);
            *reinterpret_cast<f16x4*>(static_cast<_Float16*>(a.y) + yi) = h;
        } else {
            *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.y) + yi) =
                u32x2{f32_to_bf16_rne(yv[0]) | (static_cast<uint32_t>(f32_to_bf16_rne(yv[1])) << 16),
                      f32_to_bf16_rne(yv[2]) | (static_cast<uint32_t>(f32_to_bf16_rne(yv[3])) << 16)};
        }
    } else {
        if (a.y_dt == THB_DT_F32)
            static_cast<float*>(a.y)[yi] = yv[0];
        else if (!FULL || a.y_dt == THB_DT_F16)
            static_cast<_Float16*>(a.y)[yi] = static_cast<_Float16>(yv[0]);
        else
            static_cast<uint16_t*>(a.y)[yi] = f32_to_bf16_rne(yv[0]);
    }
}

// Q^T operand of a lane: column (row, head), dims 32j + 8 a4 .. + 8 of k-step
// j, split into high and low halves.  The raw query is split (the prefill
// kernel passes pre = the sign of the score scale, an exact multiply) and the
// f32 scores are scaled afterwards, so the low half stays out of the f16
// subnormal range.  In the FULL kernels: query heads q_stride apart and,
// with rope on, the query head is first normalised (q_norm; the four lanes
// of the column add their sums of squares) and rotated at the row's
// position.  Every lane must call it (column sums).
template <int KS, class O, bool FULL>
__device__ inline void load_q(const AttnArgs& a, bool con, uint32_t row, uint32_t head, uint32_t a4,
                              typename O::in8 (&qh)[KS], typename O::in8 (&ql)[KS], float pre = 1.0f) {
    const uint32_t hd = a.head_dim;
    const uint64_t qbase = (static_cast<uint64_t>(row) * a.q_heads + head) * (FULL ? a.q_stride : hd);
    const bool rope = FULL && a.rope_on;
    if (!rope) {
        float x[KS][8];
        load_q_all<KS, FULL>(a, con, qbase, a4, x);
#pragma unroll
        for (int j = 0; j < KS; j++) {
#pragma unroll
            for (int e = 0; e < 8; e++) x[j][e] *= pre;
            O::split8(x[j], qh[j], ql[j]);
        }
        return;
    }
    // Rotary path: the lane's chunks in registers, normalised in place.
    const RopeDev& r = a.qrope;
    const uint32_t pos = con ? a.meta[8 * row] : 0u;
    float x[KS][8];
    load_q_all<KS, FULL>(a, con, qbase, a4, x);
    float inv = 1.0f;
    if (r.w) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < KS; j++) ss += sumsq8(x[j]);
        inv = rms_inv(col_sum(ss), hd, r.eps);
#pragma unroll
        for (int j = 0; j < KS; j++) {
            const uint32_t d0 = 32u * j + 8u * a4;
            if (con && d0 < hd) norm8(x[j], inv, r.w + d0);
        }
    }
    if (r.rot == hd && hd == 32u * KS) {
        // Full rotation at the template width: the partner of chunk j is
        // chunk j + KS / 2 of the same lane.
#pragma unroll
        for (int j = 0; j < KS / 2; j++) {
            float lo[8], hi[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                lo[e] = x[j][e];
                hi[e] = x[j + KS / 2][e];
            }
            const uint32_t d0 = 32u * j + 8u * a4;
            rotate8(x[j], hi, d0, pos, r);
            rotate8(x[j + KS / 2], lo, d0 + r.half, pos, r);
        }
    } else {
        // Partial rotation or a narrower head: partners from memory.
#pragma unroll
        for (int j = 0; j < KS; j++) {
            const uint32_t d0 = 32u * j + 8u * a4;
            if (con && d0 < r.rot) {
                const uint32_t dp = d0 < r.half ? d0 + r.half : d0 - r.half;
                float y[8];
                load_q8<FULL>(a, qbase, dp, y);
                if (r.w) norm8(y, inv, r.w + dp);
                rotate8(x[j], y, d0, pos, r);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < KS; j++) {
#pragma unroll
        for (int e = 0; e < 8; e++) x[j][e] *= pre;
        O::split8(x[j], qh[j], ql[j]);
    }
}

// The query operand in LDS (head_dim 512 only: QLDS), else nothing.
template <typename T, int KS, bool QLDS>
struct DecodeQLds {
    T q[KS][2][64];
};
template <typename T, int KS>
struct DecodeQLds<T, KS, false> {};

// ------------------------------------------------ split-K partition merge
// A group whose keys span several partitions has one partial result (m, l,
// o) per partition.  The partials are written with relaxed agent-scope
// atomic stores and read with relaxed agent-scope atomic loads (coherent
// across the XCDs' L2 caches: the stores reach the device's coherence point,
// the loads do not hit a stale copy), so a workgroup of the same launch can
// read another's partial once that partial's stores have completed.
__device__ inline void publish_o(float* p, const f32x4& v) {
    uint64_t* q = reinterpret_cast<uint64_t*>(p);
    __hip_atomic_store(q, (uint64_t(__float_as_uint(v[1])) << 32) | __float_as_uint(v[0]), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 1, (uint64_t(__float_as_uint(v[3])) << 32) | __float_as_uint(v[2]), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void publish_ml(float* p, float m, float l) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), (uint64_t(__float_as_uint(l)) << 32) | __float_as_uint(m),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool COH>
__device__ inline uint64_t load_u64(const float* p) {
    const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
    if constexpr (COH)
        return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        return *q;
}
template <bool COH>
__device__ inline f32x4 load_o(const float* p) {
    const uint64_t lo = load_u64<COH>(p), hi = load_u64<COH>(p + 2);
    return f32x4{__uint_as_float(static_cast<uint32_t>(lo)), __uint_as_float(static_cast<uint32_t>(lo >> 32)),
                 __uint_as_float(static_cast<uint32_t>(hi)), __uint_as_float(static_cast<uint32_t>(hi >> 32))};
}

// Weights of W wave states (running max m, sum l) of one column, their
// common max M and combined sum L: waves in order, one rounding per step.
// Written with explicit fused multiply-adds, as are the sums over o that use
// the weights, so that the merge in one workgroup's LDS and the merge of
// states from memory (attn_spread) give the same bits.
template <int W>
__device__ __forceinline__ void wave_weights(const float (&m)[W], const float (&l)[W], float (&f)[W], float& M,
                                             float& L) {
    M = m[0];
#pragma unroll
    for (int w = 1; w < W; w++) M = fmaxf(M, m[w]);
    L = 0.0f;
#pragma unroll
    for (int w = 0; w < W; w++) {
        f[w] = fast_exp2(m[w] - M);
        L = __builtin_fmaf(l[w], f[w], L);
    }
}
// acc + x * f, element by element.
__device__ __forceinline__ f32x4 fma4(const f32x4& x, float f, const f32x4& acc) {
    return f32x4{__builtin_fmaf(x[0], f, acc[0]), __builtin_fmaf(x[1], f, acc[1]), __builtin_fmaf(x[2], f, acc[2]),
                 __builtin_fmaf(x[3], f, acc[3])};
}

// Combines the partitions of one (group, KV head) in partition order.  Each
// of NT threads owns 4-dimension units of the group's outputs (unit u:
// column u / q4, dims 4 (u % q4) .. + 4) and reads its column's (m, l)
// itself; up to U partitions are requested at once, (m, l) and o together.
// The arithmetic does not depend on NT or on where it runs (the merge
// kernel, or the workgroup of the group's last partition), so neither does
// the output.
template <int HD, bool FULL, int NT, bool COH>
__device__ __forceinline__ void merge_group(const AttnArgs& a, uint32_t r0, uint32_t R, uint32_t h0, uint32_t H,
                                            uint32_t n_parts, uint32_t item0, uint32_t kvh, uint32_t tid) {
    const uint32_t ncols = R * H, hd = a.head_dim, q4 = hd >> 2;
    const uint64_t base = static_cast<uint64_t>(item0) * a.n_kvh + kvh;  // partition pi: base + pi * n_kvh
    const uint64_t mstep = 2 * static_cast<uint64_t>(a.n_kvh) * kCols;   // (m, l) of the next partition
    const uint64_t ostep = static_cast<uint64_t>(a.n_kvh) * kCols * HD;  // o of the next partition
    constexpr uint32_t U = 8, NU = (kCols * HD / 4 + NT - 1) / NT;
    for (uint32_t u0 = 0; u0 < NU; u0++) {
        const uint32_t u = tid + NT * u0;
        if (u >= ncols * q4) break;
        const uint32_t c = u / q4, d = 4u * (u - c * q4);
        const float* ml = a.part_ml + 2 * (base * kCols + c);
        const float* op = a.part_o + (base * kCols + c) * HD + d;
        float M = kFloor;
        if (n_parts > U) {  // long merges: the maximum first
            for (uint32_t p0 = 0; p0 < n_parts; p0 += U) {
                float mv[U];
#pragma unroll
                for (uint32_t k = 0; k < U; k++)
                    mv[k] = p0 + k < n_parts ? __uint_as_float(static_cast<uint32_t>(load_u64<COH>(ml + (p0 + k) * mstep)))
                                             : kFloor;
#pragma unroll
                for (uint32_t k = 0; k < U; k++) M = fmaxf(M, mv[k]);
            }
        }
        float L = 0.0f;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t p0 = 0; p0 < n_parts; p0 += U) {
            float mv[U], lv[U];
            f32x4 ov[U];
#pragma unroll
            for (uint32_t k = 0; k < U; k++) {
                const bool in = p0 + k < n_parts;
                const uint64_t w = in ? load_u64<COH>(ml + (p0 + k) * mstep) : 0ull;
                mv[k] = in ? __uint_as_float(static_cast<uint32_t>(w)) : kFloor;
                lv[k] = in ? __uint_as_float(static_cast<uint32_t>(w >> 32)) : 0.0f;
                ov[k] = in ? load_o<COH>(op + (p0 + k) * ostep) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            if (n_parts <= U) {
#pragma unroll
                for (uint32_t k = 0; k < U; k++) M = fmaxf(M, mv[k]);
            }
#pragma unroll
            for (uint32_t k = 0; k < U; k++) {
                if (p0 + k >= n_parts) break;
                const float w = fast_exp2(mv[k] - M);
                L = __builtin_fmaf(w, lv[k], L);
                acc = fma4(ov[k], w, acc);
            }
        }
        const float inv = 1.0f / L;
        const float yv[4] = {acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
        const uint32_t rr = c / H, hh = c - rr * H;
        store_y<4, FULL>(a, r0 + rr, kvh * a.nq_per_kv + h0 + hh, d, yv);
    }
}

// Run by every thread of a decode workgroup of a group with several
// partitions once its partial is published: the workgroup that finishes
// the group's last partition combines them all (merge_group) and clears the
// group's counter for the next launch.  Each thread waits until its partial
// stores have completed before the barrier, the counter add (relaxed, agent
// scope) is issued after it, and the combining loads only after the add has
// returned, so the last workgroup's loads find every partition's stores
// done.  No workgroup waits for another.  Every partial store and merge load
// is an agent-scope atomic (sc1 on gfx950: not held in an XCD's L2), so this
// is the memory model's agent-scope release/acquire sequence without the L2
// write-back and invalidate, which only plain accesses need.
template <int HD, bool FULL, int NT>
__device__ __forceinline__ void merge_if_last(const AttnArgs& a, uint32_t& s_arrived, uint32_t r0, uint32_t R,
                                              uint32_t h0, uint32_t H, uint32_t n_parts, uint32_t item0,
                                              uint32_t kvh, uint32_t tid) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint32_t* cnt = a.merge_cnt + static_cast<uint64_t>(item0) * a.n_kvh + kvh;
    if (tid == 0) s_arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_arrived + 1u != n_parts) return;
    merge_group<HD, FULL, NT, true>(a, r0, R, h0, H, n_parts, item0, kvh, tid);
    if (tid == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The last wave of a group over a spread launch (attn_spread): combines the
// W wave states of each partition as the one-workgroup merge does, then the
// partitions as merge_group does.  State (item, KV head, wave): (m, l) and o
// of the group's columns.  One wave; each lane takes UN units of 4
// dimensions at a time so that their states are requested together.
template <int HD, bool FULL, int W>
__device__ __forceinline__ void merge_spread(const AttnArgs& a, uint32_t r0, uint32_t R, uint32_t h0, uint32_t H,
                                             uint32_t n_parts, uint32_t item0, uint32_t kvh, uint32_t lane) {
    const uint32_t ncols = R * H, hd = a.head_dim, q4 = hd >> 2, units = ncols * q4;
    constexpr uint32_t UN = 2;
    for (uint32_t u0 = lane; u0 < units; u0 += 64u * UN) {
        uint32_t c[UN], d[UN];
#pragma unroll
        for (uint32_t n = 0; n < UN; n++) {
            const uint32_t u = min(u0 + 64u * n, units - 1u);
            c[n] = u / q4;
            d[n] = 4u * (u - c[n] * q4);
        }
        // Partition p's combined state of unit n.
        auto part = [&](uint32_t p, float (&M)[UN], float (&Lp)[UN], f32x4 (&acc)[UN]) {
            const uint64_t st = (static_cast<uint64_t>(item0 + p) * a.n_kvh + kvh) * W;
            uint64_t ml[UN][W];
            f32x4 ov[UN][W];
#pragma unroll
            for (uint32_t n = 0; n < UN; n++)
#pragma unroll
                for (int w = 0; w < W; w++) {
                    ml[n][w] = load_u64<true>(a.part_ml + 2 * ((st + w) * kCols + c[n]));
                    ov[n][w] = load_o<true>(a.part_o + ((st + w) * kCols + c[n]) * HD + d[n]);
                }
#pragma unroll
            for (uint32_t n = 0; n < UN; n++) {
                float m[W], l[W], f[W];
#pragma unroll
                for (int w = 0; w < W; w++) {
                    m[w] = __uint_as_float(static_cast<uint32_t>(ml[n][w]));
                    l[w] = __uint_as_float(static_cast<uint32_t>(ml[n][w] >> 32));
                }
                wave_weights<W>(m, l, f, M[n], Lp[n]);
                acc[n] = ov[n][0] * f[0];
#pragma unroll
                for (int w = 1; w < W; w++) acc[n] = fma4(ov[n][w], f[w], acc[n]);
            }
        };
        float L[UN];
        f32x4 acc[UN];
        if (n_parts == 1) {
            float M[UN];
            part(0, M, L, acc);
        } else {
            float M[UN];
#pragma unroll
            for (uint32_t n = 0; n < UN; n++) {
                M[n] = kFloor;
                L[n] = 0.0f;
                acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                for (uint32_t p = 0; p < n_parts; p++) {
                    const uint64_t st = (static_cast<uint64_t>(item0 + p) * a.n_kvh + kvh) * W;
                    float mv[W];
#pragma unroll
                    for (int w = 0; w < W; w++)
                        mv[w] = __uint_as_float(
                            static_cast<uint32_t>(load_u64<true>(a.part_ml + 2 * ((st + w) * kCols + c[n]))));
#pragma unroll
                    for (int w = 0; w < W; w++) M[n] = fmaxf(M[n], mv[w]);
                }
            }
            for (uint32_t p = 0; p < n_parts; p++) {
                float Mp[UN], Lp[UN];
                f32x4 ap[UN];
                part(p, Mp, Lp, ap);
#pragma unroll
                for (uint32_t n = 0; n < UN; n++) {
                    const float w = fast_exp2(Mp[n] - M[n]);
                    L[n] = __builtin_fmaf(w, Lp[n], L[n]);
                    acc[n] = fma4(ap[n], w, acc[n]);
                }
            }
        }
#pragma unroll
        for (uint32_t n = 0; n < UN; n++) {
            if (u0 + 64u * n >= units) break;
            const f32x4 yv = acc[n] * (1.0f / L[n]);
            const float v4[4] = {yv[0], yv[1], yv[2], yv[3]};
            const uint32_t rr = c[n] / H, hh = c[n] - rr * H;
            store_y<4, FULL>(a, r0 + rr, kvh * a.nq_per_kv + h0 + hh, d[n], v4);
        }
    }
}

// LDS of one decode workgroup.  The W waves' states are merged in one step
// (every state in LDS, each wave merging and storing its own 16-dimension
// tiles) up to head_dim 256 (128 KiB at 8 waves); head_dim 512 uses a fixed
// tree over W / 2 states.
template <int HD, bool F16, int W>
struct DecodeLds : DecodeQLds<typename Ops<F16>::in8, HD / 32, q_in_lds(HD)> {
    static constexpr bool FLAT = HD <= 256;
    static constexpr int NSTATE = FLAT ? W : (W / 2 > 0 ? W / 2 : 1);
    uint32_t page[kMaxPartPages];
    f32x4 o[NSTATE][HD / 16][64];
    float m[NSTATE][64];
    float l[NSTATE][64];
    uint32_t arrived;  // partitions of the group finished before this one
};

// LDS of one wave of a spread launch: its ring of tiles and the pages of its
// run.
template <int HD, int W, bool LEAN = false>
struct SpreadLds {
    __attribute__((aligned(16))) uint8_t ring[spread_ring(HD)][64 * HD];
    uint32_t page[kMaxPartPages / W + 4];
    u32x4 ql[LEAN ? HD / 32 : 1][LEAN ? 64 : 1];  // LEAN: the query's low halves
};
template <int HD, bool F16, int W, bool SPREAD, bool LEAN>
struct DecodeLdsOf {
    typedef DecodeLds<HD, F16, W> type;
};
template <int HD, bool F16, int W, bool LEAN>
struct DecodeLdsOf<HD, F16, W, true, LEAN> {
    typedef SpreadLds<HD, W, LEAN> type;
};

// One (group, partition, KV head) per workgroup of W waves.  NB tiles of
// loads are kept in flight per wave: tile i + NB is requested as soon as
// tile i has been consumed.  SPREAD: this is one of the W waves, which run in
// workgroups of their own (attn_spread, attn_pick) and whose states meet in
// memory.  G: the item's record; tid: the thread among the item's (SPREAD: the
// lane).  LEAN: within 256 registers at head_dim 256 (attn_pick): the query's low
// halves stay in LDS, and V's operands are read from it behind QK^T.
template <int HD, bool F16, int W, int NB, bool FULL, bool SPREAD, bool LEAN = false>
__device__ __forceinline__ void decode_item(const AttnArgs& a, const uint32_t* G, uint32_t kvh, uint32_t wave,
                                            typename DecodeLdsOf<HD, F16, W, SPREAD, LEAN>::type& L, uint32_t tid) {
    using O = Ops<F16>;
    typedef typename O::in8 in8;
    typedef typename O::in4 in4;
    constexpr int KS = HD / 32;  // QK k-steps of 32 dimensions
    constexpr int MT = HD / 16;  // PV tiles of 16 dimensions
    constexpr bool FLAT = DecodeLds<HD, F16, W>::FLAT;
    static_assert(!SPREAD || FLAT, "spread launches merge in one step");
    auto& s_page = L.page;

    const uint32_t lane = tid & 63u;
    const uint32_t a4 = lane >> 4, c = lane & 15u;
    const uint32_t r0 = G[0], R = G[1], h0 = G[2], H = G[3], seq = G[4];
    const uint32_t glo = G[5], ghi = G[6], n_parts = G[7], gbase = G[8], P = G[9], item0 = G[10];
    const uint32_t part = G[kGroupWords] & ((1u << kRecRun) - 1u), part_slot = item0 + part;  // the partition, its partial-result slot
    // A device-planned call's fixed grid holds slots past a group's last
    // partition (and groups past the call's last): they do nothing.
    if (part >= n_parts) return;
    const uint32_t pbeg = gbase + part * P;
    const uint32_t tb = max(glo, pbeg), te = min(ghi, pbeg + P);
    const uint32_t hd = a.head_dim;
    const uint32_t pshift = a.page_shift;
    const uint32_t pmask = (1u << pshift) - 1u;

    // This wave's run of 16-token tiles inside [tb, te).  For groups of
    // several rows, and with the rotary embedding, runs are handed out last
    // key first: wave 0 takes the run that ends at te, which holds the rows'
    // new tokens, so a fused append's stores (~3.5 us for a 4-row verify
    // chunk at head_dim 256) delay the older wave of its SIMD pair, which
    // the SIMD's issue arbiter favours (over equal runs the younger waves
    // 4-7 take 9-14% longer).  The order depends on the group and the call's
    // kind only, not on whether the append is fused, so fused and separate
    // calls stay bit-identical.
    const uint32_t tb16 = tb & ~15u;
    const uint32_t span = te > tb16 ? te - tb16 : 0u;
    const uint32_t run = ((span + W - 1) / W + 15u) & ~15u;
    const bool last_first = R > 1 || (FULL && a.rope_on);
    const uint32_t ws = tb16 + (last_first ? W - 1u - wave : wave) * run;
    const uint32_t we = min(ws + run, te);

    // Physical pages of this partition (SPREAD: of this wave's run) that hold
    // keys of the group.
    const uint32_t lp0 = (SPREAD ? ws : pbeg) >> pshift;
    {
        const uint32_t kb = SPREAD ? max(ws, tb) : tb, ke = SPREAD ? we : te;
        const uint32_t npg = SPREAD ? (we > ws ? ((we - 1u) >> pshift) - lp0 + 1u : 0u) : P >> pshift;
        const uint32_t* trow = a.table + static_cast<uint64_t>(seq) * a.max_pages;
        for (uint32_t i = tid; i < npg; i += SPREAD ? 64 : 64 * W) {
            const uint32_t lp = lp0 + i;
            const bool used = kb < ke && (lp << pshift) < ke && ((lp + 1) << pshift) > kb;
            const uint32_t pg = used ? trow[lp] : 0u;
            s_page[i] = pg < a.pages ? pg : 0u;  // block_pages: a page outside the pool reads page 0
        }
    }

    // Column c of this lane: row r0 + c / H, head h0 + c % H of the KV head.
    const uint32_t ncols = R * H;
    const bool con = c < ncols;
    const uint32_t rr = con ? c / H : 0u;
    const uint32_t row = r0 + rr;
    const uint32_t head = kvh * a.nq_per_kv + h0 + (con ? c - rr * H : 0u);
    uint32_t clo = 0, chi = 0;
    if (con) {
        clo = max(a.ranges[2 * row], tb);
        chi = min(a.ranges[2 * row + 1], te);
    }
    // Key t is read iff t - clo < cspan (SPREAD: tiles past the run repeat its
    // last one).
    if (SPREAD) chi = min(chi, we);
    const uint32_t cspan = chi > clo ? chi - clo : 0u;

    // Q^T operand: lane (a4, c) holds q[c][32j + 8a4 .. +8], split hi/lo; at
    // head_dim 512 in LDS (wave 0 writes it before the barrier below).
    constexpr bool QLDS = q_in_lds(HD);
    [[maybe_unused]] in8 qh[QLDS ? 1 : KS], ql[QLDS ? 1 : KS];
    if constexpr (QLDS) {
        if (wave == 0) {
            in8 th[KS], tl[KS];
            load_q<KS, O, FULL>(a, con, row, head, a4, th, tl);
#pragma unroll
            for (int j = 0; j < KS; j++) {
                L.q[j][0][lane] = th[j];
                L.q[j][1][lane] = tl[j];
            }
        }
    } else {
        load_q<KS, O, FULL>(a, con, row, head, a4, qh, ql);
        if constexpr (LEAN) {
#pragma unroll
            for (int j = 0; j < KS; j++) L.ql[j][lane] = __builtin_bit_cast(u32x4, ql[j]);
        }
    }


    // Fused append (thb_attn_append).  A row's new token sits at position
    // hi - 1 of the row, and the only wave that ever loads it is the wave
    // whose run holds that position.  That wave encodes and stores the row's
    // K and V of this KV head (exactly as kv_store) before its first tile
    // load; one wave's accesses to an address are ordered, so its tile loads
    // read the stored token.  Work item t of the group: row t / (2 cpr), K or
    // V, 8-element chunk.
    const uint32_t cpr = hd >> 3;
    const uint32_t app_items = a.k_src != nullptr ? R * 2 * cpr : 0u;
    constexpr uint32_t KVE = F16 ? THB_KV_F16_RNE : THB_KV_BF16_TRUNC;
    auto app_decode = [&](uint32_t t, uint32_t& pos, bool& is_v, uint32_t& d, uint64_t& e) -> bool {
        const uint32_t ar = t / (2 * cpr), rem = t - ar * 2 * cpr;
        is_v = rem >= cpr;
        d = (is_v ? rem - cpr : rem) << 3;
        pos = a.ranges[2 * (r0 + ar) + 1] - 1;
        e = (static_cast<uint64_t>(r0 + ar) * a.n_kvh + kvh) * hd + d;
        return pos >= ws && pos < we;
    };
    auto app_store_at = [&](uint32_t page, uint32_t pos, bool is_v, uint32_t d, const uint4& w) {
        const uint64_t base = ((static_cast<uint64_t>(page) * hd) << pshift) + static_cast<uint64_t>(kvh) * a.plane;
        if (!is_v) {
            *reinterpret_cast<uint4*>(a.k + base + k_off(pos & pmask, d, hd, pshift)) = w;
        } else {
            uint16_t* dst = a.v + base + v_off(pos & pmask, d, hd);  // dim d + e at + 4 e
            const uint32_t ws4[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int q2 = 0; q2 < 4; q2++) {
                dst[8 * q2] = static_cast<uint16_t>(ws4[q2] & 0xffffu);
                dst[8 * q2 + 4] = static_cast<uint16_t>(ws4[q2] >> 16);
            }
        }
    };
    auto app_store = [&](uint32_t pos, bool is_v, uint32_t d, const uint4& w) {
        app_store_at(s_page[(pos >> pshift) - lp0], pos, is_v, d, w);
    };
    // The first kAppLane items of each lane (items lane + 64 k): their
    // positions, and the sources of the items this wave owns, are loaded
    // beside the query loads, before the barrier (the source loads overlap
    // the page-table round trips the barrier waits for); the owning lanes
    // encode and store them after the barrier, before the first tile load.
    // A 4-row verify chunk at head_dim 256 (256 items, all in one wave's
    // run) thus costs one round trip instead of four in a row.  The tile
    // loop then holds no store.
    constexpr int kAppLane = 4;
    uint32_t app_pos[kAppLane], app_d[kAppLane];
    uint64_t app_e[kAppLane];
    bool app_v[kAppLane], app_own[kAppLane];
    Raw8 app_raw[kAppLane];
    const bool rope = FULL && a.rope_on;
#pragma unroll
    for (int k = 0; k < kAppLane; k++) {
        const uint32_t t = lane + 64u * k;
        app_own[k] = false;
        if (t < app_items && !rope) {
            app_own[k] = app_decode(t, app_pos[k], app_v[k], app_d[k], app_e[k]);
            if (app_own[k]) app_raw[k] = load_raw8_rt(a.src_dtype, app_v[k] ? a.v_src : a.k_src, app_e[k]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kAppLane; k++)
        if (app_own[k]) app_store(app_pos[k], app_v[k], app_d[k], encode8_rt<KVE>(a.src_dtype, app_raw[k]));
    if (rope) {
        if (app_items != 0) {
            // Rotary append: the key head of each row this wave owns, one chunk
            // of 8 dims per lane (the norm and the rotation need the whole head),
            // exactly as kv_store_rope_kernel.
            for (uint32_t ar = 0; ar < R; ar++) {
                const uint32_t pos = a.ranges[2 * (r0 + ar) + 1] - 1;
                if (pos < ws || pos >= we) continue;  // wave-uniform
                const uint64_t e = (static_cast<uint64_t>(r0 + ar) * a.n_kvh + kvh) * hd + 8u * lane;
                float x[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                if (lane < cpr) load8_f32(a.src_dtype, a.k_src, e, x);
                rope_head_seg(x, lane, cpr, 0, pos, a.krope);
                if (lane < cpr) {
                    uint32_t w[4];
#pragma unroll
                    for (int q2 = 0; q2 < 4; q2++) {
                        if (a.src_dtype == THB_DT_F16)
                            w[q2] = conv16<THB_DT_F16, KVE>(f32_to_f16_rne(x[2 * q2])) |
                                    (conv16<THB_DT_F16, KVE>(f32_to_f16_rne(x[2 * q2 + 1])) << 16);
                        else
                            w[q2] = conv32<KVE>(__float_as_uint(x[2 * q2])) |
                                    (conv32<KVE>(__float_as_uint(x[2 * q2 + 1])) << 16);
                    }
                    app_store(pos, false, 8u * lane, make_uint4(w[0], w[1], w[2], w[3]));
                    app_store(pos, true, 8u * lane, load_encode8_rt<KVE>(a.src_dtype, a.v_src, e));
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    } else if (app_items > 64u * kAppLane) {
        for (uint32_t t = lane + 64u * kAppLane; t < app_items; t += 64) {
            uint32_t pos2, d2;
            uint64_t e2;
            bool v2;
            if (app_decode(t, pos2, v2, d2, e2))
                app_store(pos2, v2, d2, load_encode8_rt<KVE>(a.src_dtype, v2 ? a.v_src : a.k_src, e2));
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }

    float m = kFloor, l = 0.0f;
    f32x4 o[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) o[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* kplane = a.k + static_cast<uint64_t>(kvh) * a.plane;
    const uint16_t* vplane = a.v + static_cast<uint64_t>(kvh) * a.plane;
    const uint32_t last = te > 0 ? te - 1 : 0;
    const uint32_t page_elems = hd << pshift;

    // Loads one 16-token tile with buffer loads.  Tokens outside [tb, te)
    // are clamped into it (their scores are masked).  The tile's tokens lie
    // in the pages of its first and last clamped token (one page unless
    // page_len is 8); the buffer resource starts at the lower of the two, so
    // every lane's byte offset is non-negative (below 4 GiB: the pool checks
    // the plane size for page_len 8).  A tile past the wave's run gets a
    // resource of size 0 and a lane past head_dim an offset beyond the size:
    // such loads return zeros without touching memory (K dims past head_dim
    // must be zeros: the query is zero there).  Every load is thus
    // issued unconditionally, and the compiler's wait counts stay exact
    // through the tile loop (a skipped load would force a full drain).
    // K pages hold 32-dimension groups ([hd/32][page_len][32]): for a fixed
    // k-step j the 64 lanes read 16 tokens x 64 bytes, 1 KiB contiguous.  V
    // pages hold 4-slot groups ([page_len/4][hd][4]): a lane's 4 slots of one
    // dim are 8 bytes, and 16 lanes read 128 contiguous bytes.  The loads are
    // non-temporal (every byte is read once).
    struct TileRes {
        __amdgpu_buffer_rsrc_t k, v;
        uint32_t pa, pb, pmin, first_lp;
    };
    auto tile_res = [&](uint32_t t0) {
        TileRes r;
        const bool on = t0 < we;  // then tb <= tf <= tl <= last: pages of the partition
        const uint32_t tf = min(max(t0, tb), last), tl = min(max(t0 + 15u, tb), last);
        r.first_lp = tf >> pshift;
        r.pa = __builtin_amdgcn_readfirstlane(s_page[on ? r.first_lp - lp0 : 0u]);
        r.pb = __builtin_amdgcn_readfirstlane(s_page[on ? (tl >> pshift) - lp0 : 0u]);
        r.pmin = min(r.pa, r.pb);
        const uint32_t nrec = on ? (max(r.pa, r.pb) - r.pmin + 1u) * 2u * page_elems : 0u;
        const uint64_t off = static_cast<uint64_t>(r.pmin) * page_elems;
        r.k = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kplane + off), 0, nrec, kBufferFlags);
        r.v = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vplane + off), 0, nrec, kBufferFlags);
        return r;
    };
    // Byte offset of token t's page from the resource base.
    auto page_bytes_off = [&](const TileRes& r, uint32_t t) {
        return ((t >> pshift) == r.first_lp ? r.pa - r.pmin : r.pb - r.pmin) * 2u * page_elems;
    };
    auto load_k = [&](uint32_t t0, u32x4 (&kr)[KS]) {
        const TileRes r = tile_res(t0);
        const uint32_t tk = min(max(t0 + c, tb), last);
        const uint32_t base = page_bytes_off(r, tk);
#pragma unroll
        for (int j = 0; j < KS; j++) {
            const uint32_t d0 = 32u * j + 8u * a4;
            const uint32_t off = d0 < hd ? base + 2u * k_off(tk & pmask, d0, hd, pshift) : kBufferOob;
            kr[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r.k, off, 0, kBufferNt));
        }
    };
    auto load_v = [&](uint32_t t0, u32x2 (&vr)[MT]) {
        const TileRes r = tile_res(t0);
        const uint32_t tv = min(max(t0 + 4u * a4, tb & ~3u), last & ~3u);
        const uint32_t base = page_bytes_off(r, tv) + 2u * v_off(tv & pmask, 0, hd);
        // Dims past head_dim read whatever lies there (or zeros): each PV
        // output row is one dim, so they only reach outputs never stored.
#pragma unroll
        for (int i = 0; i < MT; i++)
            vr[i] = __builtin_bit_cast(
                u32x2, __builtin_amdgcn_raw_buffer_load_b64(r.v, base + 8u * (16u * i + c), 0, kBufferNt));
    };
    auto load = [&](uint32_t t0, u32x4 (&kr)[KS], u32x2 (&vr)[MT]) {
        load_k(t0, kr);
        load_v(t0, vr);
    };

    const float qscale = a.qscale, cap2 = a.cap2;
    // The tile arithmetic in parts: QK^T, the masked scores and their lane
    // maximum, the lazy rescale, probabilities and PV.
    auto qk = [&](const u32x4 (&kr)[KS]) {
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < KS; j++) {
            if constexpr (QLDS) {
                s = O::qk(kr[j], L.q[j][0][lane], s);
                s = O::qk(kr[j], L.q[j][1][lane], s);
            } else {
                s = O::qk(kr[j], qh[j], s);
                s = O::qk(kr[j], ql[j], s);
            }
        }
        return s;
    };
    auto scores = [&](uint32_t t0, const f32x4& s, float (&sv)[4]) {  // t0: the lane's first key
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float x = s[e] * qscale;
            if (FULL && cap2 != 0.0f) x = cap2 * tanh_approx(x);  // soft-cap: FULL kernels only
            const uint32_t t = t0 + e;
            x = t - clo < cspan ? x : -INFINITY;
            sv[e] = x;
            mx = fmaxf(mx, x);
        }
        return mx;
    };
    // The column max (two cross-lane steps) is taken only when some score
    // beats its column's running max by more than kTau; without one, no
    // column rescales, exactly as if the max had been taken.
    auto rescale = [&](float mx) {
        if (__builtin_amdgcn_ballot_w64(mx > m + kTau) != 0) {
            mx = col_max(mx);
            if (mx > m + kTau) {
                const float alpha = fast_exp2(m - mx);
                l *= alpha;
#pragma unroll
                for (int i = 0; i < MT; i++) o[i] *= alpha;
                m = mx;
            }
        }
    };
    auto probs = [&](const float (&sv)[4], in4& ph, in4& pl) {
        float p[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            p[e] = fast_exp2(sv[e] - m);
            l += p[e];
        }
        O::split4(p, ph, pl);
    };
    auto pv = [&](const u32x2 (&vr)[MT], const in4& ph, const in4& pl) {
#pragma unroll
        for (int i = 0; i < MT; i++) {
            o[i] = O::pv(vr[i], ph, o[i]);
            o[i] = O::pv(vr[i], pl, o[i]);
        }
    };
    // after_qk runs once the tile's K operands are consumed (one tile in
    // flight: the next tile's K is requested there, before the softmax and
    // the PV products of this one).
    auto compute = [&](uint32_t t0, const u32x4 (&kr)[KS], const u32x2 (&vr)[MT], auto&& after_qk) {
        const f32x4 s = qk(kr);
        after_qk();
        float sv[4];
        rescale(scores(t0 + 4u * a4, s, sv));
        in4 ph, pl;
        probs(sv, ph, pl);
        pv(vr, ph, pl);
    };

    if constexpr (SPREAD) {
        // Tiles come through a ring of NB in LDS, requested NB tiles ahead.
        // (A tile loaded into registers in operand order touches 16 rows of 64
        // bytes per K load: one CU takes in 37 GB/s that way, 80-100 GB/s
        // through direct-to-LDS loads of 1 KiB.)  One tile is HD / 32 blocks of
        // K (16 tokens x 32 dims, as the page holds them) and as many KiB of V
        // (4 slot groups); 16-byte units are swizzled so that an operand read
        // spreads over the banks: K unit u of token t at u ^ t / 4, V unit u of
        // slot group g at u ^ 8 (g odd).
        constexpr int U = spread_step(HD), TL = HD / 16;  // tiles per step, loads per tile
        constexpr uint32_t kTileB = 64u * HD, kUnits = HD / 2;
        const uint32_t ring0 = __builtin_amdgcn_readfirstlane(lds_offset(&L.ring[0][0]));
        const uint32_t k_lane = 2u * (32u * (lane >> 2) + 8u * ((lane & 3u) ^ (lane >> 4)));
        const uint32_t t_end = (we + 15u) & ~15u;  // past the run's last tile
        // Lane offsets (bytes) of V's loads inside a tile.
        uint32_t v_lane[KS];
#pragma unroll
        for (uint32_t i = 0; i < static_cast<uint32_t>(KS); i++) {
            const uint32_t pos = 64u * i + lane, grp = pos / kUnits;
            v_lane[i] = 2u * (4u * HD * grp + 8u * ((pos % kUnits) ^ (8u * (grp & 1u))));
        }
        // A tile to request: past the run its last one again, so that the wait
        // counts stay exact.  next() reads its page (early: an LDS round trip),
        // request() issues its n-th load.
        struct Next {
            const uint16_t *k, *v;
            uint32_t v_lane[KS];
        };
        auto next_page = [&](uint32_t t) { return s_page[(min(t, t_end - 16u) >> pshift) - lp0]; };
        auto next = [&](uint32_t t, uint32_t page) {
            t = min(t, t_end - 16u);
            const uint64_t pbase = (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(page)) * HD) << pshift;
            Next x;
            x.k = kplane + pbase + 32u * (t & pmask);
            x.v = vplane + pbase + HD * (t & pmask);
#pragma unroll
            for (int i = 0; i < KS; i++) x.v_lane[i] = v_lane[i];
            if (t < tb || t + 16u > te) {
                // Slot groups outside [tb, te) are replaced by the first or
                // last one inside (their probabilities are zero, their slots
                // may hold anything).
                const uint32_t g0 = t >> 2, gmin = max(tb >> 2, g0) - g0, gmax = min(last >> 2, g0 + 3u) - g0;
#pragma unroll
                for (uint32_t i = 0; i < static_cast<uint32_t>(KS); i++) {
                    const uint32_t grp = (64u * i + lane) / kUnits;
                    x.v_lane[i] += 8u * HD * (min(max(grp, gmin), gmax) - grp);
                }
            }
            return x;
        };
        // Non-temporal, as load()'s: every byte is read once.  (Eight rows of
        // 3000 keys, 8 KV heads of 128, rotated: 33.4 us per layer of a
        // replayed step with plain loads, 29.1 so; eight of 1600 at
        // head_dim 256 34.0, 29.7; the shortest the same.)
        auto request = [&](const Next& x, uint32_t slot, int n) {
            const uint32_t to = ring0 + slot * kTileB + 1024u * n;
            if (n < KS)
                dma16_from<true>(x.k + ((32u * n) << pshift), k_lane, to);
            else
                dma16_from<true>(x.v, x.v_lane[n - KS], to);
        };
        const uint32_t k_rd = 64u * c + 16u * (a4 ^ (c >> 2));
        if (ws < we) {
            for (uint32_t b = 0; b < static_cast<uint32_t>(NB); b++) {
                const Next x = next(ws + 16u * b, next_page(ws + 16u * b));
#pragma unroll
                for (int n = 0; n < TL; n++) request(x, b, n);
            }
            uint32_t slot = 0;
            for (uint32_t t0 = ws; t0 < we; t0 += 16u * U) {
                wait_vm<(NB - U) * TL>();
                u32x4 kr[U][KS];
                u32x2 vr[U][MT];
                uint32_t page[U];
#pragma unroll
                for (int u = 0; u < U; u++) page[u] = next_page(t0 + 16u * (NB + u));
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int j = 0; j < KS; j++)
                        kr[u][j] = *reinterpret_cast<const u32x4*>(L.ring[slot + u] + 1024u * j + k_rd);
                auto read_v = [&]() {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const uint8_t* vt = L.ring[slot + u] + 32u * HD + 8u * HD * a4 + 8u * c;
#pragma unroll
                        for (int i = 0; i < MT; i++)
                            vr[u][i] = *reinterpret_cast<const u32x2*>(vt + ((128u * i) ^ (128u * (a4 & 1u))));
                    }
                };
                if constexpr (!LEAN) read_v();
                // QK^T, the tiles' chains side by side.
                f32x4 s[U];
#pragma unroll
                for (int u = 0; u < U; u++) s[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < KS; j++) {
#pragma unroll
                    for (int u = 0; u < U; u++) s[u] = O::qk(kr[u][j], qh[j], s[u]);
#pragma unroll
                    for (int u = 0; u < U; u++) s[u] = O::qk(kr[u][j], LEAN ? __builtin_bit_cast(in8, L.ql[j][lane]) : ql[j], s[u]);
                }
                if constexpr (LEAN) {
                    __builtin_amdgcn_sched_barrier(0);
                    read_v();
                }
                Next x[U];
#pragma unroll
                for (int u = 0; u < U; u++) x[u] = next(t0 + 16u * (NB + u), page[u]);
                float sv[U][4], mx[U], top = -INFINITY;
#pragma unroll
                for (int u = 0; u < U; u++) {
                    mx[u] = scores(t0 + 16u * u + 4u * a4, s[u], sv[u]);
                    top = fmaxf(top, mx[u]);
                }
                in4 ph[U], pl[U];
                // Where a step reaches past the run, its repeated tile is left out
                // of the products (zero probabilities of an infinite value would
                // make NaNs).
                const bool past = U > 1 && t0 + 16u * (U - 1) >= we;
                const bool move = past || __builtin_amdgcn_ballot_w64(top > m + kTau) != 0;
                if (!move) {
#pragma unroll
                    for (int u = 0; u < U; u++) probs(sv[u], ph[u], pl[u]);
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tiles are read: request into their slots
                if (!move) {
                    // No tile of the step rescales (the common case): their
                    // products side by side, each output's sums in the order
                    // of one tile at a time, the requests in between (a wave
                    // issues in order).
                    constexpr int kBlk = 4, kProd = MT * 2 * U, kReq = U * TL;
#pragma unroll
                    for (int f = 0; f < kProd; f++) {  // blocks of 4 outputs: tile 0 high, low, tile 1 high, ...
                        const int b = f / kBlk, u = b % (2 * U) / 2, i = b / (2 * U) * kBlk + f % kBlk;
                        o[i] = O::pv(vr[u][i], b & 1 ? pl[u] : ph[u], o[i]);
#pragma unroll
                        for (int n = f * kReq / kProd; n < (f + 1) * kReq / kProd; n++)
                            request(x[n / TL], slot + n / TL, n % TL);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        if (u == 0 || t0 + 16u * u < we) {
                            rescale(mx[u]);
                            probs(sv[u], ph[u], pl[u]);
                            pv(vr[u], ph[u], pl[u]);
                        }
#pragma unroll
                        for (int n = 0; n < TL; n++) request(x[u], slot + u, n);
                    }
                }
                slot = slot + U == NB ? 0u : slot + U;
            }
        }
    } else {
        // NB tiles in flight per wave.  Loads of tiles past the run are
        // issued too (they read nothing), so every iteration issues the same
        // loads and only the products are skipped.
        u32x4 kr[NB][KS];
        u32x2 vr[NB][MT];
#pragma unroll
        for (int b = 0; b < NB; b++) load(ws + 16u * b, kr[b], vr[b]);
        for (uint32_t t0 = ws; t0 < we; t0 += 16u * NB) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const uint32_t t = t0 + 16u * b, tn = t + 16u * NB;
                if constexpr (NB == 1 && HD < 512) {
                    // One tile in flight: the next tile's K goes out as soon
                    // as this tile's K is consumed, its V after the PV.  (At
                    // head_dim 512 the next K beside this tile's V and the
                    // 128 output registers spilled ~90 registers: 246 us for
                    // a 16 x 4096-token decode, against 106 us with the whole
                    // next tile requested after the PV, below.)
                    compute(t, kr[b], vr[b], [&]() { load_k(tn, kr[b]); });
                    load_v(tn, vr[b]);
                } else {
                    if (t < we) compute(t, kr[b], vr[b], []() {});
                    load(tn, kr[b], vr[b]);
                }
            }
        }
    }
    l = col_sum(l);

    if constexpr (SPREAD) {
        // ---- publish this wave's state; the group's last wave merges -----
        if (con) {
            const uint64_t st = ((static_cast<uint64_t>(part_slot) * a.n_kvh + kvh) * W + wave) * kCols + c;
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const uint32_t d = 16u * i + 4u * a4;
                if (d < hd) publish_o(a.part_o + st * HD + d, o[i]);
            }
            if (a4 == 0) publish_ml(a.part_ml + 2 * st, m, l);
        }
        // As merge_if_last: stores complete, then the arrival, then the loads.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t* cnt = a.merge_cnt + static_cast<uint64_t>(item0) * a.n_kvh + kvh;
        uint32_t arrived = 0;
        if (lane == 0) arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        arrived = __builtin_amdgcn_readfirstlane(arrived);
        if (arrived + 1u != n_parts * W) return;
        merge_spread<HD, FULL, W>(a, r0, R, h0, H, n_parts, item0, kvh, lane);
        if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    } else {

    auto& s_o = L.o;
    auto& s_m = L.m;
    auto& s_l = L.l;
    auto& s_arrived = L.arrived;
    if constexpr (FLAT) {
        // ---- merge the W waves' states in one step ----------------------
#pragma unroll
        for (int i = 0; i < MT; i++) s_o[wave][i][lane] = o[i];
        s_m[wave][lane] = m;
        s_l[wave][lane] = l;
        __syncthreads();
        float wm[W], wl[W], f[W], M, L;
#pragma unroll
        for (int w = 0; w < W; w++) {
            wm[w] = s_m[w][lane];
            wl[w] = s_l[w][lane];
        }
        wave_weights<W>(wm, wl, f, M, L);
        const uint64_t pb = (static_cast<uint64_t>(part_slot) * a.n_kvh + kvh) * kCols + c;
        for (uint32_t i = wave; i < static_cast<uint32_t>(MT); i += W) {  // this wave's tiles
            f32x4 acc = s_o[0][i][lane] * f[0];
#pragma unroll
            for (int w = 1; w < W; w++) acc = fma4(s_o[w][i][lane], f[w], acc);
            const uint32_t d = 16u * i + 4u * a4;
            if (!con || d >= hd) continue;
            if (n_parts == 1) {
                const f32x4 yv = acc * (1.0f / L);
                const float v4[4] = {yv[0], yv[1], yv[2], yv[3]};
                store_y<4, FULL>(a, row, head, d, v4);
            } else {
                // several partitions: publish this one's (m, l, o) for the
                // workgroup of the last partition (or the merge kernel)
                publish_o(a.part_o + pb * HD + d, acc);
            }
        }
        if (n_parts > 1 && wave == 0 && con && a4 == 0) publish_ml(a.part_ml + 2 * pb, M, L);
        if (n_parts > 1 && a.merge_cnt)
            merge_if_last<HD, FULL, 64 * W>(a, s_arrived, r0, R, h0, H, n_parts, item0, kvh, tid);
        return;
    }

    // ---- merge the W waves' states through LDS (fixed tree) -------------
    for (uint32_t half = W / 2; half >= 1; half >>= 1) {
        if (wave >= half && wave < 2 * half) {
            const uint32_t sl = wave - half;
#pragma unroll
            for (int i = 0; i < MT; i++) s_o[sl][i][lane] = o[i];
            s_m[sl][lane] = m;
            s_l[sl][lane] = l;
        }
        __syncthreads();
        if (wave < half) {
            const float m2 = s_m[wave][lane], l2 = s_l[wave][lane];
            const float M = fmaxf(m, m2);
            const float f1 = fast_exp2(m - M), f2 = fast_exp2(m2 - M);
#pragma unroll
            for (int i = 0; i < MT; i++) o[i] = o[i] * f1 + s_o[wave][i][lane] * f2;
            l = l * f1 + l2 * f2;
            m = M;
        }
        __syncthreads();
    }
    if (wave == 0 && con) {
        if (n_parts == 1) {
            const float inv = 1.0f / l;
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const uint32_t d = 16u * i + 4u * a4;
                if (d >= hd) continue;
                const f32x4 yv = o[i] * inv;
                const float v4[4] = {yv[0], yv[1], yv[2], yv[3]};
                store_y<4, FULL>(a, row, head, d, v4);
            }
        } else {
            // Several partitions: publish this one's (m, l, o) for the
            // workgroup of the last partition (or the merge kernel).
            const uint64_t pb = (static_cast<uint64_t>(part_slot) * a.n_kvh + kvh) * kCols + c;
#pragma unroll
            for (int i = 0; i < MT; i++) publish_o(a.part_o + pb * HD + 16u * i + 4u * a4, o[i]);
            if (a4 == 0) publish_ml(a.part_ml + 2 * pb, m, l);
        }
    }
    if (n_parts > 1 && a.merge_cnt)
        merge_if_last<HD, FULL, 64 * W>(a, s_arrived, r0, R, h0, H, n_parts, item0, kvh, tid);
    }
}

// A workgroup of W waves of a 1-D grid, KV head fastest: consecutive
// workgroups share a work item, and items are ordered longest first (the host
// sorts them).  tid: threadIdx.x (opaque in attn_list).
template <int HD, bool F16, int W, int NB, bool FULL>
__device__ __forceinline__ void decode_wg(const AttnArgs& a, uint32_t bid, DecodeLds<HD, F16, W>& L, uint32_t tid) {
    const uint32_t item = bid / a.n_kvh, kvh = bid - item * a.n_kvh;
    const uint32_t* G = a.items + static_cast<uint64_t>(item) * kItemWords;
    decode_item<HD, F16, W, NB, FULL, false>(a, G, kvh, __builtin_amdgcn_readfirstlane(tid >> 6), L, tid);
}

}  // namespace
}  // namespace thb
