// The attention consumer's projection on the matrix cores: y[rows, n] =
// x[rows, k] . w[n, k]^T, plus y's old value when acc (ops::gemm_acc,
// crates/thuban_model/src/ops/gemm.rs:113-131; rows == 1 is the reference's
// gemv; the model calls it for o_proj with acc = "add into the residual",
// transformer/forward.rs:338-351).  Weights are bf16 or f16; x is f32 (the
// reference's activations), f16 or bf16 (the attention output the fused
// step writes for this product); y is f32.
//
// Precision: the matrix cores multiply two 16-bit operands.  An x that does
// not fit the weight's type exactly (f32, or f16 against bf16 weights) is
// split into a high and a low part of that type (hi = RNE(x), lo = RNE(x -
// hi)) and both are multiplied, so every product carries ~16 (bf16) or ~22
// (f16) bits of x against the exact weight, accumulated in f32.
//
// Two kernels, no state between calls, a row's sums independent of the other
// rows' values:
//  * gemm_rows (rows <= 16; an x that is converted: up to 64): one workgroup
//    per 16 output columns, its waves splitting K.
//  * gemm_tile (more rows): output tiles of 32 x 16 to 128 x 256, the largest
//    that fills the CUs.
// Both add K up in levels, short chains first.  From 65 rows on every tile
// shape adds in the same order, so a row's bits do not depend on how many rows
// its call has (of an x of the weight's type: nor among 17 to 64 rows).
#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "lds_dma.hpp"

namespace thb {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct GemmArgs {
    const void* x;      // [m, k] of x_dt
    const uint16_t* w;  // [n, k] bf16 or f16
    float* y;           // [m, n]
    uint32_t m, n, k, acc;
};

// Matrix-core operands of one weight type.
template <bool WF16>
struct WOps;

template <>
struct WOps<false> {
    typedef bf16x8 v8;
    typedef __bf16 e;
    __device__ static f32x4 mfma(const v8& a, const v8& b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};

template <>
struct WOps<true> {
    typedef f16x8 v8;
    typedef _Float16 e;
    __device__ static f32x4 mfma(const v8& a, const v8& b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// x elements fit the weight's operand type exactly (one product), or need
// a low part (two products).
constexpr bool same_type(uint32_t xt, bool wf16) {
    return (xt == THB_DT_BF16 && !wf16) || (xt == THB_DT_F16 && wf16);
}
constexpr bool needs_lo(uint32_t xt, bool wf16) {
    return xt == THB_DT_F32 || (xt == THB_DT_F16 && !wf16);
}
// 32-bit words holding 8 x elements.
constexpr int x_words(uint32_t xt) { return xt == THB_DT_F32 ? 8 : 4; }

// Element i of 8 x elements held as words, as f32.
template <uint32_t XT>
__device__ inline float x_elem(const uint32_t* w, int i) {
    if constexpr (XT == THB_DT_F32) {
        return __uint_as_float(w[i]);
    } else {
        const uint32_t h = (w[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
        if constexpr (XT == THB_DT_BF16)
            return __uint_as_float(h << 16);
        else
            return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h)));
    }
}

// The high (and low) operand of 8 x elements in the weight's type.
template <uint32_t XT, bool WF16>
__device__ inline void x_operands(const uint32_t* w, typename WOps<WF16>::v8& hi, typename WOps<WF16>::v8& lo) {
    using E = typename WOps<WF16>::e;
    if constexpr (same_type(XT, WF16)) {
        hi = __builtin_bit_cast(typename WOps<WF16>::v8, u32x4{w[0], w[1], w[2], w[3]});
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float v = x_elem<XT>(w, i);
            const E h = static_cast<E>(v);
            hi[i] = h;
            if constexpr (needs_lo(XT, WF16)) lo[i] = static_cast<E>(v - static_cast<float>(h));
        }
    }
}

// More than 16 rows: output tiles of BM rows (m) x BN columns (n) per
// workgroup, WM x WN waves of NJ x NI products per k-step of 32.
//  * k-tiles of 64 enter LDS without passing through registers (direct-to-LDS
//    loads, ST stages, requested ST - 1 k-tiles ahead): W [row][8 chunks of
//    16 bytes], x likewise in its own type, converted as it is read; a chunk
//    is swizzled by its row so that the 16 rows of an operand read spread
//    over the banks.
//  * The requests go out between the products: a wave issues in order and the
//    CU's address unit takes 16 cycles per direct load, so requests ahead of
//    the products would hold them all back.
//  * Two waves per SIMD, so that one's products run beside the other's LDS
//    reads and waits (one wave per SIMD with 64 x 128 outputs, software
//    pipelined, measured 181 us at 4096^3, this 153 us).
//  * One barrier per k-tile.
// Measured (us per call, bf16 x and W resident in cache, the 128 x 128 tiles
// and split-K kernels before): 32 x 4096 x 4096 12.2 -> 10.1, 128: 59.7 ->
// 15.3, 300: 71.6 -> 23.9, 1000: 77.1 -> 39.3, 1500 x 5120 x 5120 109 -> 87;
// f32 x 266 -> 151.
struct TileArgs {
    GemmArgs g;
    uint32_t mt, nt;  // tiles
};

constexpr uint32_t kBK = 64, kPanel = 1024;  // k of a tile, rows of a panel of tiles
// An output's products add up in chains of kChain k-tiles (16 k-steps), whose
// sums add up in turn; in calls of up to 64 rows (DEEP; half as many k-tiles
// where a low part doubles the products) in runs of kChain2 chains first.  A
// chain's error grows with the square root of its length: at k = 4096 one
// chain over all of K is 4.0e-7 of the result off (bf16; f32 x with f16 W
// 5.8e-7), chains of 8 tiles 1.4e-7 (2.2e-7), DEEP 1.3e-7 (1.7e-7), at k =
// 28672 1.1e-6, 1.9e-7 and 1.6e-7.  Same time with and without, us: bf16 500 x
// 4096 x 4096 24.8 / 25.5, 1500 x 5120 x 5120 86 / 87, f32 150 / 154.
constexpr uint32_t kChain = 8, kChain2 = 4;

// Position swizzle of row r in LDS tiles of 64 k: 128-byte rows (8 positions
// of 16 bytes) cover the 64 banks in pairs, 256-byte rows (f32) each.
template <uint32_t XE>
__device__ inline uint32_t swizzle(uint32_t r) {
    return XE == 4 ? r & 15u : (r >> 1) & 7u;
}
// The 8 x elements at k = 8 u .. of row c of a 16-row block staged at xb.
template <uint32_t XT>
__device__ inline void read_x8(const uint8_t* xb, uint32_t u, uint32_t c, uint32_t* out) {
    constexpr uint32_t XE = XT == THB_DT_F32 ? 4 : 2, H = XE / 2;
#pragma unroll
    for (uint32_t h = 0; h < H; h++) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(xb + c * 64u * XE + ((H * u + h) ^ swizzle<XE>(c)) * 16u);
#pragma unroll
        for (int e = 0; e < 4; e++) out[4 * h + e] = v[e];
    }
}

template <uint32_t XT, bool WF16, int BM, int BN, int WM, int WN, int ST, bool DEEP>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_tile(TileArgs ta) {
    using O = WOps<WF16>;
    using v8 = typename O::v8;
    constexpr bool LO = needs_lo(XT, WF16);
    constexpr int XW = x_words(XT), NT = 64 * WM * WN;
    constexpr int NI = BN / WN / 16, NJ = BM / WM / 16;     // products of 16 n, of 16 m per wave
    constexpr uint32_t XE = XT == THB_DT_F32 ? 4 : 2, kXRow = 64u * XE, kPos = kXRow / 16u;
    constexpr uint32_t kWB = BN * 128, kStage = kWB + BM * kXRow;  // bytes of a W tile, of a stage
    constexpr int WL = BN * 8 / NT, XL = BM * kPos / NT, ND = WL + XL;  // loads per thread of W, x, a k-tile
    __shared__ __attribute__((aligned(16))) uint8_t lds[ST * kStage];
    const GemmArgs& a = ta.g;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane & 15u, g = lane >> 4, wn = wave % WN, wm = wave / WN;
    // Workgroups are dealt to the 8 XCDs in turn: each XCD takes a run of
    // consecutive tiles, in panels of kPanel rows (m) with m fastest, so that
    // the workgroups it runs at once share few rows of x and of W in its L2.
    const uint32_t total = ta.mt * ta.nt, per = (total + 7u) / 8u;
    const uint32_t tile = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (tile >= total || (blockIdx.x >> 3) >= per) return;
    constexpr uint32_t kPT = kPanel / BM;
    const uint32_t p0 = tile / (kPT * ta.nt) * kPT, pm = min(kPT, ta.mt - p0);
    const uint32_t pt = tile - p0 * ta.nt, nb = pt / pm, mb = p0 + pt - nb * pm;
    const uint32_t n0 = nb * BN, m0 = mb * BM;
    const uint32_t tiles = a.k / kBK;

    // Staging: thread t moves chunks t + NT i; the chunk at position p of row
    // r holds chunk p ^ swizzle(r) of the row.  Rows past the matrix read its
    // last row (their outputs are not stored).
    const uint16_t* wp[WL];
    const uint8_t* xp[XL];
#pragma unroll
    for (int i = 0; i < WL; i++) {
        const uint32_t s = tid + NT * i, r = s >> 3, ch = (s & 7u) ^ swizzle<2>(r);
        wp[i] = a.w + static_cast<uint64_t>(min(n0 + r, a.n - 1u)) * a.k + 8u * ch;
    }
#pragma unroll
    for (int i = 0; i < XL; i++) {
        const uint32_t s = tid + NT * i, r = s / kPos, ch = (s % kPos) ^ swizzle<XE>(r);
        xp[i] = static_cast<const uint8_t*>(a.x) + static_cast<uint64_t>(min(m0 + r, a.m - 1u)) * a.k * XE + 16u * ch;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_offset(lds));
    auto request = [&](uint32_t st, int n) {  // the n-th load of a k-tile
        if (n < WL)
            dma16(wp[n], lds0 + st * kStage + (NT * n + 64u * wave) * 16u);
        else
            dma16(xp[n - WL], lds0 + st * kStage + kWB + (NT * (n - WL) + 64u * wave) * 16u);
    };
    uint32_t issued = 0;  // k-tiles requested; past the last one, the last again (the counts stay exact)
    auto advance = [&]() {
        const uint32_t step = ++issued < tiles ? kBK : 0u;
#pragma unroll
        for (int i = 0; i < WL; i++) wp[i] += step;
#pragma unroll
        for (int i = 0; i < XL; i++) xp[i] += step * XE;
    };
    constexpr uint32_t kFlush = DEEP && LO ? kChain / 2 : kChain;
    // A chain's sums are added between the first products of the next one, in
    // the products' shadow; of 16 outputs per lane in front of them (between
    // them 40 to 138 registers spilled).
    constexpr bool FOLD = NI * NJ <= 8;
    f32x4 d[NI][NJ], sum[NI][NJ], top[DEEP ? NI : 1][DEEP ? NJ : 1];
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            d[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (DEEP) top[i][j] = d[i][j];
        }
    auto flush = [&]() {
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) sum[i][j] += d[i][j];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto flush_top = [&]() {
        if constexpr (DEEP)
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    top[i][j] += sum[i][j];
                    sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
    };
#pragma unroll
    for (uint32_t st = 0; st < ST - 1; st++) {
#pragma unroll
        for (int n = 0; n < ND; n++) request(st, n);
        advance();
    }
    uint32_t rs = 0, qs = ST - 1;  // stage read, stage requested
    auto k_tile = [&](auto first_c) {
        constexpr bool first = decltype(first_c)::value;  // of a chain
        // This wave's part of the k-tile has landed (the ST - 2 tiles after it
        // stay in flight) and its reads of the last one, whose stage the next
        // requests overwrite, are complete; the barrier makes both true of
        // every wave.
        wait_vm<(ST - 2) * ND>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint8_t* wb = lds + rs * kStage + (BN / WN * wn + c) * 128u;
        const uint8_t* xb = lds + rs * kStage + kWB + BM / WM * wm * kXRow;
        u32x4 wv[2][NI];
        uint32_t xv[2][NJ][XW];
#pragma unroll
        for (uint32_t ks = 0; ks < 2; ks++) {
            const uint32_t u = 4u * ks + g;  // the lane's 8 k
#pragma unroll
            for (int j = 0; j < NJ; j++) read_x8<XT>(xb + 16u * j * kXRow, u, c, xv[ks][j]);
#pragma unroll
            for (int i = 0; i < NI; i++)
                wv[ks][i] = *reinterpret_cast<const u32x4*>(wb + 2048u * i + (u ^ swizzle<2>(c)) * 16u);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            v8 xh[NJ], xl[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) x_operands<XT, WF16>(xv[ks][j], xh[j], xl[j]);
#pragma unroll
            for (int i = 0; i < NI; i++) {
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    if (first && ks == 0) {
                        if constexpr (FOLD) sum[i][j] += d[i][j];
                        d[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                    d[i][j] = O::mfma(__builtin_bit_cast(v8, wv[ks][i]), xh[j], d[i][j]);
                    if constexpr (LO) d[i][j] = O::mfma(__builtin_bit_cast(v8, wv[ks][i]), xl[j], d[i][j]);
                }
#pragma unroll
                for (int n = 0; n < ND; n++)
                    if (n * 2 * NI / ND == ks * NI + i) request(qs, n);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        advance();
        rs = rs == ST - 1 ? 0u : rs + 1u;
        qs = qs == ST - 1 ? 0u : qs + 1u;
    };
    for (uint32_t kt = 0; kt < tiles; kt += kFlush) {
        if (DEEP && kt / kFlush % kChain2 == 1u) flush_top();
        if (!FOLD && kt) flush();
        k_tile(std::true_type{});
        for (uint32_t n = min(kFlush, tiles - kt) - 1u; n; n--) k_tile(std::false_type{});
    }
    flush();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the redundant last requests
    auto& out = [&]() -> auto& {
        if constexpr (DEEP) {
            flush_top();
            return top;
        } else {
            return sum;
        }
    }();
    // out[i][j]: n-tile i, m-tile j; lane (c, g) holds D[n = 4 g + r][m = c].
    const uint32_t nw = n0 + BN / WN * wn;             // the wave's first column
    if (nw >= a.n) return;
    const int ni = min((a.n - nw) / 16u, static_cast<uint32_t>(NI));
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const uint32_t row = m0 + BM / WM * wm + 16u * j + c;
        if (row >= a.m) continue;
        f32x4* yp = reinterpret_cast<f32x4*>(a.y + static_cast<uint64_t>(row) * a.n + nw + 4u * g);
        f32x4 old[NI];
        if (a.acc)
#pragma unroll
            for (int i = 0; i < NI; i++) old[i] = yp[4 * min(i, ni - 1)];
#pragma unroll
        for (int i = 0; i < NI; i++)
            if (i < ni) yp[4 * i] = a.acc ? out[i][j] + old[i] : out[i][j];
    }
}

// Few rows (decode; the gemv included): one workgroup per 16 output columns
// and all rows, its NW waves taking the k-chunks of 64 in turn.  What bounds
// it is the weight stream, and before that how fast one CU takes in its
// share: an operand read straight into registers touches 16 rows of 64 bytes
// per load, which the CU's address unit serves at 37 GB/s (L2-resident, same
// for any number of waves), a direct-to-LDS load of 8 rows of 128 bytes at
// 120-140 GB/s.  So both operands go through LDS: each wave keeps a ring of R
// chunks of its own ([16 W rows | 16 MT x rows], x in its own type, converted
// as it is read), waits for its own loads only, and the loop has no barrier.
// A chain of products spans kRowsChain chunks; the chains' sums add up in each
// wave, the waves' through LDS in wave order: one launch, no atomics,
// deterministic.  A wave requests no chunk past its last.
//
// Up to 16 rows W's loads are non-temporal, as each byte is read once: kept in
// L2 it would push out the code, tables and inputs of the kernels between two
// products (a captured layer of one row of 200 keys, head_dim 128: 22.5 us with
// W kept, 19.6 so; of f32 x 23.4, 20.8).  A W that the calls repeat stays in
// cache only with plain loads (16 rows 5.2 us, so 5.9; 1 row 4.4, 4.9): those of
// calls of more rows are plain, as 31 rows of f32 x a repeated W of 52 MiB lose
// too much (21.8, 28.2).
//
// Measured at k = n = 4096, each call with a W of its own, us per call (loads
// straight into registers before): 1 row of bf16 8.7 -> 7.1, 16 11.7 -> 8.0, 16
// of f32 15.2 -> 10.0, 32 18.9 -> 13.9; 896 x 896, 1 row of f32 3.7 -> 3.6.
constexpr uint32_t kRowsChain = 8, kCus = 256;

template <uint32_t XT, int MT, bool WIDE>
struct RowsShape {
    static constexpr uint32_t kXE = XT == THB_DT_F32 ? 4 : 2;
    static constexpr uint32_t kChunk = 2048u + 16u * MT * 64u * kXE;  // bytes of a chunk of W and x
    // 64 KiB of LDS for the smallest chunk (two workgroups per CU where n / 16
    // exceeds the CUs: 5120 columns at one row 15.2 -> 14.1 us), else three
    // chunks in flight of 8 waves or two of 4.  WIDE (n / 16 exceeds the CUs):
    // half the waves where that gives two workgroups per CU, so that one loads
    // while the other starts or ends (one row of f32 x, 65536 columns 116 -> 100
    // us, 32 rows of f16 x with bf16 W, 16384: 37 -> 26).
    static constexpr int NW = kChunk <= 4096 || (kChunk <= 6144 && !WIDE) ? 8 : 4;
    static constexpr int R = kChunk > 4096 && kChunk <= 6144 ? 3 : 2;
};

template <uint32_t XT, bool WF16, int MT, bool WIDE>
__global__ __launch_bounds__((64 * RowsShape<XT, MT, WIDE>::NW)) void gemm_rows(GemmArgs a) {
    using O = WOps<WF16>;
    using v8 = typename O::v8;
    using Sh = RowsShape<XT, MT, WIDE>;
    constexpr bool LO = needs_lo(XT, WF16);
    constexpr int XW = x_words(XT), NW = Sh::NW, R = Sh::R;
    constexpr uint32_t XE = Sh::kXE, kXRow = 64u * XE;     // bytes of a chunk's x row
    constexpr uint32_t kPos = kXRow / 16u, kRpl = 64u / kPos;  // 16-byte positions of it, x rows per load
    constexpr int XL = 16 * MT / kRpl, CN = 2 + XL;        // loads of x, of a chunk
    constexpr size_t kRing = static_cast<size_t>(R) * Sh::kChunk, kRed = sizeof(f32x4) * MT * 64;
    __shared__ __attribute__((aligned(16))) uint8_t lds[NW * (kRing > kRed ? kRing : kRed)];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane & 15u, g = lane >> 4, n0 = blockIdx.x * 16u;
    const uint32_t all = a.k / 64u, cnt = wave < all ? (all - wave + NW - 1u) / NW : 0u;
    // The accumulated y of the writing waves is requested first.
    f32x4 y_old[(MT + NW - 1) / NW];
#pragma unroll
    for (int t = 0; t < (MT + NW - 1) / NW; t++) {
        const uint32_t row = 16u * (wave + NW * t) + c;
        if (a.acc && row < a.m)
            y_old[t] = *reinterpret_cast<const f32x4*>(a.y + static_cast<uint64_t>(row) * a.n + n0 + 4u * g);
    }
    // Lane addresses of the loads at k = 0: W row 8 i + lane / 8, x row kRpl
    // i + lane / kPos, the 16 bytes whose position in LDS is the lane's,
    // swizzled so that the 16 rows of an operand read spread over the banks.
    const uint16_t* wp[2];
    const uint8_t* xp[XL];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t r = 8u * i + (lane >> 3);
        wp[i] = a.w + static_cast<uint64_t>(n0 + r) * a.k + 8u * ((lane & 7u) ^ swizzle<2>(r));
    }
#pragma unroll
    for (int i = 0; i < XL; i++) {
        const uint32_t r = kRpl * i + lane / kPos;
        const uint32_t pos = lane % kPos ^ swizzle<XE>(r);
        xp[i] = static_cast<const uint8_t*>(a.x) + static_cast<uint64_t>(min(r, a.m - 1u)) * a.k * XE + 16u * pos;
    }
    const uint32_t ring0 = __builtin_amdgcn_readfirstlane(lds_offset(lds)) + wave * static_cast<uint32_t>(kRing);
    // Chunk i of this wave.  The workgroups of an XCD (every eighth) start at
    // different chunks, so that they read different lines of x, and channels
    // of its L2, at once: by blockIdx.x itself they start at one or two where
    // cnt is a power of two (one row of bf16, k = 8192: 24.3 us, this 13.6).
    const uint32_t rot = cnt ? (blockIdx.x >> 3) % cnt : 0u;
    auto request = [&](uint32_t i, uint32_t slot) {
        const uint32_t ii = i + rot, j = ii >= cnt ? ii - cnt : ii;
        const uint64_t ke = static_cast<uint64_t>(wave + NW * j) * 64u;
        const uint32_t to = ring0 + slot * Sh::kChunk;
#pragma unroll
        for (int n = 0; n < 2; n++) dma16<MT == 1>(wp[n] + ke, to + 1024u * n);
#pragma unroll
        for (int n = 0; n < XL; n++) dma16(xp[n] + ke * XE, to + 2048u + 1024u * n);
    };
    // One chain per k-step of a chunk, added up every kRowsChain chunks.
    f32x4 d[2][MT], sum[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) d[0][t] = d[1][t] = sum[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto add_up = [&]() {
#pragma unroll
        for (int t = 0; t < MT; t++) {
            sum[t] += d[0][t] + d[1][t];
            d[0][t] = d[1][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    if (cnt != 0) {
#pragma unroll
        for (int i = 0; i < R; i++)
            if (static_cast<uint32_t>(i) < cnt) request(i, i);
        uint32_t slot = 0;
        auto chunk = [&](uint32_t i) {
            const bool more = i + R < cnt;
            if (i + R <= cnt)  // as many chunks after this one are in flight
                wait_vm<(R - 1) * CN>();
            else if (R == 3 && i + 1 < cnt)
                wait_vm<CN>();
            else
                wait_vm<0>();
            const uint8_t* wb = lds + wave * kRing + slot * Sh::kChunk;
            const uint8_t* xb = wb + 2048u;
            u32x4 wv[2];
            uint32_t xv[2][MT][XW];
#pragma unroll
            for (uint32_t ks = 0; ks < 2; ks++) {
                const uint32_t u = 4u * ks + g;  // the lane's 8 k
                wv[ks] = *reinterpret_cast<const u32x4*>(wb + c * 128u + (u ^ swizzle<2>(c)) * 16u);
#pragma unroll
                for (int t = 0; t < MT; t++) read_x8<XT>(xb + 16u * t * kXRow, u, c, xv[ks][t]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot is read: request into it
            if (more) request(i + R, slot);
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    v8 bh, bl;
                    x_operands<XT, WF16>(xv[ks][t], bh, bl);
                    d[ks][t] = O::mfma(__builtin_bit_cast(v8, wv[ks]), bh, d[ks][t]);
                    if constexpr (LO) d[ks][t] = O::mfma(__builtin_bit_cast(v8, wv[ks]), bl, d[ks][t]);
                }
            slot = slot == R - 1 ? 0u : slot + 1u;
        };
        for (uint32_t i0 = 0; i0 < cnt; i0 += kRowsChain) {
            for (uint32_t i = i0; i < min(i0 + kRowsChain, cnt); i++) chunk(i);
            add_up();
        }
    }
    // Lane (c, g) holds D[n = 4 g + r][m = c] of each m-tile: add the waves'
    // sums in order and write y[16 t + c][n0 + 4 g .. + 4].
    __syncthreads();  // every ring is idle: the sums take its place
    f32x4* red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int t = 0; t < MT; t++) red[(wave * MT + t) * 64u + lane] = sum[t];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < (MT + NW - 1) / NW; t++) {
        const uint32_t mt = wave + NW * t, row = 16u * mt + c;
        if (mt >= static_cast<uint32_t>(MT) || row >= a.m) continue;
        f32x4 s = red[mt * 64u + lane];
#pragma unroll
        for (int q = 1; q < NW; q++) s += red[(q * MT + mt) * 64u + lane];
        if (a.acc) s += y_old[t];
        *reinterpret_cast<f32x4*>(a.y + static_cast<uint64_t>(row) * a.n + n0 + 4u * g) = s;
    }
}

template <uint32_t XT, bool WF16, int BM, int BN, int WM, int WN, int ST, bool DEEP = false>
void launch_tile_as(const GemmArgs& a, hipStream_t s) {
    TileArgs ta;
    ta.g = a;
    ta.mt = (a.m + BM - 1) / BM;
    ta.nt = (a.n + BN - 1) / BN;
    const dim3 grid((ta.mt * ta.nt + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_tile<XT, WF16, BM, BN, WM, WN, ST, DEEP>), grid, dim3(64 * WM * WN), 0, s, ta);
}

// Tile shapes, largest first, and a shape's time per k-tile with one workgroup
// per CU.  launch_tile takes the shape with the shortest estimate, rounds of
// 256 workgroups x that time: a k-tile of a smaller shape costs less, but not
// in proportion (its LDS reads and requests per product grow), so the largest
// shape that fills the CUs wins.  Measured in us per call: 1500 x 5120 x 5120
// 90 on 128 x 256, 110 on 128 x 128, 140 on 128 x 64; 1000 x 4096 x 4096 59 /
// 42 / 57; 512 rows 58 / 39 / 29; 128 rows 59 / 39 / 28, 21 on 64 x 64, 17 on
// 64 x 32; 64 rows 14.4 on 64 x 32, 12.3 on 32 x 32; 32 rows 12.1 on 32 x 32,
// 10.2 on 32 x 16.
struct TileShape {
    uint32_t m, n;
    float us;
};
constexpr TileShape kShapes[] = {{128, 256, 1.1f}, {128, 128, 0.66f}, {128, 64, 0.44f}, {64, 64, 0.31f},
                                 {64, 32, 0.25f},  {32, 32, 0.185f},  {32, 16, 0.155f}};
// For an x that is converted (its waves own whole rows: no row is converted
// twice).
constexpr TileShape kShapesConv[] = {{128, 256, 2.3f}, {128, 128, 1.25f}, {64, 128, 0.85f}, {64, 64, 0.53f},
                                     {64, 32, 0.42f},  {32, 32, 0.39f}};
// Up to 64 rows: no wave of more than 8 outputs per lane, whose third level of
// sums would not fit the registers (64 x 65536 x 4096 of bf16 122 us on 64 x 64,
// 127 on 64 x 128, 132 on 64 x 256 and before, one chain on 128 x 256).
constexpr TileShape kDeep[] = {{64, 64, 0.31f}, {64, 32, 0.25f}, {32, 32, 0.185f}, {32, 16, 0.155f}};
constexpr TileShape kDeepConv[] = {{64, 128, 0.85f}, {64, 64, 0.53f}, {64, 32, 0.42f}, {32, 32, 0.39f}};

template <uint32_t XT, bool WF16>
void launch_tile(const GemmArgs& a, hipStream_t s) {
    auto best = [&](const auto& shapes) {
        int b = 0, i = 0;
        float us = INFINITY;
        for (const TileShape& t : shapes) {
            const uint64_t n = static_cast<uint64_t>((a.m + t.m - 1) / t.m) * ((a.n + t.n - 1) / t.n);
            const float e = static_cast<float>((n + 255) / 256) * t.us;
            if (e < us) {
                us = e;
                b = i;
            }
            i++;
        }
        return b;
    };
    constexpr bool F = XT == THB_DT_F32;
    if (a.m <= 64) {
        if constexpr (same_type(XT, WF16)) {
            switch (best(kDeep)) {
                case 0: return launch_tile_as<XT, WF16, 64, 64, 2, 2, 6, true>(a, s);
                case 1: return launch_tile_as<XT, WF16, 64, 32, 2, 1, 8, true>(a, s);
                case 2: return launch_tile_as<XT, WF16, 32, 32, 2, 2, 8, true>(a, s);
                default: return launch_tile_as<XT, WF16, 32, 16, 2, 1, 12, true>(a, s);
            }
        } else {
            switch (best(kDeepConv)) {
                case 0: return launch_tile_as<XT, WF16, 64, 128, 4, 1, 4, true>(a, s);
                case 1: return launch_tile_as<XT, WF16, 64, 64, 4, 1, F ? 5 : 6, true>(a, s);
                case 2: return launch_tile_as<XT, WF16, 64, 32, 4, 1, F ? 6 : 8, true>(a, s);
                default: return launch_tile_as<XT, WF16, 32, 32, 2, 1, F ? 6 : 8, true>(a, s);
            }
        }
    }
    if constexpr (same_type(XT, WF16)) {
        switch (best(kShapes)) {
            case 0: return launch_tile_as<XT, WF16, 128, 256, 2, 4, 3>(a, s);
            case 1: return launch_tile_as<XT, WF16, 128, 128, 2, 4, 4>(a, s);
            case 2: return launch_tile_as<XT, WF16, 128, 64, 2, 2, 4>(a, s);
            case 3: return launch_tile_as<XT, WF16, 64, 64, 2, 2, 6>(a, s);
            case 4: return launch_tile_as<XT, WF16, 64, 32, 2, 1, 8>(a, s);
            case 5: return launch_tile_as<XT, WF16, 32, 32, 2, 2, 8>(a, s);
            default: return launch_tile_as<XT, WF16, 32, 16, 2, 1, 12>(a, s);
        }
    } else {
        switch (best(kShapesConv)) {
            case 0: return launch_tile_as<XT, WF16, 128, 256, 4, 2, F ? 2 : 3>(a, s);
            case 1: return launch_tile_as<XT, WF16, 128, 128, 8, 1, F ? 3 : 4>(a, s);
            case 2: return launch_tile_as<XT, WF16, 64, 128, 4, 1, 4>(a, s);
            case 3: return launch_tile_as<XT, WF16, 64, 64, 4, 1, F ? 5 : 6>(a, s);
            case 4: return launch_tile_as<XT, WF16, 64, 32, 4, 1, F ? 6 : 8>(a, s);
            default: return launch_tile_as<XT, WF16, 32, 32, 2, 1, F ? 6 : 8>(a, s);
        }
    }
}

template <uint32_t XT, bool WF16, int MT>
void launch_rows(const GemmArgs& a, hipStream_t s) {
    auto go = [&](auto wide) {
        constexpr bool WIDE = decltype(wide)::value;
        hipLaunchKernelGGL((gemm_rows<XT, WF16, MT, WIDE>), dim3(a.n / 16), dim3(64 * RowsShape<XT, MT, WIDE>::NW), 0, s, a);
    };
    if constexpr (RowsShape<XT, MT, true>::NW != RowsShape<XT, MT, false>::NW)
        if (a.n / 16 > kCus) return go(std::true_type{});
    go(std::false_type{});
}

// gemm_rows reads all of x in every workgroup: up to 16 rows, where that is
// no more than its W.  Of an x that is converted, which gemm_tile's small
// shapes feed to their few waves slowly, up to a chunk of 10 KiB (64 rows of
// f16: 16.4 us against 24.2 on 32 x 32 tiles), and with the larger ones (33 to
// 64 rows of f32) where every workgroup has a CU of its own: 48 rows, 4096
// columns, k = 4096 18.1 us against 25.4, k = 8192 30 against 48; 5120 columns
// equal, 11008 38.6 against 31.4.
template <uint32_t XT, bool WF16>
void launch_gemm(const GemmArgs& a, hipStream_t s) {
    if (a.m <= 16) return launch_rows<XT, WF16, 1>(a, s);
    if constexpr (!same_type(XT, WF16)) {
        if (a.m <= 32) return launch_rows<XT, WF16, 2>(a, s);
        if (XT != THB_DT_F32 || a.n <= 16u * kCus) {
            if (a.m <= 48) return launch_rows<XT, WF16, 3>(a, s);
            if (a.m <= 64) return launch_rows<XT, WF16, 4>(a, s);
        }
    }
    launch_tile<XT, WF16>(a, s);
}

template <bool WF16>
void launch_w(uint32_t x_dt, const GemmArgs& a, hipStream_t s) {
    switch (x_dt) {
        case THB_DT_F32: launch_gemm<THB_DT_F32, WF16>(a, s); break;
        case THB_DT_F16: launch_gemm<THB_DT_F16, WF16>(a, s); break;
        default: launch_gemm<THB_DT_BF16, WF16>(a, s); break;
    }
}

}  // namespace
}  // namespace thb

using namespace thb;

extern "C" {

int thb_check_gemm_dims(uint32_t n, uint32_t k) {
    // ops::check_gemm_dims (crates/thuban_model/src/ops/gemm.rs:133-146)
    if (n % 16 != 0 || k % 64 != 0)
        return fail(THB_ERR_CONFIG, "dimension pair (N=" + std::to_string(n) + ", K=" + std::to_string(k) +
                                        ") does not satisfy N%16 and K%64");
    return THB_OK;
}

int thb_gemm_acc(const void* x, uint32_t x_dtype, const void* w, uint32_t w_dtype, float* y, uint32_t rows,
                 uint32_t n, uint32_t k, uint32_t acc, void* stream) {
    if (int rc = thb_check_gemm_dims(n, k)) return rc;
    if (rows == 0 || n == 0 || k == 0) return THB_OK;
    if (!x || !w || !y) return fail(THB_ERR_INVALID, "null x, w or y");
    if (x_dtype > THB_DT_BF16) return fail(THB_ERR_INVALID, "unknown x_dtype " + std::to_string(x_dtype));
    if (w_dtype != THB_DT_BF16 && w_dtype != THB_DT_F16)
        return fail(THB_ERR_INVALID, "weights must be THB_DT_BF16 or THB_DT_F16 (w_dtype " + std::to_string(w_dtype) +
                                         ")");
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y)) & 15u)
        return fail(THB_ERR_INVALID, "x, w and y must be 16-byte aligned");
    if (static_cast<uint64_t>(rows) * k >= (1ull << 40) || static_cast<uint64_t>(n) * k >= (1ull << 40))
        return fail(THB_ERR_INVALID, "gemm operands too large");
    return guarded([&]() -> int {
        GemmArgs a;
        a.x = x;
        a.w = static_cast<const uint16_t*>(w);
        a.y = y;
        a.m = rows;
        a.n = n;
        a.k = k;
        a.acc = acc ? 1u : 0u;
        hipStream_t s = as_stream(stream);
        if (w_dtype == THB_DT_F16)
            launch_w<true>(x_dtype, a, s);
        else
            launch_w<false>(x_dtype, a, s);
        THB_HIP(hipGetLastError());
        return THB_OK;
    });
}

}  // extern "C"
