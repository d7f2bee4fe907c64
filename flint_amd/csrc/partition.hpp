// Split-K partitions of a key span and the rule for decode calls of few items,
// shared by the host planner and the device planner (and pinned on the CPU by
// tests/test_abi.py, tests/test_prefill_plan.py).
#pragma once

#include <cstdint>

namespace thb {

// Partitions of a key span (a function of the span only, so a group's
// arithmetic does not depend on the rest of the call): ceil(span / PL)
// rounded up to a power of two, as n_parts equal pieces of plen keys (a
// multiple of align), the last one shorter.  A span at most PL / 64 per
// piece over k * PL (k >= 2) counts as k pieces, each up to PL + PL / 64
// long: Gemma-2's global layers (8192 + 4 keys) then take 2 partitions
// instead of 4, one round of workgroups instead of two.  (k = 1 keeps two
// pieces: a span just over PL on one piece would leave half the CUs idle
// where a call holds few groups.)  Rounding down in general (pieces up to
// ~2 PL) measured faster on those layers and slower on the ragged Qwen3
// batch and the 131072-token Qwen2.5 contexts.
__host__ __device__ inline void part_split(uint64_t span, uint32_t PL, uint32_t align, uint32_t& n_parts,
                                           uint32_t& plen) {
    uint32_t n = static_cast<uint32_t>((span + PL - 1) / PL);
    const uint64_t k = span / PL;
    if (n > 2 && span - k * PL <= k * (PL / 64)) n = static_cast<uint32_t>(k);
    if (n > 1) n = 1u << (32 - __builtin_clz(n - 1));
    plen = static_cast<uint32_t>(((span + n - 1) / n + align - 1) / align * align);
    n_parts = static_cast<uint32_t>((span + plen - 1) / plen);
}

// part_split for 0 < span < 2^31 and a power-of-two align, in 32-bit
// arithmetic with shifts for the power-of-two divisors (n and align): the
// device planner's form (a 64-bit division is a long instruction sequence
// on the GPU).  Same results as part_split.
__host__ __device__ inline void part_split32(uint32_t span, uint32_t PL, uint32_t align, uint32_t& n_parts,
                                             uint32_t& plen) {
    const uint32_t k = span / PL;
    uint32_t n = k + (span - k * PL != 0 ? 1u : 0u);
    if (n > 2 && span - k * PL <= k * (PL / 64)) n = k;
    uint32_t sh = 0;
    if (n > 1) {
        sh = 32 - __builtin_clz(n - 1);
        n = 1u << sh;
    }
    plen = (((span + n - 1) >> sh) + align - 1) & ~(align - 1);
    n_parts = (span + plen - 1) / plen;
}

// Keys [tb, te) of a prefill block's range [lo, hi) in its partition of plen
// keys from pbeg: the work item's first 32-key step and its tiles of `tile`
// keys.  No tile without a key: a block cut from a larger one keeps its
// partitions, whose pages an item that holds none of them must not look up.
struct BlockKeys {
    uint32_t tb, te, first, tiles;
};
__host__ __device__ inline BlockKeys block_keys(uint32_t lo, uint32_t hi, uint32_t pbeg, uint32_t plen,
                                                uint32_t tile) {
    BlockKeys k;
    k.tb = lo > pbeg ? lo : pbeg;
    k.te = hi < pbeg + plen ? hi : pbeg + plen;
    k.first = k.tb & ~31u;
    k.tiles = k.te > k.tb ? (k.te - k.first + tile - 1) / tile : 0u;
    return k;
}

// Items x KV heads that a spread launch takes at most.
constexpr uint32_t kSpreadMax = 64;

// Whether n_items decode items x n_kvh KV heads, of up to `cols` query vectors
// and `parts` partitions a group, whose longest holds `keys` keys, run one wave
// per workgroup (attn_spread, attn_pick): when they leave three quarters of the
// 256 CUs idle and are long enough to pay for the wave states' way through
// memory (~1.3 us, more where a state is larger than 4 KiB).  Measured, us per
// fused call, one workgroup per item / one per wave (8 KV heads of 128, 4
// columns): one sequence of 512 keys 10.2 / 10.4, 1000 13.2 / 12.3, 4000 34.9 /
// 21.5; eight (64 items) 512 10.4 / 12.4, 1000 14.0 / 14.5, 2000 25.0 / 19.5;
// 128 items of 2000 28.5 / 36.  head_dim 64, 7 columns, 8 items: 1000 10.4 /
// 10.6, 2000 14.3 / 12.6; 256, 2 columns, 8 items: 256 11.7 / 10.6, 4000 63.6 /
// 32; 256, 8 columns (8 KiB states), 16 items: 512 18.3 / 20.5, 2000 38.7 /
// 31.9.  (One per wave with plain loads, here and below; non-temporal ones take
// up to 13 % less above ~1500 keys and the same on short items.)
//
// More than half of 64 items, or states of more than 4 KiB, need longer items:
// 2 rows x 4 columns, rotated, 1500 keys: 32 items 21.3 / 20.9, 48 23.3 / 24.3,
// 64 24.7 / 25.4; 64 of 5 columns, 1800 keys 25.5 / 21.6.  Where an item's keys
// are split into parts, one workgroup combines the waves' states of all parts,
// a serial chain that grows with parts x columns: head_dim 128, parts of 3900
// keys: 4 columns x 2 38.7 / 28.2, x 4 45.3 / 32.7, x 8 49.5 / 41.2; 8 columns
// x 2 39.0 / 34.6, x 4 45.6 / 41.5 (a gated call of two sequences with parts of
// ~3000 keys 45.0 / 48.5), x 8 50.3 / 54.9; 16 columns x 2 44.5 / 44.9, x 4
// 51.8 / 56.9.  head_dim 256: 4 columns x 4 82.6 / 46.2, 8 x 2 75.9 / 45.8; 64:
// 7 x 4 28.8 / 24.0, x 8 30.7 / 30.7.
__host__ __device__ inline bool spread_rule(uint32_t hd, uint32_t cols, uint64_t n_items, uint32_t n_kvh,
                                            uint64_t keys, uint32_t parts) {
    const uint64_t wgs = n_items * n_kvh;
    const uint64_t least = (cols * hd > 1024 ? 256u : wgs > kSpreadMax / 2 ? 208u : 128u) * 1024u;
    if (parts > 1 && parts * cols > (cols * hd <= 512 ? 32u : 16u)) return false;
    return wgs <= kSpreadMax && keys * hd >= least;
}
// The layers and pages the spread form takes.
inline bool spread_head_dim(uint32_t hd, uint32_t page_len) {
    return (hd == 64 || hd == 128 || hd == 256) && page_len >= 16;
}

}  // namespace thb
