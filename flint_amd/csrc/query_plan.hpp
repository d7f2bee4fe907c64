// The host planner's geometry of a call: the rows' key ranges, the query
// groups and the prefill blocks.  Host code without HIP, so that
// tests/test_prefill_plan.py pins it on the CPU.
#pragma once

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

#include "../../include/thuban_hip.h"
#include "partition.hpp"

namespace thb {

constexpr uint32_t kCols = 16;        // query vectors per group (MFMA N)
constexpr uint32_t kGroupWords = 11;  // r0, R, h0, H, seq, lo, hi, n_parts, base, plen, item0
constexpr uint32_t kBlockWords = 9;   // g0, ng, seq, lo, hi, n_parts, base, plen, bitem0

// Per-row key ranges (attn.wgsl:78-88,169).  A chunk is the whole call when
// the sequence is fixed (reference mode, one dispatch per sequence chunk,
// forward.rs:316-336), else each maximal run of rows with equal seq.
struct RowPlan {
    std::vector<uint32_t> lo, hi, seq;
    std::vector<std::pair<uint32_t, uint32_t>> chunks;  // [start, end)
};

inline RowPlan plan_rows(const uint32_t* args, uint32_t m, uint32_t seq_fixed, bool causal, uint32_t window) {
    RowPlan rp;
    rp.lo.resize(m);
    rp.hi.resize(m);
    rp.seq.resize(m);
    uint32_t start = 0;
    while (start < m) {
        const uint32_t seq = seq_fixed != THB_SEQ_PER_ROW ? seq_fixed : args[8 * start + 1];
        uint32_t end = start + 1;
        if (seq_fixed == THB_SEQ_PER_ROW)
            while (end < m && args[8 * end + 1] == seq) end++;
        else
            end = m;
        const uint32_t n = end - start;
        for (uint32_t i = 0; i < n; i++) {
            const uint32_t r = start + i;
            const uint32_t pos = args[8 * r];
            const uint32_t blk_last = std::min((i / 8) * 8 + 8, n);
            const uint64_t kv_len = causal ? uint64_t(args[8 * (start + blk_last - 1)]) + 1
                                           : uint64_t(args[8 * (end - 1)]) + 1;
            uint64_t ws = 0;
            if (causal && window != 0 && uint64_t(pos) + 1 > window) ws = uint64_t(pos) + 1 - window;
            uint64_t h = kv_len;
            if (causal && uint64_t(pos) + 1 < h) h = uint64_t(pos) + 1;
            rp.lo[r] = static_cast<uint32_t>(ws);
            rp.hi[r] = static_cast<uint32_t>(std::min<uint64_t>(h, 0xFFFFFFFFull));
            rp.seq[r] = seq;
        }
        rp.chunks.push_back({start, end});
        start = end;
    }
    return rp;
}

// The query groups and prefill blocks of a call's rows.
struct QueryPlan {
    std::vector<uint32_t> groups, blocks;  // kGroupWords, kBlockWords each
    std::vector<uint8_t> in_block;         // by group: a block's member
    uint32_t max_parts = 0;
    uint64_t max_span = 0;
    bool any_split = false;
};

// Partitions of a group (or of a prefill block) start at its first key
// (rounded down to the page and tile size) and split its span into
// n equal parts (part_split: n = ceil(span / part_len) rounded up to a
// power of two, then lowered if the aligned part length leaves trailing
// parts empty): a function of its own key range only.  G: query heads per KV
// head; PL: part_len; align: a part's length is a multiple of it; WB: query
// groups per block.
inline QueryPlan plan_groups(const RowPlan& rp, uint32_t G, uint32_t PL, uint32_t align, uint32_t WB) {
    QueryPlan qp;
    auto& groups = qp.groups;
    auto& blocks = qp.blocks;
    auto& in_block = qp.in_block;
    auto partition = [&](uint32_t& lo, uint32_t& hi, uint32_t& base, uint32_t& n_parts, uint32_t& plen) {
        base = 0;
        n_parts = 1;
        plen = align;
        if (hi <= lo || lo == 0xFFFFFFFFu) {
            lo = hi = 0;  // no keys: one empty partition, output 0/0 = NaN
        } else {
            base = lo & ~(align - 1);
            const uint64_t span = uint64_t(hi) - base;
            qp.max_span = std::max(qp.max_span, span);
            part_split(span, PL, align, n_parts, plen);
        }
        qp.max_parts = std::max(qp.max_parts, n_parts);
        qp.any_split = qp.any_split || n_parts > 1;
    };
    auto add_group = [&](uint32_t r0, uint32_t R, uint32_t h0, uint32_t H, uint32_t seq) {
        uint32_t lo = 0xFFFFFFFFu, hi = 0;
        for (uint32_t r = r0; r < r0 + R; r++) {
            if (rp.hi[r] <= rp.lo[r]) continue;
            lo = std::min(lo, rp.lo[r]);
            hi = std::max(hi, rp.hi[r]);
        }
        uint32_t base, n_parts, plen;
        partition(lo, hi, base, n_parts, plen);
        groups.insert(groups.end(), {r0, R, h0, H, seq, lo, hi, n_parts, base, plen, 0u});
    };
    // A chunk that needs at least 4 groups (a prefill chunk) is cut into
    // blocks of WB consecutive groups for attn_prefill; the others go to the
    // decode kernel.
    for (auto& c : rp.chunks) {
        const uint32_t seq = rp.seq[c.first];
        const uint32_t first = static_cast<uint32_t>(groups.size() / kGroupWords);
        if (G <= kCols) {
            const uint32_t rg = kCols / G;
            for (uint32_t r = c.first; r < c.second; r += rg) add_group(r, std::min(rg, c.second - r), 0, G, seq);
        } else {
            for (uint32_t r = c.first; r < c.second; r++)
                for (uint32_t h0 = 0; h0 < G; h0 += kCols) add_group(r, 1, h0, std::min(kCols, G - h0), seq);
        }
        const uint32_t ncg = static_cast<uint32_t>(groups.size() / kGroupWords) - first;
        in_block.resize(first + ncg, 0);
        if (G > kCols || ncg < 4) continue;
        for (uint32_t b = 0; b < ncg; b += WB) {
            const uint32_t g0 = first + b, ng = std::min(WB, ncg - b);
            uint32_t lo = 0xFFFFFFFFu, hi = 0;
            for (uint32_t g = g0; g < g0 + ng; g++) {
                const uint32_t* gr = &groups[static_cast<size_t>(g) * kGroupWords];
                in_block[g] = 1;
                if (gr[6] <= gr[5]) continue;
                lo = std::min(lo, gr[5]);
                hi = std::max(hi, gr[6]);
            }
            uint32_t base, n_parts, plen;
            partition(lo, hi, base, n_parts, plen);
            for (uint32_t g = g0; g < g0 + ng; g++) {  // members share the block's partitions
                uint32_t* gr = &groups[static_cast<size_t>(g) * kGroupWords];
                gr[7] = n_parts;
                gr[8] = base;
                gr[9] = plen;
            }
            blocks.insert(blocks.end(), {g0, ng, seq, lo, hi, n_parts, base, plen, 0u});
        }
    }
    return qp;
}

// Few blocks leave CUs idle: cut them into smaller ones (waves without a
// group of their own only load) while those still run in one round beside
// the call's decode items.  A smaller block keeps its parent's partitions,
// and 32-key steps start at multiples of 32, so no column's arithmetic
// changes (a partition may hold no key of a smaller block: that work item
// runs no tile, block_keys).  A block's time is its serial chain over the
// keys, which shrinks with its groups (64 keys of head_dim 128, f32 queries:
// 3.2 us with 10 groups, two in some waves, 2.6 with 8 or fewer), and short
// chunks need several CUs per KV head.
// Measured, us per call, uncut / cut (8 KV heads of 128 x 4): one chunk of
// 100 rows 23.5 / 10.0, 512 42.5 / 24.7, 1000 64.6 / 44.2; 200 rows after
// 3000 keys (f32 queries) 323 / 130; four chunks of 250 32.9 / 17.7;
// head_dim 256 x 2, 777 rows after 3001 keys 412 / 177, and 232 where the
// cut stops at 8 groups.  A cut into more than one round gains nothing: what
// runs second waits for the first.
// dec: decode work items of the same launch.
inline void cut_blocks(QueryPlan& qp, uint32_t WB, uint64_t dec, uint32_t kv_heads, uint32_t cus) {
    const auto& groups = qp.groups;
    auto& blocks = qp.blocks;
    auto count = [&](uint32_t bg) {
        uint64_t n = 0;
        for (size_t b = 0; b < blocks.size(); b += kBlockWords)
            n += static_cast<uint64_t>((blocks[b + 1] + bg - 1) / bg) * blocks[b + 5];
        return n;
    };
    uint32_t bg = WB;
    while (bg > 1 && (dec + count(bg / 2)) * kv_heads <= cus) bg /= 2;
    if (bg < WB) {
        std::vector<uint32_t> cut;
        for (size_t b = 0; b < blocks.size(); b += kBlockWords) {
            const uint32_t* bk = &blocks[b];
            for (uint32_t g = bk[0]; g < bk[0] + bk[1]; g += bg) {
                const uint32_t ng = std::min(bg, bk[0] + bk[1] - g);
                uint32_t lo = 0xFFFFFFFFu, hi = 0;
                for (uint32_t i = g; i < g + ng; i++) {
                    const uint32_t* gr = &groups[static_cast<size_t>(i) * kGroupWords];
                    if (gr[6] <= gr[5]) continue;
                    lo = std::min(lo, gr[5]);
                    hi = std::max(hi, gr[6]);
                }
                if (hi <= lo) lo = hi = 0;
                cut.insert(cut.end(), {g, ng, bk[2], lo, hi, bk[5], bk[6], bk[7], 0u});
            }
        }
        blocks.swap(cut);
    }
}

}  // namespace thb
