"""Runs the host planner's geometry (flint_amd/csrc/query_plan.hpp and
partition.hpp) on the CPU, for tests that ask which form a call takes."""

import functools
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "query_plan.hpp"
using namespace thb;
// heads per KV head, KV heads, head_dim, page, part_len, window, rows, then (position, sequence) of each:
// build_plan's choice for a causal call (plan.spread)
int main() {
    unsigned G, kvh, hd, page, part_len, window, m;
    while (std::scanf("%u %u %u %u %u %u %u", &G, &kvh, &hd, &page, &part_len, &window, &m) == 7) {
        std::vector<uint32_t> args(8 * m, 0);
        for (uint32_t i = 0; i < m; i++)
            if (std::scanf("%u %u", &args[8 * i], &args[8 * i + 1]) != 2) return 1;
        const RowPlan rp = plan_rows(args.data(), m, THB_SEQ_PER_ROW, true, window);
        const QueryPlan qp = plan_groups(rp, G, part_len, page > 16 ? page : 16, hd > 128 ? 8 : 16);
        uint64_t items = 0, keys = 0;
        uint32_t cols = 0;
        for (size_t g = 0; g < qp.in_block.size(); g++) {
            const uint32_t* gr = &qp.groups[g * kGroupWords];
            if (qp.in_block[g]) continue;
            items += gr[7];
            keys = std::max<uint64_t>(keys, std::min(gr[9], gr[6] - gr[8]));
            cols = std::max(cols, gr[1] * gr[3]);
        }
        std::printf("%d\n", int(items && qp.blocks.empty() && spread_head_dim(hd, page) &&
                                spread_rule(hd, cols, items, kvh, keys, qp.max_parts)));
    }
    return 0;
}
"""


@functools.lru_cache(None)
def _exe():
    d = tempfile.mkdtemp(prefix="plan")
    src, exe = os.path.join(d, "plan.cpp"), os.path.join(d, "plan")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__host__=", "-D__device__=", "-I",
                    os.path.join(ROOT, "flint_amd", "csrc"), src, "-o", exe], check=True)
    return exe


def takes_spread(g, kv_heads, head_dim, page, part_len, window, positions, seqs):
    """Whether a causal, host-planned call runs one wave per workgroup."""
    call = [g, kv_heads, head_dim, page, part_len or 4096, window, len(positions)]
    call += [x for p in zip(positions, seqs) for x in p]
    out = subprocess.run([_exe()], input=" ".join(map(str, call)), capture_output=True, text=True, check=True).stdout
    return out.strip() == "1"
