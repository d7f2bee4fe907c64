"""The host planner's prefill blocks (flint_amd/csrc/query_plan.hpp and
block_keys of partition.hpp, what build_plan and the prefill kernel use),
without a GPU: a block cut into smaller ones keeps its groups' partitions, so
a partition may hold no key of a smaller block.  Its work item then has no
tile; every other item's tiles cover exactly the keys its groups read there,
and every key they load lies in the partition, whose staged pages they index."""

import os
import random
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "query_plan.hpp"
using namespace thb;
int main() {
    unsigned page, part_len, kvh, G, WB, window, causal, prefix, chunk, tile;
    while (std::scanf("%u %u %u %u %u %u %u %u %u %u", &page, &part_len, &kvh, &G, &WB, &window, &causal, &prefix,
                      &chunk, &tile) == 10) {
        std::vector<uint32_t> args(8 * chunk, 0);
        for (uint32_t i = 0; i < chunk; i++) args[8 * i] = prefix + i;
        const RowPlan rp = plan_rows(args.data(), chunk, THB_SEQ_PER_ROW, causal, window);
        QueryPlan qp = plan_groups(rp, G, part_len, page > 16 ? page : 16, WB);
        const size_t uncut = qp.blocks.size();
        if (!qp.blocks.empty()) cut_blocks(qp, WB, 0, kvh, 256);
        std::printf("call %d\n", int(qp.blocks.size() > uncut));
        for (size_t b = 0; b < qp.blocks.size(); b += kBlockWords) {
            const uint32_t* B = &qp.blocks[b];
            for (uint32_t p = 0; p < B[5]; p++) {
                const uint32_t pbeg = B[6] + p * B[7];
                const BlockKeys k = block_keys(B[3], B[4], pbeg, B[7], tile);
                // the keys the item's groups read in this partition
                uint32_t lo = 0xFFFFFFFFu, hi = 0, same = 1;
                for (uint32_t g = B[0]; g < B[0] + B[1]; g++) {
                    const uint32_t* gr = &qp.groups[g * kGroupWords];
                    same &= gr[7] == B[5] && gr[8] == B[6] && gr[9] == B[7];
                    const uint32_t gl = std::max(gr[5], pbeg), gh = std::min(gr[6], pbeg + B[7]);
                    if (gl < gh) { lo = std::min(lo, gl); hi = std::max(hi, gh); }
                }
                std::printf("%u %u %u %u %u %u %u %u %u\n", pbeg, B[7], k.tb, k.te, k.first, k.tiles, lo, hi, same);
            }
        }
    }
    return 0;
}
"""

# page, part_len, kv heads, q heads per kv head, groups per block, window, causal, prefix, chunk, keys per tile
KNOWN = [
    # partitions of 528 keys; the last one starts 6 keys before the chunk's end
    (16, 1024, 2, 4, 16, 0, 1, 33226, 64, 64),
    (16, 2048, 1, 5, 16, 0, 1, 152366, 48, 64),
    (16, 4096, 1, 1, 16, 0, 1, 266050, 256, 64),
    # partitions of 48 keys, one group per block
    (16, 64, 8, 4, 16, 0, 1, 20, 64, 64),
    (16, 128, 8, 1, 16, 0, 1, 0, 200, 64),
    # a window: the last blocks hold no key of the first partition
    (16, 64, 8, 4, 16, 60, 1, 100, 64, 64),
    (8, 64, 4, 2, 8, 100, 1, 37, 129, 64),
]


def _plan(tmp_path, cases):
    src = tmp_path / "plan.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "plan"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__host__=", "-D__device__=", "-I",
                    os.path.join(ROOT, "flint_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, c)) for c in cases), capture_output=True,
                         text=True, check=True).stdout
    calls = []
    for line in out.splitlines():
        if line.startswith("call"):
            calls.append((line.endswith("1"), []))
        else:
            calls[-1][1].append(tuple(map(int, line.split())))
    assert len(calls) == len(cases)
    return calls


def test_prefill_items_load_only_keys_of_their_partition(tmp_path):
    rng = random.Random(3)
    cases = list(KNOWN)
    for _ in range(4000):
        g = rng.choice([1, 2, 3, 4, 5, 7, 8, 16])
        part_len = rng.choice([32, 64, 128, 256, 1024, 4096])
        cases.append((rng.choice([8, 16, 16, 32]), part_len, rng.choice([1, 2, 4, 8]), g, rng.choice([8, 16]),
                      rng.choice([0, 0, rng.randrange(1, 4 * part_len)]), int(rng.random() < 0.9),
                      rng.choice([0, rng.randrange(0, 30 * part_len)]), rng.randrange(1, 700), 64))
    without_keys = cuts = 0
    for case, (cut, items) in zip(cases, _plan(tmp_path, cases)):
        cuts += cut
        for pbeg, plen, tb, te, first, tiles, lo, hi, same in items:
            item = (case, pbeg, plen, tb, te, first, tiles)
            assert same, item
            if lo >= hi:  # no query of the block reads a key here
                without_keys += 1
                assert tiles == 0, item
                continue
            assert tiles > 0 and pbeg <= tb <= lo and hi <= te <= pbeg + plen, item
            assert first <= tb < first + 32 and first % 32 == 0, item
            assert first + tiles * case[9] >= te > first + (tiles - 1) * case[9], item
    assert cuts > 1000 and without_keys > 100, (cuts, without_keys)


def test_known_calls_reach_partitions_without_keys(tmp_path):
    """Each of these calls is cut so that some block has no key in one of its
    partitions (the items are checked by the sweep above)."""
    for case, (cut, items) in zip(KNOWN, _plan(tmp_path, KNOWN)):
        assert cut and any(lo >= hi for *_, lo, hi, _ in items), case
