"""A prefill call of few blocks is cut into smaller ones, unpaired, to reach
more CUs.  The cut keeps every query's partitions and 32-key steps, so a
chunk's outputs are the same bits alone (cut) and beside enough other chunks
that nothing is cut and blocks run as pairs; and they are the oracle's exact
softmax.  Blocks of at most 8 groups run one group on each wave at head_dim <=
128, the batch's blocks two: the same bits, in each form of the query (f16,
rotated, f32).  Sizes: last groups with fewer rows or heads than a tile, chunks
just above the decode kernel's, one short of and one past a block, a prefix,
windows, soft-cap, several partitions, and no causal mask."""

import math
import random

import pytest

import oracle
from gpu_util import fill, make_pool, oracle_layer, say, scattered_alloc

pytestmark = pytest.mark.gpu

# name, head_dim, kv heads, q heads per kv head, page, kv type, part_len, window, softcap, causal, chunk, prefix
CASES = [
    ("hd128-four-groups", 128, 8, 4, 16, "f16", 0, 0, 0.0, True, 13, 0),
    ("hd128-block-and-one-row", 128, 8, 4, 16, "f16", 0, 0, 0.0, True, 65, 300),
    ("hd128-block-less-one-bf16", 128, 4, 4, 32, "bf16", 0, 0, 0.0, True, 63, 1),
    ("hd128-window-parts", 128, 4, 8, 16, "f16", 1024, 1500, 0.0, True, 77, 2900),
    ("hd128-all-keys", 128, 4, 5, 16, "bf16", 0, 0, 0.0, False, 70, 500),
    ("hd64-seven-columns", 64, 2, 7, 16, "f16", 0, 0, 0.0, True, 101, 33),
    ("hd64-parts", 64, 4, 1, 16, "f16", 1024, 0, 0.0, True, 200, 2000),
    ("hd256-softcap-window", 256, 4, 2, 16, "f16", 0, 333, 50.0, True, 129, 700),
    ("hd256-parts-bf16", 256, 4, 4, 32, "bf16", 1024, 0, 30.0, True, 40, 2100),
    ("hd64-softcap-bf16", 64, 4, 4, 16, "bf16", 0, 0, 30.0, True, 45, 100),
    # smaller blocks with no key in one of their partitions, before or after it
    ("hd128-parts-without-keys", 128, 8, 4, 16, "f16", 64, 0, 0.0, True, 64, 20),
    ("hd128-parts-without-keys-window", 128, 8, 4, 16, "f16", 64, 60, 0.0, True, 64, 100),
    ("hd64-parts-without-keys", 64, 8, 1, 16, "bf16", 128, 0, 0.0, True, 200, 0),
    # no second item, and a range from an odd 16 keys, where the page list begins
    ("hd128-window-from-16", 128, 8, 4, 16, "f16", 0, 100, 0.0, True, 64, 115),
    ("hd80-ragged", 80, 4, 3, 16, "f16", 0, 0, 0.0, True, 50, 61),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_chunk_alone_matches_chunk_in_a_batch(torch_cuda, case):
    torch = torch_cuda
    from flint_amd import ops
    from flint_amd.pool import RowMeta
    from flint_amd.rope import Rope

    name, hd, nkv, g, page, kv, part_len, window, cap, causal, chunk, prefix = case
    say("prefill cut", name)
    # Others: chunks of one block each, so that blocks * kv heads exceeds two
    # rounds of the CUs.
    others = 1024 // nkv
    per = 64
    lens = [prefix + chunk] + [per] * others
    pool = make_pool(lens, kv_heads=nkv, head_dim=hd, page_len=page, kv_dtype=kv, part_len=part_len)
    scattered_alloc(pool, lens, random.Random(11), page)
    fill(torch, pool, RowMeta(4096), lens, seed=3)
    pos = [prefix + i for i in range(chunk)] + [i for _ in range(others) for i in range(per)]
    seq = [0] * chunk + [1 + s for s in range(others) for _ in range(per)]
    nq = g * nkv
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    q = torch.randn(len(pos), nq, hd, device="cuda", generator=gen)
    for rope, dt in ((None, torch.float16), (Rope.from_theta(max(lens), hd, 1e4), torch.float32), (None, torch.float32)):
        out = []
        for m in (chunk, len(pos)):
            rows = RowMeta(m)
            rows.write(pos[:m], seq[:m])
            y = torch.full((m, nq, hd), 7.0, device="cuda")
            spec = ops.AttnSpec(q_heads=nq, window=window, scale=1.5 / math.sqrt(hd), m=m, causal=causal, seq=None,
                                args=rows, softcap=cap)
            ops.attn_step(pool, 0, spec, q[:m].to(dt).contiguous(), y, rope=rope)
            torch.cuda.synchronize()
            out.append(y[:chunk])
        assert torch.equal(out[0], out[1]), (name, dt, float((out[0] - out[1]).abs().max()))
    want = oracle_layer(torch, pool).attn(q[:chunk].cpu().numpy(), oracle.row_meta(pos[:chunk], seq[:chunk]), chunk,
                                          nq, spec.scale, window=window, softcap=cap, causal=causal)
    err = float(abs(out[0].cpu().numpy() - want).max())
    say(name, "max abs err vs oracle", err)
    # f32 queries and probabilities go through the matrix cores as exact 16-bit
    # halves: only f32 rounding of sums of a few thousand terms is left.
    assert err <= 1e-4, (name, err)
