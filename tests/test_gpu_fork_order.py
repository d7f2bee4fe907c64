"""Decode over forked sequences: work items whose keys lie in the same pages
follow one another in the launch.  The order changes no result: forks that
share a prefix give the same bits as sequences of the same keys in pages of
their own, over several partitions, forks of different lengths, sequences that
share nothing between them, query groups split over the heads, the fused
append, a prefill chunk beside them, and repeated launches."""

import math

import pytest

from gpu_util import make_pool, say

pytestmark = pytest.mark.gpu

# name, head_dim, kv heads, q heads per kv head, page, kv type, part_len, rows per sequence, chunk rows
CASES = [
    ("hd128-parts", 128, 8, 4, 16, "f16", 1024, 1, 0),
    ("hd128-verify-bf16", 128, 2, 4, 32, "bf16", 0, 3, 0),
    ("hd64-mixed", 64, 2, 7, 16, "f16", 1024, 1, 90),
    ("hd128-heads-split", 128, 1, 24, 16, "f16", 1024, 1, 0),
    ("hd256-parts", 256, 4, 2, 16, "bf16", 1024, 1, 0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_forks_match_unshared_sequences(torch_cuda, case):
    torch = torch_cuda
    from flint_amd import ops
    from flint_amd.pool import RowMeta

    name, hd, nkv, g, page, kv, part_len, rps, chunk = case
    say("fork order", name)
    # Sequence 0 and 2 are sources; 1, 4, 5 fork 0 (5 after its first 1500
    # tokens), 3 forks 2; 6 holds the prefill chunk.
    src = {0: 2500, 2: 1900}
    forks = {1: (0, 2500), 4: (0, 2500), 5: (0, 1500), 3: (2, 1900)}
    lens = [src[s] if s in src else forks[s][1] for s in range(6)]
    budget = [n + rps for n in lens] + [max(chunk, 1)]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(21)
    data = {s: [torch.randn(n, nkv, hd, device="cuda", generator=gen) for _ in range(2)] for s, n in src.items()}
    pools = [make_pool(budget, kv_heads=nkv, head_dim=hd, page_len=page, kv_dtype=kv, part_len=part_len)
             for _ in range(2)]
    for shared, pool in zip((True, False), pools):
        for s in list(src) + ([] if shared else list(forks)):
            n = lens[s]
            pool.alloc(s, 0, n)
            k, v = data[s if s in src else forks[s][0]]
            rows = RowMeta(n)
            rows.write(range(n), [s] * n)
            ops.kv_store(k[:n].contiguous(), v[:n].contiguous(), pool, 0, n, rows)
        for s, (frm, n) in forks.items():
            if shared:
                pool.fork(frm, s, n)
        for s in range(6):
            pool.alloc(s, lens[s], rps)
        if chunk:
            pool.alloc(6, 0, chunk)
    pos = [lens[s] + i for s in range(6) for i in range(rps)] + list(range(chunk))
    seq = [s for s in range(6) for _ in range(rps)] + [6] * chunk
    m, nq = len(pos), g * nkv
    q = torch.randn(m, nq, hd, device="cuda", generator=gen)
    k, v = (torch.randn(m, nkv, hd, device="cuda", generator=gen) for _ in range(2))
    out = []
    for pool in pools:
        rows = RowMeta(m)
        rows.write(pos, seq)
        spec = ops.AttnSpec(q_heads=nq, window=0, scale=1.5 / math.sqrt(hd), m=m, causal=True, seq=None, args=rows)
        for _ in range(2):
            y = torch.full_like(q, 7.0)
            ops.attn_step(pool, 0, spec, q, y, k_src=k, v_src=v)
        z = torch.full_like(q, 8.0)
        ops.attn(q, pool, 0, z, spec)
        torch.cuda.synchronize()
        assert torch.equal(y, z), name
        out.append(y)
    assert torch.equal(out[0], out[1]), (name, float((out[0] - out[1]).abs().max()))
