"""Device plans of few rows choose at every build, from the rows' keys, whether
an item runs on one workgroup or each of its waves on its own (attn_pick): one
plan, rebuilt while the rows move from a few keys to several partitions and
back, gives bit for bit what host-planned calls give, whatever the pool's
budget allows; with more rows than the spread form takes, rows without pages,
layers of several head_dims, pages of 8 and grids that end inside a KV head's
slots; and in a captured graph."""

import math
import random

import pytest

from gpu_util import fill, make_pool, say, scattered_alloc

pytestmark = pytest.mark.gpu

# name, head_dim, kv heads, q heads per kv head, sequences, page, kv type, part_len, budget, lengths in turn
CASES = [
    ("hd128-one", 128, 8, 4, 1, 16, "f16", 0, 32768, [[5], [1023], [1024], [1100], [4099], [300]]),
    ("hd128-eight", 128, 8, 4, 8, 16, "f16", 0, 4096,
     [[40 + s for s in range(8)], [1663] * 8, [1700 - 200 * s for s in range(8)], [3000] * 8, [9] * 8]),
    ("hd128-budget-just-enough", 128, 4, 8, 3, 32, "bf16", 0, 0, [[700, 3100, 50], [1, 2, 3]]),
    ("hd128-parts", 128, 1, 4, 2, 16, "f16", 2048, 20000, [[6000, 100], [4097, 8300], [17, 2049]]),
    ("hd128-three-kv-heads", 128, 3, 5, 4, 16, "bf16", 0, 8192, [[2500, 1, 1800, 900], [60, 70, 80, 90]]),
    ("hd64", 64, 2, 7, 8, 16, "f16", 0, 8192, [[2100] * 8, [2047] * 8, [4096, 5, 3000, 8, 2500, 1, 40, 4000]]),
    ("hd256", 256, 8, 2, 2, 16, "f16", 0, 4096, [[400, 511], [512, 30], [3000, 2000], [4, 4]]),
    ("hd256-parts-bf16", 256, 1, 8, 2, 32, "bf16", 1024, 6000, [[3000, 900], [1025, 2040], [10, 20]]),
    ("hd128-too-many-rows", 128, 8, 4, 9, 16, "f16", 0, 4096, [[2500] * 9, [30] * 9]),
    ("hd80", 80, 4, 3, 3, 16, "f16", 0, 4096, [[2500, 10, 3000]]),
    ("hd128-page8", 128, 2, 4, 3, 8, "f16", 0, 4096, [[2500, 10, 3000]]),
]


@pytest.mark.parametrize("rotary", [False, True], ids=["plain", "rotary"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_rebuilt_plan_matches_host_plans(torch_cuda, case, rotary):
    torch = torch_cuda
    from flint_amd import ops
    from flint_amd.pool import RowMeta
    from flint_amd.rope import Rope

    name, hd, nkv, g, b, page, kv, part_len, budget, turns = case
    say("dplan pick", name, rotary)
    most = [max(t[s] for t in turns) + 1 for s in range(b)]
    nq = g * nkv
    pools = []
    for _ in range(2):
        p = make_pool(most, kv_heads=nkv, head_dim=hd, page_len=page, kv_dtype=kv, part_len=part_len,
                      seq_lens=[budget or n for n in most])
        scattered_alloc(p, most, random.Random(5), page)
        fill(torch, p, RowMeta(256), most, seed=6)
        pools.append(p)
    rope = Rope.from_theta(max(most), hd, 1e4) if rotary else None
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    plan = ops.DevicePlan(pools[0], max_m=b, q_heads=nq, append=True)
    if rope is not None:
        plan.set_pos_limit(rope.max_pos)
    for turn in turns:
        rows = RowMeta(b)
        rows.write(turn, list(range(b)))
        q = torch.randn(b, nq, hd, device="cuda", generator=gen)
        k, v = (torch.randn(b, nkv, hd, device="cuda", generator=gen) for _ in range(2))
        spec = ops.AttnSpec(q_heads=nq, window=0, scale=1.5 / math.sqrt(hd), m=b, causal=True, seq=None, args=rows)
        want = torch.full_like(q, 7.0)
        ops.attn_step(pools[1], 0, spec, q, want, k_src=k, v_src=v, rope=rope)
        got = torch.full_like(q, 8.0)
        plan.build(spec, q, got)
        for _ in range(3):  # every launch leaves its counters at zero
            got.fill_(9.0)
            plan.step(0, q, got, k_src=k, v_src=v, rope=rope)
            torch.cuda.synchronize()
            assert torch.equal(got, want), (name, turn, float((got - want).abs().max()))
    for a, c in zip(pools[0].layer_tensors(0), pools[1].layer_tensors(0)):
        assert torch.equal(a, c), name
    plan.close()


def test_layers_of_several_head_dims(torch_cuda):
    """One plan serves layers that take the spread form, each by its own
    head_dim's rule, and layers that do not."""
    torch = torch_cuda
    from flint_amd import ops
    from flint_amd.pool import RowMeta

    dims, nkv, g, lens = [64, 256, 80, 128, 256], 4, 2, [1500, 700, 40]
    pool = make_pool([n + 1 for n in lens], kv_heads=nkv, head_dim=dims[0], layers=len(dims), head_dims=dims,
                     seq_lens=[4096] * 3)
    scattered_alloc(pool, [n + 1 for n in lens], random.Random(2), 16)
    for layer in range(len(dims)):
        fill(torch, pool, RowMeta(256), [n + 1 for n in lens], layer=layer, seed=layer)
    plan = ops.DevicePlan(pool, max_m=3, q_heads=nkv * g)
    for pos in (lens, [1100, 2, 3], [9, 8, 7], lens):
        rows = RowMeta(3)
        rows.write(pos, [0, 1, 2])
        for layer, hd in enumerate(dims):
            say("dplan head_dims", pos, hd)
            q = torch.randn(3, nkv * g, hd, device="cuda")
            spec = ops.AttnSpec(q_heads=nkv * g, window=0, scale=0.1, m=3, causal=True, seq=None,
                                args=rows)
            want, got = torch.full_like(q, 7.0), torch.full_like(q, 8.0)
            ops.attn(q, pool, layer, want, spec)
            if layer == 0:
                plan.build(spec, q, got)
            plan.attn(layer, q, got)
            torch.cuda.synchronize()
            assert torch.equal(got, want), (pos, hd)


@pytest.mark.parametrize("hd,nkv,g", [(128, 8, 4), (64, 2, 7)])
def test_captured_step_follows_the_rows(torch_cuda, hd, nkv, g):
    """One graph of build and step, captured at a few keys, replayed while the
    rows grow past the spread form's threshold and shrink again."""
    torch = torch_cuda
    from flint_amd import ops
    from flint_amd.pool import RowMeta

    b, most = 4, 3001
    pool = make_pool([most] * b, kv_heads=nkv, head_dim=hd, seq_lens=[4096] * b)
    scattered_alloc(pool, [most] * b, random.Random(3), 16)
    fill(torch, pool, RowMeta(256), [most] * b, seed=4)
    rows, other = RowMeta(b), RowMeta(b)
    q = torch.randn(b, nkv * g, hd, device="cuda")
    y = torch.zeros_like(q)

    def spec(r):
        return ops.AttnSpec(q_heads=nkv * g, window=0, scale=1.0 / math.sqrt(hd), m=b, causal=True, seq=None, args=r)

    plan = ops.DevicePlan(pool, max_m=b, q_heads=nkv * g)
    rows.write([20] * b, list(range(b)))

    def body():
        plan.build(spec(rows), q, y)
        for _ in range(2):
            plan.attn(0, q, y)

    body()
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            body()
    torch.cuda.current_stream().wait_stream(side)
    for pos in ([20] * b, [3000] * b, [2999, 5, 1800, 900], [100, 200, 300, 50], [3000] * b):
        say("dplan captured", hd, pos)
        rows.write(pos, list(range(b)))
        q.normal_()
        for _ in range(2):
            y.fill_(9.0)
            graph.replay()
            torch.cuda.synchronize()
        other.write(pos, list(range(b)))
        want = torch.zeros_like(q)
        ops.attn(q, pool, 0, want, spec(other))
        torch.cuda.synchronize()
        assert torch.equal(y, want), pos
    del graph
    plan.close()
