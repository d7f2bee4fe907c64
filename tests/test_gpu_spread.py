"""Decode calls of few, long work items run one wave per workgroup
(attn_spread): bit for bit the result of the one-workgroup form, which
thb_attn_noalloc always takes, and the oracle's exact softmax, over head_dims,
KV types, page lengths, runs that end anywhere in a tile or hold no key,
windows that start inside a tile or page, soft-cap, several partitions and
rows per sequence; the fused append against kv_store followed by attn and against the
device-planned append, with rotation against kv_store_rope followed by attn_rope
of a call with too many rows for the form; infinite values; repeated launches
(the arrival counters)."""

import ctypes
import math
import random

import pytest

import oracle
from gpu_util import fill, make_pool, oracle_layer, say, scattered_alloc
from plan_util import takes_spread

pytestmark = pytest.mark.gpu

# name, head_dim, kv heads, q heads per kv head, rows, page, kv type, part_len, window, softcap, contexts
CASES = [
    ("hd128-one-tile-over", 128, 8, 4, 1, 16, "f16", 0, 0, 0.0, [1025]),
    ("hd128-bf16-page32-ragged", 128, 2, 4, 1, 32, "bf16", 0, 0, 0.0, [1500, 37, 4095]),
    ("hd128-parts", 128, 1, 5, 1, 16, "f16", 2048, 0, 0.0, [3900, 2049]),
    ("hd128-eight-parts", 128, 1, 4, 1, 16, "bf16", 1040, 0, 0.0, [8300, 700]),
    ("hd64-more-parts-than-combined", 64, 1, 7, 1, 16, "f16", 2048, 0, 0.0, [9000]),
    ("hd128-window", 128, 4, 8, 1, 16, "f16", 0, 1333, 0.0, [4099, 1400]),
    ("hd64-long", 64, 2, 7, 1, 16, "f16", 0, 0, 0.0, [2049, 4000, 5]),
    ("hd64-page256", 64, 1, 1, 1, 256, "bf16", 0, 0, 0.0, [3001]),
    ("hd256-one-column", 256, 1, 1, 1, 16, "f16", 0, 0, 30.0, [700]),
    ("hd256-verify-window", 256, 2, 2, 4, 16, "f16", 0, 1500, 50.0, [2600, 1333]),
    ("hd256-parts-bf16", 256, 1, 4, 1, 32, "bf16", 1024, 0, 0.0, [4000, 3000]),
    ("hd256-verify-parts", 256, 1, 4, 2, 16, "f16", 2048, 0, 0.0, [4000]),
]


NOT_SPREAD = ("hd64-more-parts-than-combined",)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_spread_matches_one_workgroup(torch_cuda, case):
    torch = torch_cuda
    from flint_amd import _lib, ops
    from flint_amd.pool import RowMeta, _stream_ptr
    from flint_amd.rope import Rope, attn_rope, kv_store_rope

    name, hd, nkv, g, rps, page, kv, part_len, window, cap, lens = case
    say("spread", name)
    budget = [n + rps for n in lens] + [1, 1]  # (two sequences of one token, for rows beside the call's)
    pools = []
    for _ in range(2):
        p = make_pool(budget, kv_heads=nkv, head_dim=hd, page_len=page, kv_dtype=kv, extra_pages=1, part_len=part_len)
        scattered_alloc(p, budget, random.Random(7), page)
        fill(torch, p, RowMeta(256), lens + [1, 1], seed=7)
        pools.append(p)
    m, nq = rps * len(lens), g * nkv
    rows = RowMeta(m)
    pos, seq = [n + i for n in lens for i in range(rps)], [s for s in range(len(lens)) for _ in range(rps)]
    rows.write(pos, seq)
    shape = (g, nkv, hd, page, part_len, window)
    assert takes_spread(*shape, pos, seq) == (name not in NOT_SPREAD), name
    gen = torch.Generator(device="cuda")
    gen.manual_seed(8)
    q = torch.randn(m, nq, hd, device="cuda", generator=gen)
    k, v = (torch.randn(m, nkv, hd, device="cuda", generator=gen) for _ in range(2))
    spec = ops.AttnSpec(q_heads=nq, window=window, scale=1.5 / math.sqrt(hd), m=m, causal=True, seq=None, args=rows,
                        softcap=cap)
    y, z = torch.full_like(q, 7.0), torch.full_like(q, 8.0)
    for rope in (None, Rope.from_theta(max(budget), hd, 1e4)):
        for _ in range(3):  # every launch leaves its counters at zero
            ops.attn_step(pools[0], 0, spec, q, y, k_src=k, v_src=v, rope=rope)
        if rope is None:
            ops.kv_store(k, v, pools[1], 0, m, rows)
            c = ops._spec_c(spec, q, z)
            rc = _lib.lib().thb_attn_noalloc(pools[1].handle, 0, q.data_ptr(), z.data_ptr(), ctypes.byref(c),
                                             rows.handle, _stream_ptr(None))
            assert rc == 0, _lib.lib().thb_last_error()
            torch.cuda.synchronize()
            assert torch.equal(y, z), (name, float((y - z).abs().max()))
            layer = oracle_layer(torch, pools[1])
            plan = ops.DevicePlan(pools[1], max_m=m, q_heads=nq, append=True)
            plan.build(spec, q, z)
            for _ in range(2):
                z.fill_(9.0)
                plan.attn_append(0, k, v, q, z)
                torch.cuda.synchronize()
                assert torch.equal(y, z), name
            plan.close()
            want = layer.attn(q.cpu().numpy(), oracle.row_meta(pos, seq), m, nq, spec.scale, window=window, softcap=cap)
            err = float(abs(y.cpu().numpy() - want).max())
            say(name, "max abs err vs oracle", err)
            assert err <= 1e-4, (name, err)
        else:
            # The rotary append by itself, then the one-workgroup form: the same
            # rows in a call with too many items to spread.
            kv_store_rope(k, v, pools[1], 0, m, rows, rope)
            more, last = 65, len(lens)
            pos2, seq2 = pos + [0] * more, seq + [last + i % 2 for i in range(more)]
            assert not takes_spread(*shape, pos2, seq2)
            big = RowMeta(m + more)
            big.write(pos2, seq2)
            q2 = torch.cat([q, q[:1].expand(more, nq, hd)]).contiguous()
            z2 = torch.full_like(q2, 8.0)
            attn_rope(q2, pools[1], 0, z2, ops.AttnSpec(q_heads=nq, window=window, scale=spec.scale, m=m + more,
                                                        causal=True, seq=None, args=big, softcap=cap), rope)
            z.copy_(z2[:m])
        torch.cuda.synchronize()
        assert torch.equal(y, z), name
        for a, b in zip(pools[0].layer_tensors(0), pools[1].layer_tensors(0)):
            assert torch.equal(a, b), name


def test_infinite_values(torch_cuda):
    """An infinite value whose key has a probability, in the last tile of a run
    that ends inside a step of two tiles: infinities and NaNs as the
    one-workgroup form gives them."""
    torch = torch_cuda
    from flint_amd import _lib, ops
    from flint_amd.pool import RowMeta, _stream_ptr

    for hd, g, n in ((128, 4, 1090), (64, 7, 2100)):
        say("spread infinite values", hd)
        pool = make_pool([n], kv_heads=2, head_dim=hd)
        pool.alloc(0, 0, n)
        rows = RowMeta(n)
        rows.write(list(range(n)), [0] * n)
        gen = torch.Generator(device="cuda")
        gen.manual_seed(3)
        k, v = (torch.randn(n, 2, hd, device="cuda", generator=gen) for _ in range(2))
        run = -(-n // 8) + 15 & ~15
        assert run // 16 % 2 == 1
        for t in range(run - 1, n, 2 * run):  # every second run's last key
            v[t, :, ::3] = math.inf
        ops.kv_store(k, v, pool, 0, n, rows)
        one = RowMeta(1)
        one.write([n - 1], [0])
        assert takes_spread(g, 2, hd, 16, 0, 0, [n - 1], [0])
        q = torch.randn(1, 2 * g, hd, device="cuda", generator=gen) * 0.1
        y, z = torch.full_like(q, 7.0), torch.full_like(q, 8.0)
        spec = ops.AttnSpec(q_heads=2 * g, window=0, scale=0.1, m=1, causal=True, seq=None, args=one)
        ops.attn(q, pool, 0, y, spec)
        c = ops._spec_c(spec, q, z)
        assert _lib.lib().thb_attn_noalloc(pool.handle, 0, q.data_ptr(), z.data_ptr(), ctypes.byref(c), one.handle,
                                           _stream_ptr(None)) == 0
        torch.cuda.synchronize()
        assert torch.equal(torch.isnan(y), torch.isnan(z)), (hd, int(torch.isnan(y).sum()), int(torch.isnan(z).sum()))
        assert torch.equal(torch.nan_to_num(y), torch.nan_to_num(z)), hd
