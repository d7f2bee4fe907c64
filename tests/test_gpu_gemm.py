"""GPU parity of thb_gemm_acc (ops::gemm_acc, the o_proj product after
attention) against the oracle's restatement of cpu_ref::gemm / gemv
(crates/thuban_backend/tests/support/cpu_ref.rs:11-35).

* The reference's own bf16-weight cases, inputs drawn from its LCG:
  gemm_coop_bf16_acc and gemm_coop_bf16_multi_tile (kernels.rs:472-536),
  gemv_bf16 / gemv_bf16_wide_k (kernels.rs:630-680), and the shapes and
  seeds of gemm_acc_case (kernels.rs:542-598, which uses Q8_0 weights there;
  here the weights are bf16 draws of the same LCG), each within the
  reference's tolerance (rel 2e-2, abs 5e-2) of cpu_ref::gemm.
* A tight check against the oracle's double-precision sums: |gpu - exact|
  <= 2^-15 * sum |x w| + 1e-6 (the high/low split keeps ~16 bits of x against
  the exact weight), for every x type (f32, f16, bf16) x weight type (bf16,
  f16) over row counts that take both kernels and their edges.
* Identity weights give y = x exactly for an x of the weight's type;
  results are deterministic (two runs, same bits)."""

import zlib

import numpy as np
import pytest

import oracle
from gpu_util import say

pytestmark = pytest.mark.gpu


def _bf16_round(v):
    """bf16_round of kernels.rs:126-130: the upper 16 bits."""
    return (np.asarray(v, np.float32).view(np.uint32) & 0xFFFF0000).view(np.float32)


def _run(torch, x, w16, y0, acc, x_dtype=None, w_dtype=None):
    from flint_amd import ops

    m, k = x.shape
    tx = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    if x_dtype is not None:
        tx = tx.to(x_dtype)
    tw = torch.from_numpy(np.ascontiguousarray(w16)).cuda().to(w_dtype or torch.bfloat16)
    ty = torch.from_numpy(np.ascontiguousarray(y0, np.float32)).cuda()
    ops.gemm_acc(tx, tw, ty, m, acc)
    torch.cuda.synchronize()
    return ty.cpu().numpy()


def _agree(got, want, rel, abs_):
    diff = np.abs(got - want)
    assert np.all(diff <= rel * np.abs(want) + abs_), float(np.max(diff - rel * np.abs(want)))


# (name, seed, m, n, k, acc): the reference's cases (kernels.rs lines above)
REF_CASES = [
    ("gemm_coop_bf16_acc", 13, 128, 128, 256, True),
    ("gemm_coop_bf16_multi_tile", 29, 128, 256, 1024, False),
    ("gemv_bf16", 31, 1, 32, 128, False),
    ("gemv_bf16_wide_k", 47, 1, 32, 1024, False),
    ("gemm_acc_coop_full", 31, 128, 128, 256, False),
    ("gemm_acc_coop_tail", 37, 144, 128, 256, False),
    ("gemm_acc_coop_tail_accumulates", 39, 144, 128, 256, True),
    ("gemm_acc_coop_long_k", 41, 128, 128, 8192, False),
    ("gemm_classic_segs_long_k", 43, 64, 64, 8192, False),
]


@pytest.mark.parametrize("case", REF_CASES, ids=[c[0] for c in REF_CASES])
def test_reference_cases(torch_cuda, case):
    torch = torch_cuda
    name, seed, m, n, k, acc = case
    say("gemm reference case", name)
    if name.startswith("gemm_coop_bf16") or name.startswith("gemv_bf16"):
        # one Rng: x, then w, then y0 (kernels.rs:479-482, 512-514, 633-634)
        draws = oracle.lcg_fill(seed, m * k + n * k + (m * n if acc else 0))
        x, w = draws[:m * k].reshape(m, k), draws[m * k:m * k + n * k].reshape(n, k)
        y0 = draws[m * k + n * k:].reshape(m, n) if acc else np.zeros((m, n), np.float32)
    else:
        # gemm_acc_case: Rng(seed) for x then y0; weights from seed ^ 0x1234
        draws = oracle.lcg_fill(seed, m * k + m * n)
        x, y0 = draws[:m * k].reshape(m, k), draws[m * k:].reshape(m, n)
        w = oracle.lcg_fill(seed ^ 0x1234, n * k).reshape(n, k)
        if not acc:
            y0 = np.zeros((m, n), np.float32)
    wb = _bf16_round(w)
    got = _run(torch, x, wb, y0, acc)
    want = oracle.gemm(x, wb, m, n, k, y0=y0 if acc else None)
    _agree(got, want, 2e-2, 5e-2)
    exact = oracle.gemm(x, wb, m, n, k, y0=y0 if acc else None, exact=True)
    scale = np.abs(x).astype(np.float64) @ np.abs(wb).astype(np.float64).T
    err = float(np.max(np.abs(got - exact) - 2.0 ** -15 * scale))
    say(name, "max |gpu - exact| over the bound", err)
    assert err <= 1e-6


@pytest.mark.parametrize("wt", ["bf16", "f16"])
@pytest.mark.parametrize("xt", ["f32", "f16", "bf16"])
def test_every_type_and_row_count(torch_cuda, xt, wt):
    torch = torch_cuda
    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    rng = np.random.default_rng(zlib.crc32(f"{xt}-{wt}".encode()))  # the same inputs in every process
    n, k = 192, 512
    w = rng.standard_normal((n, k)).astype(np.float32)
    w = _bf16_round(w) if wt == "bf16" else w.astype(np.float16).astype(np.float32)
    for m in (1, 5, 16, 17, 32, 33, 48, 64, 65, 130):
        x = rng.standard_normal((m, k)).astype(np.float32)
        xq = torch.from_numpy(x).to(tdt[xt]).float().numpy()  # x as the kernel sees it
        y0 = rng.standard_normal((m, n)).astype(np.float32)
        got = _run(torch, x, w, y0, True, x_dtype=tdt[xt], w_dtype=tdt[wt])
        exact = oracle.gemm(xq, w, m, n, k, y0=y0, exact=True)
        scale = np.abs(xq).astype(np.float64) @ np.abs(w).astype(np.float64).T
        err = float(np.max(np.abs(got - exact) - 2.0 ** -15 * scale))
        assert err <= 1e-6, (xt, wt, m, err)
    say("gemm types", xt, wt, "ok")


def test_identity_weights_and_determinism(torch_cuda):
    torch = torch_cuda
    from flint_amd import ops

    k = 256
    eye = torch.eye(k, device="cuda", dtype=torch.bfloat16)
    for m in (3, 32, 100):
        x = torch.randn(m, k, device="cuda").to(torch.bfloat16)
        y = torch.zeros(m, k, device="cuda")
        ops.gemm_acc(x, eye, y, m, False)
        torch.cuda.synchronize()
        assert torch.equal(y, x.float()), m
    # Llama-3-8B o_proj at batch 32 (bf16 attention output into the residual)
    x = torch.randn(32, 4096, device="cuda").to(torch.bfloat16)
    w = (torch.randn(4096, 4096, device="cuda") * 0.02).to(torch.bfloat16)
    y0 = torch.randn(32, 4096, device="cuda")
    ya, yb = y0.clone(), y0.clone()
    ops.gemm_acc(x, w, ya, 32, True)
    ops.gemm_acc(x, w, yb, 32, True)
    torch.cuda.synchronize()
    assert torch.equal(ya, yb)
    exact = oracle.gemm(x.float().cpu().numpy(), w.float().cpu().numpy(), 32, 4096, 4096, y0=y0.cpu().numpy(),
                        exact=True)
    err = float(np.max(np.abs(ya.cpu().numpy() - exact)))
    say("o_proj 32 x 4096 x 4096 max abs err", err)
    assert err <= 1e-4


# (m, n, k): each tile shape with ragged last tiles in both directions and k
# of one k-tile, of a full and of a part group of k-tiles; the last rows and
# the first past each limit of the few-row kernel; fewer columns than a tile;
# few rows of more columns than 16 per CU.
SHAPES = [(1987, 4064, 192), (990, 4064, 64), (500, 4064, 576), (250, 4064, 512), (120, 4064, 640), (60, 4064, 1088),
          (30, 4064, 64), (16, 4064, 64), (17, 16, 64), (33, 48, 1024), (64, 16, 192), (65, 5120, 128), (1, 32, 64),
          (7, 5120, 320), (25, 4112, 1152)]


@pytest.mark.parametrize("types", ["bf16-bf16", "f16-f16", "f32-bf16", "f16-bf16", "bf16-f16"])
def test_every_tile_shape(torch_cuda, types):
    torch = torch_cuda
    xt, wt = types.split("-")
    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    rng = np.random.default_rng(zlib.crc32(types.encode()))
    for m, n, k in SHAPES:
        x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(tdt[xt])
        w = torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to(tdt[wt])
        y0 = rng.standard_normal((m, n)).astype(np.float32)
        acc = bool((m + n) & 1) or m > 64
        got = _run(torch, x.float().numpy(), w.float().numpy(), y0, acc, x_dtype=tdt[xt], w_dtype=tdt[wt])
        x64, w64 = x.double().numpy(), w.double().numpy()
        exact = x64 @ w64.T + (y0 if acc else 0.0)
        scale = np.abs(x64) @ np.abs(w64).T + np.abs(y0)
        err = float(np.max(np.abs(got - exact) - 2.0 ** -15 * scale))
        assert err <= 1e-6, (types, m, n, k, err)
    say("gemm tile shapes", types, "ok")


def test_gemm_errors(torch_cuda):
    torch = torch_cuda
    from flint_amd import ThubanError, ops

    x = torch.zeros(2, 96, device="cuda")
    w = torch.zeros(32, 96, device="cuda", dtype=torch.bfloat16)
    y = torch.zeros(2, 32, device="cuda")
    with pytest.raises(ThubanError) as e:
        ops.gemm_acc(x, w, y, 2, False)
    assert str(e.value) == "dimension pair (N=32, K=96) does not satisfy N%16 and K%64"
    assert e.value.kind == "Config"
    with pytest.raises(ThubanError):
        ops.check_gemm_dims([(4096, 4096), (40, 64)])
    ops.check_gemm_dims([(4096, 4096), (32, 128)])


LEVEL_CASES = [  # x, weights, rows, n, k
    ("bf16", "bf16", 33, 65536, 4096),
    ("f32", "f16", 33, 65536, 4096),
    ("f16", "f16", 64, 512, 28672),
    ("f16", "bf16", 64, 512, 28672),
    ("f32", "f16", 20, 512, 28672),
    ("bf16", "bf16", 300, 4096, 4096),
    ("f32", "f16", 1000, 4096, 4096),
]


@pytest.mark.parametrize("case", LEVEL_CASES, ids=["-".join(map(str, c)) for c in LEVEL_CASES])
def test_sums_add_up_in_levels(torch_cuda, case):
    """The error against 64 bits of wide and of long products (types whose
    products are exact to well below f32's rounding).  A chain of c additions
    of terms of random signs, each rounded by up to 2^-24 of a partial sum,
    loses about sqrt(c / 6) units of 2^-24 of its result.  The kernels' levels
    make c = 20 + k / 1024, above 64 rows 32 + k / 512 (chains of 512 k, twice
    the products with a low part, whose sums add up).  The bound is 1.5 times
    that, with 2 under the root for the matrix cores' own sums of 32 products:
    at k = 4096, 2.2e-7 and 2.6e-7, where one chain over all of K loses 4.0e-7,
    with a low part 5.8e-7."""
    torch = torch_cuda
    from flint_amd import ops

    xt, wt, m, n, k = case
    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    say("gemm levels", case)
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).to(dt[xt])
    w = (torch.randn(n, k, device="cuda", generator=g) * 0.02).to(dt[wt])
    y = torch.full((m, n), 5.0, device="cuda")
    ops.gemm_acc(x, w, y, m, False)
    err = ref = 0.0
    for c in range(0, n, 8192):
        want = torch.matmul(x.double(), w[c:c + 8192].double().t().contiguous())
        err += float((y[:, c:c + 8192].double() - want).square().sum())
        ref += float(want.square().sum())
    rel = (err / ref) ** 0.5
    sums = 20 + k / 1024 if m <= 64 else 32 + k / 512
    bound = 1.5 * 2.0 ** -24 * (sums / 6 + 2) ** 0.5
    say(case, "relative error", rel, "bound", bound)
    assert rel <= bound, (case, rel, bound)


@pytest.mark.parametrize("wt", ["bf16", "f16"])
@pytest.mark.parametrize("xt", ["f32", "f16", "bf16"])
def test_row_bits_do_not_depend_on_the_row_count(torch_cuda, xt, wt):
    """Above 64 rows every tile shape adds K up in the same order (a last chain
    of one k-tile included), as do all calls of 17 to 64 rows of the weight's
    type."""
    torch = torch_cuda
    from flint_amd import ops

    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    n, k = 4096, 1088
    g = torch.Generator(device="cuda")
    g.manual_seed(17)
    x = torch.randn(3000, k, device="cuda", generator=g).to(dt[xt])
    w = (torch.randn(n, k, device="cuda", generator=g) * 0.02).to(dt[wt])
    for counts in ((65, 130, 300, 1000, 3000),) + (((17, 33, 64),) if xt == wt else ()):
        first = None
        for m in counts:
            y = torch.full((m, n), 5.0, device="cuda")
            ops.gemm_acc(x[:m].contiguous(), w, y, m, False)
            first = y if first is None else first
            assert torch.equal(y[:counts[0]], first), (xt, wt, m)
