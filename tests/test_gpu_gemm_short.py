"""GPU parity of the INT8 GEMMs' short ping-pong tiles (192 or 128 rows, alone or behind 256-row tiles) and of
256-row tiles in place of 128 x 128 ones: int32 sums against an exact product, the epilogues against the same
IEEE operations in torch, bit for bit, and the workspace's counters zero after every launch."""

import pytest
import torch

import mx_qlinear._lib as L
from _util import bits, gen
from mx_qlinear.ops import _p, _stream
from oracle import convrot as cr

pytestmark = pytest.mark.gpu

# (m, n, k): rows of the short tile, claimed or not. K in whole stages and with a tail, columns whole and
# ragged (n % 4 != 0 stores element by element), last tiles of one and of almost all their rows.
SHAPES = [(513, 16001, 2064, 192, False), (576, 16384, 2048, 192, False), (1044, 21504, 2048, 128, True),
          (1025, 21506, 2160, 128, True), (8129, 5120, 4112, 192, True), (8192, 4990, 4096, 192, True),
          (2310, 5120, 4112, 256, False), (5000, 3001, 2176, 256, False), (8129, 3001, 2064, 256, True)]
# The same for the gated residual, whose rule has costs of its own.
GATED = [(2971, 28333, 2064, 128, True), (907, 24818, 2064, 192, True), (793, 28352, 2064, 192, True),
         (258, 22467, 7184, 192, False), (390, 25509, 14352, 256, False)]


def _case(dev, m, n, k, table=0):
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the shapes are chosen for 256 CUs")
    a = torch.randint(-128, 128, (m, k), generator=gen(m + k), dtype=torch.int8).to(dev)
    w = torch.randint(-128, 128, (n, k), generator=gen(n + k), dtype=torch.int8).to(dev)
    acc = torch.empty((m, n), dtype=torch.int32, device=dev)
    for r in range(0, m, 1024):
        acc[r:r + 1024] = (a[r:r + 1024].double() @ w.double().t()).to(torch.int32)  # exact: below 2^53
    space = torch.zeros(L.GEMM_WORKSPACE_BYTES, dtype=torch.uint8, device=dev)
    xs = (torch.rand(m, generator=gen(4)) * 0.1 + 0.01).to(dev)
    ws = (torch.rand(n, generator=gen(3)) * 0.01 + 0.001).to(dev)
    return a, w, acc, space, xs, ws, torch.randn(n, generator=gen(5)).to(dev)


def _dequant(acc, xs, ws, bias, dtype):
    return ((acc.float() * (xs[:, None] * ws)).to(dtype).float() + bias.to(dtype).float()).to(dtype)


@pytest.mark.parametrize("m,n,k,rows,queued", SHAPES)
def test_short_tiles(dev, m, n, k, rows, queued):
    print(f"short tiles m={m} n={n} k={k} rows={rows}", flush=True)
    plan = L.gemm_short_plan(m, n, k)
    a, w, acc, space, xs, ws, bias = _case(dev, m, n, k)
    assert (plan["rows"], plan["queued"]) == (rows, queued), plan
    ld = (n + 8) // 8 * 8
    st = _stream(dev)
    for _ in range(2):  # the second launch finds the counters as the first left them
        c = torch.full((m, ld), 7, dtype=torch.int32, device=dev)
        L.call("mxq_int8_gemm_i32", _p(a), _p(w), _p(c), m, n, k, ld, _p(space), space.numel(), st)
        assert torch.equal(c[:, :n], acc) and bool((c[:, n:] == 7).all())
        assert int(space.count_nonzero()) == 0
    for code, dtype in ((L.DTYPE_F32, torch.float32), (L.DTYPE_F16, torch.float16), (L.DTYPE_BF16, torch.bfloat16)):
        b = bias.to(dtype)
        y = torch.zeros((m, n), dtype=dtype, device=dev)
        L.call("mxq_int8_gemm_dequant", _p(a), _p(w), _p(xs), _p(ws), n, _p(b), _p(y), m, n, k, n, code, _p(space),
               space.numel(), st)
        assert torch.equal(y, _dequant(acc, xs, ws, bias, dtype))
    _check_gated(dev, a, w, acc, space, xs, ws, bias)


def _check_gated(dev, a, w, acc, space, xs, ws, bias):
    (m, k), n, st = a.shape, w.shape[0], _stream(dev)
    b, gate = bias.bfloat16(), torch.randn(3, n, generator=gen(6)).bfloat16().to(dev)
    grow = torch.randint(0, 3, (m,), generator=gen(7), dtype=torch.int32).to(dev)
    res = torch.randn(m, n, generator=gen(8)).bfloat16().to(dev)
    y = _dequant(acc, xs, ws, bias, torch.bfloat16)
    want = (res.float() + y.float() * gate[grow.long()].float()).bfloat16()
    L.call("mxq_int8_gemm_gated_residual", _p(a), _p(w), _p(xs), _p(ws), n, _p(b), _p(res), n, _p(gate), n, 3, _p(grow),
           m, n, k, _p(space), space.numel(), st)
    assert torch.equal(res, want) and int(space.count_nonzero()) == 0


@pytest.mark.parametrize("m,n,k,rows,queued", GATED)
def test_short_gated_residual(dev, m, n, k, rows, queued):
    print(f"short gated residual m={m} n={n} k={k} rows={rows}", flush=True)
    case = _case(dev, m, n, k)
    plan = L.gemm_short_plan(m, n, k, L.PLAN_GATED_RESIDUAL)
    assert (plan["rows"], plan["queued"]) == (rows, queued), plan
    for _ in range(2):  # the second launch finds the counters as the first left them
        _check_gated(dev, *case)


@pytest.mark.parametrize("m,f,k,rows,queued", [(333, 14336, 2064, 192, False), (129, 14336, 2048, 128, False),
                                               (1025, 10752, 2064, 128, True), (1314, 14336, 2064, 192, True)])
def test_short_swiglu(dev, m, f, k, rows, queued):
    print(f"short swiglu m={m} f={f} k={k} rows={rows}", flush=True)
    import mx_qlinear as mx

    plan = L.gemm_short_plan(m, 2 * f, k, 2)
    a, w, acc, space, xs, ws, bias = _case(dev, m, 2 * f, k)
    assert (plan["rows"], plan["queued"]) == (rows, queued), plan
    fc1 = mx.prepare_swiglu_fc1(w, ws, bias.bfloat16())
    h = mx.int8_swiglu_fc1(a, xs[:, None], fc1)
    pick = torch.unique(torch.cat([torch.arange(0, m, 61), torch.tensor([0, m - 1])]))  # every height's tiles
    y = _dequant(acc[pick.to(dev)], xs[pick.to(dev)], ws, bias, torch.bfloat16)
    assert (bits(h[pick.to(dev)].cpu()) == cr.swiglu_bf16(bits(y.cpu()))).all()
