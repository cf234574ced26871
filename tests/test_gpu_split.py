"""GPU parity of the split-K route of the INT8 GEMMs: problems of few tiles, given the workspace the
library asks for, run K slices and a summing epilogue; every output must equal the unsplit kernel's (a
workspace of the tile-queue counters alone), bit for bit, and the int32 sums an int64 product."""

import pytest
import torch

import mx_qlinear._lib as L
from _util import gen
from mx_qlinear.ops import _gemm_ws, _p, _stream

pytestmark = pytest.mark.gpu

# (m, n, k): both sides of every tile height, ragged columns (n % 4 != 0 stores element by element), K tails
# inside the last slice's stage, a last slice shorter than the others, one column tile.
SHAPES = [(1, 5376, 7168), (2, 1001, 14336), (31, 130, 2064), (32, 512, 4112), (33, 3, 20480), (64, 1000, 7184),
          (65, 2050, 5120), (128, 5120, 5376), (129, 516, 14336), (300, 1030, 20480), (7, 1, 131056)]


def _i8(shape, seed, dev):
    return torch.randint(-128, 128, shape, generator=gen(seed), dtype=torch.int8).to(dev)


def _spaces(dev, m, n, k, table=0):
    """(workspace args, keep-alive) without and with room for the split."""
    need = L.gemm_workspace_bytes(m, n, k, table)
    assert need > L.GEMM_WORKSPACE_BYTES, "the shape is meant to split"
    small = torch.zeros(L.GEMM_WORKSPACE_BYTES, dtype=torch.uint8, device=dev)
    large = torch.full((need,), 0x5A, dtype=torch.uint8, device=dev)
    large[: L.GEMM_WORKSPACE_BYTES] = 0
    return small, large


def _factors(m, n, dev, dtype, scalar):
    ws = (torch.rand(1 if scalar else n, generator=gen(3)) * 0.01 + 0.001).to(dev)
    xs = (torch.rand(m, generator=gen(4)) * 0.1 + 0.01).to(dev)
    return ws, xs, torch.randn(n, generator=gen(5)).to(dtype).to(dev)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_split_sums_and_dequant(dev, m, n, k):
    print(f"split m={m} n={n} k={k}", flush=True)
    a, w = _i8((m, k), m + k, dev), _i8((n, k), n + k, dev)
    small, large = _spaces(dev, m, n, k)
    ld = n + 5  # a row stride that is no multiple of 4 elements
    out = []
    for space in (small, large):
        c = torch.full((m, ld), 7, dtype=torch.int32, device=dev)
        L.call("mxq_int8_gemm_i32", _p(a), _p(w), _p(c), m, n, k, ld, _p(space), space.numel(), _stream(dev))
        out.append(c)
    assert torch.equal(out[0], out[1])
    want = (a[:, :].cpu().double() @ w.cpu().double().t()).to(torch.int64)  # exact: below 2^53
    assert torch.equal(out[1][:, :n].cpu().to(torch.int64), want) and bool((out[1][:, n:] == 7).all())
    for code, dtype in ((L.DTYPE_F32, torch.float32), (L.DTYPE_F16, torch.float16), (L.DTYPE_BF16, torch.bfloat16)):
        ws, xs, bias = _factors(m, n, dev, dtype, code == L.DTYPE_F16)
        for ldd in (ld, (n + 7) // 8 * 8):  # element and run stores
            got = []
            for space in (small, large):
                y = torch.zeros((m, ldd), dtype=dtype, device=dev)
                L.call("mxq_int8_gemm_dequant", _p(a), _p(w), _p(xs), _p(ws), ws.numel(),
                       _p(bias) if code != L.DTYPE_F32 else None, _p(y), m, n, k, ldd, code, _p(space), space.numel(),
                       _stream(dev))
                got.append(y)
            assert torch.equal(got[0], got[1]), (dtype, ldd)
    assert int(large[: L.GEMM_WORKSPACE_BYTES].max()) == 0  # the counters stay zero


@pytest.mark.parametrize("m,n,k", [(1, 5376, 7168), (33, 1001, 14336), (130, 2050, 14336)])
@pytest.mark.parametrize("pad", [0, 3])
def test_split_gated_residual(dev, m, n, k, pad):
    a, w = _i8((m, k), 1, dev), _i8((n, k), 2, dev)
    small, large = _spaces(dev, m, n, k)
    ws, xs, bias = _factors(m, n, dev, torch.bfloat16, False)
    gate = torch.randn(3, n, generator=gen(6)).to(torch.bfloat16).to(dev)
    rows = torch.randint(0, 3, (m,), generator=gen(7), dtype=torch.int32).to(dev)
    res0 = torch.randn(m, n + pad, generator=gen(8)).to(torch.bfloat16).to(dev)
    got = []
    for space in (small, large):
        r = res0.clone()
        L.call("mxq_int8_gemm_gated_residual", _p(a), _p(w), _p(xs), _p(ws), ws.numel(), _p(bias), _p(r), n + pad, _p(gate),
               n, 3, _p(rows), m, n, k, _p(space), space.numel(), _stream(dev))
        got.append(r)
    assert torch.equal(got[0], got[1]) and torch.equal(got[1][:, n:], res0[:, n:]) and not torch.equal(got[1], res0)


@pytest.mark.parametrize("m,n,k", [(1, 28672, 5376), (40, 2080, 5376), (77, 8192, 3072), (129, 96, 4112)])
def test_split_swiglu(dev, m, n, k):
    """With SwiGLU also one slice alone takes the two-launch form (28672 columns at one row)."""
    a, w = _i8((m, k), 1, dev), _i8((n, k), 2, dev)
    small, large = _spaces(dev, m, n, k, 2)
    ws, xs, bias = _factors(m, n, dev, torch.bfloat16, False)
    xs[0] = float("nan") if m > 1 else xs[0]
    got = []
    for space in (small, large):
        h = torch.zeros((m, n // 2 + 3), dtype=torch.bfloat16, device=dev)
        L.call("mxq_int8_gemm_dequant_swiglu", _p(a), _p(w), _p(xs), _p(ws), ws.numel(), _p(bias), _p(h), m, n, k,
               n // 2 + 3, _p(space), space.numel(), _stream(dev))
        got.append(h.view(torch.int16))
    assert torch.equal(got[0], got[1])


def test_split_calls_on_two_streams_and_in_a_graph(dev):
    """Each call's partial sums are its own: calls overlap on two streams, and a captured one replays."""
    import mx_qlinear as mx

    m, n, k = 24, 5376, 7168
    assert _gemm_ws(dev, m, n, k)[1] > L.GEMM_WORKSPACE_BYTES
    w = _i8((n, k), 2, dev)
    ws = torch.rand(n, generator=gen(3)).to(dev) * 0.01
    xs = [torch.randn(m, k, generator=gen(10 + i)).to(torch.bfloat16).to(dev) for i in range(6)]
    want = [mx.int8_linear(x, w, ws) for x in xs]
    torch.cuda.synchronize(dev)
    streams = [torch.cuda.Stream(dev), torch.cuda.Stream(dev)]
    got = []
    for i, x in enumerate(xs):
        with torch.cuda.stream(streams[i % 2]):
            got.append(mx.int8_linear(x, w, ws))
    torch.cuda.synchronize(dev)
    assert all(torch.equal(g, r) for g, r in zip(got, want))
    graph, x = torch.cuda.CUDAGraph(), xs[0].clone()
    with torch.cuda.graph(graph):
        y = mx.int8_linear(x, w, ws)
    for i in (3, 1, 5):
        x.copy_(xs[i])
        mx.int8_linear(xs[2], w, ws)  # eager work between the replays
        graph.replay()
        torch.cuda.synchronize(dev)
        assert torch.equal(y, want[i])
