"""GPU parity of fc2 with the gated residual epilogue against the oracle (bit-exact bf16):
int8_linear followed by the per-segment addcmul_ of the reference."""

import numpy as np
import pytest
import torch

from _util import activations, bf16_vec, bits, gen, int8_weight
from oracle import convrot as cr
from oracle import eager_np

pytestmark = pytest.mark.gpu


def _mx():
    import mx_qlinear

    return mx_qlinear


def _segments(m, parts):
    cuts = sorted({0, m, *[(m * i) // parts for i in range(1, parts)]})
    return tuple((a, b, i % 3) for i, (a, b) in enumerate(zip(cuts[:-1], cuts[1:])))


def _expected(res, x, w, ws, b, gate, rows, g=0, act=None):
    if g or act:
        q, s, _ = cr.convrot_quantize_bf16(bits(x), g, act)
    else:
        q, s = eager_np.quantize_int8_rowwise(bits(x))
    y = eager_np.dequant_epilogue(eager_np.int8_matmul(q, w.numpy()), s, ws.numpy(),
                                  None if b is None else bits(b), "bf16")
    from oracle.bf16 import bf16_bits

    return eager_np.gated_residual_bf16(bits(res), bf16_bits(y), bits(gate), rows)


@pytest.mark.parametrize("m,n,k,bias", [(300, 512, 1024, True), (257, 200, 640, False), (1, 256, 256, True),
                                        (64, 3072, 3072, True), (515, 776, 208, True)])
def test_gated_residual_matches_oracle(dev, m, n, k, bias):
    print(f"gated residual m={m} n={n} k={k} bias={bias}", flush=True)
    x = activations(m, k, m + n)
    w, ws = int8_weight(n, k, k)
    b = bf16_vec(n, 5, 0.02) if bias else None
    gate = torch.randn(3, n, generator=gen(7)).to(torch.bfloat16)
    res = activations(m, n, 8) * 3
    segs = _segments(m, 4)
    rows = eager_np.segment_row_map(m, segs)
    out = res.to(dev)
    r = _mx().int8_linear_gated_residual_(out, x.to(dev), w.to(dev), ws.to(dev), None if b is None else b.to(dev),
                                          gate.to(dev), segs)
    assert r is out
    assert np.array_equal(bits(out), _expected(res, x, w, ws, b, gate, rows))


def test_gated_residual_equals_linear_then_addcmul_on_device(dev):
    """The fused update equals the reference's two-step composition run with torch on the GPU."""
    m, n, k = 200, 384, 512
    x = activations(m, k, 1).to(dev)
    w, ws = int8_weight(n, k, 2)
    w, ws = w.to(dev), ws.to(dev)
    b = bf16_vec(n, 3, 0.02).to(dev)
    gate = torch.randn(2, n, generator=gen(4)).to(dev)          # float32 gate, rounded per use
    res = (activations(m, n, 5) * 2).to(dev)
    segs = ((0, 50, 1), (50, 200, 0))
    ref = res.clone()
    y = _mx().int8_linear(x, w, ws, b)
    for a, c, row in segs:
        ref[a:c].addcmul_(y[a:c], gate[row].to(y.dtype))
    _mx().int8_linear_gated_residual_(res, x, w, ws, b, gate, segs)
    assert torch.equal(res, ref)


def test_gated_residual_strided_residual_and_row_tensor(dev):
    """A residual that is a column slice of a wider buffer (row stride > N, unaligned start,
    so the element-wise store path runs) and gate rows passed as a tensor."""
    m, n, k = 130, 200, 256
    x = activations(m, k, 11)
    w, ws = int8_weight(n, k, 12)
    gate = torch.randn(4, n, generator=gen(13)).to(torch.bfloat16)
    rows = torch.randint(0, 4, (m,), generator=gen(14), dtype=torch.int32)
    base = (activations(m, n + 9, 15) * 2)
    res = base[:, 3:3 + n]
    want = _expected(res, x, w, ws, None, gate, rows.numpy())
    dbase = base.to(dev)
    dres = dbase[:, 3:3 + n]
    _mx().int8_linear_gated_residual_(dres, x.to(dev), w.to(dev), ws.to(dev), None, gate.to(dev), rows.to(dev))
    assert np.array_equal(bits(dres), want)
    # the columns outside the slice are untouched
    assert torch.equal(dbase[:, :3].cpu(), base[:, :3]) and torch.equal(dbase[:, 3 + n:].cpu(), base[:, 3 + n:])


def test_fused_down_gated_residual_swiglu_convrot(dev):
    m, inner, n = 96, 1024, 512
    hidden = activations(m, 2 * inner, 21, outlier_frac=0.0)
    w, ws = int8_weight(n, inner, 22)
    b = bf16_vec(n, 23, 0.01)
    gate = torch.randn(2, n, generator=gen(24)).to(torch.bfloat16)
    res = activations(m, n, 25)
    segs = ((0, 32, 1), (32, 96, 0))
    rows = _mx().segment_row_map(m, segs, dev)
    out = res.to(dev)
    _mx().fused_down_gated_residual(hidden.to(dev), out, gate.to(dev), rows, w.to(dev), ws.to(dev), b.to(dev))
    want = _expected(res, hidden, w, ws, b, gate, rows.cpu().numpy(), g=256, act="swiglu")
    assert np.array_equal(bits(out), want)


def test_gated_residual_rejects_bad_maps(dev):
    m, n, k = 16, 64, 64
    x = activations(m, k, 1).to(dev)
    w, ws = int8_weight(n, k, 2)
    gate = torch.zeros(2, n, dtype=torch.bfloat16, device=dev)
    res = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):
        _mx().int8_linear_gated_residual_(res, x, w.to(dev), ws.to(dev), None, gate,
                                          torch.full((m,), 2, dtype=torch.int32))
    with pytest.raises(ValueError):
        _mx().int8_linear_gated_residual_(res, x, w.to(dev), ws.to(dev), None, gate, ((0, 8, 0), (9, 16, 1)))
    with pytest.raises(ValueError):
        _mx().int8_linear_gated_residual_(res[:8], x, w.to(dev), ws.to(dev), None, gate, ((0, 16, 0),))


# ---- RMS adaLN (+ ConvRot quantizer) -----------------------------------------------------------

def _rms_inputs(m, d, seed):
    x = activations(m, d, seed) * 2
    w = (1 + 0.2 * torch.randn(d, generator=gen(seed + 1))).to(torch.bfloat16)
    scale = (0.1 * torch.randn(3, d, generator=gen(seed + 2))).to(torch.bfloat16)
    shift = (0.1 * torch.randn(3, d, generator=gen(seed + 3))).to(torch.bfloat16)
    return x, w, scale, shift


def _check_rms_adaln_bound(y, x, w, scale, shift, rows, eps):
    """Modulated bf16 within 2 ulp(n·t) + ulp(y) of the oracle. The mean of squares is a
    reduction whose order differs from torch's CPU kernel, so the normalised value n may differ
    by one bf16 ulp; a = bf16(n·t) then differs by at most ulp(n)·t plus the two half-ulp
    roundings (<= 2 ulp(n·t)), and y = bf16(a + shift) by that plus the two half-ulp roundings
    of y (ulp(y)). Over 27 M elements a few reach more than 1 ulp(n·t); none exceed this."""
    from oracle.bf16 import bf16_bits, bf16_to_f32, bf16_ulp

    ref = eager_np.rms_adaln(bits(x), bits(w), eps, bits(scale), bits(shift), rows)
    yv, rv = bf16_to_f32(bits(y)), bf16_to_f32(ref)
    n64 = eager_np.rms_norm_f64(bits(x), bits(w), eps)
    t = bf16_to_f32(bf16_bits(np.float32(1.0) + bf16_to_f32(bits(scale))[rows]))
    tol = 2 * bf16_ulp(np.abs(n64 * t).astype(np.float32)) + bf16_ulp(np.maximum(np.abs(rv), np.abs(yv)))
    assert np.all(np.abs(yv - rv) <= tol)
    mismatch = float(np.mean(bits(y) != ref))
    print(f"rms_adaln bf16 mismatch rate vs torch CPU: {mismatch:.2e}")
    assert mismatch <= RMS_ADALN_MISMATCH_BOUND
    return mismatch


# Elements of the RMS adaLN bf16 output that differ from torch's CPU rms_norm composition.
# Measured on MI355X against the host's torch: 3.5e-6 of 22 M elements (4096 x 5376). The
# large-sample bound is about twice that; RMS_ADALN_MISMATCH_BOUND covers the small tests.
RMS_ADALN_MISMATCH_BOUND = 5e-5
RMS_ADALN_MISMATCH_LARGE = 7e-6


def test_rms_adaln_mismatch_rate_large_sample(dev):
    m, d, eps = 4096, 5376, 1e-6
    print(f"rms_adaln mismatch sample m={m} d={d}", flush=True)
    x, w, scale, shift = _rms_inputs(m, d, 4343)
    segs = _segments(m, 3)
    rows = eager_np.segment_row_map(m, segs)
    y = _mx().rms_adaln(x.to(dev), (w.to(dev), eps), shift.to(dev), scale.to(dev), segs)
    rate = _check_rms_adaln_bound(y, x, w, scale, shift, rows, eps)
    print(f"rms_adaln mismatch vs torch CPU over {m * d} elements: bf16 {rate:.3e}", flush=True)
    assert rate <= RMS_ADALN_MISMATCH_LARGE


@pytest.mark.parametrize("m,d,eps", [(64, 5120, 1e-6), (33, 1024, 1e-5), (7, 3072, 1e-6), (300, 5120, 1e-6)])
def test_rms_adaln_matches_oracle(dev, m, d, eps):
    print(f"rms_adaln m={m} d={d}", flush=True)
    x, w, scale, shift = _rms_inputs(m, d, m + d)
    segs = _segments(m, 3)
    rows = eager_np.segment_row_map(m, segs)
    y = _mx().rms_adaln(x.to(dev), (w.to(dev), eps), shift.to(dev), scale.to(dev), segs)
    _check_rms_adaln_bound(y, x, w, scale, shift, rows, eps)


@pytest.mark.parametrize("g", [256, 0])
def test_rms_adaln_quantize_matches_oracle(dev, g):
    m, d, eps = 150, 5120, 1e-6
    x, w, scale, shift = _rms_inputs(m, d, 9 + g)
    segs = ((0, 20, 2), (20, 64, 1), (64, 150, 0))
    rows = eager_np.segment_row_map(m, segs)

    class Norm:  # the reference's RMSNorm attributes
        weight = w.to(dev)
        eps = 1e-6

    q, s, y = _mx().rms_adaln_quantize_int8(x.to(dev), Norm, shift.to(dev), scale.to(dev), segs,
                                            convrot_groupsize=g, return_modulated=True)
    _check_rms_adaln_bound(y, x, w, scale, shift, rows, eps)
    # the quantizer of the kernel's own modulated rows is bit-exact
    qr, sr, _ = cr.convrot_quantize_bf16(bits(y), g)
    assert np.array_equal(q.cpu().numpy(), qr) and np.array_equal(s.cpu().numpy(), sr)
    # the standalone norm and the fused path agree exactly; a row map tensor is the same as segments
    y2 = _mx().rms_adaln(x.to(dev), Norm, shift.to(dev), scale.to(dev), torch.from_numpy(rows))
    assert torch.equal(y, y2)
    q3, s3 = _mx().rms_adaln_quantize_int8(x.to(dev), Norm, shift.to(dev), scale.to(dev), segs, convrot_groupsize=g)
    assert torch.equal(q3, q) and torch.equal(s3, s)


def test_rms_adaln_rejects_bad_segments(dev):
    x, w, scale, shift = _rms_inputs(16, 256, 3)
    args = (x.to(dev), (w.to(dev), 1e-6), shift.to(dev), scale.to(dev))
    with pytest.raises(ValueError):
        _mx().rms_adaln(*args, ((0, 8, 0), (9, 16, 1)))
    with pytest.raises(ValueError):
        _mx().rms_adaln(*args, ((0, 16, 3),))
    with pytest.raises(ValueError):
        _mx().rms_adaln_quantize_int8(*args, ((0, 16, 0),), convrot_groupsize=1024)


@pytest.mark.parametrize("mapping", ["segments", "random"])
def test_rms_adaln_quantize_h3_width_many_rows(dev, mapping):
    """5000 rows of the H3 hidden size (27 M elements) under three modulation segments or a
    random row map that changes the modulation row on most rows: the modulated rows within the
    stated bound, the quantized rows bit-exact, the standalone norm identical."""
    m, d, eps = 5000, 5376, 1e-6
    print(f"rms_adaln quant h3 width m={m} d={d} mapping={mapping}", flush=True)
    x, w, scale, shift = _rms_inputs(m, d, 77)
    if mapping == "segments":
        segs = ((0, 1700, 2), (1700, 3400, 0), (3400, m, 1))
        rows = eager_np.segment_row_map(m, segs)
    else:
        rows = torch.randint(0, 3, (m,), generator=gen(78), dtype=torch.int32).numpy()
        segs = torch.from_numpy(rows)
    q, s, y = _mx().rms_adaln_quantize_int8(x.to(dev), (w.to(dev), eps), shift.to(dev), scale.to(dev), segs,
                                            convrot_groupsize=256, return_modulated=True)
    _check_rms_adaln_bound(y, x, w, scale, shift, rows, eps)
    qr, sr, _ = cr.convrot_quantize_bf16(bits(y), 256)
    assert np.array_equal(q.cpu().numpy(), qr) and np.array_equal(s.cpu().numpy(), sr)
    y2 = _mx().rms_adaln(x.to(dev), (w.to(dev), eps), shift.to(dev), scale.to(dev), segs)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("m,ld_pad", [(777, 0), (777, 40), (3, 40)])
def test_rms_adaln_modulation_workspace_changes_nothing(dev, m, ld_pad):
    """Through the C-ABI: the same call with the modulation workspace (bf16(1 + scale) formed
    once per call), with one 16 bytes too small and with none gives identical q, scales and y,
    also for scale / shift rows strided beyond the hidden size, and in a three-row launch (one
    unit of 256 columns per 16-lane group); the quantizer of the modulated rows is bit-exact."""
    from mx_qlinear import _lib
    from mx_qlinear.ops import _p, _stream

    d, eps, mods = 5376, 1e-6, 5
    print(f"rms_adaln workspace m={m} d={d} ld_pad={ld_pad}", flush=True)
    x, w, _, _ = _rms_inputs(m, d, 91 + ld_pad)
    ld = d + ld_pad
    scale = (0.1 * torch.randn(mods, ld, generator=gen(92))).to(torch.bfloat16).to(dev)
    shift = (0.1 * torch.randn(mods, ld, generator=gen(93))).to(torch.bfloat16).to(dev)
    rows = torch.randint(0, mods, (m,), generator=gen(94), dtype=torch.int32).to(dev)
    x, w = x.to(dev), w.to(dev)
    outs = []
    for ws_bytes in (mods * ld * 2, mods * ld * 2 - 16, 0):
        ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=dev)
        q = torch.empty((m, d), dtype=torch.int8, device=dev)
        s = torch.empty((m, 1), dtype=torch.float32, device=dev)
        y = torch.empty((m, d), dtype=torch.bfloat16, device=dev)
        _lib.call("mxq_rms_adaln_quantize_int8", _p(x), _p(w), _p(scale), _p(shift), ld, mods, _p(rows), eps, _p(y),
                  _p(q), _p(s), m, d, 256, _p(ws) if ws_bytes else None, ws_bytes, _stream(dev))
        torch.cuda.synchronize()
        outs.append((q, s, y))
    for q, s, y in outs[1:]:
        assert torch.equal(q, outs[0][0]) and torch.equal(s, outs[0][1]) and torch.equal(y, outs[0][2])
    qr, sr, _ = cr.convrot_quantize_bf16(bits(outs[0][2].cpu()), 256)
    assert np.array_equal(outs[0][0].cpu().numpy(), qr) and np.array_equal(outs[0][1].cpu().numpy().reshape(-1), sr.reshape(-1))
    # and the modulated rows are the oracle's within the stated bound
    _check_rms_adaln_bound(outs[0][2].cpu(), x.cpu(), w.cpu(), scale[:, :d].contiguous().cpu(), shift[:, :d].contiguous().cpu(),
                           rows.cpu().numpy(), eps)


@pytest.mark.parametrize("over", [0, 1])
def test_rms_adaln_modulation_table_from_many_rows(dev, over):
    """The workspace holds bf16(1 + scale) after a call of more than RMS_ADALN_TABLE_ROWS rows and is untouched by one
    of that many; q, scales and y are those of a call without it, for modulation rows strided beyond the hidden size."""
    from mx_qlinear import _lib
    from mx_qlinear.ops import _p, _stream

    m, d, eps, mods, ld = _lib.RMS_ADALN_TABLE_ROWS + over, 768, 1e-6, 5, 768 + 40
    print(f"rms_adaln table m={m} d={d}", flush=True)
    x, w, _, _ = _rms_inputs(m, d, 95)
    scale = (0.1 * torch.randn(mods, ld, generator=gen(96))).to(torch.bfloat16).to(dev)
    shift = (0.1 * torch.randn(mods, ld, generator=gen(97))).to(torch.bfloat16).to(dev)
    rows = torch.randint(0, mods, (m,), generator=gen(98), dtype=torch.int32).to(dev)
    x, w = x.to(dev), w.to(dev)
    outs = []
    for ws_bytes in (mods * ld * 2, mods * ld * 2 - 16, 0):
        ws = torch.full((max(ws_bytes, 1),), 0x5A, dtype=torch.uint8, device=dev)
        q = torch.empty((m, d), dtype=torch.int8, device=dev)
        s = torch.empty((m, 1), dtype=torch.float32, device=dev)
        y = torch.empty((m, d), dtype=torch.bfloat16, device=dev)
        _lib.call("mxq_rms_adaln_quantize_int8", _p(x), _p(w), _p(scale), _p(shift), ld, mods, _p(rows), eps, _p(y),
                  _p(q), _p(s), m, d, 256, _p(ws) if ws_bytes else None, ws_bytes, _stream(dev))
        outs.append((q, s, y))
        if over and ws_bytes == mods * ld * 2:
            table = ws.view(torch.bfloat16).reshape(mods, ld)[:, :d]
            assert torch.equal(table, (1 + scale[:, :d].float()).to(torch.bfloat16))
        else:
            assert bool((ws == 0x5A).all())
    for q, s, y in outs[1:]:
        assert torch.equal(q, outs[0][0]) and torch.equal(s, outs[0][1]) and torch.equal(y, outs[0][2])
    pick = torch.arange(0, m, 97)
    qr, sr, _ = cr.convrot_quantize_bf16(bits(outs[0][2][pick.to(dev)].cpu()), 256)
    assert np.array_equal(outs[0][0][pick.to(dev)].cpu().numpy(), qr)
    assert np.array_equal(outs[0][1][pick.to(dev)].cpu().numpy().reshape(-1), sr.reshape(-1))
