"""GPU parity of the reference-format int4 routes: the decode through tables of 16 levels against the
oracle, also for scales and codebooks that are not finite, and the few-row GEMM that decodes in
registers against the decode + GEMM route (one column per chunk leaves no room for its sums), bit for
bit, with the workspace read back to see which of the two ran."""

import numpy as np
import pytest
import torch

import mx_qlinear as mx
import mx_qlinear._lib as L
from _util import bf16_vec, gen, packed_int4
from mx_qlinear.ops import _p, _stream
from oracle import eager_np

pytestmark = pytest.mark.gpu

CODEBOOK = torch.tensor([-0.98, -0.79, -0.63, -0.5, -0.37, -0.26, -0.15, -0.05, 0.0, 0.15, 0.26, 0.38, 0.5, 0.64, 0.79, 0.98])


def _scales(n, groups, e4m3, seed):
    if e4m3:  # every byte value, NaN included
        return torch.randint(0, 256, (n, groups), generator=gen(seed), dtype=torch.uint8).view(torch.float8_e4m3fn)
    s = torch.randn(n, groups, generator=gen(seed)) * 60
    s.view(-1)[::7] = 0.5  # ties
    s.view(-1)[::11] = torch.tensor([float("inf"), float("-inf"), float("nan"), 3e38, 1e-45, -0.0])[
        torch.arange(s.view(-1)[::11].numel()) % 6]
    return s


@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("codebook", ["none", "finite", "inf"])
# Few weights; many by levels in whole rows of one piece and of several, and in pieces of rows (the last of one vector).
@pytest.mark.parametrize("n,k,g", [(7, 272, 4), (5, 160, 8), (1, 16, 16), (5, 1040, 16), (3, 4112, 16), (9, 1536, 48), (70, 2048, 64),
                                   (6800, 1552, 16), (4099, 4112, 16), (1281, 8208, 48)])
def test_decode_levels(dev, n, k, g, codebook, e4m3):
    qd, s = packed_int4(n, k, k + g), _scales(n, k // g, e4m3, n + k)
    cb = None if codebook == "none" else CODEBOOK.clone()
    if codebook == "inf":
        cb[3], cb[9] = float("inf"), float("nan")
    w8 = mx.dequantize_int4_grouped_to_int8(qd.to(dev), s.to(dev), None if cb is None else cb.to(dev), g).cpu().numpy()
    codes = eager_np.unpack_int4(qd.numpy())
    v = (codes - 8).astype(np.float32) if cb is None else cb.numpy()[codes]
    with np.errstate(all="ignore"):
        prod = v * np.repeat(s.float().numpy(), g, axis=1)
        want = np.where(np.isnan(prod), 0, np.clip(np.rint(prod), -127, 127)).astype(np.int8)  # a NaN decodes to 0
    assert np.array_equal(w8, want)


def _slices(work, acc, n):
    """How many slices of int32 sums [m, n padded to a multiple of 4] at the front of ``work`` add up to acc; 0: none do."""
    m, ldp = acc.shape[0], (n + 3) // 4 * 4
    room = work.numel() // (4 * m * ldp)
    part = work.reshape(-1)[: 4 * room * m * ldp].view(torch.int32).reshape(room, m, ldp)[:, :, :n].to(torch.int64).cumsum(0)
    hits = [s + 1 for s in range(room) if torch.equal(part[s], acc)]
    return hits[0] if hits else 0


# Both sides of each row block and of the split, ragged columns, one stage, an uneven last slice, two and three 128-row
# tiles with one slice and with several. Past 128 rows fp32 scales of group 16 decode to memory by rule; the workspace
# shows which route ran: the slices' sums, or the decoded weights.
@pytest.mark.parametrize("m,n,k", [(1, 257, 256), (20, 1000, 2304), (32, 130, 5376), (33, 255, 512), (64, 513, 2816),
                                   (65, 3, 1024), (128, 300, 4352), (129, 260, 1280), (300, 258, 1536), (384, 514, 1792),
                                   (384, 130, 5376), (385, 130, 5376)])
@pytest.mark.parametrize("g,e4m3", [(16, True), (32, True), (64, True), (16, False), (32, False), (64, False)])
def test_few_row_gemm(dev, m, n, k, g, e4m3):
    print(f"few rows m={m} n={n} k={k} g={g} e4m3={e4m3}", flush=True)
    xq = torch.randint(-128, 128, (m, k), generator=gen(m + k), dtype=torch.int8).to(dev)
    xs = (torch.rand(m, generator=gen(1)) * 1e-2).to(dev)
    qd = packed_int4(n, k, n).to(dev)
    s = torch.rand(n, k // g, generator=gen(2)) * 100 + 40
    s = (s.to(torch.float8_e4m3fn) if e4m3 else s).to(dev)
    sch = (torch.rand(n, generator=gen(3)) * 1e-3).to(dev)
    cb = CODEBOOK.to(dev)
    bias = bf16_vec(n, 5, 0.01).to(dev) if n % 2 else None
    w8 = mx.dequantize_int4_grouped_to_int8(qd, s, cb, g)
    acc = (xq.cpu().double() @ w8.cpu().double().t()).to(torch.int64)  # exact
    outs = []
    for chunk in (n, 1):
        work = torch.full((chunk, k), 0x5A, dtype=torch.int8, device=dev)
        y = torch.zeros((m, n), dtype=torch.bfloat16, device=dev)
        L.call("mxq_w4a8_codebook_gemm", _p(xq), _p(qd), _p(s), L.DTYPE_E4M3 if e4m3 else L.DTYPE_F32, _p(cb), _p(sch),
               _p(xs), _p(bias), _p(work), _p(y), m, n, k, g, chunk, L.DTYPE_BF16, None, 0, _stream(dev))
        outs.append(y)
        if chunk == n and (m <= 128 or (m <= 384 and (e4m3 or g > 16))):
            assert _slices(work.cpu(), acc, n) > 0, "the sums of the few-row GEMM are not in the workspace"
        else:
            assert torch.equal(work, w8[n - chunk:]), "the last chunk's decoded weights are not in the workspace"
    assert torch.equal(outs[0], outs[1])
    want = (acc.float() * (xs.cpu()[:, None] * sch.cpu()[None, :])).to(torch.bfloat16)  # (float32 of the sum, rounded once)
    if n % 2:
        want = (want.float() + bias.cpu().float()).to(torch.bfloat16)
    assert torch.equal(outs[0].cpu(), want)
