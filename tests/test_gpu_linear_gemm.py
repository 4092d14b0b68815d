"""The matrix-core linear (linear_gemm.hip) behind tsa_gguf_matvec, tsa_mxfp4_matvec and
tsa_router_logits for many bf16 tokens: tile edges, ragged sizes, every tile shape, rows that
start inside a super-block, unaligned weights and results that are not finite."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import gguf as og
from oracle import mxfp4 as omx
from tests.helpers import dev_u8
from tinyserve_amd import ops, synth

pytestmark = pytest.mark.gpu


def _x(rng, T, K):
    xt = torch.from_numpy(rng.normal(0.0, 1.0, (T, K)).astype(np.float32)).to(torch.bfloat16)
    return xt.double().numpy(), xt.cuda()


def _check(y, x, w, bias=None):
    """Each result within one bf16 rounding (2^-9, twice that for a rounding on the edge) plus
    the split weights' 2^-17 and fp32 summation (K 2^-24) of the sum of absolute products."""
    ref, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    if bias is not None:
        ref, mag = ref + bias, mag + np.abs(bias)
    d = np.abs(y.double().cpu().numpy() - ref)
    bound = 2.0 ** -8 * np.abs(ref) + (2.0 ** -17 + w.shape[1] * 2.0 ** -24) * mag
    assert (d <= bound).all(), f"worst {np.max(d / np.maximum(bound, 1e-30)):.3f} of the bound"


SMALL = [(8, 32, 9), (40, 96, 33), (33, 256, 65), (130, 512, 64), (96, 2880, 129), (24, 1120, 32), (31, 1280, 10)]
# 256 CUs pick each of the five tiles: 32 x 32 rows, then 32 x 64, 64 x 64, 64 x 128, 128 x 128
TILES = [(4096, 256, 20), (4096, 256, 96), (4096, 256, 130), (4096, 256, 500), (4096, 256, 1500), (4096, 96, 1500)]


@pytest.mark.parametrize("gtype", [8, 12, 13, 14])
@pytest.mark.parametrize("N,K,T", SMALL + TILES)
def test_gguf_linear(gtype, N, K, T):
    rng = np.random.default_rng(N + 3 * K + T + gtype)
    data = synth.make_gguf(rng, gtype, N * K) if gtype == 8 or N * K % 256 == 0 else None
    if data is None:
        pytest.skip("not a whole number of super-blocks")
    x, xd = _x(rng, T, K)
    _check(ops.gguf_matvec(xd, dev_u8(data), gtype, N, K), x, og.dequant_tensor(data, gtype, (N, K)).astype(np.float64))


@pytest.mark.parametrize("gtype,K", [(8, 96), (14, 512), (14, 288)])
@pytest.mark.parametrize("offset", [2, 6, 14])
def test_gguf_linear_2byte_aligned(gtype, K, offset):
    rng = np.random.default_rng(K + offset)
    N, T = 64, 40
    data = synth.make_gguf(rng, gtype, N * K)
    x, xd = _x(rng, T, K)
    _check(ops.gguf_matvec(xd, dev_u8(data, offset=offset), gtype, N, K), x,
           og.dequant_tensor(data, gtype, (N, K)).astype(np.float64))


@pytest.mark.parametrize("N,K,T,offset", [(33, 32, 40, 0), (100, 96, 33, 1), (5760, 2880, 12, 0), (1536, 2080, 77, 2),
                                          (2880, 160, 700, 3)])
def test_mxfp4_linear(N, K, T, offset):
    rng = np.random.default_rng(N + K + T)
    blocks = rng.integers(0, 256, size=(N, K // 32, 16), dtype=np.uint8)
    scales = rng.integers(110, 130, size=(N, K // 32), dtype=np.uint8)
    bias = rng.normal(0.0, 0.5, N).astype(np.float32)
    x, xd = _x(rng, T, K)
    w = omx.dequant_mxfp4_no_transpose(blocks, scales, "f32").astype(np.float64)
    y = ops.mxfp4_matvec(xd, torch.from_numpy(blocks).cuda(), dev_u8(scales, offset=offset).view(N, K // 32),
                         torch.from_numpy(bias).cuda())
    _check(y, x, w, bias.astype(np.float64))


@pytest.mark.parametrize("E,H,T", [(1, 32, 5), (60, 2048, 31), (33, 96, 200), (128, 2880, 700)])
def test_router_batch(E, H, T):
    rng = np.random.default_rng(E + H + T)
    x, xd = _x(rng, T, H)
    w = torch.from_numpy(rng.normal(0.0, H ** -0.5, (E, H)).astype(np.float32)).to(torch.bfloat16)
    b = torch.from_numpy(rng.normal(0.0, 0.1, E).astype(np.float32)).to(torch.bfloat16)
    _check(ops.router_logits(xd, w.cuda(), b.cuda()), x, w.double().numpy(), b.double().numpy())


@pytest.mark.parametrize("fmt", [8, 12, 13, 14, "mxfp4", "router"])
def test_not_finite(fmt):
    """Infinite and NaN activations give what the plain products give: inf where every product
    with the value has one sign, NaN where a weight is zero or signs meet."""
    rng = np.random.default_rng(9)
    N, K, T = 48, 512, 40
    x, xd = _x(rng, T, K)
    for t, k, v in ((3, 17, np.inf), (7, 300, -np.inf), (9, 5, np.nan), (11, 0, np.inf), (11, 511, np.inf)):
        x[t, k] = v
        xd[t, k] = v
    if fmt == "mxfp4":
        blocks = rng.integers(0, 256, size=(N, K // 32, 16), dtype=np.uint8)
        scales = rng.integers(119, 126, size=(N, K // 32), dtype=np.uint8)
        w = omx.dequant_mxfp4_no_transpose(blocks, scales, "f32")
        y = ops.mxfp4_matvec(xd, torch.from_numpy(blocks).cuda(), torch.from_numpy(scales).cuda())
    elif fmt == "router":
        wt = torch.from_numpy(rng.normal(size=(N, K)).astype(np.float32)).to(torch.bfloat16)
        w = wt.float().numpy()
        y = ops.router_logits(xd, wt.cuda())
    else:
        data = synth.make_gguf(rng, fmt, N * K)
        w = og.dequant_tensor(data, fmt, (N, K))
        y = ops.gguf_matvec(xd, dev_u8(data), fmt, N, K)
    with np.errstate(invalid="ignore"):
        ref = np.stack([(x[t] * w.astype(np.float64)).sum(1) for t in range(T)])
    y = y.double().cpu().numpy()
    for t in (3, 7, 9, 11):
        assert np.array_equal(np.isnan(y[t]), np.isnan(ref[t])) and np.array_equal(y[t][np.isinf(ref[t])], ref[t][np.isinf(ref[t])])
    fine = [t for t in range(T) if t not in (3, 7, 9, 11)]
    _check(torch.from_numpy(y[fine]), x[fine], w.astype(np.float64))
