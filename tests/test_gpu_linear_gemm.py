"""The matrix-core linear (linear_gemm.hip) behind tsa_gguf_matvec, tsa_mxfp4_matvec and
tsa_router_logits for many bf16 tokens: tile edges, ragged sizes, every tile shape, rows that
start inside a super-block, unaligned weights and results that are not finite."""
from __future__ import annotations

import os
import re

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
    fp32 summation (K 2^-24) of the sum of absolute products."""
    ref, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    if bias is not None:
        ref, mag = ref + bias, mag + np.abs(bias)
    d = np.abs(y.double().cpu().numpy() - ref)
    bound = 2.0 ** -8 * np.abs(ref) + w.shape[1] * 2.0 ** -24 * mag
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


def _tile(N, T, mxfp4):
    """The tile lg_pick takes (32 x first tokens, 256 / second rows), from the source's table."""
    src = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinyserve_amd", "csrc",
                            "linear_gemm.hip")).read()
    table = re.findall(r"\{(\d), (\d), (?:MX \? (\d+) : )?(\d+)\}", re.search(r"constexpr Tile tiles\[5\] = (.*);", src)[1])
    assert len(table) == 5
    cus = torch.cuda.get_device_properties(0).multi_processor_count

    def cost(mt, kw, mx, other):
        wgs = -(-N // (256 // int(kw))) * -(-T // (32 * int(mt)))
        return -(-wgs // cus) * int(mx if mx and mxfp4 else other)

    return min(((int(mt), int(kw)) for mt, kw, *_ in table), key={(int(t[0]), int(t[1])): cost(*t) for t in table}.get)


@pytest.mark.parametrize("tile,T", [((1, 8), 20), ((1, 4), 95), ((2, 4), 130), ((2, 2), 499), ((4, 2), 1020)])
@pytest.mark.parametrize("fmt,K", [(8, 1312), (12, 1280), (13, 1280), (14, 1280), (12, 1312), (13, 1312), (14, 1312),
                                   ("mxfp4", 1312), ("bf16", 1312)])
def test_tiles(fmt, K, tile, T):
    """Each tile over several K steps (1024, 512 or 256 values each) with a partial last one wherever
    the format allows it, in whole and straddling rows, with ragged rows and tokens."""
    N = 4088
    assert _tile(N, T, fmt == "mxfp4") == tile
    rng = np.random.default_rng(K + T)
    x, xd = _x(rng, T, K)
    if fmt == "mxfp4":
        blocks = rng.integers(0, 256, size=(N, K // 32, 16), dtype=np.uint8)
        scales = rng.integers(110, 130, size=(N, K // 32), dtype=np.uint8)
        w = omx.dequant_mxfp4_no_transpose(blocks, scales, "f32")
        y = ops.mxfp4_matvec(xd, torch.from_numpy(blocks).cuda(), torch.from_numpy(scales).cuda())
    elif fmt == "bf16":
        wt = torch.from_numpy(rng.normal(0.0, K ** -0.5, (N, K)).astype(np.float32)).to(torch.bfloat16)
        w, y = wt.float().numpy(), ops.router_logits(xd, wt.cuda())
    else:
        data = synth.make_gguf(rng, fmt, N * K)
        w, y = og.dequant_tensor(data, fmt, (N, K)), ops.gguf_matvec(xd, dev_u8(data), fmt, N, K)
    _check(y, x, w.astype(np.float64))


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
                                          (2880, 160, 700, 3), (64, 8192, 64, 0), (65, 8192, 64, 0), (33, 4128, 33, 2)])
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


@pytest.mark.parametrize("E,H,T", [(1, 32, 5), (60, 2048, 31), (33, 96, 200), (128, 2880, 700), (128, 512, 7), (128, 512, 8),
                                   (33, 544, 5)])
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


def _us(fn, n=20):
    best = float("inf")
    for _ in range(4):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(n):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / n)
    return best


def test_not_finite_cost():
    """One NaN token must not hold up the call: its results are NaN after one look at the token (a
    thread forming 8 results one after the other in fp32 took 60 times the call's time)."""
    rng = np.random.default_rng(3)
    N, K, T = 2048, 4096, 24
    w = dev_u8(synth.make_gguf(rng, 14, N * K))
    _, x = _x(rng, T, K)
    y = ops.gguf_matvec(x, w, 14, N, K)
    t0 = _us(lambda: ops.gguf_matvec(x, w, 14, N, K))
    x[5, 17] = float("nan")
    z = ops.gguf_matvec(x, w, 14, N, K)
    t1 = _us(lambda: ops.gguf_matvec(x, w, 14, N, K))
    rest = [t for t in range(T) if t != 5]
    assert z[5].isnan().all() and torch.equal(z[rest], y[rest])
    assert t1 < 4 * t0, f"{t0:.1f} us, with a NaN token {t1:.1f}"


@pytest.mark.parametrize("gtype", [8, 12, 14])
@pytest.mark.parametrize("N,T", [(64, 16), (32, 33)])
def test_few_rows_long_k(gtype, N, T):
    """Few rows of a long K, where the GEMM has one or two workgroups, take the row kernel, as fp32
    tokens do (the GEMM took 2.5 to 5 times as long)."""
    rng = np.random.default_rng(gtype + N)
    K = 16384
    data = synth.make_gguf(rng, gtype, N * K)
    x, xd = _x(rng, T, K)
    w, xf = dev_u8(data), xd.float()
    _check(ops.gguf_matvec(xd, w, gtype, N, K), x, og.dequant_tensor(data, gtype, (N, K)).astype(np.float64))
    t0, t1 = _us(lambda: ops.gguf_matvec(xf, w, gtype, N, K)), _us(lambda: ops.gguf_matvec(xd, w, gtype, N, K))
    assert t1 < 1.6 * t0, f"{t1:.1f} us, fp32 tokens {t0:.1f}"


@pytest.mark.parametrize("gtype", [8, 12, 13, 14])
@pytest.mark.parametrize("T", [9, 70, 130])
def test_weights_whole(gtype, T):
    """Weights enter with all their fp32 bits. Rows hold a block at the scales 1707, 1706 and 1 x 2^-10
    (the last with codes of its own) against tokens +-1 with the signs +, -, -, so the sums cancel to
    2^-10 of their products. All products are multiples of 2^-10 whose absolute sum stays under 2^14:
    fp32 adds them exactly in any order, and every result is the exact sum's nearest bf16."""
    rng = np.random.default_rng(gtype + T)
    N, (be, ts), dof = 64, ops.gguf_block_info(gtype), 208 if gtype == 14 else 0
    base = synth.make_gguf(rng, gtype, 2 * N * be).reshape(2, N, ts)
    if gtype == 14:
        base[:, :, 192:208] = rng.integers(-15, 16, (2, N, 16)).astype(np.int8).view(np.uint8)
    blocks = np.stack([base[0], base[0], base[1]], 1)  # [N, 3, ts]
    for i, d in enumerate((1707, 1706, 1)):
        blocks[:, i, dof:dof + 2] = np.array([d * 2.0 ** -10], np.float16).view(np.uint8)
        if gtype in (12, 13):
            blocks[:, i, 2:4] = blocks[:, i, 0:2]  # dmin
    w = og.dequant_tensor(blocks.reshape(-1), gtype, (N, 3 * be)).astype(np.float64)
    x = np.zeros((T, 3, be))
    for k in rng.permutation(be):
        s = rng.choice([-1.0, 1.0], T)
        x[:, 0, k], x[:, 1, k], x[:, 2, k] = s, -s, -s
        if (np.abs(x[0]).reshape(-1) @ np.abs(w).T).max() >= 2.0 ** 14:
            x[:, :, k] = 0.0
            break
    x = x.reshape(T, -1)
    assert (w * 2 ** 10 == np.round(w * 2 ** 10)).all() and np.count_nonzero(x[0]) >= 6
    y = ops.gguf_matvec(torch.from_numpy(x).to(torch.bfloat16).cuda(), dev_u8(blocks.reshape(-1)), gtype, N, 3 * be)
    ref = torch.from_numpy((x @ w.T).astype(np.float32)).to(torch.bfloat16)
    assert torch.equal(y.cpu(), ref)
