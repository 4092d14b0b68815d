"""The performance cases of this library: what a serving program has it do.

Two model shapes run through it, the ones the benchmark and the tests use: an MXFP4 MoE layer
(hidden = inter = 2880, 32 experts, top-4, clamped SwiGLU with biases, slots in the tile order)
and GGUF MoE layers (hidden 2048, inter 768, 128 experts, top-8; and hidden = inter = 2880, 32
experts, top-4, whose rows straddle super-blocks). Around them: the GGUF linears of the
attention and shared-expert projections (``GGMLLinear``), the standalone MXFP4 linear of a
template expert, the router linear, and dequantisation of whole tensors.

Weights are random codes with scales that give them the size real weights have; activations are
N(0, 1) with a few larger channels, as the residual stream has. A case is a dict of plain values;
``prepare`` builds a program's state from it, ``run`` makes one pass, ``exact`` is the same
result in 64 bits from plain torch.
"""
from __future__ import annotations

import numpy as np
import torch

from tinyserve_amd import ops, synth
from tinyserve_amd.expert_forward import gguf_expert_layout, mxfp4_expert_layout
from tinyserve_amd.ggml_linear import GGMLLinear
from tinyserve_amd.mxfp4 import mxfp4_linear

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
MXFP4 = 0  # not a ggml type id: the MXFP4 format, where a case may name either
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}  # values, bytes
WSTD = 0.03  # the weights' standard deviation

MX_MOE = {"H": 2880, "I": 2880, "E": 32, "k": 4, "gate": MXFP4, "down": MXFP4}
GG_MOE = {"H": 2048, "I": 768, "E": 128, "k": 8, "gate": Q5_K, "down": Q6_K}
GG_MOE_2880 = {"H": 2880, "I": 2880, "E": 32, "k": 4, "gate": Q4_K, "down": Q6_K}


# ----------------------------------------------------------------------------- the cases
def listed() -> list[dict]:
    return [
        # one projection of a decode step, called by itself: launch and call latency
        {"name": "linear q8_0 decode", "op": "linear", "type": Q8_0, "N": 2880, "K": 2880, "T": 1, "dtype": "bf16",
         "bias": False},
        # the same layer for a decode batch of 24 sequences
        {"name": "linear q6_k batch", "op": "linear", "type": Q6_K, "N": 2048, "K": 4096, "T": 24, "dtype": "bf16",
         "bias": False},
        # the query projection over a prompt of 512 tokens
        {"name": "linear q4_k prefill", "op": "linear", "type": Q4_K, "N": 4096, "K": 2048, "T": 512, "dtype": "bf16",
         "bias": False},
        # an expert's gate_up as a module of its own, over the tokens a prompt sends to it
        {"name": "mxfp4 linear", "op": "mxlinear", "N": 5760, "K": 2880, "T": 77},
        # the router of a layer over a long prompt
        {"name": "router prefill", "op": "router", "E": 128, "H": 2048, "T": 2048},
        # a projection's weights decoded to bf16 (a program that wants them in full)
        {"name": "dequant q5_k", "op": "dequant", "type": Q5_K, "N": 8192, "K": 4096, "dtype": "bf16"},
        # one token through a stack of MoE layers, as a captured decode step replays it
        {"name": "mxfp4 decode", "op": "decode", **MX_MOE, "layers": 8, "T": 1},
        {"name": "gguf decode", "op": "decode", **GG_MOE, "layers": 8, "T": 1},
        # a decode batch of 24 sequences through one MoE layer
        {"name": "mxfp4 moe batch", "op": "moe", **MX_MOE, "T": 24},
        # prompts: the benchmark's long one, its GGUF ones, and one of odd length
        {"name": "mxfp4 moe prefill", "op": "moe", **MX_MOE, "T": 2048},
        {"name": "gguf moe prefill", "op": "moe", **GG_MOE, "T": 1024},
        {"name": "gguf moe prefill 2880", "op": "moe", **GG_MOE_2880, "T": 301},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng) -> dict:
    """One more case of the same kinds: token counts over the logarithm of their range."""
    op = rng.choice(["linear", "linear", "mxlinear", "router", "dequant", "decode", "moe", "moe", "moe"])
    if op == "linear":
        N, K = rng.choice([(2880, 2880), (4096, 2048), (2048, 4096), (512, 2048), (768, 2048), (2880, 4096),
                           (4096, 2880)])
        T = _log_int(rng, 1, 1536)
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"]) if T <= 8 else "bf16"
        return {"op": op, "type": rng.choice([Q8_0, Q4_K, Q5_K, Q6_K]), "N": N, "K": K, "T": T, "dtype": dtype,
                "bias": rng.random() < 0.25}
    if op == "mxlinear":
        N, K = rng.choice([(5760, 2880), (2880, 2880), (1536, 2048), (2048, 768)])
        return {"op": op, "N": N, "K": K, "T": _log_int(rng, 1, 700)}
    if op == "router":
        E, H = rng.choice([(32, 2880), (128, 2048), (64, 4096), (60, 2048)])
        return {"op": op, "E": E, "H": H, "T": _log_int(rng, 1, 4096)}
    if op == "dequant":
        N, K = rng.choice([(4096, 2048), (5760, 2880), (8192, 4096), (2880, 2880)])
        return {"op": op, "type": rng.choice([MXFP4, Q8_0, Q4_K, Q5_K, Q6_K]), "N": N, "K": K,
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"])}
    if op == "decode":
        shape = rng.choice([MX_MOE, GG_MOE, {**GG_MOE, "gate": Q4_K}, GG_MOE_2880])
        return {"op": op, **shape, "layers": 8, "T": rng.randint(1, 4)}
    shape = rng.choice([MX_MOE, MX_MOE, GG_MOE, {**GG_MOE, "gate": Q4_K}, {**GG_MOE, "gate": Q8_0, "down": Q8_0},
                        GG_MOE_2880])
    return {"op": op, **shape, "T": _log_int(rng, 5, 2047 if shape["gate"] == MXFP4 else 1023)}


# ----------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _acts(g, *shape, dtype=torch.bfloat16) -> torch.Tensor:
    """N(0, 1), one channel in 256 six times larger."""
    x = torch.randn(shape, device=DEV, generator=g)
    x *= torch.where(torch.rand(shape[-1], device=DEV, generator=g) < 1 / 256, 6.0, 1.0)
    return x.to(dtype)


def _bytes(g, *shape, lo: int = 0, hi: int = 256) -> torch.Tensor:
    return torch.randint(lo, hi, shape, dtype=torch.uint8, device=DEV, generator=g)


def _half(g, n: int, mid: float) -> torch.Tensor:
    """n fp16 scales around mid, as bytes [n, 2]."""
    v = (mid * (1.0 + 0.25 * torch.randn(n, device=DEV, generator=g))).abs().to(torch.float16)
    return v.view(torch.uint8).view(n, 2)


def _gguf(g, ty: int, n: int) -> torch.Tensor:
    """n values as GGUF blocks of random codes, as bytes; standard deviation about WSTD."""
    be, ts = BLOCK[ty]
    nb = n // be
    b = _bytes(g, nb, ts)
    if ty == Q8_0:
        b[:, 0:2] = _half(g, nb, WSTD / 74)
    elif ty == Q6_K:  # signed sub-scales of either sign
        s = torch.randint(32, 128, (nb, 16), device=DEV, generator=g)
        s *= 2 * torch.randint(0, 2, (nb, 16), device=DEV, generator=g) - 1
        b[:, 192:208] = s.to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _half(g, nb, WSTD / (84 * 18.5))
    else:  # equal sub-scales and mins: codes centred on zero by dmin = d * half the code range
        top = 15 if ty == Q4_K else 31
        d = _half(g, nb, WSTD / (40 * top * 0.29)).view(torch.float16).view(nb)
        b[:, 0:2] = d.view(torch.uint8).view(nb, 2)
        b[:, 2:4] = (d.float() * (top / 2)).to(torch.float16).view(torch.uint8).view(nb, 2)
        s = _bytes(g, nb, 8, lo=16, hi=64)
        lo4, hi4 = s[:, :4], s[:, 4:]
        b[:, 4:8] = lo4 | ((hi4 >> 4) << 6)
        b[:, 8:12] = lo4 | ((hi4 >> 4) << 6)
        b[:, 12:16] = (hi4 & 15) | ((hi4 & 15) << 4)
    return b.view(-1)


def _gguf64(raw: torch.Tensor, ty: int, N: int, K: int) -> torch.Tensor:
    """The values of GGUF blocks in 64 bits, [N, K]."""
    be, ts = BLOCK[ty]
    b = raw.reshape(-1)[: N * K // be * ts].view(-1, ts)

    def half(o):
        return b[:, o : o + 2].contiguous().view(torch.float16).double()

    def sbyte(t):
        return t.contiguous().view(torch.int8).double()

    if ty == Q8_0:
        v = half(0) * sbyte(b[:, 2:34])
    elif ty == Q6_K:
        ql, qh, sc = b[:, :128].view(-1, 2, 64), b[:, 128:192].view(-1, 2, 32), sbyte(b[:, 192:208])
        q = torch.stack([((ql[:, :, 32 * (t & 1) : 32 * (t & 1) + 32] >> (4 * (t >> 1))) & 15) |
                         (((qh >> (2 * t)) & 3) << 4) for t in range(4)], 2)  # [nb, half, t, 32]
        v = (q.double() - 32).view(-1, 16, 16) * (half(208) * sc).unsqueeze(2)
    else:
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:12] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, ts - 128 :].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        if ty == Q5_K:
            q = q | (torch.stack([(b[:, 16:48] >> u) & 1 for u in range(8)], 1) << 4)
        v = (half(0) * sc).unsqueeze(2) * q.double() - (half(2) * mn).unsqueeze(2)
    return v.reshape(N, K)


def _mxfp4(g, N: int, K: int) -> tuple[torch.Tensor, torch.Tensor]:
    """MXFP4 blocks [N, K/32, 16] and e8m0 scales [N, K/32], checkpoint order."""
    return _bytes(g, N, K // 32, 16), _bytes(g, N, K // 32, lo=117, hi=123)


def _mxfp4_64(blocks: torch.Tensor, scales: torch.Tensor) -> torch.Tensor:
    lut = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=DEV)
    lut = torch.cat([lut, -lut])
    q = torch.stack([blocks & 15, blocks >> 4], -1).flatten(-2)  # [N, G, 32]
    v = lut[q.long()] * torch.exp2(scales.double() - 127).unsqueeze(-1)
    return v.reshape(blocks.shape[0], -1)


def _bias(g, *shape) -> torch.Tensor:
    return (0.02 * torch.randn(shape, device=DEV, generator=g)).to(torch.bfloat16)


def _layer(case: dict, seed: int) -> dict:
    """One MoE layer's experts as a checkpoint holds them: a tensor per matrix, expert first."""
    g = _gen(seed)
    H, I, E = case["H"], case["I"], case["E"]
    if case["gate"] == MXFP4:
        gu, dn = _mxfp4(g, E * 2 * I, H), _mxfp4(g, E * H, I)
        return {"gu": gu, "dn": dn, "gub": _bias(g, E, 2 * I), "dnb": _bias(g, E, H)}
    return {"gate": _gguf(g, case["gate"], E * H * I).view(E, -1), "up": _gguf(g, case["gate"], E * H * I).view(E, -1),
            "down": _gguf(g, case["down"], E * H * I).view(E, -1)}


def _pool(case: dict, layer: dict) -> tuple[torch.Tensor, object]:
    """(slot pool, layout): the layer's experts resident, expert e in slot e."""
    H, I, E = case["H"], case["I"], case["E"]
    if case["gate"] == MXFP4:
        lay = synth.mxfp4_tiled_layout(H, I)
        pool = torch.empty((E, lay.total_bytes), dtype=torch.uint8, device=DEV)
        parts = {"gate_up_proj_bias": layer["gub"].view(torch.uint8), "down_proj_bias": layer["dnb"].view(torch.uint8)}
        for name, m in (("gate_up_proj", layer["gu"]), ("down_proj", layer["dn"])):
            parts[name], parts[name + "_scales"] = ops.mxfp4_tile(*m)
        L = mxfp4_expert_layout(lay, tiled=True)
    else:
        types = (case["gate"], case["gate"], case["down"])
        lay = synth.gguf_layout(H, I, *types)
        pool = torch.empty((E, lay.total_bytes), dtype=torch.uint8, device=DEV)
        parts = layer
        L = gguf_expert_layout(lay, dict(zip(("gate", "up", "down"), types)),
                               {"gate": (H, I), "up": (H, I), "down": (I, H)})
    for name, t in parts.items():
        o = lay.offsets[name]
        pool[:, o : o + lay.sizes[name]] = t.reshape(E, -1)
    return pool, L


def _mode(case: dict) -> str:
    return "topk_then_softmax" if case["E"] == 32 else "softmax_then_topk"


def _logits(g, case: dict, T: int, dtype) -> torch.Tensor:
    """Router logits: N(0, 1) and a popularity of the experts that falls as rank^-1.1."""
    rank = torch.randperm(case["E"], device=DEV, generator=g) + 1
    return (torch.randn((T, case["E"]), device=DEV, generator=g) - 1.1 * rank.double().log().float()).to(dtype)


def _decode_inputs(case: dict, seed: int) -> list[tuple[torch.Tensor, torch.Tensor]]:
    g, T = _gen(seed + 7), case["T"]
    return [(_acts(g, T, case["H"]), _logits(g, case, T, torch.bfloat16)) for _ in range(case["layers"])]


def _layer_seed(seed: int, i: int) -> int:
    return 1000003 * (seed + 1) + i


def prepare(case: dict, seed: int) -> dict:
    g, op = _gen(seed), case["op"]
    s = {"op": op, "case": case}
    if op == "linear":
        raw = _gguf(g, case["type"], case["N"] * case["K"])
        bias = _bias(g, case["N"]).to(DTYPES[case["dtype"]]) if case["bias"] else None
        s["layer"] = GGMLLinear(raw, case["type"], case["N"], case["K"], bias=bias)
        s["x"] = _acts(g, case["T"], case["K"], dtype=DTYPES[case["dtype"]])
    elif op == "mxlinear":
        s["w"], s["bias"] = _mxfp4(g, case["N"], case["K"]), _bias(g, case["N"])
        s["x"] = _acts(g, case["T"], case["K"])
    elif op == "router":
        s["w"] = (torch.randn((case["E"], case["H"]), device=DEV, generator=g) * case["H"] ** -0.5).to(torch.bfloat16)
        s["bias"], s["x"] = _bias(g, case["E"]), _acts(g, case["T"], case["H"])
    elif op == "dequant":
        N, K = case["N"], case["K"]
        s["w"] = _mxfp4(g, N, K) if case["type"] == MXFP4 else _gguf(g, case["type"], N * K)
    elif op == "moe":
        s["pool"], s["L"] = _pool(case, _layer(case, _layer_seed(seed, 0)))
        s["slot"] = torch.arange(case["E"], dtype=torch.int32, device=DEV)
        s["x"], s["logits"] = _acts(g, case["T"], case["H"]), _logits(g, case, case["T"], torch.float32)
    else:  # a decode step over the layers, captured once and replayed
        H, T, k = case["H"], case["T"], case["k"]
        layers = [_pool(case, _layer(case, _layer_seed(seed, i))) for i in range(case["layers"])]
        slot = torch.arange(case["E"], dtype=torch.int32, device=DEV)
        ins = _decode_inputs(case, seed)
        y = torch.empty((case["layers"], T, H), dtype=torch.bfloat16, device=DEV)
        ws = ops.moe_decode_workspace(layers[0][1], T, k, DEV)

        def step():
            return [ops.moe_decode_routed(L, pool, slot, lg, x, k, _mode(case), out=y[i], workspace=ws,
                                          return_routing=True)
                    for i, ((pool, L), (x, lg)) in enumerate(zip(layers, ins))]

        step()
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            out = step()
        s["out"] = {"y": y, "idx": [o[1] for o in out], "w": [o[2] for o in out]}
        s["keep"] = (layers, slot, ins, ws)
    return s


def run(s: dict):
    op, case = s["op"], s["case"]
    if op == "linear":
        return s["layer"](s["x"])
    if op == "mxlinear":
        return mxfp4_linear(s["x"], *s["w"], s["bias"])
    if op == "router":
        return ops.router_logits(s["x"], s["w"], s["bias"])
    if op == "dequant":
        dt = DTYPES[case["dtype"]]
        if case["type"] == MXFP4:
            return ops.mxfp4_dequant(*s["w"], dtype=dt)
        return ops.gguf_dequant(s["w"], case["type"], (case["N"], case["K"]), dtype=dt)
    if op == "moe":
        idx, w = ops.route_topk(s["logits"], case["k"], _mode(case))
        y = ops.moe_prefill(s["L"], s["pool"], s["slot"], idx, w, s["x"])
        return {"y": y, "idx": idx, "w": w}
    s["graph"].replay()
    return s["out"]


# ----------------------------------------------------------------------------- work and tolerance
def _expert_bytes(case: dict) -> float:
    n = case["H"] * case["I"]
    if case["gate"] == MXFP4:
        return 3 * n * 17 / 32 + 2 * (2 * case["I"] + case["H"])
    be, ts = BLOCK[case["gate"]]
    bd, td = BLOCK[case["down"]]
    return 2 * n * ts / be + n * td / bd


def _distinct(case: dict) -> float:
    """Experts that T tokens' top-k selections reach, on average."""
    rng = np.random.default_rng(1)
    E, k, got = case["E"], case["k"], []
    for _ in range(8):
        lg = rng.normal(size=(case["T"], E)) - 1.1 * np.log(rng.permutation(E) + 1)
        got.append(len(np.unique(np.argpartition(-lg, k - 1, axis=1)[:, :k])))
    return float(np.mean(got))


def work(case: dict) -> dict:
    op, T = case["op"], case.get("T", 0)
    if op in ("linear", "mxlinear", "dequant"):
        n = case["N"] * case["K"]
        ty = case.get("type", MXFP4)
        wb = n * 17 / 32 if ty == MXFP4 else n * BLOCK[ty][1] / BLOCK[ty][0]
        es = torch.empty(0, dtype=DTYPES[case.get("dtype", "bf16")]).element_size()
        if op == "dequant":
            return {"bytes": wb + n * es, "flops": 0}
        return {"bytes": wb + es * T * (case["N"] + case["K"]), "flops": 2 * n * T}
    if op == "router":
        return {"bytes": 2 * (case["E"] * case["H"] + T * case["H"] + T * case["E"]), "flops": 2 * T * case["E"] * case["H"]}
    layers = case.get("layers", 1)
    flops = 2 * T * case["k"] * 3 * case["H"] * case["I"]
    per = _distinct(case) * _expert_bytes(case) + T * (4 * case["H"] + 4 * case["E"])
    return {"bytes": layers * per, "flops": layers * flops}


def tolerance(case: dict):
    op = case["op"]
    if op == "dequant":
        return "exact"
    if op in ("linear", "mxlinear", "router"):
        # one rounding to the output type; f32 results differ by the order of the sums and,
        # up to 8 tokens, by activations carried in 16 significant bits
        if case.get("dtype", "bf16") == "f32":
            return {"rel": 1e-4, "max": 1e-3}
        if case.get("dtype", "bf16") == "f16":
            return {"rel": 1e-3, "max": 5e-3}
        return {"rel": 6e-3, "max": 2e-2}
    # two roundings to bf16 (h and y); prefill also rounds each expert's output, and its
    # operands: two fp6 terms per activation (MXFP4), bf16 weights (GGUF)
    return {"rel": 1e-2, "max": 6e-2, "differ": 1e-3}


# ----------------------------------------------------------------------------- 64-bit results
def _route64(logits: torch.Tensor, k: int, mode: str) -> tuple[torch.Tensor, torch.Tensor]:
    v, idx = torch.sort(logits.double(), dim=-1, descending=True, stable=True)
    w = torch.softmax(v[:, :k], -1)  # either mode: the full softmax renormalised over the k is this
    return idx[:, :k], w


def _moe64(case: dict, layer: dict, x: torch.Tensor, idx: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    H, I = case["H"], case["I"]
    x, y = x.double(), torch.zeros((x.shape[0], H), dtype=torch.float64, device=DEV)
    for e in torch.unique(idx).tolist():
        t, j = (idx == e).nonzero(as_tuple=True)
        if case["gate"] == MXFP4:
            gu = x[t] @ _mxfp4_64(*(m[e * 2 * I : (e + 1) * 2 * I] for m in layer["gu"])).t() + layer["gub"][e].double()
            gate, up = gu[:, 0::2].clamp(max=7.0), gu[:, 1::2].clamp(-7.0, 7.0)
            h = (up + 1) * gate * torch.sigmoid(1.702 * gate)
            o = h @ _mxfp4_64(*(m[e * H : (e + 1) * H] for m in layer["dn"])).t() + layer["dnb"][e].double()
        else:
            gate = x[t] @ _gguf64(layer["gate"][e], case["gate"], I, H).t()
            up = x[t] @ _gguf64(layer["up"][e], case["gate"], I, H).t()
            o = (torch.nn.functional.silu(gate) * up) @ _gguf64(layer["down"][e], case["down"], H, I).t()
        y.index_add_(0, t, w[t, j].unsqueeze(1) * o)
    return y


def exact(case: dict, seed: int):
    s_op = case["op"]
    g = _gen(seed)
    if s_op == "linear":
        W = _gguf64(_gguf(g, case["type"], case["N"] * case["K"]), case["type"], case["N"], case["K"])
        b = _bias(g, case["N"]).to(DTYPES[case["dtype"]]).double() if case["bias"] else 0.0
        return _acts(g, case["T"], case["K"], dtype=DTYPES[case["dtype"]]).double() @ W.t() + b
    if s_op == "mxlinear":
        W, b = _mxfp4_64(*_mxfp4(g, case["N"], case["K"])), _bias(g, case["N"])
        return _acts(g, case["T"], case["K"]).double() @ W.t() + b.double()
    if s_op == "router":
        W = (torch.randn((case["E"], case["H"]), device=DEV, generator=g) * case["H"] ** -0.5).to(torch.bfloat16)
        b, x = _bias(g, case["E"]), _acts(g, case["T"], case["H"])
        return x.double() @ W.double().t() + b.double()
    if s_op == "dequant":
        N, K = case["N"], case["K"]
        return _mxfp4_64(*_mxfp4(g, N, K)) if case["type"] == MXFP4 else _gguf64(_gguf(g, case["type"], N * K),
                                                                                 case["type"], N, K)
    if s_op == "moe":
        x, logits = _acts(g, case["T"], case["H"]), _logits(g, case, case["T"], torch.float32)
        idx, w = _route64(logits, case["k"], _mode(case))
        return {"y": _moe64(case, _layer(case, _layer_seed(seed, 0)), x, idx, w), "idx": None, "w": w}
    ys, ws = [], []
    for i, (x, lg) in enumerate(_decode_inputs(case, seed)):
        idx, w = _route64(lg, case["k"], _mode(case))
        ys.append(_moe64(case, _layer(case, _layer_seed(seed, i)), x, idx, w))
        ws.append(w)
    return {"y": torch.stack(ys), "idx": [None] * case["layers"], "w": ws}
