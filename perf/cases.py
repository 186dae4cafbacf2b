"""The calls whose speed is measured: what a program that uses this package has it do, one call per case.

The sizes are the ones of ``bench.py`` and of the tests (K = 4096 with N = 4096 and 14336, the 256^3
CHAIN graphs, C = 256 x 32 heads, B = 8, T = 4096, H = 32) and ragged or smaller ones of the same
ranges: prompts of a few hundred rows, decode batches of 1 to 16 rows, short single sequences.

``prepare`` makes the operands on the GPU from the seed alone and holds the prepared op, as a program
that loads its weights once does; ``run`` is the one call; ``exact`` is the same result in 64 bits
with plain torch.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from qcom_htp_amd import _lib, cases, gdn
from qcom_htp_amd.qmm import QuantMatmul, weight_format_of

D = 128  # GDN head dimension
DRAIN_SA, DRAIN_ST = 2.770166930875267e-05, 6.103701895199438e-05  # GdnSolve scales of the reference's gate


def listed():
    return [
        # the reference's own benchmark graph: 8 dependent 256^3 matmuls with the integer contract; latency
        {"name": "chain8_u8i8_256", "kind": "chain", "family": "u8i8", "m": 256, "k": 256, "chain": 8},
        # one decode step of one sequence through a 4096 x 14336 layer: streams the int4 weights
        {"name": "decode_w4a8_lpbq_m1", "kind": "linear", "family": "w4a8_lpbq", "m": 1, "k": 4096, "n": 14336, "block": 64},
        # one decode step of a batch of 16 through the same layer, 16-bit activations
        {"name": "decode_w4a16_lpbq_m16", "kind": "linear", "family": "w4a16_lpbq", "m": 16, "k": 4096, "n": 14336, "block": 64},
        # a short prompt (ragged) through the same layer, 16-bit activations
        {"name": "prompt_w4a16_lpbq_m200", "kind": "linear", "family": "w4a16_lpbq", "m": 200, "k": 4096, "n": 14336, "block": 32},
        # a prompt through a square layer, 8-bit activations: the headline size
        {"name": "prefill_w4a8_4096", "kind": "linear", "family": "w4a8_per_channel", "m": 4096, "k": 4096, "n": 4096, "block": 0},
        # the same with 8-bit weights and 16-bit activations: the largest call
        {"name": "prefill_w8a16_4096", "kind": "linear", "family": "w8a16", "m": 4096, "k": 4096, "n": 4096, "block": 0},
        # a prompt of ordinary length through a per-group (K64) quantised square layer
        {"name": "prompt_w4a8_group_m500", "kind": "linear", "family": "w4a8_per_group", "m": 500, "k": 4096, "n": 4096, "block": 0},
        # 16-bit weights and activations with their integer output contract, a layer of ordinary size
        {"name": "contract_w16a16_1024", "kind": "contract", "family": "w16a16", "m": 1024, "k": 1024, "n": 1024},
        # the triangular solve alone at the size it is quoted on, float32
        {"name": "solve_c256_h32_fp32", "kind": "solve", "heads": 32, "c": 256, "bits": 32, "precision": "fp32"},
        # the GdnSolve op on u16 codes over many chunk-heads of 64 tokens
        {"name": "solve_u16_c64_h2048", "kind": "solve", "heads": 2048, "c": 64, "bits": 16, "precision": "fp32"},
        # the gated-delta-rule prefill of a full batch of long sequences, default (float32) precision
        {"name": "gdn_prefill_b8_t4096", "kind": "prefill", "b": 8, "t": 4096, "h": 32, "precision": "fp32", "state": False},
        # one sequence of ragged length continued from a carried state, bf16 products
        {"name": "gdn_prefill_b1_t1000", "kind": "prefill", "b": 1, "t": 1000, "h": 16, "precision": "bf16", "state": True},
    ]


GEMM_FAMILIES = ("u8i8", "w4a8_per_channel", "w4a8_lpbq", "w8a16", "w4a16_per_channel", "w4a16_lpbq")
GROUP_FAMILIES = ("w4a8_per_group", "w4a16_per_group")
CHAIN_FAMILIES = ("u8i8", "w4a8_per_channel", "w4a8_lpbq", "w8a16", "w4a16_lpbq", "w16a16")
MOST_PRODUCTS = 3 * 4096 ** 3  # int8 products of the largest listed call


def _log(rng, lo, hi, step=1):
    """A size in [lo, hi], uniform over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(("decode", "prompt", "prompt", "group", "contract", "chain", "solve", "prefill"))
    if kind in ("decode", "prompt", "group"):
        family = rng.choice(GROUP_FAMILIES if kind == "group" else GEMM_FAMILIES)
        m = rng.randint(1, 16) if kind == "decode" else _log(rng, 17, 4096)
        align = 64 if kind == "group" else 32
        while True:
            k, n = _log(rng, 512, 4096, align), _log(rng, 512, 14336, 32)
            planes = 4 if family == "w4a16_per_group" else 3 if "a16" in family else 2 if kind == "group" else 1
            if planes * m * k * n <= MOST_PRODUCTS // (4 if kind == "group" else 1):
                break
            m = max(17, m // 2)
        block = rng.choice((32, 64)) if family.endswith("lpbq") else 0
        if block and k % block:
            k += 32
        return {"kind": "linear", "family": family, "m": m, "k": k, "n": n, "block": block}
    if kind == "contract":
        return {"kind": "contract", "family": rng.choice(("w16a16", "u8i8", "w8a16")), "m": _log(rng, 17, 2048),
                "k": _log(rng, 256, 2048, 32), "n": _log(rng, 256, 2048, 32)}
    if kind == "chain":
        return {"kind": "chain", "family": rng.choice(CHAIN_FAMILIES), "m": _log(rng, 16, 1024),
                "k": rng.choice((128, 192, 256)), "chain": rng.randint(2, 8)}
    if kind == "solve":
        c = rng.choice((16, 32, 48, 64, 128, 192, 256))
        bits = rng.choice((16, 32))
        return {"kind": "solve", "heads": _log(rng, 8, 2048 * 64 // c), "c": c, "bits": bits,
                "precision": "fp32" if bits == 16 else rng.choice(("fp32", "bf16"))}
    return {"kind": "prefill", "b": _log(rng, 1, 8), "t": _log(rng, 64, 4096), "h": _log(rng, 2, 32),
            "precision": rng.choice(("fp32", "bf16")), "state": rng.random() < 0.5}


# ---------------------------------------------------------------------------------- operands


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (int(seed) + 1))
    return g


def _ints(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=dtype)


def _codes(g, bits, shape, spread):
    """Activation codes ~ N(zero point, spread), clipped: int32 on the GPU."""
    zp = float(1 << (bits - 1))
    return (torch.randn(shape, generator=g, device="cuda") * spread + zp).round_().clamp_(0, 2 * zp - 1).to(torch.int32)


def _as_act(codes, bits):
    return codes.to(torch.uint8) if bits == 8 else codes.to(torch.uint16)


def _linear_operands(case, seed):
    """The operands of a requantised matmul: activations ~ N(zp, 40) or N(zp, 10000), uniform weight codes,
    scales ~ U(1e-3, 1e-2), LPBQ block scales in [1, 15], and the output scale that the result needs."""
    fam = cases.FAMILIES[case["family"]]
    m, k, n = case["m"], case["k"], case["n"]
    g = _gen(seed)
    o = {"fam": fam, "act": _codes(g, fam.act_bits, (m, k), 40.0 if fam.act_bits == 8 else 10000.0)}
    o["sa"] = 0.02 if fam.act_bits == 8 else 1e-4
    q = fam.weight_qmax
    o["w"] = _ints(g, -q, q, (n, k), torch.int8)
    group = fam.weight_schema == "per_group"
    o["ws"] = torch.rand((n, k // 64) if group else (n,), generator=g, device="cuda") * 9e-3 + 1e-3
    o["block"] = _ints(g, 1, 15, (n, k // case["block"]), torch.uint8) if case["block"] else None
    o["bias"] = (torch.rand((n,), generator=g, device="cuda") - 0.5) if group else _ints(g, -(1 << 15), 1 << 15, (n,), torch.int32)
    # output scale: the range of the first 16 rows on the family's fixed zero point
    t = _dequantised(o, rows=16)
    o["so"] = cases.affine_scale_from_minmax(float(t.min()), float(t.max()), 0, fam.out_qmax, fam.out_zp)
    return o


def _dequantised(o, rows=None):
    """(x_deq @ w_deq.T + bias) in float64, w_deq a float32 product of the integer weight and its scale."""
    fam = o["fam"]
    w = o["w"].float()
    if o["block"] is not None:
        w = w * o["block"].float().repeat_interleave(w.shape[1] // o["block"].shape[1], dim=1)
    ws = o["ws"] if o["ws"].dim() == 2 else o["ws"][:, None]
    w = (w * ws.repeat_interleave(w.shape[1] // ws.shape[1], dim=1)).double()
    x = (o["act"][:rows].double() - fam.act_zp) * o["sa"]
    bias = o["bias"].double() if ws.shape[1] > 1 else o["bias"].double() * (o["sa"] * o["ws"].double())
    return x @ w.t() + bias


def _contract_operands(case, seed):
    """Integer operands of the output contracts, spread so that most outputs fall inside their range."""
    fam, m, k, g = case["family"], case["m"], case["k"], _gen(seed)
    n = case.get("n", k)
    bits = 8 if "a8" in fam or fam == "u8i8" else 16
    o = {"bits": bits, "wbits": 16 if fam == "w16a16" else 8 if fam in ("u8i8", "w8a16") else 4}
    o["act"] = _codes(g, bits, (m, k), 40.0 if bits == 8 else 3000.0)
    if o["wbits"] == 16:
        o["w"] = (torch.randn((n, k), generator=g, device="cuda") * 4000.0).round_().clamp_(-32767, 32767).to(torch.int16)
    else:
        q = 7 if o["wbits"] == 4 or fam == "u8i8" else 127
        o["w"] = _ints(g, -q, q, (n, k), torch.int8)
    o["block"] = _ints(g, 1, 3, (n, k // 32), torch.uint8) if fam.endswith("lpbq") else None
    o["bias"] = _ints(g, 0, 255, (n,), torch.int32) if bits == 8 else torch.zeros(n, dtype=torch.int32, device="cuda")
    o["contract"], o["divisor"] = {8: ("clip_i32", 1)}.get(bits, ("div_rint", {16: 32767, 8: 127, 4: 7}[o["wbits"]]))
    return o


def _gdn_keys(g, *shape):
    """bf16 q / k / v rows, float32 per-token log decays and betas, as a gated delta rule layer makes them."""
    q, k, v = (torch.randn((*shape, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    beta = torch.sigmoid(torch.randn(shape, generator=g, device="cuda"))
    gc = torch.nn.functional.logsigmoid(torch.randn(shape, generator=g, device="cuda") + 3.0)
    return q, k, v, gc, beta


def _solve_a(case, seed):
    """The strictly lower A of `heads` chunks of c tokens (float64)."""
    _, k, _, gc, beta = _gdn_keys(_gen(seed), case["heads"], case["c"])
    return _build_a(k.double(), gc.double(), beta.double())


def _build_a(k, gc, beta):
    k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    s = gc.cumsum(-1)
    a = -(beta[..., :, None] * (k @ k.transpose(-1, -2).contiguous())) * torch.exp(s[..., :, None] - s[..., None, :])
    return torch.tril(a, -1)


def _codes16(a):
    return (torch.round(a / DRAIN_SA) + 32768).clamp(0, 65535)


PRECISION = {"fp32": gdn.FP32, "bf16": gdn.BF16}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        o = _linear_operands(case, seed)
        fam, fmt = o["fam"], weight_format_of(o["fam"])
        group = fam.weight_schema == "per_group"
        host = lambda x: None if x is None else x.cpu().numpy()  # noqa: E731
        op = QuantMatmul(host(o["w"]), host(o["ws"]), np.zeros(case["n"], np.int32) if group else host(o["bias"]),
                         act_bits=fam.act_bits, out_bits=fam.out_bits, act_scale=o["sa"], out_scale=o["so"], act_zp=fam.act_zp,
                         out_zp=fam.out_zp, weight_format=fmt, lpbq_block_scale=host(o["block"]), lpbq_block=case["block"],
                         bias_float=host(o["bias"]) if group else None)
        return {"kind": kind, "op": op, "act": _as_act(o["act"], fam.act_bits)}
    if kind in ("contract", "chain"):
        o = _contract_operands(case, seed)
        bits = o["bits"]
        fmt = (_lib.QH_WEIGHT_I16 if o["wbits"] == 16 else _lib.QH_WEIGHT_I4_LPBQ if o["block"] is not None else
               _lib.QH_WEIGHT_I8 if o["wbits"] == 8 else _lib.QH_WEIGHT_I4)
        op = QuantMatmul(o["w"].cpu().numpy(), np.ones(o["w"].shape[0], np.float32), o["bias"].cpu().numpy(), act_bits=bits,
                         out_bits=bits, act_scale=1.0, out_scale=1.0, act_zp=1 << (bits - 1), out_zp=32768 if bits == 16 else 0,
                         weight_format=fmt, lpbq_block_scale=None if o["block"] is None else o["block"].cpu().numpy(), lpbq_block=32)
        return {"kind": kind, "op": op, "act": _as_act(o["act"], bits), "contract": o["contract"], "divisor": o["divisor"],
                "chain": case.get("chain", 1)}
    if kind == "solve":
        a = _solve_a(case, seed)
        a = _codes16(a).to(torch.int32).to(torch.uint16) if case["bits"] == 16 else a.float()
        return {"kind": kind, "a": a.contiguous(), "bits": case["bits"], "precision": PRECISION[case["precision"]]}
    g = _gen(seed)
    q, k, v, gc, beta = _gdn_keys(g, case["b"], case["t"], case["h"])
    s0 = 0.1 * torch.randn((case["b"], case["h"], D, D), generator=g, device="cuda") if case["state"] else None
    return {"kind": kind, "args": (q, k, v, gc, beta), "s0": s0, "precision": PRECISION[case["precision"]]}


def _bits(codes):
    """uint16 codes as int16 of the same bits: torch indexes no uint16 tensors on the GPU."""
    return codes.view(torch.int16) if codes.dtype == torch.uint16 else codes


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return _bits(state["op"](state["act"]))
    if kind == "contract":
        return _bits(state["op"].run_contract(state["act"], state["contract"], state["divisor"]))
    if kind == "chain":
        return _bits(state["op"].chain(state["act"], state["chain"], state["contract"], state["divisor"]))
    if kind == "solve":
        if state["bits"] == 16:
            return _bits(gdn.GdnSolve(state["a"], 32768, DRAIN_SA, 32768, DRAIN_ST, precision=state["precision"]))
        return gdn.gdn_solve(state["a"], precision=state["precision"])
    return gdn.gdn_prefill(*state["args"], initial_state=state["s0"], precision=state["precision"])


# ---------------------------------------------------------------------------------- work, tolerance, exact


def work(case):
    kind = case["kind"]
    if kind in ("linear", "contract", "chain"):
        fam = case["family"]
        m, k, n = case["m"], case["k"], case.get("n", case["k"])
        ab = 1 if "a8" in fam or fam == "u8i8" else 2
        wbits = 16 if fam == "w16a16" else 8 if fam in ("u8i8", "w8a16") else 4
        scales = n * k // 64 * 4 if "group" in fam else 4 * n + (n * k // (case.get("block") or 32) if "lpbq" in fam else 0)
        return {"bytes": m * k * ab + n * k * wbits // 8 + scales + 4 * n + m * n * ab, "flops": 2 * m * k * n * case.get("chain", 1)}
    if kind == "solve":
        h, c = case["heads"], case["c"]
        return {"bytes": h * (c * (c - 1) // 2 + c * c) * case["bits"] // 8, "flops": h * c ** 3 // 3}
    b, t, h, c = case["b"], case["t"], case["h"], 64
    rows = b * t * h
    per_chunk = 3 * 2 * c * c * D + c ** 3 // 3 + 2 * (2 * c * c * D + 3 * c * D * D)
    return {"bytes": rows * (4 * 2 * D + 8) + b * h * D * D * 4 * (2 if case["state"] else 1), "flops": rows * per_chunk // c}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "contract", "chain"):
        return "exact"  # the outputs are codes with one right value
    if kind == "solve":
        if case["bits"] == 16:  # a float32 sum in another order moves a T code at a rounding boundary: 1.3e-4 of them seen
            return {"rel": 0.0, "differ": 1e-3}
        return {"rel": 2e-6, "max": 1e-4} if case["precision"] == "fp32" else {"rel": 1e-3, "max": 4e-2}
    # bf16 stage-A products and bf16 outputs in both precisions: 3.3e-3 from 64 bits, so 2.4e-3 times sqrt 2 apart
    return {"rel": 1e-2, "max": 2e-1}


def _requantised(t, fam, so):
    return _as_act(torch.clamp(torch.round(t / so + fam.out_zp), 0, fam.out_qmax).to(torch.int32), fam.out_bits)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        o = _linear_operands(case, seed)
        return _bits(_requantised(_dequantised(o), o["fam"], o["so"]))
    if kind in ("contract", "chain"):
        o = _contract_operands(case, seed)
        bits = o["bits"]
        w = o["w"].double()
        if o["block"] is not None:
            w = w * o["block"].double().repeat_interleave(32, dim=1)
        a = o["act"].double()
        for _ in range(case.get("chain", 1)):  # every product and sum is an integer below 2^53
            acc = (a - (1 << (bits - 1))) @ w.t().contiguous()
            if o["contract"] == "clip_i32":
                a = torch.clamp(acc + o["bias"].double(), 0, 255)
            else:
                a = torch.clamp(torch.round(acc / o["divisor"] + 32768), 0, 65535)
        return _bits(_as_act(a.to(torch.int32), bits))
    if kind == "solve":
        a = _solve_a(case, seed)
        a = (_codes16(a) - 32768) * float(np.float32(DRAIN_SA)) if case["bits"] == 16 else a.float().double()
        eye = torch.eye(case["c"], dtype=torch.float64, device="cuda").expand_as(a).contiguous()
        t = torch.linalg.solve_triangular(eye - torch.tril(a, -1), eye, upper=False, unitriangular=True)
        if case["bits"] == 16:
            t = torch.clamp(torch.round(t / float(np.float32(DRAIN_ST))) + 32768, 0, 65535)
            return _bits(t.to(torch.int32).to(torch.uint16))
        return t
    return _exact_prefill(case, seed)


def _exact_prefill(case, seed):
    """The chunked gated delta rule in float64, chunks of 64, over [B, H, T, D]."""
    s = prepare(case, seed)
    B, T, H = case["b"], case["t"], case["h"]
    pad = -T % 64
    q, k, v = (torch.nn.functional.pad(x.double().permute(0, 2, 1, 3), (0, 0, 0, pad)).contiguous() for x in s["args"][:3])
    gc, beta = (torch.nn.functional.pad(x.double().permute(0, 2, 1), (0, pad)).contiguous() for x in s["args"][3:])
    S = torch.zeros((B, H, D, D), dtype=torch.float64, device="cuda") if s["s0"] is None else s["s0"].double()
    out = []
    eye = torch.eye(64, dtype=torch.float64, device="cuda").expand(B, H, 64, 64).contiguous()
    for c in range(0, T + pad, 64):
        qc, kc, vc, bc = q[:, :, c:c + 64], k[:, :, c:c + 64], v[:, :, c:c + 64], beta[:, :, c:c + 64]
        g = gc[:, :, c:c + 64].cumsum(-1)
        qh = qc / torch.sqrt((qc * qc).sum(-1, keepdim=True) + 1e-6) / math.sqrt(D)
        kh = kc / torch.sqrt((kc * kc).sum(-1, keepdim=True) + 1e-6)
        kt = kh.transpose(-1, -2).contiguous()
        rhs = torch.cat((bc[..., None] * torch.exp(g)[..., None] * kh, bc[..., None] * vc), dim=-1)
        wu = torch.linalg.solve_triangular(eye - _build_a(kc, gc[:, :, c:c + 64], bc), rhs, upper=False, unitriangular=True)
        vn = wu[..., D:] - wu[..., :D].contiguous() @ S
        p = torch.tril((qh @ kt) * torch.exp(g[..., :, None] - g[..., None, :]))
        out.append((qh * torch.exp(g)[..., None]) @ S + p @ vn)
        S = S * torch.exp(g[..., -1])[..., None, None] + (kt * torch.exp(g[..., -1:] - g)[..., None, :]) @ vn
    return torch.cat(out, dim=2)[:, :, :T].permute(0, 2, 1, 3).contiguous(), S
