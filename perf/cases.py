"""The work that a program using this library has it do, as cases to be timed.

A serving engine on one MI355X calls the library in a handful of ways, and the
cases cover each of them from its smallest calls to its largest:

  route      moe_route on the router logits of a batch
  matmul     dense quantized projections: decode (m <= 8, GEMV), batched
             decode (m of 9 to 64: concurrent sequences or draft tokens),
             prompt chunks and whole prompts (m up to 4096)
  moe        moe_route followed by moe_ffn: decode, batched decode, prompts

A decode step goes through many layers, each with weights of its own, so a
decode case's pass runs `layers` projections (or expert sets) one after
another: enough of them that the weights come from HBM and not from the
256 MB Infinity Cache.  Engines replay such steps as a HIP graph that they
captured once, and so do the cases with `graph`; prompts are launched
eagerly.

Weights are seeded random GGUF blocks (every bit pattern of the quants and
sub-block scales) whose f16 scales give weights of about 0.03, centred on
zero, as in trained projections; activations and router logits are N(0, 1),
prompts' logits with Zipf-skewed expert popularity.  `exact` decodes the
blocks and multiplies in 64 bits with plain torch.
"""
from __future__ import annotations

import math
import pathlib
import re

import torch

from r9v_amd import ffi

SCHEMES = {"q4_k": ffi.Q4_K, "iq4_xs": ffi.IQ4_XS, "q6_k": ffi.Q6_K, "q8_0": ffi.Q8_0, "iq3_s": ffi.IQ3_S}
# GGUF wire formats: bytes and weights of a block, the f16 scale's offset
BLOCK = {"q4_k": (144, 256, 0), "iq4_xs": (136, 256, 0), "q6_k": (210, 256, 208), "q8_0": (34, 32, 0),
         "iq3_s": (110, 256, 0)}
# the f16 scale at which such blocks' weights have a standard deviation of 0.03
SCALE = {"q4_k": 1.2e-4, "iq4_xs": 2.3e-5, "q6_k": 2.2e-5, "q8_0": 4e-4, "iq3_s": 1.9e-4}
DEV = "cuda"


# ------------------------------------------------------------------ the cases

def _matmul(name, scheme, m, k, n, x="bf16", out="f32", epilogue="none", graph=False):
    return {"name": name, "kind": "matmul", "scheme": scheme, "m": m, "k": k, "n": n, "x": x, "out": out,
            "epilogue": epilogue, "layers": _layers(_row_bytes(scheme, k) * n * (2 if epilogue == "swiglu" else 1))
            if graph else 1, "graph": graph}


def _moe(name, t, e, top_k, dm, dff, gate_up="iq4_xs", down="q4_k", shared=0, zipf=0.0, layers=1, graph=False):
    return {"name": name, "kind": "moe", "t": t, "e": e, "top_k": top_k, "dm": dm, "dff": dff, "gate_up": gate_up,
            "down": down, "shared": shared, "zipf": zipf, "layers": layers, "graph": graph}


def listed():
    return [
        # the smallest call: the router of one MTP-verify step (1 + 4 draft tokens), launched on its own
        {"name": "route_t5", "kind": "route", "t": 5, "e": 512, "top_k": 10, "scoring": "softmax", "zipf": 0.0},
        # one token through the attention output projections of a 4096-wide model, f32 residual stream
        _matmul("decode_q4k_m1_f32", "q4_k", 1, 4096, 4096, x="f32", graph=True),
        # five tokens (MTP verify) through a fused QKV-sized projection of a 2048-wide model
        _matmul("decode_iq4xs_m5", "iq4_xs", 5, 2048, 5120, graph=True),
        # the gated half of a dense FFN at decode, gate and up in one launch
        _matmul("decode_swiglu_q4k_m3", "q4_k", 3, 4096, 14336, out="bf16", epilogue="swiglu", graph=True),
        # 32 concurrent sequences through the widest projection of the same FFN
        _matmul("batch_q4k_m32", "q4_k", 32, 4096, 14336, out="bf16", graph=True),
        # an odd number of sequences through the FFN's down projection, added to the residual stream
        _matmul("batch_q6k_m57_residual", "q6_k", 57, 14336, 4096, epilogue="residual", graph=True),
        # a ragged prompt chunk of a 2048-wide model
        _matmul("chunk_iq4xs_m300", "iq4_xs", 300, 2048, 5120, out="bf16"),
        # a prompt chunk through an 8-bit attention projection with a bias
        _matmul("chunk_q8_0_m777_bias", "q8_0", 777, 4096, 4096, epilogue="bias"),
        # a whole prompt through the widest projection
        _matmul("prefill_q4k_m2048", "q4_k", 2048, 4096, 14336, out="bf16"),
        # an MTP-verify step of a 512-expert model: router, routed experts and the shared expert
        _moe("moe_decode_t5", 5, 512, 10, 2048, 512, shared=1, layers=4, graph=True),
        # 48 concurrent sequences of the same model: most experts active, one or two rows each
        _moe("moe_batch_t48", 48, 512, 10, 2048, 512, shared=1),
        # a long prompt of the same model, experts of very unequal popularity
        _moe("moe_prefill_t8192", 8192, 512, 10, 2048, 512, zipf=1.1),
    ]


def draw(rng):
    """One more case of the same ranges."""
    def log_int(lo, hi):
        return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))

    def k256(lo, hi):
        return 256 * log_int(lo // 256, hi // 256)

    scheme = rng.choice(["q4_k", "q4_k", "q4_k", "iq4_xs", "iq4_xs", "q6_k", "q8_0", "iq3_s"])
    kind = rng.choice(["route", "decode", "decode", "swiglu", "batch", "batch", "chunk", "chunk", "prefill",
                       "moe_decode", "moe_batch", "moe_prefill"])
    if kind == "route":
        e = rng.choice([64, 128, 160, 256, 512])
        c = {"kind": "route", "t": log_int(1, 8192), "e": e, "top_k": rng.randint(2, 10),
             "scoring": rng.choice(["softmax", "softmax", "sigmoid"]), "zipf": rng.choice([0.0, 1.1])}
    elif kind.startswith("moe"):
        e = rng.choice([16, 64, 128, 256, 512])
        dm, dff = k256(1024, 4096), k256(256, 2048)
        while e * 3 * dm * dff > 1.75e9:  # expert sets of up to about 1 GB
            e //= 2
        t = log_int(1, 8) if kind == "moe_decode" else log_int(9, 128) if kind == "moe_batch" else log_int(129, 8192)
        top_k = rng.randint(2, min(10, e // 2))
        while 6.0 * t * top_k * dm * dff > 5e11:
            t = t * 3 // 4
        gate_up, down = rng.choice([("iq4_xs", "q4_k"), ("iq4_xs", "q4_k"), ("q4_k", "q4_k"), ("q4_k", "q6_k"),
                                    ("iq4_xs", "iq4_xs"), ("q8_0", "q8_0")])
        c = _moe("", t, e, top_k, dm, dff, gate_up, down, rng.choice([0, 1]),
                 1.1 if kind == "moe_prefill" else 0.0, 2 if kind == "moe_decode" else 1, kind == "moe_decode")
    else:
        k, n = k256(1024, 14336), log_int(512, 16384)
        if rng.random() < 0.75:  # most projections are a multiple of 64 wide, some (heads, padded vocabularies) are not
            n = max(512, n // 64 * 64)
        x = "f32" if kind == "decode" and scheme in ("q4_k", "iq4_xs") and rng.random() < 0.3 else "bf16"
        out = rng.choice(["f32", "bf16"])
        epilogue = "swiglu" if kind == "swiglu" else rng.choice(["none", "none", "none", "bias", "residual"])
        m = (log_int(1, 8) if kind in ("decode", "swiglu") else log_int(9, 64) if kind == "batch" else
             log_int(65, 1024) if kind == "chunk" else log_int(1025, 4096))
        while 2.0 * m * n * k > 2.4e11:
            m = m * 3 // 4
        c = _matmul("", scheme, m, k, n, x, out, epilogue, kind in ("decode", "swiglu", "batch"))
    c.pop("name", None)
    return c


def _row_bytes(scheme, k):
    nbytes, length, _ = BLOCK[scheme]
    return k // length * nbytes


def _layers(weight_bytes):
    """Projections of a decode pass: about 300 MB of weights, at most 48 of them."""
    return max(1, min(48, round(300e6 / weight_bytes)))


# ------------------------------------------------------------------ inputs

def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(seed)


def _wire(scheme, rows, k, g):
    """Random GGUF blocks of a [rows, k] weight, uint8 [blocks, bytes of a block]."""
    nbytes, length, at = BLOCK[scheme]
    blocks = rows * (k // length)
    w = torch.randint(0, 2 ** 31 - 1, ((blocks * nbytes + 3) // 4,), dtype=torch.int32, device=DEV, generator=g)
    w = (w ^ (w << 7)).view(torch.uint8)[: blocks * nbytes].view(blocks, nbytes)  # every bit of a byte is random
    d = SCALE[scheme] * (0.5 + torch.rand(blocks, device=DEV, generator=g))
    w[:, at:at + 2] = d.half().view(torch.uint8).view(blocks, 2)
    if scheme == "q4_k":  # the mins centre the weights on zero
        w[:, 2:4] = (7.5 * d).half().view(torch.uint8).view(blocks, 2)
    return w


def _device_weight(scheme, rows, k, g):
    """The weight as a program keeps it on the GPU: (blocks or body, f16 scales or None)."""
    w = _wire(scheme, rows, k, g)
    if scheme in ("q4_k", "iq4_xs"):
        return w.view(-1), None
    return ffi.repack(w.view(-1), SCHEMES[scheme], rows, k)


def _logits(c, g, device=DEV):
    z = torch.randn((c["t"], c["e"]), device=device, generator=g)
    if c["zipf"]:
        rank = torch.randperm(c["e"], device=device, generator=g)
        z = z - c["zipf"] * torch.log(rank.float() + 1.0)[None, :]
    return z


def _inputs(c, seed):
    """What a case's pass reads, apart from its weights."""
    g = _gen(seed)
    s = {}
    if c["kind"] == "matmul":
        dt = torch.float32 if c["x"] == "f32" else torch.bfloat16
        s["x"] = torch.randn((c["layers"], c["m"], c["k"]), device=DEV, generator=g).to(dt)
        if c["epilogue"] == "bias":
            s["bias"] = [torch.randn(c["n"], device=DEV, generator=g) for _ in range(c["layers"])]
        if c["epilogue"] == "residual":
            s["residual"] = [torch.randn((c["m"], c["n"]), device=DEV, generator=g) for _ in range(c["layers"])]
    elif c["kind"] == "moe":
        s["logits"] = [_logits(c, g) for _ in range(c["layers"])]
        s["x"] = torch.randn((c["layers"], c["t"], c["dm"]), device=DEV, generator=g).to(torch.bfloat16)
    else:
        s["logits"] = [_logits(c, g)]
    return s


def _weight_gen(seed, layer, part=0):
    return _gen(seed * 1000003 + 64 * layer + part + 1)


def _expert_rows(c):
    experts = c["e"] + c["shared"]
    return experts * 2 * c["dff"], experts * c["dm"]


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    s["case"] = c
    if c["kind"] == "matmul":
        rows = c["n"] * (2 if c["epilogue"] == "swiglu" else 1)
        s["w"] = [_device_weight(c["scheme"], rows, c["k"], _weight_gen(seed, i)) for i in range(c["layers"])]
        if c["graph"]:
            s["y"] = [torch.empty((c["m"], c["n"]), device=DEV, dtype=torch.float32 if c["out"] == "f32"
                                  else torch.bfloat16) for _ in range(c["layers"])]
    else:
        n = c.get("layers", 1)
        s["ids"] = torch.empty((n, c["t"], c["top_k"]), dtype=torch.int32, device=DEV)
        s["weights"] = torch.empty((n, c["t"], c["top_k"]), device=DEV)
        s["status"] = torch.zeros(1, dtype=torch.int32, device=DEV)
        if c["kind"] == "moe":
            gu, dn = _expert_rows(c)
            s["gu"] = [_device_weight(c["gate_up"], gu, c["dm"], _weight_gen(seed, i, 1)) for i in range(n)]
            s["dn"] = [_device_weight(c["down"], dn, c["dff"], _weight_gen(seed, i, 2)) for i in range(n)]
            s["y"] = torch.empty((n, c["t"], c["dm"]), device=DEV)
            st = ffi.ffn_static(c["t"], c["e"], c["top_k"], c["dm"], c["dff"], c["shared"], SCHEMES[c["gate_up"]],
                                SCHEMES[c["down"]])
            s["workspace"] = torch.empty(ffi.ffn_workspace_bytes(st), dtype=torch.uint8, device=DEV)
    if c.get("graph"):
        _pass(s)  # once eagerly, as before any capture
        torch.cuda.synchronize()
        s["replay"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["replay"]):
            s["out"] = _pass(s)
    return s


# ------------------------------------------------------------------ a pass

def _pass(s):
    c = s["case"]
    if c["kind"] == "matmul":
        return [ffi.matmul(w, SCHEMES[c["scheme"]], c["n"], c["k"], s["x"][i],
                           out_dtype=ffi.F32 if c["out"] == "f32" else ffi.BF16,
                           bias=s["bias"][i] if "bias" in s else None,
                           residual=s["residual"][i] if "residual" in s else None,
                           y=s["y"][i] if "y" in s else None, w_scales=scales, swiglu=c["epilogue"] == "swiglu")
                for i, (w, scales) in enumerate(s["w"])]
    for i, logits in enumerate(s["logits"]):
        ids, weights = ffi.moe_route(logits, c["top_k"], scoring=ffi.SCORING_SIGMOID if c.get("scoring") == "sigmoid"
                                     else ffi.SCORING_SOFTMAX, ids=s["ids"][i], weights=s["weights"][i],
                                     status=s["status"])
        if c["kind"] == "moe":
            ffi.moe_ffn(s["x"][i], ids, weights, s["gu"][i][0], s["dn"][i][0], c["e"], c["dff"], shared=c["shared"],
                        gate_up_scheme=SCHEMES[c["gate_up"]], down_scheme=SCHEMES[c["down"]], y=s["y"][i],
                        workspace=s["workspace"], w_gate_up_scales=s["gu"][i][1], w_down_scales=s["dn"][i][1])
    out = {"ids": s["ids"], "weights": s["weights"]}
    if c["kind"] == "moe":
        out["y"] = s["y"]
    return out


def run(state):
    if "replay" in state:
        state["replay"].replay()
        return state["out"]
    return _pass(state)


# ------------------------------------------------------------------ what a pass cannot do without

def _active_experts(c):
    z = _logits(c, _gen(1, "cpu"), "cpu")
    return int(torch.unique(torch.topk(z, c["top_k"], dim=1).indices).numel()) + c["shared"]


def work(case):
    c = case
    if c["kind"] == "route":
        return {"bytes": c["t"] * (4.0 * c["e"] + 8.0 * c["top_k"]), "flops": c["t"] * (4.0 * c["e"] + 3.0 * c["top_k"])}
    if c["kind"] == "matmul":
        rows = c["n"] * (2 if c["epilogue"] == "swiglu" else 1)
        per = (rows * _row_bytes(c["scheme"], c["k"]) + c["m"] * c["k"] * (4 if c["x"] == "f32" else 2) +
               c["m"] * c["n"] * (4 if c["out"] == "f32" else 2))
        per += 4 * c["n"] if c["epilogue"] == "bias" else 4 * c["m"] * c["n"] if c["epilogue"] == "residual" else 0
        return {"bytes": float(c["layers"] * per), "flops": 2.0 * c["layers"] * c["m"] * rows * c["k"]}
    expert = 2 * c["dff"] * _row_bytes(c["gate_up"], c["dm"]) + c["dm"] * _row_bytes(c["down"], c["dff"])
    per = _active_experts(c) * expert + c["t"] * (4 * c["e"] + 8 * c["top_k"] + 6 * c["dm"])
    return {"bytes": float(c["layers"] * per),
            "flops": 6.0 * c["layers"] * c["t"] * (c["top_k"] + c["shared"]) * c["dm"] * c["dff"]}


def tolerance(case):
    c = case
    if c["kind"] == "route":  # bit-exact by contract, ids and weights
        return "exact"
    if c["kind"] == "matmul":
        if c["out"] == "bf16":  # one rounding of the result to 8 bits
            return {"rel": 8e-3, "max": 0.03}
        if c["m"] <= 8:  # f32 sums of exact products
            return {"rel": 1e-5, "max": 2e-4}
        return {"rel": 1e-3, "max": 2e-2}  # fp16 weights (11 bits) with f32 sums
    return {"rel": 2e-3, "max": 2e-2}  # the same, and fp16 SwiGLU rows and expert outputs between the two products


# ------------------------------------------------------------------ the same in 64 bits, in plain torch

_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _iq3s_grid():
    """The format's codebook: 512 words of four byte values."""
    text = (pathlib.Path(ffi.__file__).parent / "csrc" / "r9vx_iq3s_grid.h").read_text()
    words = [int(v, 16) for v in re.findall(r"0x([0-9a-fA-F]{8})", text)][:512]
    return torch.tensor([[(v >> (8 * i)) & 0xFF for i in range(4)] for v in words], dtype=torch.float64, device=DEV)


def _decode(scheme, w, rows, k):
    """GGUF wire blocks [blocks, bytes] -> f64 [rows, k]."""
    def bits(a, shift, mask):
        return (a >> shift) & mask

    if scheme == "q8_0":
        v = _f16(w[:, 0:2]) * w[:, 2:34].contiguous().view(torch.int8).double()
    elif scheme == "q4_k":
        s, q = w[:, 4:16].int(), w[:, 16:144].view(-1, 4, 1, 32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6) << 4], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6) << 4], 1).double()
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        v = (_f16(w[:, 0:2]) * sc)[:, :, None] * q - (_f16(w[:, 2:4]) * mn)[:, :, None]
    elif scheme == "iq4_xs":
        high, low = w[:, 2].int() | w[:, 3].int() << 8, w[:, 4:8].int()
        c = torch.arange(8, device=DEV)
        ls = bits(low[:, c // 2], 4 * (c % 2), 15) | bits(high[:, None], 2 * c, 3) << 4
        q = w[:, 8:136].view(-1, 8, 16)
        q = torch.cat([q & 15, q >> 4], 2).long()
        kv = torch.tensor(_IQ4, dtype=torch.float64, device=DEV)[q]
        v = (_f16(w[:, 0:2]) * (ls - 32).double())[:, :, None] * kv
    elif scheme == "q6_k":
        ql, qh = w[:, 0:128].view(-1, 2, 2, 32), w[:, 128:192].view(-1, 2, 32)
        lo = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        hi = torch.stack([bits(qh, 2 * i, 3) for i in range(4)], 2)
        q = (lo | hi << 4).reshape(-1, 16, 16).double() - 32
        v = (_f16(w[:, 208:210]) * w[:, 192:208].contiguous().view(torch.int8).double())[:, :, None] * q
    else:
        c, b = torch.arange(8, device=DEV), torch.arange(32, device=DEV)
        idx = w[:, 2:66].view(-1, 8, 8).long() | bits(w[:, 66:74].long()[:, :, None], c, 1) << 8
        sign = bits(w[:, 74:106].view(-1, 8, 4).int()[:, :, b // 8], b % 8, 1)
        db = _f16(w[:, 0:2]) * (1 + 2 * bits(w[:, 106:110].int()[:, c // 2], 4 * (c % 2), 15)).double()
        v = db[:, :, None] * _iq3s_grid()[idx].view(-1, 8, 32) * (1 - 2 * sign).double()
    return v.reshape(rows, k)


def _exact_route(logits, top_k, sigmoid):
    z = logits.double()
    p = torch.sigmoid(z) if sigmoid else torch.softmax(z, 1)
    # the top experts of a row in descending score, the lower id first where scores are equal
    ids = torch.argsort(p if sigmoid else z, dim=1, descending=True, stable=True)[:, :top_k]
    w = torch.gather(p, 1, ids)
    return ids, w / w.sum(1, keepdim=True)


def exact(case, seed):
    c, s = case, _inputs(case, seed)
    if c["kind"] == "matmul":
        gated = c["epilogue"] == "swiglu"
        rows, ys = c["n"] * (2 if gated else 1), []
        for i in range(c["layers"]):
            w = _decode(c["scheme"], _wire(c["scheme"], rows, c["k"], _weight_gen(seed, i)), rows, c["k"])
            y = s["x"][i].double() @ w.t().contiguous()
            if gated:
                y = torch.nn.functional.silu(y[:, :c["n"]]) * y[:, c["n"]:]
            y = y + s["bias"][i] if "bias" in s else y + s["residual"][i] if "residual" in s else y
            ys.append(y)
        return ys
    routed = [_exact_route(z, c["top_k"], c.get("scoring") == "sigmoid") for z in s["logits"]]
    out = {"ids": None, "weights": torch.stack([w for _, w in routed])}
    if c["kind"] == "route":
        return out
    ys = []
    dm, dff = c["dm"], c["dff"]
    gu_rows, dn_rows = _expert_rows(c)
    for i, (ids, weights) in enumerate(routed):
        gu = _wire(c["gate_up"], gu_rows, dm, _weight_gen(seed, i, 1)).view(c["e"] + c["shared"], -1, BLOCK[c["gate_up"]][0])
        dn = _wire(c["down"], dn_rows, dff, _weight_gen(seed, i, 2)).view(c["e"] + c["shared"], -1, BLOCK[c["down"]][0])
        x, y = s["x"][i].double(), torch.zeros((c["t"], dm), dtype=torch.float64, device=DEV)
        for e in sorted(set(ids.flatten().tolist()) | set(range(c["e"], c["e"] + c["shared"]))):
            if e < c["e"]:
                tok, slot = (ids == e).nonzero(as_tuple=True)
                share = weights[tok, slot][:, None]
            else:
                tok, share = torch.arange(c["t"], device=DEV), 1.0
            w = _decode(c["gate_up"], gu[e], 2 * dff, dm)
            g = x[tok] @ w.t().contiguous()
            h = torch.nn.functional.silu(g[:, :dff]) * g[:, dff:]
            y[tok] += share * (h @ _decode(c["down"], dn[e], dm, dff).t().contiguous())
        ys.append(y)
    out["y"] = torch.stack(ys)
    return out
