"""The work that a program built on this framework has it do, as cases that can be timed.

Every case goes through the modules and functions that such a program calls (VQLinear,
VQSparseMoeBlock, VQEmbedding, codepack.pack_codes). Four kinds:

  linear  one VQ-coded dense linear, y = x . W^T: the decode GEMV (up to 32 rows), short and
          long prompts (decode-then-GEMM)
  moe     one VQ-coded MoE block: softmax top-k routing, the routed experts' SwiGLU, the
          weighted combine, and a shared expert where the layer has one; decode (a few
          tokens), the verify batch of speculative decoding, prompts
  embed   rows of a VQ-coded embedding table, by token id
  pack    codes packed to their bit width, with the round trip that the packer checks

Weights are what the artifacts hold: uniform codes, an fp16 codebook ~ N(0, 0.02), fp16 scales
~ U(0.5, 1.5) per row and group of 64 columns; activations and router logits are N(0, 1).
"""
from __future__ import annotations

import math

import torch

from vqlab_amd import codepack, vq_pack
from vqlab_amd.moe import VQSparseMoeBlock, VQSwitchGLU
from vqlab_amd.vq_dense import VQEmbedding, VQLinear
from vqlab_amd.vq_switch import VQSwitchLinear

G = 64                                          # columns per scale group
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


# ------------------------------------------------------------------ cases
def listed():
    return [
        # one token through an attention-sized projection: launch and first-byte latency
        dict(name="linear_decode_4096", kind="linear", rows=1, inp=4096, out=4096, d=2, K=256,
             packed=False, dtype="bf16"),
        # twenty sequences decoded together through an MLP gate in 12-bit packed codes
        dict(name="linear_decode_20_rows", kind="linear", rows=20, inp=5120, out=17408, d=4, K=4096,
             packed=True, dtype="bf16"),
        # a short prompt of odd length through an MLP down projection
        dict(name="linear_prompt_333", kind="linear", rows=333, inp=17408, out=5120, d=4, K=4096,
             packed=True, dtype="fp16"),
        # a long prompt (or one chunk of it) through an MLP gate of the 2-bit format
        dict(name="linear_prompt_2048", kind="linear", rows=2048, inp=5120, out=17408, d=8, K=65536,
             packed=False, dtype="bf16"),
        # one token through a layer of 256 small experts: the inner loop of decoding
        dict(name="moe_decode_e256", kind="moe", tokens=1, hidden=2048, inter=512, experts=256,
             top_k=8, shared=False, d=4, K=4096, dead=0.0, dtype="bf16"),
        # one token through a layer of 512 larger experts whose table is larger than LDS
        dict(name="moe_decode_e512", kind="moe", tokens=1, hidden=4096, inter=1024, experts=512,
             top_k=10, shared=True, d=8, K=16384, dead=0.0, dtype="bf16"),
        # the same layer for four sequences
        dict(name="moe_decode_e512_batch4", kind="moe", tokens=4, hidden=4096, inter=1024,
             experts=512, top_k=10, shared=True, d=8, K=16384, dead=0.0, dtype="bf16"),
        # its verify batch in speculative decoding, a fifth of the code rows dead (skipzero)
        dict(name="moe_verify_e512_64", kind="moe", tokens=64, hidden=4096, inter=1024, experts=512,
             top_k=10, shared=True, d=8, K=16384, dead=0.2, dtype="bf16"),
        # a prompt of odd length through that layer: ten pairs or so for each expert
        dict(name="moe_prompt_e512_509", kind="moe", tokens=509, hidden=4096, inter=1024,
             experts=512, top_k=10, shared=True, d=8, K=16384, dead=0.0, dtype="bf16"),
        # a long prompt through the layer of small experts: 64 pairs for each expert
        dict(name="moe_prompt_e256_2048", kind="moe", tokens=2048, hidden=2048, inter=512,
             experts=256, top_k=8, shared=False, d=4, K=4096, dead=0.0, dtype="bf16"),
        # the embedding rows of that prompt
        dict(name="embed_2048", kind="embed", ids=2048, rows=131072, inp=4096, d=4, K=4096,
             dtype="bf16"),
        # the codes of one expert stack packed to 12 bits when an artifact is written
        dict(name="pack_e256", kind="pack", experts=256, out=512, nsub=512, K=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi):
    """A model dimension: mostly a multiple of 256, else of the scale group."""
    step = 256 if rng.random() < 0.75 else G
    return max(step, int(_log_int(rng, lo, hi) / step + 0.5) * step)


# (d, K, packed): the formats artifacts are written in
FORMATS = [(2, 256, False), (2, 1024, True), (4, 256, False), (4, 1024, True), (4, 4096, True),
           (4, 8192, True), (8, 4096, True), (8, 16384, True), (8, 65536, False)]


def _draw_linear(rng):
    d, K, packed = rng.choice(FORMATS)
    inp, out = _dim(rng, 1024, 17408), _dim(rng, 1024, 17408)
    if rng.random() < 0.3:
        out += rng.randrange(1, 64)             # a head's or a split's odd row count
    rows = rng.choice([_log_int(rng, 1, 32), _log_int(rng, 33, 2048)])
    rows = max(1, min(rows, 2048 * 5120 * 17408 // (inp * out)))
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if dtype == "fp32" and rows > 32:
        rows = max(33, rows // 3)
    return dict(kind="linear", rows=rows, inp=inp, out=out, d=d, K=K, packed=packed, dtype=dtype)


def _draw_moe(rng):
    d, K = rng.choice([(4, 1024), (4, 4096), (4, 4096), (8, 4096), (8, 16384), (8, 16384)])
    experts = rng.choice([64, 96, 128, 160, 256] + ([384, 512] if d == 8 else []))
    top_k = rng.choice([4, 6, 8, 10])
    hidden, inter = 256 * rng.randint(4, 16), 256 * rng.randint(1, 4)
    tokens = rng.choice([_log_int(rng, 1, 8), _log_int(rng, 9, 128), _log_int(rng, 129, 2048)])
    cap = 509 * 10 * 4096 * 1024 // (top_k * hidden * inter)      # the largest listed layer's work
    shared = rng.random() < 0.4
    dead = 0.2 if rng.random() < 0.25 else 0.0
    return dict(kind="moe", tokens=max(1, min(tokens, cap)), hidden=hidden, inter=inter,
                experts=experts, top_k=top_k, shared=shared, d=d, K=K, dead=dead,
                dtype=rng.choice(["bf16", "bf16", "fp16"]))


def _draw_embed(rng):
    d, K = rng.choice([(4, 4096), (8, 4096), (8, 16384)])
    return dict(kind="embed", ids=_log_int(rng, 1, 2048), rows=rng.randrange(30000, 131073),
                inp=_dim(rng, 1024, 5120), d=d, K=K, dtype="bf16")


def _draw_pack(rng):
    return dict(kind="pack", experts=rng.randint(8, 256), out=rng.randint(100, 512),
                nsub=32 * rng.randint(4, 16), K=1 << rng.choice([9, 10, 11, 12, 13, 14]))


def draw(rng):
    return rng.choice([_draw_linear, _draw_linear, _draw_linear, _draw_moe, _draw_moe, _draw_moe,
                       _draw_embed, _draw_pack])(rng)


# ---------------------------------------------------------------- weights
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(0x5EED + 7919 * int(seed))


def _bits(K):
    return (K - 1).bit_length()


def _codes(g, lead, nsub, K, packed):
    """Uniform codes [*lead, nsub] as stored: bytes, 16-bit words, or packed words."""
    if not packed:
        if K <= 256:
            return torch.randint(0, K, (*lead, nsub), dtype=torch.uint8, device="cuda", generator=g)
        return torch.randint(-32768, 32768, (*lead, nsub), dtype=torch.int16, device="cuda",
                             generator=g).view(torch.uint16)       # K = 65536
    bits = _bits(K)
    if nsub % 32 == 0:                          # every bit pattern is 32 codes
        return torch.randint(-2**31, 2**31, (*lead, nsub // 32 * bits), dtype=torch.int32,
                             device="cuda", generator=g)
    c = torch.randint(0, K, (1, math.prod(lead), nsub), dtype=torch.int32, device="cuda", generator=g)
    return vq_pack.pack(c, bits).reshape(*lead, -1)


def _table(g, K, d):
    return (torch.randn(K, d, device="cuda", generator=g) * 0.02).half()


def _scales(g, *shape):
    return (torch.rand(*shape, device="cuda", generator=g) + 0.5).half()


def _linear(g, case, rows):
    inp, d, K = case["inp"], case["d"], case["K"]
    packed = case.get("packed", True)
    return dict(codes=_codes(g, (rows,), inp // d, K, packed), codebook=_table(g, K, d),
                vq_scales=_scales(g, rows, inp // G), group_size=G,
                pack_bits=_bits(K) if packed else 0, in_features=inp if packed else None)


def _experts(g, case, E, out, inp, dead):
    d, K = case["d"], case["K"]
    if not dead:
        return dict(codes=_codes(g, (E, out), inp // d, K, True), codebook=_table(g, K, d),
                    vq_scales=_scales(g, E, out, inp // G), group_size=G, pack_bits=_bits(K),
                    in_features=inp)
    # skipzero: a fixed share of the rows is dead, the others are stored without them
    n_live = E * out - int(dead * E * out)
    live = torch.randperm(E * out, device="cuda", generator=g)[:n_live].sort().values
    table = torch.full((E * out,), -1, dtype=torch.int32, device="cuda")
    table[live] = torch.arange(n_live, dtype=torch.int32, device="cuda")
    return dict(codes=_codes(g, (n_live,), inp // d, K, True), codebook=_table(g, K, d),
                vq_scales=_scales(g, n_live, inp // G), group_size=G, pack_bits=_bits(K),
                in_features=inp, row_table=table.reshape(E, out))


def _block(g, case):
    """The layer's weights: {"gate" | "up" | "down": module arguments}, the shared expert's, its gate."""
    H, I, E = case["hidden"], case["inter"], case["experts"]
    dims = {"gate": (I, H), "up": (I, H), "down": (H, I)}
    routed = {n: _experts(g, case, E, o, i, case["dead"]) for n, (o, i) in dims.items()}
    shared = gate = None
    if case["shared"]:
        shared = {n: _experts(g, case, 1, o, i, 0.0) for n, (o, i) in dims.items()}
        gate = (torch.randn(H, device="cuda", generator=g) / math.sqrt(H)).to(DTYPES[case["dtype"]])
    return routed, shared, gate


def _acts(g, case, *shape):
    return torch.randn(*shape, device="cuda", generator=g).to(DTYPES[case["dtype"]])


def _inputs(case, seed):
    """Every tensor of the case, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        return dict(x=_acts(g, case, case["rows"], case["inp"]), w=_linear(g, case, case["out"]))
    if kind == "moe":
        x = _acts(g, case, case["tokens"], case["hidden"])
        logits = torch.randn(case["tokens"], case["experts"], device="cuda", generator=g)
        return dict(x=x, logits=logits, w=_block(g, case))
    if kind == "embed":
        ids = torch.randint(0, case["rows"], (case["ids"],), device="cuda", generator=g)
        return dict(ids=ids, w=_linear(g, case, case["rows"]))
    codes = torch.randint(0, case["K"], (case["experts"], case["out"], case["nsub"]),
                          dtype=torch.int32, device="cuda", generator=g)
    return dict(codes=codes.to(torch.int16))


# -------------------------------------------------------------- one pass
def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "linear":
        s["module"] = VQLinear(**s.pop("w"))
    elif case["kind"] == "moe":
        routed, shared, gate = s.pop("w")

        def glu(w):
            return VQSwitchGLU(*(VQSwitchLinear(**w[n]) for n in ("gate", "up", "down")))
        s["module"] = VQSparseMoeBlock(glu(routed), top_k=case["top_k"],
                                       shared_expert=glu(shared) if shared else None,
                                       shared_expert_gate=gate)
    elif case["kind"] == "embed":
        s["module"] = VQEmbedding(**s.pop("w"), out_dtype=DTYPES[case["dtype"]])
    return s


@torch.no_grad()
def run(state):
    kind = state["case"]["kind"]
    if kind == "linear":
        return state["module"](state["x"])
    if kind == "moe":
        return state["module"](state["x"], state["logits"])
    if kind == "embed":
        return state["module"](state["ids"])
    return codepack.pack_codes("experts", state["codes"], state["case"]["K"])[0]


# ------------------------------------------------------------------ work
def _weight_bytes(case, out, inp):
    nsub = inp // case["d"]
    if case["kind"] == "linear" and not case["packed"]:
        row = nsub * (1 if case["K"] <= 256 else 2)
    else:
        row = -(-nsub // 32) * _bits(case["K"]) * 4
    return out * (row + inp // G * 2)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        r, i, o = case["rows"], case["inp"], case["out"]
        act = 4 if case["dtype"] == "fp32" else 2
        return dict(bytes=_weight_bytes(case, o, i) + case["K"] * case["d"] * 2 + r * (i + o) * act,
                    flops=2 * r * i * o)
    if kind == "moe":
        T, H, I, E, k = (case[n] for n in ("tokens", "hidden", "inter", "experts", "top_k"))
        touched = E * (1 - (1 - k / E) ** T)                       # expected, of uniform routing
        per = 2 * _weight_bytes(case, I, H) + _weight_bytes(case, H, I)
        sh = 1 if case["shared"] else 0
        tables = 3 * case["K"] * case["d"] * 2
        live = 1 - case["dead"]
        return dict(bytes=int(touched * per * live + sh * per + (1 + sh) * tables
                              + T * (2 * H * 2 + E * 4)),
                    flops=int(6 * T * H * I * (k * live + sh)))
    if kind == "embed":
        return dict(bytes=_weight_bytes(case, case["ids"], case["inp"]) + case["K"] * case["d"] * 2
                    + case["ids"] * (case["inp"] * 2 + 8), flops=case["ids"] * case["inp"])
    n = case["experts"] * case["out"] * case["nsub"]
    return dict(bytes=n * 2 + n * _bits(case["K"]) // 8, flops=n)


# --------------------------------------------------------------- results
def tolerance(case):
    if case["kind"] in ("embed", "pack"):
        return "exact"
    # about four times the measured distance from the 64-bit result: one rounding of the outputs;
    # rows that enter the products as fp16 (short fp32 inputs, a layer's SwiGLU rows); weights
    # that enter them as bf16 (long bf16 inputs) or with their scale unrounded (decode)
    long = case["kind"] == "linear" and case["rows"] > 64
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.04} if long else {"rel": 7e-3, "max": 0.02}
    if case["dtype"] == "fp32" and long:
        return {"rel": 2e-5, "max": 1e-4}
    return {"rel": 2e-3, "max": 8e-3} if case["kind"] == "moe" else {"rel": 1.2e-3, "max": 5e-3}


def _unpacked(codes, nsub, K, packed):
    """Stored code rows [R, *] -> integer codes [R, nsub]."""
    if not packed:
        c = codes.view(torch.int16).to(torch.int64) & 0xFFFF if codes.dtype == torch.uint16 else codes
        return c.to(torch.int64)
    bits = _bits(K)
    w = codes.to(torch.int64).reshape(codes.shape[0], -1, bits) & 0xFFFFFFFF
    pos = torch.arange(32, device=codes.device) * bits
    lo, sh = pos // 32, pos % 32
    c = w[..., lo] >> sh
    c = c | torch.where(sh + bits > 32, w[..., (lo + 1).clamp(max=bits - 1)] << (32 - sh), 0)
    return (c & ((1 << bits) - 1)).reshape(codes.shape[0], -1)[:, :nsub]


def _dense(w, codes, scales):
    """fp16(codebook entry * scale), the decoded weight rows, in 64 bits."""
    d = w["codebook"].shape[1]
    K, inp = w["codebook"].shape[0], scales.shape[1] * G
    c = _unpacked(codes, inp // d, K, bool(w["pack_bits"]))
    v = w["codebook"].double()[c].reshape(codes.shape[0], inp)
    return (v * scales.double().repeat_interleave(G, 1)).half().double()


def _expert(w, e):
    """Decoded rows of expert e, dead rows zero."""
    if w.get("row_table") is None:
        return _dense(w, w["codes"][e], w["vq_scales"][e])
    r = w["row_table"][e].long()
    live = r >= 0
    out = torch.zeros(r.numel(), w["vq_scales"].shape[-1] * G, dtype=torch.float64, device=r.device)
    out[live] = _dense(w, w["codes"][r[live]], w["vq_scales"][r[live]])
    return out


def _glu(ws, e, x):
    g, u = x @ _expert(ws["gate"], e).T, x @ _expert(ws["up"], e).T
    return (g * torch.sigmoid(g) * u) @ _expert(ws["down"], e).T


@torch.no_grad()
def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        w = s["w"]
        x = s["x"].double()
        return torch.cat([x @ _dense(w, w["codes"][r:r + 1024], w["vq_scales"][r:r + 1024]).T
                          for r in range(0, case["out"], 1024)], 1)
    if kind == "moe":
        routed, shared, gate = s["w"]
        x = s["x"].double()
        p, ids = torch.topk(torch.softmax(s["logits"].double(), -1), case["top_k"], dim=-1)
        p = p / p.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e in ids.unique().tolist():
            t, j = (ids == e).nonzero(as_tuple=True)
            y.index_add_(0, t, p[t, j, None] * _glu(routed, e, x[t]))
        if shared:
            y += torch.sigmoid(x @ gate.double())[:, None] * _glu(shared, 0, x)
        return y
    return None                                 # whole values: compared as they are
