"""Performance cases of the routed-expert MXFP4 path on one MI355X.

A case is a dict of plain values; its "kind" names the entry point that `run`
calls.  Sizes are the library's two presets (K3: hidden 3584, intermediate
3072, SiTU, fp32; preset 2: hidden 7168, intermediate 2048, SiLU-GLU, bf16),
the K3 MoE block around them, and generic widths between.

  gemv          one MXFP4 matrix against 1..16 activation rows (moe.mxfp4_gemv)
  expert        one expert for a batch of activation rows (moe.moe_launch)
  layer         one token through caller-routed experts (moe.moe_layer)
  route_layer   one token, the router on the device (moe.moe_route_layer)
  verify_route  draft tokens, the router on the device (moe.moe_verify_route)
  verify        draft tokens with a caller route, a different number of experts
                per position, experts shared between positions (moe.moe_verify)
  proj          a resident spine projection, BF16 or row-int8 weights
                (spine.bf16_gemv / spine.int8_gemv)
  block         the whole K3 MoE block, router to output (spine.moe_block)
"""
from __future__ import annotations

import math
import random

import torch

from deltafin_amd import moe, spine

K3 = (3584, 3072)        # preset 1: hidden, intermediate
WIDE = (7168, 2048)      # preset 2
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
_SCALE_LO, _SCALE_HI = 117, 121   # E8M0 bytes: weights of about 1/sqrt(columns)
_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


# ------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # one dequant-GEMV of a gate matrix: the smallest call, launch bound
        dict(name="gemv_one", kind="gemv", rows=2048, cols=7168, batch=1, x="f32", out="f32"),
        # one expert over a small batch of rows, as a host that groups a draft
        # batch by expert calls it (an odd batch)
        dict(name="expert_rows7", kind="expert", hidden=K3[0], inter=K3[1], act="situ", batch=7),
        # one routed expert of a bf16 model, batch 1
        dict(name="layer_one", kind="layer", hidden=WIDE[0], inter=WIDE[1], act="silu", n=1,
             bank=32, x="bf16", out="bf16"),
        # the K3 decode layer: 16 caller-routed experts, fp32
        dict(name="layer_k3", kind="layer", hidden=K3[0], inter=K3[1], act="situ", n=16,
             bank=128, x="f32", out="f32"),
        # the decode layer with the router on the device: 16 of 384, bf16
        dict(name="decode_384", kind="route_layer", hidden=WIDE[0], inter=WIDE[1], act="silu",
             n=16, bank=384, x="bf16", out="bf16"),
        # speculative verify of 8 draft tokens, independent routes
        dict(name="verify_384_m8", kind="verify_route", hidden=WIDE[0], inter=WIDE[1],
             act="silu", n=16, bank=384, m=8, x="bf16", out="bf16"),
        # speculative verify with a caller route: 5 tokens whose routes share
        # most of a pool of experts, fewer experts at some positions
        dict(name="verify_shared_m5", kind="verify", hidden=K3[0], inter=K3[1], act="situ",
             n=16, pool=28, m=5, x="f32", out="f32"),
        # spine projections on their own: a draft batch through BF16 weights,
        # and a wider one through row-int8 weights
        dict(name="proj_bf16_p4", kind="proj", weights="bf16", rows=3584, cols=7168, m=4),
        dict(name="proj_int8_p16", kind="proj", weights="int8", rows=7168, cols=6144, m=16),
        # the whole K3 MoE block: decode of one token, a draft batch over the
        # packed int8 spine, and the widest verify batch
        dict(name="block_p1", kind="block", weights="bf16", bank=896, n=16, m=1),
        dict(name="block_int8_p4", kind="block", weights="int8", bank=896, n=16, m=4),
        dict(name="block_p16", kind="block", weights="bf16", bank=896, n=16, m=16),
    ]


def draw(rng: random.Random) -> dict:
    def log_int(lo: int, hi: int, step: int = 1) -> int:
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min(hi, max(lo, step * round(v / step)))

    def geometry() -> dict:
        which = rng.randrange(4)
        if which == 0:
            return dict(hidden=K3[0], inter=K3[1], act="situ")
        if which == 1:
            return dict(hidden=WIDE[0], inter=WIDE[1], act="silu")
        return dict(hidden=log_int(1024, 7168, 256), inter=log_int(512, 3072, 256),
                    act=rng.choice(("situ", "silu")))

    dtypes = lambda: dict(x=rng.choice(("f32", "bf16")), out=rng.choice(("f32", "bf16")))
    kind = rng.choice(("gemv", "expert", "layer", "route_layer", "verify_route", "verify",
                       "proj", "proj", "block"))
    if kind == "gemv":
        return dict(kind=kind, rows=log_int(500, 12288), cols=log_int(1024, 8192, 32),
                    batch=log_int(1, 16), **dtypes())
    if kind == "expert":
        return dict(kind=kind, batch=log_int(1, 16), **geometry())
    if kind == "layer":
        n = log_int(1, 16)
        return dict(kind=kind, n=n, bank=max(32, 8 * n), **geometry(), **dtypes())
    if kind == "route_layer":
        return dict(kind=kind, n=rng.choice((4, 8, 16)), bank=rng.randrange(64, 385),
                    **geometry(), **dtypes())
    if kind == "verify_route":
        return dict(kind=kind, n=rng.choice((8, 16)), bank=rng.randrange(64, 385),
                    m=log_int(2, 16), **geometry(), **dtypes())
    if kind == "verify":
        return dict(kind=kind, n=16, pool=rng.randrange(20, 65), m=log_int(2, 16), **geometry(),
                    **dtypes())
    if kind == "proj":
        return dict(kind=kind, weights=rng.choice(("bf16", "int8")), rows=log_int(500, 12288),
                    cols=log_int(1024, 7168, 64), m=log_int(1, 64))
    return dict(kind=kind, weights=rng.choice(("bf16", "int8")), bank=rng.randrange(256, 897),
                n=16, m=log_int(1, 16))


# ------------------------------------------------------------------ inputs
def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _geometry(case: dict):
    act = moe.K3_ACT_SITU if case["act"] == "situ" else moe.K3_ACT_SILU
    return moe.geometry(case["hidden"], case["inter"], act)


def _block_case(case: dict) -> dict:
    """The expert geometry inside the K3 MoE block."""
    return dict(case, hidden=K3[0], inter=K3[1], act="situ")


def _bank(g, n: int, gen: torch.Generator) -> torch.Tensor:
    """n expert spans: uniform E2M1 codes, uniform scales in [_SCALE_LO, _SCALE_HI]."""
    off = moe.span_offsets(g)
    bank = torch.empty(n, off["span"], dtype=torch.uint8, device="cuda")
    for e0 in range(0, n, 64):
        part = bank[e0:e0 + 64]
        part.random_(0, 256, generator=gen)
        for lo, hi in (("w1s", "w2p"), ("w2s", "w3p"), ("w3s", "span")):
            part[:, off[lo]:off[hi]].random_(_SCALE_LO, _SCALE_HI + 1, generator=gen)
    return bank


def _randn(*shape: int, gen: torch.Generator, dtype: torch.dtype = torch.float32) -> torch.Tensor:
    return torch.randn(*shape, generator=gen, device="cuda").to(dtype)


def _weights(n: int, rng: random.Random) -> list[float]:
    w = [rng.random() + 0.05 for _ in range(n)]
    return [v / sum(w) for v in w]


def _matrix(weights: str, rows: int, cols: int, gen: torch.Generator):
    """(weights, row scales or None) of a spine matrix."""
    if weights == "bf16":
        return _randn(rows, cols, gen=gen).mul_(cols ** -0.5).to(torch.bfloat16), None
    q = torch.empty(rows, cols, dtype=torch.int8, device="cuda").random_(-127, 128, generator=gen)
    s = torch.rand(rows, generator=gen, device="cuda").add_(0.5).mul_(cols ** -0.5 / 73.0)
    return q, s


def prepare(case: dict, seed: int) -> dict:
    gen, rng = _generator(seed), random.Random(seed)
    kind = case["kind"]
    st = dict(case=case)
    if kind == "gemv":
        rows, cols, b = case["rows"], case["cols"], case["batch"]
        st["packed"] = torch.empty(rows, cols // 2, dtype=torch.uint8,
                                   device="cuda").random_(0, 256, generator=gen)
        st["scales"] = torch.empty(rows, cols // 32, dtype=torch.uint8, device="cuda").random_(
            _SCALE_LO, _SCALE_HI + 1, generator=gen)
        st["x"] = _randn(b, cols, gen=gen, dtype=_DTYPES[case["x"]])
        return st
    if kind == "proj":
        st["w"], st["s"] = _matrix(case["weights"], case["rows"], case["cols"], gen)
        st["x"] = _randn(case["m"], case["cols"], gen=gen)
        return st
    if kind == "block":
        H, R, S, E = 7168, K3[0], 6144, case["bank"]
        st["g"] = _geometry(_block_case(case))
        st["bank"] = _bank(st["g"], E, gen)
        mats = {}
        for name, r, c in (("router", E, H), ("routed_down", R, H), ("routed_up", H, R),
                           ("shared_gate", S, H), ("shared_up", S, H), ("shared_down", H, S)):
            mats[name] = _matrix(case["weights"], r, c, gen)
        scales = {k: v[1] for k, v in mats.items()} if case["weights"] == "int8" else None
        st["spine"] = spine.MoeSpine(
            case["weights"], router_bias=_randn(E, gen=gen).mul_(0.02),
            routed_norm=_randn(R, gen=gen).mul_(0.1).add_(1.0), scales=scales, top_k=case["n"],
            **{k: v[0] for k, v in mats.items()})
        st["x"] = _randn(case["m"], H, gen=gen)
        st["ws"] = spine.moe_block_workspace(st["spine"], st["g"], case["m"])
        return st
    g = st["g"] = _geometry(case)
    xdt = _DTYPES[case.get("x", "f32")]
    if kind == "expert":
        st["bank"] = _bank(g, 1, gen)
        st["x"] = _randn(case["batch"], g.hidden, gen=gen)
    elif kind == "layer":
        st["bank"] = _bank(g, case["bank"], gen)
        st["ids"] = rng.sample(range(case["bank"]), case["n"])
        st["spans"] = [st["bank"][i].data_ptr() for i in st["ids"]]
        st["w"] = _weights(case["n"], rng)
        st["x"] = _randn(g.hidden, gen=gen, dtype=xdt)
        st["ws"] = moe.workspace(g, case["n"])
    elif kind == "route_layer":
        st["bank"] = _bank(g, case["bank"], gen)
        st["logits"] = _randn(case["bank"], gen=gen)
        st["x"] = _randn(g.hidden, gen=gen, dtype=xdt)
        st["ws"] = moe.workspace(g, case["n"])
    elif kind == "verify_route":
        m = case["m"]
        st["bank"] = _bank(g, case["bank"], gen)
        st["logits"] = _randn(m, case["bank"], gen=gen)
        st["x"] = _randn(m, g.hidden, gen=gen, dtype=xdt)
        st["ws"] = moe.workspace(g, m * case["n"], m)
    else:  # verify
        m = case["m"]
        st["bank"] = _bank(g, case["pool"], gen)
        st["ids"], st["w"], st["offs"] = [], [], [0]
        for p in range(m):
            n = case["n"] - (p * 3) % 5
            st["ids"] += rng.sample(range(case["pool"]), n)
            st["w"] += _weights(n, rng)
            st["offs"].append(len(st["ids"]))
        st["spans"] = [st["bank"][i].data_ptr() for i in st["ids"]]
        st["x"] = _randn(m, g.hidden, gen=gen, dtype=xdt)
        st["ws"] = moe.workspace(g, len(st["ids"]), m)
    return st


# ------------------------------------------------------------------ one pass
def run(st: dict):
    case = st["case"]
    kind = case["kind"]
    if kind == "gemv":
        return moe.mxfp4_gemv(st["packed"], st["scales"], st["x"], case["rows"], case["cols"],
                              out_dtype=_DTYPES[case["out"]])
    if kind == "proj":
        if case["weights"] == "bf16":
            return spine.bf16_gemv(st["w"], st["x"])
        return spine.int8_gemv(st["w"], st["s"], st["x"])
    g = st["g"]
    if kind == "expert":
        return moe.moe_launch(g, st["bank"], st["x"])
    if kind == "block":
        return spine.moe_block(st["spine"], g, st["bank"], g.expert_span, st["x"],
                               workspace=st["ws"])
    odt = _DTYPES[case["out"]]
    if kind == "layer":
        return moe.moe_layer(g, st["spans"], st["w"], st["x"], st["ws"], out_dtype=odt)
    if kind == "route_layer":
        return moe.moe_route_layer(g, st["bank"], g.expert_span, case["bank"], st["logits"],
                                   case["n"], st["x"], st["ws"], out_dtype=odt)
    if kind == "verify_route":
        return moe.moe_verify_route(g, st["bank"], g.expert_span, case["bank"], st["logits"],
                                    case["n"], st["x"], st["ws"], out_dtype=odt)
    return moe.moe_verify(g, st["spans"], st["w"], st["offs"], st["x"], st["ws"], out_dtype=odt)


# ------------------------------------------------------------------ what a pass needs
def _positions(case: dict) -> list[int]:
    """Experts of each position."""
    kind = case["kind"]
    if kind == "expert":
        return [1] * case["batch"]
    if kind in ("layer", "route_layer"):
        return [case["n"]]
    if kind == "verify":
        return [case["n"] - (p * 3) % 5 for p in range(case["m"])]
    return [case["n"]] * case["m"]


def work(case: dict) -> dict:
    kind = case["kind"]
    xb = 2 if case.get("x") == "bf16" else 4
    ob = 2 if case.get("out") == "bf16" else 4
    if kind == "gemv":
        r, c, b = case["rows"], case["cols"], case["batch"]
        return dict(bytes=r * c // 2 + r * c // 32 + b * (c * xb + r * ob), flops=2 * r * c * b)
    if kind == "proj":
        r, c, m = case["rows"], case["cols"], case["m"]
        per_row = 2 * c if case["weights"] == "bf16" else c + 4
        return dict(bytes=r * per_row + 4 * m * (c + r), flops=2 * r * c * m)
    geo = _block_case(case) if kind == "block" else case
    H, I = geo["hidden"], geo["inter"]
    per_pos = _positions(case)
    m, edges = len(per_pos), sum(per_pos)
    span = 3 * H * I // 2 + 3 * H * I // 32
    if kind == "expert":
        unique = 1.0
    else:  # the expected number of distinct experts of independent routes
        pool = case["pool"] if kind == "verify" else case["bank"]
        unique = pool * (1.0 - math.prod(1.0 - n / pool for n in per_pos))
    flops = 6 * H * I * edges
    if kind == "block":
        B, S, E = 7168, 6144, case["bank"]
        params = E * B + 2 * H * B + 3 * S * B
        matrices = 2 * params if case["weights"] == "bf16" else params + 4 * (
            E + H + B + 2 * S + B)
        return dict(bytes=int(unique * span) + matrices + 8 * m * B + 8 * edges,
                    flops=flops + 2 * m * params)
    extra = m * H * (xb + ob)
    if kind == "expert":
        extra += 4 * m * I
    if kind in ("route_layer", "verify_route"):
        extra += 4 * m * case["bank"] + 8 * edges
    return dict(bytes=int(unique * span) + extra, flops=flops)


# ------------------------------------------------------------------ tolerances
def tolerance(case: dict) -> dict:
    """About four times the distance from the 64-bit result measured on the card."""
    # a route can differ where two experts tie within the logits' rounding
    if case.get("out") == "bf16":
        return dict(rel=7e-3, differ=0.01)    # one bf16 rounding of the result (1.7e-3)
    if case["kind"] in ("verify", "verify_route") or (case["kind"] == "block" and case["m"] > 1):
        # batches whose experts are shared keep h in 12-bit block-scaled terms (3.1e-5)
        return dict(rel=1.3e-4, differ=0.01)
    return dict(rel=2e-6, differ=0.01)        # fp32 sums (1.0e-7 to 3.9e-7)


# ------------------------------------------------------------------ 64-bit results
def _dequant(packed: torch.Tensor, scales: torch.Tensor, rows: int, cols: int) -> torch.Tensor:
    lut = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device="cuda")
    p = packed.reshape(rows, cols // 2)
    v = torch.stack((lut[(p & 15).long()], lut[(p >> 4).long()]), dim=-1)
    s = torch.exp2(scales.reshape(rows, cols // 32).double() - 127.0)
    return (v.reshape(rows, cols // 32, 32) * s.unsqueeze(-1)).reshape(rows, cols)


def _expert64(span: torch.Tensor, H: int, I: int, act: str, x: torch.Tensor):
    """(h, output) of one expert for x [rows, H], in 64 bits."""
    n13, s13 = I * H // 2, I * (H // 32)
    span = span.reshape(-1)
    parts = torch.split(span, [n13, s13, n13, s13, n13, s13])
    gate = x @ _dequant(parts[0], parts[1], I, H).t()
    up = x @ _dequant(parts[4], parts[5], I, H).t()
    if act == "situ":
        h = 4.0 * torch.tanh(gate / 4.0) * torch.sigmoid(gate) * (25.0 * torch.tanh(up / 25.0))
    else:
        h = gate * torch.sigmoid(gate) * up
    return h, h @ _dequant(parts[2], parts[3], H, I).t()


def _routed64(bank: torch.Tensor, geo: dict, x: torch.Tensor, routes: list[list[int]],
              weights: list[list[float]]) -> torch.Tensor:
    """sum over each position's route of weight * expert(x), each expert once."""
    out = torch.zeros(x.shape[0], geo["hidden"], dtype=torch.float64, device="cuda")
    users: dict[int, list[tuple[int, float]]] = {}
    for p, (ids, ws) in enumerate(zip(routes, weights)):
        for i, w in zip(ids, ws):
            users.setdefault(i, []).append((p, w))
    for i, rows in users.items():
        pos = torch.tensor([p for p, _ in rows], device="cuda")
        w = torch.tensor([w for _, w in rows], dtype=torch.float64, device="cuda")
        _, y = _expert64(bank[i], geo["hidden"], geo["inter"], geo["act"], x[pos])
        out.index_add_(0, pos, y * w.unsqueeze(1))
    return out


def _top_k(v: torch.Tensor, k: int) -> torch.Tensor:
    """The k largest of each row, descending, the lower index first on ties."""
    return torch.sort(v, dim=-1, descending=True, stable=True).indices[..., :k]


def exact(case: dict, seed: int):
    st = prepare(case, seed)
    kind = case["kind"]
    x = st["x"].double()
    if kind == "gemv":
        return x @ _dequant(st["packed"], st["scales"], case["rows"], case["cols"]).t()
    if kind == "proj":
        y = x @ st["w"].double().t()
        return y * st["s"].double() if case["weights"] == "int8" else y
    if kind == "expert":
        return _expert64(st["bank"], case["hidden"], case["inter"], case["act"], x)
    if kind == "layer":
        return _routed64(st["bank"], case, x.unsqueeze(0), [st["ids"]], [st["w"]])[0]
    if kind == "verify":
        cut = list(zip(st["offs"], st["offs"][1:]))
        return _routed64(st["bank"], case, x, [st["ids"][a:b] for a, b in cut],
                         [st["w"][a:b] for a, b in cut])
    if kind in ("route_layer", "verify_route"):
        logits = st["logits"].double().reshape(-1, case["bank"])
        ids = _top_k(logits, case["n"])
        w = torch.softmax(torch.gather(logits, 1, ids), dim=1)
        out = _routed64(st["bank"], case, x.reshape(-1, case["hidden"]), ids.tolist(), w.tolist())
        if kind == "route_layer":
            return out[0], ids[0], w[0]
        return out, ids, w
    sp = st["spine"]

    def mul(name: str, v: torch.Tensor) -> torch.Tensor:
        y = v @ getattr(sp, name).double().t()
        return y * sp.scales[name].double() if case["weights"] == "int8" else y

    scores = torch.sigmoid(mul("router", x))
    ids = _top_k(scores + sp.router_bias.double(), case["n"])
    w = torch.gather(scores, 1, ids)
    w = w / (w.sum(dim=1, keepdim=True) + 1e-20)
    routed = _routed64(st["bank"], _block_case(case), mul("routed_down", x), ids.tolist(),
                       w.tolist())
    normed = sp.routed_norm.double() * routed * torch.rsqrt(
        routed.square().mean(dim=1, keepdim=True) + 1e-5)
    gate, up = mul("shared_gate", x), mul("shared_up", x)
    h = 4.0 * torch.tanh(gate / 4.0) * torch.sigmoid(gate) * (25.0 * torch.tanh(up / 25.0))
    return mul("routed_up", normed) + mul("shared_down", h), ids, w
