"""The work a user of this package has it do, as measurable cases.

Three model-layer formats are served: K4 trellis experts, joined-MXFP4 experts (what a K4 layer becomes
in optimised mode) and K3 trellis experts (the multi-token-prediction layer), all at the GLM-5.3 layer
shape (hidden 6144, 256 routed experts with top-8 plus one shared expert, intermediate 2048).  A case is

  decode   the routed block of 1..8 token rows through a bound decode call (router, top-8, experts,
           combine): single-token decoding, and verification of a few speculated tokens, whose
           neighbouring rows are alike (pairs around one vector, each with `noise` of its own)
  layer    the post-attention half of a decoder layer for 1..8 rows: residual add, RMSNorm and the
           routed block, through a bound layer call
  block    MoEBlock on 9..2048 rows: batched decoding of many sequences (9..32 rows), short prompts
           and full prefill chunks; with a Zipf-skewed or an even expert popularity
  encode   the load-time conversion of a layer's K4 experts to joined MXFP4

Inputs are seeded random weights and activations of those shapes.  Rows whose top-9 corrected router
scores hold a near tie are drawn again, so that the selected experts do not hang on the last bit of a
32-bit sum.
"""
import math
from types import SimpleNamespace

import torch

from mlxlr8_amd.experts import ExpertLayer
from mlxlr8_amd.joined_mxfp4 import JoinedMXFP4, encode
from mlxlr8_amd.model import MoEArgs, MoEBlock

H, M, ROUTED, EXPERTS, TOP = 6144, 2048, 256, 257, 8
WIDTH = {"k4": 4, "k3": 3}
EPS = 1e-5


def listed():
    return [
        # one decoded token per layer call: the K4 layer, the joined-MXFP4 layer, the K3 draft layer
        {"name": "k4_decode_1", "kind": "decode", "format": "k4", "rows": 1, "noise": 0.0, "zipf": False},
        {"name": "mx_decode_1", "kind": "decode", "format": "mx", "rows": 1, "noise": 0.0, "zipf": False},
        {"name": "k3_decode_1", "kind": "decode", "format": "k3", "rows": 1, "noise": 0.0, "zipf": False},
        # verification of speculated tokens: neighbouring rows are alike, so experts repeat
        {"name": "k4_verify_8", "kind": "decode", "format": "k4", "rows": 8, "noise": 0.5, "zipf": False},
        {"name": "mx_verify_5", "kind": "decode", "format": "mx", "rows": 5, "noise": 0.5, "zipf": False},
        # a decoder layer's post-attention half for three sequences
        {"name": "k4_layer_3", "kind": "layer", "format": "k4", "rows": 3, "noise": 0.0, "zipf": True},
        # batched decoding of more sequences than one decode call takes
        {"name": "k4_block_13", "kind": "block", "format": "k4", "rows": 13, "zipf": False},
        {"name": "mx_block_24", "kind": "block", "format": "mx", "rows": 24, "zipf": False},
        # prefill chunks: the usual short one, a ragged long one, a full one
        {"name": "mx_block_512", "kind": "block", "format": "mx", "rows": 512, "zipf": True},
        {"name": "k4_block_1501", "kind": "block", "format": "k4", "rows": 1501, "zipf": True},
        {"name": "mx_block_2048", "kind": "block", "format": "mx", "rows": 2048, "zipf": True},
        # loading a K4 layer in optimised mode
        {"name": "encode_257", "kind": "encode", "experts": EXPERTS},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "layer", "block", "block", "block", "encode"])
    if kind in ("decode", "layer"):
        return {"kind": kind, "format": rng.choice(["k4", "mx", "k3"]) if kind == "decode" else "k4",
                "rows": rng.randint(1, 8), "noise": round(rng.uniform(0.3, 1.2), 3), "zipf": rng.random() < 0.5}
    if kind == "block":
        fmt = rng.choice(["k4", "mx", "mx", "k3"])
        most = {"k4": 1500, "mx": 2000, "k3": 900}[fmt]
        return {"kind": kind, "format": fmt, "rows": _log_int(rng, 9, most), "zipf": rng.random() < 0.5}
    return {"kind": kind, "experts": _log_int(rng, 16, 256)}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _bytes(g, n):
    return torch.randint(0, 256, (n,), generator=g, device="cuda", dtype=torch.uint8)


def _signs(g, *shape):
    return (torch.randint(0, 2, shape, generator=g, device="cuda", dtype=torch.int32) * 2 - 1).half()


def _signed_scale(g, mu, *shape):
    return (torch.exp(_randn(g, *shape) * 0.3 + mu) * _signs(g, *shape).float()).half()


def _trellis(g, k, experts):
    """Packed gate/up/down and their (in, out) side vectors: uniform random bitstreams, +-1 input signs,
    signed lognormal output scales around 1 / sqrt(hidden)."""
    mu = -0.5 * math.log(H)
    packed, scales = {}, {}
    for p in ("gate", "up", "down"):
        a, b = (M, H) if p == "down" else (H, M)
        packed[p] = _bytes(g, experts * H * M * k // 8)
        scales[p] = (_signs(g, experts, a), _signed_scale(g, mu, experts, b))
    return packed, scales


def _joined(g):
    """Joined MXFP4 experts: random e2m1 codes, e8m0 scales that give values of about 1 / sqrt(hidden)."""
    base = 127 + math.floor(math.log2(1.0 / math.sqrt(H) / math.sqrt(8.5625)))
    weights = {}
    for name, (n, k) in (("gate_up", (2 * M, H)), ("down", (H, M))):
        codes = _bytes(g, EXPERTS * n * k // 2).view(EXPERTS, n, k // 2)
        sc = torch.randint(base, base + 2, (EXPERTS, n, k // 32), generator=g, device="cuda", dtype=torch.uint8)
        weights[name] = (codes, sc)
    scales = {"gate": (None, _signed_scale(g, 0.0, EXPERTS, M)), "up": (None, _signed_scale(g, 0.0, EXPERTS, M)),
              "down": (_signs(g, EXPERTS, M), _signed_scale(g, 0.0, EXPERTS, H))}
    return weights, _signs(g, H), scales


def _routes(x, w, bias):
    """(ids [rows, 9], scores [rows, 8], clear [rows]) in 64 bits; clear: no near tie among the top 9."""
    s = torch.sigmoid(x.double() @ w.double().T)
    top, ids = torch.topk(s + bias.double(), TOP + 1, dim=-1)
    clear = (top[:, :-1] - top[:, 1:]).amin(-1)
    ids = ids[:, :TOP]
    p = torch.gather(s, 1, ids)
    shared = torch.full_like(ids[:, :1], ROUTED)
    return torch.cat([ids, shared], 1), p / p.sum(-1, keepdim=True) * 2.5, clear


def _normed(x, attn, weight):
    """(h, row) of a layer call: h = bf16(x + attn), row = bf16(weight * bf16(h / rms(h)))."""
    h = (x.double() + attn.double()).bfloat16()
    r = torch.rsqrt(h.double().square().mean(-1, keepdim=True) + EPS)
    return h, ((h.double() * r).bfloat16().double() * weight.double()).bfloat16()


def _inputs(case, seed):
    """What both a run and its 64-bit value start from."""
    g = _gen(seed)
    s = SimpleNamespace()
    if case["kind"] == "encode":
        s.packed, s.scales = _trellis(g, 4, case["experts"])
        return s
    rows = case["rows"]
    s.w = _randn(g, ROUTED, H) * 0.02
    s.bias = _randn(g, ROUTED) * 0.01
    if case.get("zipf"):
        rank = torch.randperm(ROUTED, generator=g, device="cuda").double() + 1.0
        s.bias = s.bias + (0.08 * rank.pow(-1.1)).float()
    noise = case.get("noise", 0.0)
    group = 2 if noise and rows > 1 else 1
    n = 2 * ((rows + group - 1) // group) + 32
    x = _randn(g, n, 1, H)
    if noise:
        x = x + noise * _randn(g, n, group, H)
    x = x.bfloat16().reshape(n * group, H)
    attn = _randn(g, n * group, H).bfloat16()
    s.norm = (0.5 + torch.rand(H, generator=g, device="cuda")).bfloat16()
    if case["kind"] == "layer":
        clear = _routes(_normed(x, attn, s.norm)[1], s.w, s.bias)[2] > 1e-4
    else:
        clear = _routes(x, s.w, s.bias)[2] > 1e-5
    keep = clear.view(n, group).all(-1).nonzero()[:, 0]
    at = (keep[:, None] * group + torch.arange(group, device="cuda")).reshape(-1)[:rows]
    if at.numel() != rows:
        raise RuntimeError("too few rows without near ties")
    s.x, s.other = x[at].contiguous(), attn[at].contiguous()
    if case["format"] == "mx":
        s.weights, s.unit, s.scales = _joined(g)
    else:
        s.packed, s.scales = _trellis(g, WIDTH[case["format"]], EXPERTS)
    return s


def prepare(case, seed):
    i = _inputs(case, seed)
    s = SimpleNamespace(kind=case["kind"])
    if case["kind"] == "encode":
        s.layer = ExpertLayer(i.packed, i.scales, H, M, k=4)
        return s
    if case["format"] == "mx":
        affine = JoinedMXFP4(i.weights, i.unit, i.scales, H, M)
        experts = SimpleNamespace(affine=affine, hidden=H, intermediate=M, k=4)
    else:
        affine = None
        experts = ExpertLayer(i.packed, i.scales, H, M, k=WIDTH[case["format"]])
    if case["kind"] == "decode":
        s.call = (affine or experts).prepare_decode(i.x, i.other, i.w, i.bias)
    elif case["kind"] == "layer":
        s.call = experts.prepare_layer_decode(i.x, i.norm, i.w, i.bias, attn=i.other, eps=EPS)
    else:
        s.block, s.x, s.h = MoEBlock(MoEArgs(), i.w, i.bias, experts), i.x, i.other
    return s


def run(state):
    if state.kind == "encode":
        unit, w = encode(state.layer)
        return {"unit": unit, "gate_up": w["gate_up"][:2], "down": w["down"][:2]}
    if state.kind == "block":
        return {"out": state.block(state.x, state.h)}
    state.call.run()
    return {"out": state.call.out, "ids": state.call.ids, "scores": state.call.scores}


# ---------------------------------------------------------------- bytes, operations, tolerances

def _distinct(case):
    """About how many distinct experts the rows select, the shared one included (even popularity; the
    neighbouring rows of a pair, which differ by `noise`, share a part of theirs)."""
    noise = case.get("noise", 0.0)
    n = case["rows"] * (min(1.0, 0.5 + 0.36 * noise) if noise and case["rows"] > 1 else 1.0)
    return 1 + ROUTED * (1 - (1 - TOP / ROUTED) ** n)


def work(case):
    mx_bytes = 3 * H * M * 17 / 32
    if case["kind"] == "encode":
        return {"bytes": case["experts"] * (3 * H * M / 2 + mx_bytes + 2 * 2 * H), "flops": 0}
    rows, fmt = case["rows"], case["format"]
    each = mx_bytes if fmt == "mx" else 3 * H * M * WIDTH[fmt] / 8 + 2 * 3 * (H + M)
    io = rows * H * 2 * 3
    return {"bytes": _distinct(case) * each + ROUTED * H * 4 + io, "flops": rows * 9 * 3 * 2 * H * M + rows * 2 * ROUTED * H}


def tolerance(case):
    """bf16 outputs of a bf16 path (its gate, up and value rows are bf16 too)."""
    if case["kind"] == "encode":
        return "exact"
    return {"rel": 1e-2}


# ---------------------------------------------------------------- the same in 64 bits, plain torch

_H128 = {}


def _had(x):
    """Normalised 128-point Hadamard of independent blocks of the last axis."""
    if "m" not in _H128:
        m = torch.ones((1, 1), dtype=torch.float64)
        while m.shape[0] < 128:
            m = torch.cat([torch.cat([m, m], 1), torch.cat([m, -m], 1)], 0)
        _H128["m"] = (m / math.sqrt(128)).cuda()
    return (x.reshape(-1, 128) @ _H128["m"]).reshape(x.shape)


def _codebook():
    """Value of every 16-bit trellis state: hash, sum of two halves in fp16, rounded to 4 significant bits."""
    if "book" not in _H128:
        word = (torch.arange(1 << 16, dtype=torch.int64) * 0xCBAC1FED) & 0xFFFFFFFF
        word = (word & 0x8FFF8FFF) ^ 0x3B603B60
        halves = [((word >> s) & 0xFFFF) for s in (0, 16)]
        lo, hi = (torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.float16) for v in halves)
        v = (lo.double() + hi.double()).half().double()
        _, e = torch.frexp(v.abs())
        q = torch.ldexp(torch.ones_like(v), torch.clamp(e - 1, min=-6) - 3)
        _H128["book"] = (torch.round(v / q) * q).cuda()
    return _H128["book"]


def _inner(packed, k, a, b, side):
    """[a, b] decoded weights of one packed matrix."""
    it, ot, n = a // 16, b // 16, 8 * k
    words = packed.view(torch.int32).to(torch.int64) & 0xFFFFFFFF
    if side == 2:
        words = words.view(it // 8, ot // 8, 8, 8, n).permute(0, 2, 1, 3, 4).reshape(it, ot, n)
    else:
        words = words.view(ot // 8, it, 8, n).permute(1, 0, 2, 3).reshape(it, ot, n)
    i = torch.arange(256, device=words.device)
    start = (k * (i + 1) - 16) % (256 * k)
    first = start // 32
    both = (words[..., first] << 32) | words[..., (first + 1) % n]
    values = _codebook()[(both >> (48 - start % 32)) & 0xFFFF]
    t, j = i // 8, i % 8
    row = (t % 4) * 2 + torch.tensor([0, 1, 8, 9], device=i.device)[j % 4]
    place = row * 16 + t // 4 + torch.where(j >= 4, 8, 0)
    tile = torch.empty_like(values)
    tile[..., place] = values
    return tile.view(it, ot, 16, 16).permute(0, 2, 1, 3).reshape(a, b)


def _mx(codes, scales):
    """[n, k] values of MXFP4 rows."""
    table = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=codes.device)
    table = torch.cat([table, -table])
    v = torch.stack([table[(codes & 15).long()], table[(codes >> 4).long()]], -1).view(codes.shape[0], -1, 32)
    return (v * torch.exp2(scales.double() - 127)[..., None]).view(codes.shape[0], -1)


def _expert(i, fmt, e, x):
    """[n, H] values of expert e for the rows x."""
    if fmt == "mx":
        gu = _had(x * i.unit.double()) @ _mx(i.weights["gate_up"][0][e], i.weights["gate_up"][1][e]).T
        gate, up = gu[:, :M], gu[:, M:]
        down = _mx(i.weights["down"][0][e], i.weights["down"][1][e]).T
    else:
        k = WIDTH[fmt]
        size = H * M * k // 8
        gate, up = (_had(x * i.scales[p][0][e].double()) @ _inner(i.packed[p][e * size:(e + 1) * size], k, H, M, 1)
                    for p in ("gate", "up"))
        down = _inner(i.packed["down"][e * size:(e + 1) * size], k, M, H, 2)
    gate, up = _had(gate) * i.scales["gate"][1][e].double(), _had(up) * i.scales["up"][1][e].double()
    act = gate * torch.sigmoid(gate) * up
    v = _had(act * i.scales["down"][0][e].double()) @ down
    return _had(v) * i.scales["down"][1][e].double()


def exact(case, seed):
    i = _inputs(case, seed)
    if case["kind"] == "encode":  # codes and scales are bytes
        return {"unit": torch.sign(i.scales["gate"][0][:1].double()), "gate_up": (None, None), "down": (None, None)}
    x, h = i.x, i.other
    if case["kind"] == "layer":
        h, x = _normed(x, h, i.norm)
    ids, scores, _ = _routes(x, i.w, i.bias)
    x, out = x.double(), h.double()
    weight = torch.cat([scores, torch.ones_like(scores[:, :1])], 1)
    for e in torch.unique(ids).tolist():
        row, slot = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, row, _expert(i, case["format"], e, x[row]) * weight[row, slot][:, None])
    if case["kind"] == "block":
        return {"out": out}
    return {"out": out, "ids": None, "scores": scores}
