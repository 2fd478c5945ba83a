"""Timed workloads of the VQ2 kernels: what a program that serves a vector-quantized model calls.

The model is the 2048-wide decoder of the benchmark (q 2048, k / v 512, MLP 6144, 151,936 tokens; MoE layers of 256
routed experts and a shared one, hidden 2048, intermediate 512), its packed projections at 2, 3 and 4 bits a weight,
and matrices of other and odd sizes.  Batch rows run from a single decoded token to a prompt's chunk; activations
are fp16 or bf16, codebooks fp16 (the containers') or bf16 (the runtime's), results in the activation's type, the MoE
layer's in fp32.

A case is a dict: ``kind`` (linear, qkv, gate_up, head, moe, step), ``batch``, ``act`` and ``book`` ("fp16" /
"bf16"), for packed matrices ``rows``, ``n`` and ``bits`` (2, 3, 4), for a step ``kv`` and ``inter``, its widths.
"""
import math

import torch

from compressai_amd.graph import DecodeStepGraph
from compressai_amd.moe import MoELayer
from compressai_amd.rot import get_rot
from compressai_amd.runtime import PackedLinear, PackedLMHead, PackedProjections

DEV = "cuda:0"
TYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
CFG = {2: (16,), 3: (16, 8), 4: (16, 16)}
HIDDEN, KV, INTER, VOCAB = 2048, 512, 6144, 151936
EXPERTS, TOP_K, MOE_INTER = 256, 8, 512


def listed():
    return [
        # one decoded token through the smallest packed matrix (an attention output projection): latency
        dict(name="o_b1", kind="linear", batch=1, rows=HIDDEN, n=HIDDEN, bits=2, act="fp16", book="fp16"),
        # one decoded token through all packed matrices of a dense layer, as generation loops run it: a captured graph
        dict(name="step_b1", kind="step", batch=1, kv=512, inter=6144, act="fp16", book="fp16"),
        # the MLP's down projection for 16 sequences decoded together
        dict(name="down_b16", kind="linear", batch=16, rows=HIDDEN, n=INTER, bits=4, act="fp16", book="fp16"),
        # gate and up for 64 sequences, the two-stage matrices with the small second codebook, the runtime's bf16
        dict(name="gate_up_b64", kind="gate_up", batch=64, rows=INTER, n=HIDDEN, bits=3, act="bf16", book="bf16"),
        # the next token: head and top-1 for one sequence, and for four
        dict(name="head_b1", kind="head", batch=1, rows=VOCAB, n=HIDDEN, bits=2, act="fp16", book="fp16"),
        dict(name="head_b4", kind="head", batch=4, rows=VOCAB, n=HIDDEN, bits=2, act="bf16", book="fp16"),
        # an MoE layer (router, experts, shared expert) for one token, for eight, and for a prompt's chunk
        dict(name="moe_t1", kind="moe", batch=1, act="fp16", book="fp16"),
        dict(name="moe_t8", kind="moe", batch=8, act="fp16", book="fp16"),
        dict(name="moe_t512", kind="moe", batch=512, act="bf16", book="bf16"),
        # a prompt of odd length through the attention's projections
        dict(name="qkv_p333", kind="qkv", batch=333, rows=HIDDEN, n=HIDDEN, bits=2, act="bf16", book="bf16"),
        # a short prompt through one matrix of odd height
        dict(name="linear_p100", kind="linear", batch=100, rows=2999, n=4096, bits=2, act="fp16", book="fp16"),
        # a prompt's chunk through the MLP's wide projections
        dict(name="gate_up_p1024", kind="gate_up", batch=1024, rows=INTER, n=HIDDEN, bits=4, act="fp16", book="fp16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "qkv", "qkv", "gate_up", "gate_up", "head", "head", "moe", "moe",
                       "moe", "step"])
    act = rng.choice(["fp16", "bf16"])
    book = "bf16" if act == "bf16" and rng.random() < 0.5 else "fp16"
    case = dict(kind=kind, batch=1, act=act, book=book)
    if kind == "moe":
        case["batch"] = _log_int(rng, 1, 512)
    elif kind == "step":
        case.update(kv=rng.choice([256, 512, 1024, 2048]), inter=rng.choice([2048, 4096, 6144]))
    elif kind == "head":
        case.update(batch=_log_int(rng, 1, 16), rows=_log_int(rng, 32000, VOCAB), n=HIDDEN, bits=2)
    elif kind == "linear":
        n = rng.choice([512, 1024, 2048, 4096, 6144])
        case.update(batch=_log_int(rng, 1, 1024), rows=_log_int(rng, 256, INTER), n=n, bits=rng.choice([2, 3, 4]))
    elif kind == "qkv":
        case.update(batch=_log_int(rng, 1, 1024), rows=HIDDEN, n=HIDDEN, bits=rng.choice([2, 3]))
    elif kind == "gate_up":
        rows = rng.choice([1408, 2560, 4864, INTER])
        case.update(batch=_log_int(rng, 1, 1024), rows=rows, n=HIDDEN, bits=rng.choice([2, 3, 4]))
    return case


# ------------------------------------------------------------------ inputs
def _codes(g, shape):
    return torch.randint(-32768, 32768, shape, generator=g, device=DEV, dtype=torch.int32).to(torch.int16)


def _codebook(g, rows, dtype):
    return (torch.randn(rows, 8, generator=g, device=DEV) * 0.125 ** 0.5).to(dtype)


def _scales(g, shape, n):
    """Row scales that keep a projection's results near its input's size, as trained weights do."""
    return ((torch.rand(shape, generator=g, device=DEV) + 0.5) * 2.0 * n ** -0.5).to(torch.float16)


def _books(g, dtype):
    return {"16": _codebook(g, 65536, dtype), "16_8": _codebook(g, 256, dtype), "16_16": _codebook(g, 65536, dtype)}


def _matrix(g, rows, n, bits):
    planes = [_codes(g, (rows, n // 8))]
    if bits == 3:
        planes.append(torch.randint(0, 256, (rows, n // 8), generator=g, device=DEV, dtype=torch.int32).to(torch.uint8))
    elif bits == 4:
        planes.append(_codes(g, (rows, n // 8)))
    return dict(planes=planes, scale=_scales(g, (rows,), n), rows=rows, n=n, bits=bits)


def _shapes(case):
    """(tag of the rotation, rows, n, bits) of a case's packed matrices."""
    kind = case["kind"]
    if kind == "step":
        return ([("attn", HIDDEN, HIDDEN, 2)] + [("attn", case["kv"], HIDDEN, 2)] * 2 + [("o", HIDDEN, HIDDEN, 2)]
                + [("mlp", case["inter"], HIDDEN, 4)] * 2 + [("down", HIDDEN, case["inter"], 4)])
    if kind == "qkv":
        return [("attn", r, case["n"], case["bits"]) for r in (case["rows"], KV, KV)]
    if kind == "gate_up":
        return [("mlp", case["rows"], case["n"], case["bits"])] * 2
    return [(kind, case["rows"], case["n"], case["bits"])]


def _inputs(case, seed):
    """The inputs of a case on the GPU, from the seed alone."""
    g = torch.Generator(device=DEV).manual_seed(seed * 1009 + 17)
    act, book = TYPES[case["act"]], TYPES[case["book"]]
    inp = {"books": _books(g, book)}
    if case["kind"] == "moe":
        E, H, I = EXPERTS + 1, HIDDEN, MOE_INTER
        inp.update(gu=_codes(g, (E, 2 * I, H // 8)), gu_scale=_scales(g, (E, 2 * I), H).to(torch.bfloat16),
                   dn=_codes(g, (E, H, I // 8)), dn_scale=_scales(g, (E, H), I).to(torch.bfloat16),
                   gate=(torch.randn(H, generator=g, device=DEV) * 0.02).to(torch.float16),
                   x=torch.randn(case["batch"], H, generator=g, device=DEV).to(act),
                   logits=torch.randn(case["batch"], EXPERTS, generator=g, device=DEV))
        return inp
    shapes = _shapes(case)
    inp["mats"] = [dict(_matrix(g, rows, n, bits), tag=tag) for tag, rows, n, bits in shapes]
    inp["x"] = torch.randn(case["batch"], shapes[0][2], generator=g, device=DEV).to(act)
    return inp


def _linear(m, books):
    return PackedLinear((m["rows"], m["n"]), CFG[m["bits"]], m["tag"], m["planes"], m["scale"], books, DEV)


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "moe":
        layer = MoELayer(inp["gu"], inp["gu_scale"], inp["dn"], inp["dn_scale"], inp["books"]["16"], inp["gate"],
                         top_k=TOP_K)
        return dict(call=layer, args=(inp["x"], inp["logits"]))
    lins = [_linear(m, inp["books"]) for m in inp["mats"]]
    if kind == "linear":
        return dict(call=lins[0], args=(inp["x"],))
    if kind == "head":
        return dict(call=PackedLMHead(lins[0]).argmax, args=(inp["x"],))
    if kind in ("qkv", "gate_up"):
        return dict(call=PackedProjections(lins), args=(inp["x"],))
    qkv, o, mlp, down = PackedProjections(lins[:3]), lins[3], PackedProjections(lins[4:6]), lins[6]

    def step(x):
        q, k, v = qkv(x)
        h = x + o(q)
        gate, up = mlp(h)
        return q, k, v, h + down(torch.nn.functional.silu(gate) * up)

    return dict(call=DecodeStepGraph(step, [inp["x"]]), args=(inp["x"],))


def run(state):
    return state["call"](*state["args"])


# ------------------------------------------------- what a pass cannot do without
def work(case):
    B = case["batch"]
    if case["kind"] == "moe":
        pairs, per_expert = B * (TOP_K + 1), 3 * MOE_INTER * HIDDEN
        touched = EXPERTS * (1.0 - (1.0 - TOP_K / EXPERTS) ** B) + 1
        scales = 2 * (2 * MOE_INTER + HIDDEN)
        return dict(bytes=touched * (per_expert // 4 + scales) + 65536 * 16 + B * (HIDDEN * 6 + EXPERTS * 4),
                    flops=2.0 * pairs * per_expert)
    shapes = _shapes(case)
    byte = flop = 0.0
    for _, rows, n, bits in shapes:
        byte += rows * n * bits / 8 + rows * 2 + (B * rows * 2 if case["kind"] != "head" else 0)
        flop += 2.0 * B * rows * n
    books = 65536 * (2 if max(s[3] for s in shapes) == 4 else 1)
    return dict(bytes=byte + books * 16 + B * shapes[0][2] * 2, flops=flop)


# Largest relative error of a correct implementation at the types of the path, about four times what the path shows
# against 64 bits.  Up to two rows the products are sums in fp32 of fp32 activations: only the result's type rounds
# (fp16 2.1e-4, bf16 1.7e-3); the head's logits (6e-8) and the MoE layer (2.4e-7) stay in fp32.  From three rows on
# the rotated activation is rounded to fp16 as well (2.9e-4 with an fp16 result, up to 7e-5 in the best logits).  In the
# step the roundings of its four stages add up (5.1e-4).
def tolerance(case):
    kind, B = case["kind"], case["batch"]
    if kind == "moe":
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "step":
        return {"rel": 2e-3, "max": 1e-2} if case["act"] == "fp16" else {"rel": 1.6e-2, "max": 8e-2}
    if kind == "head":
        # the best token may change where two logits lie within the rounding of the activation
        return {"rel": 1e-6, "max": 1e-6} if B == 1 else {"rel": 3e-4, "max": 1e-3, "differ": 0.25}
    if case["act"] == "fp16":
        return {"rel": 1.2e-3, "max": 8e-3}
    return {"rel": 7e-3, "max": 2e-2}


# ------------------------------------------------------------ the same in 64 bits
def _rotate(x, rot):
    """Permutation, signs and blockwise Hadamard transform, in 64 bits."""
    y = x.double()[..., rot.perm] * rot.sign.double()
    y = y.reshape(*x.shape[:-1], -1, rot.hb)
    h = 1
    while h < rot.hb:
        y = y.reshape(*x.shape[:-1], -1, rot.hb // (2 * h), 2, h)
        y = torch.stack((y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]), dim=-2)
        h *= 2
    return y.reshape(x.shape) * rot.hb ** -0.5


def _dense(planes, books, scale, cfg):
    """Rows of a packed matrix in 64 bits, the row scales as the modules hold them."""
    w = books["16"].double()[planes[0].int() & 0xFFFF]
    if len(planes) > 1:
        w = w + books["16_8" if cfg == (16, 8) else "16_16"].double()[planes[1].int() & 0xFFFF]
    return w.reshape(planes[0].shape[0], -1) * scale.to(torch.bfloat16).double()[:, None]


def _product(m, books, x):
    xr = _rotate(x, get_rot(m["tag"], m["n"], DEV))
    step = max(1, (1 << 26) // m["n"])
    return torch.cat([xr @ _dense([p[r:r + step] for p in m["planes"]], books, m["scale"][r:r + step], CFG[m["bits"]]).T
                      for r in range(0, m["rows"], step)], dim=-1)


def _moe(inp):
    x, book = inp["x"], inp["books"]["16"].double()
    rot_h, rot_i = get_rot("moe_expert_2048", HIDDEN, DEV), get_rot("moe_expert_512", MOE_INTER, DEV)
    p = torch.softmax(inp["logits"].double(), -1)
    order = torch.sort(p, dim=-1, descending=True, stable=True)
    ids, w = order.indices[:, :TOP_K], order.values[:, :TOP_K]
    w = w / w.sum(-1, keepdim=True)
    out = torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    xr = _rotate(x, rot_h)
    for e in range(EXPERTS + 1):
        if e < EXPERTS:
            t, k = torch.nonzero(ids == e, as_tuple=True)
            if not t.numel():
                continue
            we = w[t, k]
        else:
            t = torch.arange(x.shape[0], device=DEV)
            we = torch.sigmoid(x.double() @ inp["gate"].double())
        gu = xr[t] @ (book[inp["gu"][e].int() & 0xFFFF].reshape(2 * MOE_INTER, -1)
                      * inp["gu_scale"][e].double()[:, None]).T
        act = _rotate(torch.nn.functional.silu(gu[:, :MOE_INTER]) * gu[:, MOE_INTER:], rot_i)
        y = act @ (book[inp["dn"][e].int() & 0xFFFF].reshape(HIDDEN, -1) * inp["dn_scale"][e].double()[:, None]).T
        out[t] += we[:, None] * y
    return out


def exact(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "moe":
        return _moe(inp)
    mats, books, x = inp["mats"], inp["books"], inp["x"]
    if kind == "linear":
        return _product(mats[0], books, x)
    if kind == "head":
        best = _product(mats[0], books, x).max(-1)
        return best.indices, best.values
    if kind in ("qkv", "gate_up"):
        return [_product(m, books, x) for m in mats]
    q, k, v = (_product(m, books, x) for m in mats[:3])
    h = x.double() + _product(mats[3], books, q)
    gate, up = (_product(m, books, h) for m in mats[4:6])
    return q, k, v, h + _product(mats[6], books, torch.nn.functional.silu(gate) * up)
