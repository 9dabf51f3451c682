"""The measured workloads of the library: what a program that uses it has it do, through its Python entry points.

An inference engine for a block-diffusion MoE model calls the library once per layer and denoising step: a decode
step is one routing block (at most 32 tokens) that streams each chosen expert's packed weights once; batched
denoising and prefill are many blocks at once. Beside the MoE layers it runs dense W.A8 projections (qkv, attention
output) through the same kernels.

A case of kind "layer" is one pass over `layers` MoE layers of hidden 2048, intermediate 512, with weights of their
own (as in a model's stack: the weights of one layer are not in the caches when their turn comes):
  entry  "forward"   Layer.forward: A8, routing, experts, combine
         "norm"      Layer.forward_norm: the same with the residual add and the next layer's RMSNorm / rotation / A8
         "external"  quantize_a8 + Layer.dispatch + Layer.experts: tokens routed by the caller
  route  "x" the layer's own router; "zipf" / "skewed" router logits with that expert popularity, as given
  bits   "mixed" (61 / 34 / 6 % of 2 / 3 / 4-bit experts) or one width for every expert
A case of kind "dense" quantises x once and runs `layers` projections [rows, 2048] on it.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "llada2-orin-cuda_amd"))
import llmoe  # noqa: E402

H, I, GROUP, BLOCK, SCALE = 2048, 512, 128, 32, 2.5
CODE_BYTES = {2: 512, 3: 768, 4: 1024, 8: 2048}   # of one 16 x 128 tile; 48 bytes of scales and zeros follow
EPS = 1e-6


def _layer(T, *, name=None, entry="forward", route="x", bits="mixed", shared=True, pool=256, E=256, K=8, fast=False,
           outliers=False, layers=1):
    c = dict(kind="layer", T=T, entry=entry, route=route, bits=bits, shared=shared, pool=pool, E=E, K=K, fast=fast,
             outliers=outliers, layers=layers)
    return dict(c, name=name) if name else c


def _dense(T, rows, bits, layers, accumulate=False, name=None):
    c = dict(kind="dense", T=T, rows=rows, bits=bits, layers=layers, accumulate=accumulate)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: the tail of a denoised block, one token left; launches and latency
        _layer(1, name="token", pool=48, layers=4),
        # an odd remainder of a block, with the fused epilogue as an engine's layer step calls it, pool as shipped
        _layer(19, name="block19_norm", entry="norm", pool=48, layers=4),
        # one denoising block, the shipped mix, uniform routing without the pool: the usual decode step
        _layer(32, name="block32", layers=4),
        # one denoising block, every expert 4-bit, pool of 48, no shared expert
        _layer(32, name="block32_4bit", bits="4", shared=False, pool=48, layers=4),
        # a few sequences at once and a ragged last block, routed by the caller
        _layer(77, name="blocks77_external", entry="external", pool=256, layers=3),
        # prefill of 16 blocks, outlier channels, pool of 48
        _layer(512, name="prefill512", pool=48, outliers=True, layers=2),
        # 64 sequences denoised together, popular experts, exact numerics
        _layer(2048, name="batch2048_zipf", route="zipf", layers=2),
        # the same as an engine that chose the fast numerics would step it, a ragged batch
        _layer(1901, name="batch1901_fast_norm", entry="norm", route="zipf", fast=True, layers=2),
        # the largest batches: 4-bit experts with half of the slots on 16 experts; 8-bit experts
        _layer(4096, name="batch4096_4bit", route="skewed", bits="4", shared=False),
        _layer(4096, name="batch4096_8bit", bits="8", shared=False),
        # dense projections of a decode step (qkv shape) and of a prefill (attention output, added to the residual)
        _dense(32, 3072, 8, 8, name="dense32_qkv"),
        _dense(2048, 2048, 4, 4, accumulate=True, name="dense2048_out"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.2:
        T = _log_int(rng, 1, 3000)
        return _dense(T, 256 * rng.randint(2, 16), rng.choice([2, 3, 4, 8]), 8 if T <= 256 else 3, rng.random() < 0.4)
    T = _log_int(rng, 1, 3400)   # with a shared expert at most the slots of the largest listed case
    E = rng.choice([256, 256, 256, 192, 128, 64])
    K = rng.choice([8, 8, 8, 6, 4, 2])
    entry = rng.choice(["forward", "forward", "norm", "external"])
    route = "x" if entry == "external" else rng.choice(["x", "x", "zipf", "skewed"])
    return _layer(T, entry=entry, route=route, bits=rng.choice(["mixed", "mixed", "mixed", "2", "3", "4", "8"]),
                  shared=rng.random() < 0.7, pool=rng.choice([48, 48, E]), E=E, K=K, fast=rng.random() < 0.25,
                  outliers=rng.random() < 0.3, layers=4 if T <= 64 else 2 if T <= 1024 else 1)


# ---- inputs, from the seed alone (torch only) ----------------------------------------------------------------------

def _gen(seed, *what):
    g = torch.Generator(device="cuda")
    s = seed & 0xFFFFFFFF
    for w in what:
        s = (s * 1000003 + w + 1) & 0x7FFFFFFF
    g.manual_seed(s)
    return g


def _tiles(g, n, R, K, bits, symmetric):
    """n packed [R, K] matrices: random codes, scales ~U(0.005, 0.02), random zeros; symmetric 8-bit matrices have one
    scale per row, at 1/16 of the range, and zero 128. uint8 [n, R / 16, K / 128, tile bytes]."""
    wb = CODE_BYTES[bits]
    m = torch.randint(0, 256, (n, R // 16, K // GROUP, wb + 48), dtype=torch.uint8, device="cuda", generator=g)
    shape = (n, R // 16, 1 if symmetric else K // GROUP, 16)
    s = torch.rand(shape, device="cuda", generator=g) * 0.015 + 0.005
    s = (s / 16 if symmetric else s).half().expand(n, R // 16, K // GROUP, 16).contiguous()
    m[..., wb:wb + 32] = s.view(torch.uint8)
    m[..., wb + 32:] = 128 if symmetric else torch.randint(0, 1 << bits, (n, R // 16, K // GROUP, 16),
                                                           dtype=torch.uint8, device="cuda", generator=g)
    return m


def _weights(case, seed, li):
    """One layer's packed experts on the GPU: blob, offsets of gate_up and down, widths, router, bias."""
    g = _gen(seed, 1, li)
    E = case["E"]
    if case["bits"] == "mixed":
        p = torch.tensor([0.61, 0.34, 0.06], device="cuda")
        bits = [(2, 3, 4)[i] for i in torch.multinomial(p, E, replacement=True, generator=g).tolist()]
    else:
        bits = [int(case["bits"])] * E
    if case["shared"]:
        bits.append(8)
    parts, gu_off, d_off, at = [], [0] * len(bits), [0] * len(bits), 0
    for b in sorted(set(bits)):
        ids = [e for e, v in enumerate(bits) if v == b]
        gu = _tiles(g, len(ids), 2 * I, H, b, b == 8).reshape(len(ids), -1)
        dn = _tiles(g, len(ids), H, I, b, b == 8).reshape(len(ids), -1)
        parts.append(torch.cat([gu, dn], 1).reshape(-1))
        size = gu.shape[1] + dn.shape[1]
        for k, e in enumerate(ids):
            gu_off[e], d_off[e] = at + k * size, at + k * size + gu.shape[1]
        at += len(ids) * size
    router = torch.randn((H, E), device="cuda", generator=g) * 0.02
    bias = torch.rand(E, device="cuda", generator=g) * 0.2 - 0.1
    return dict(blob=torch.cat(parts), gu_off=gu_off, d_off=d_off, bits=bits, router=router, bias=bias)


def _x(case, seed):
    g = _gen(seed, 2)
    x = torch.randn((case["T"], H), device="cuda", generator=g)
    if case.get("outliers"):
        x[:, torch.randperm(H, device="cuda", generator=g)[:H // 100]] *= 20.0
    return x


def _routing(case, seed, li):
    """Router logits [T, E] (zipf, skewed), or the caller's (experts, weights), or None: the layer's own router."""
    g = _gen(seed, 3, li)
    T, E, K = case["T"], case["E"], case["K"]
    if case["entry"] == "external":
        topk = torch.rand((T, E), device="cuda", generator=g).topk(K, 1).indices.int().contiguous()
        w = torch.rand((T, K), device="cuda", generator=g) + 0.1
        return topk, (w / w.sum(1, keepdim=True) * SCALE).contiguous()
    if case["route"] == "zipf":   # Gumbel top-k: popularity rank^-1.1 over a random order of the experts
        rank = torch.randperm(E, device="cuda", generator=g) + 1
        u = torch.rand((T, E), device="cuda", generator=g).clamp_(1e-7, 1 - 1e-7)
        return -1.1 * rank.float().log() - (-u.log()).log()
    if case["route"] == "skewed":   # half of every token's experts among 16
        hot = torch.zeros(E, device="cuda")
        hot[torch.randperm(E, device="cuda", generator=g)[:16]] = 1
        r = torch.rand((T, E), device="cuda", generator=g)
        pick = (r + 10 * hot).topk(K // 2, 1).indices
        rest = (r + 10 * (1 - hot)).topk(K - K // 2, 1).indices
        lg = torch.randn((T, E), device="cuda", generator=g) - 4
        high = 4 + 0.1 * torch.randn((T, K), device="cuda", generator=g)
        return lg.scatter_(1, torch.cat([pick, rest], 1), high)
    return None


def _residual(case, seed):
    g = _gen(seed, 4)
    h = torch.randn((case["T"], case.get("rows", H)), device="cuda", generator=g)
    signs = torch.randint(0, 2, (H,), device="cuda", generator=g).float() * 2 - 1
    return h, signs


def prepare(case, seed):
    T, n = case["T"], case["layers"]
    s = {"case": case, "x": _x(case, seed)}
    if case["kind"] == "dense":
        s["layers"] = []
        for li in range(n):
            m = _tiles(_gen(seed, 1, li), 1, case["rows"], H, case["bits"], case["bits"] == 8)
            s["layers"].append(llmoe.Dense(m.reshape(-1).cpu().numpy(), case["rows"], case["bits"], max_tokens=T))
        if case["accumulate"]:
            s["h0"] = _residual(case, seed)[0]
            s["h"] = torch.empty_like(s["h0"])
        else:
            s["out"] = [torch.empty((T, case["rows"]), device="cuda") for _ in range(n)]
        return s
    s["layers"], s["routing"] = [], []
    for li in range(n):
        w = _weights(case, seed, li)
        layer = llmoe.Layer(w["blob"].cpu().numpy(), w["gu_off"], w["d_off"], w["bits"], w["bias"].cpu().numpy(),
                            w["router"].cpu().numpy(), n_experts=case["E"], top_k=case["K"], pool=case["pool"],
                            block=BLOCK, routed_scale=SCALE, has_shared=case["shared"], max_tokens=T)
        if case["fast"]:
            layer.set_numerics(True)
        s["layers"].append(layer)
        s["routing"].append(_routing(case, seed, li))
    if case["entry"] == "norm":
        s["h0"], s["signs"] = _residual(case, seed)
        s["h"] = torch.empty_like(s["h0"])
        s["next"] = [(torch.empty((T, H), dtype=torch.int8, device="cuda"), torch.empty((T, 16), device="cuda"),
                      torch.empty((T, 16), dtype=torch.int32, device="cuda")) for _ in range(n)]
    else:
        s["out"] = [torch.empty((T, H), device="cuda") for _ in range(n)]
    return s


def run(s):
    case, x = s["case"], s["x"]
    if case["kind"] == "dense":
        q = llmoe.quantize_a8(x)
        if case["accumulate"]:
            s["h"].copy_(s["h0"])   # the residual stream as this step finds it
            for d in s["layers"]:
                d.forward(*q, out=s["h"], accumulate=True)
            return {"h": s["h"]}
        return {"y": [d.forward(*q, out=o) for d, o in zip(s["layers"], s["out"])]}
    if case["entry"] == "norm":
        s["h"].copy_(s["h0"])
        nxt = [layer.forward_norm(x, s["signs"], EPS, s["h"], logits=r, out=o)
               for layer, r, o in zip(s["layers"], s["routing"], s["next"])]
        return {"h": s["h"], "q": [v[0] for v in nxt], "s": [v[1] for v in nxt], "sum": [v[2] for v in nxt]}
    if case["entry"] == "external":
        q = llmoe.quantize_a8(x)
        for layer, (topk, topw), o in zip(s["layers"], s["routing"], s["out"]):
            layer.dispatch(topk, topw)
            layer.experts(*q, out=o)
        return {"out": s["out"]}
    return {"out": [layer.forward(x, r, out=o) for layer, r, o in zip(s["layers"], s["routing"], s["out"])]}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _expert_bytes(b):
    return (2 * I * H + H * I) // (16 * GROUP) * (CODE_BYTES[b] + 48)


def work(case):
    T, n = case["T"], case["layers"]
    if case["kind"] == "dense":
        rows = case["rows"]
        w = rows // 16 * 16 * (CODE_BYTES[case["bits"]] + 48)
        y = 4 * T * rows * (2 if case["accumulate"] else 1)
        return {"bytes": 4 * T * H + n * (w + (0 if case["accumulate"] else y)) + (y if case["accumulate"] else 0),
                "flops": 2 * n * T * rows * H}
    E, K = case["E"], case["K"]
    blocks = -(-T // BLOCK)
    touched = E * (1 - (1 - K / E) ** T)
    if case["entry"] != "external" and case["pool"] < E:
        touched = min(touched, E * (1 - (1 - case["pool"] / E) ** blocks))
    share = {2: 0.61 / 1.01, 3: 0.34 / 1.01, 4: 0.06 / 1.01} if case["bits"] == "mixed" else {int(case["bits"]): 1.0}
    w = touched * sum(p * _expert_bytes(b) for b, p in share.items()) + (_expert_bytes(8) if case["shared"] else 0)
    own = case["route"] == "x" and case["entry"] != "external"
    w += 4 * H * E if own else 4 * T * (2 * K if case["entry"] == "external" else E)
    out = T * (H + 128) + 8 * T * H / n if case["entry"] == "norm" else 4 * T * H
    slots = T * (K + (1 if case["shared"] else 0))
    return {"bytes": int(4 * T * H + n * (w + out)), "flops": int(n * (6 * slots * I * H + (2 * T * H * E if own else 0)))}


def tolerance(case):
    """Against float64 the dense outputs are 32-bit sums (3e-8 .. 1e-7 measured). A layer output passes through the
    8-bit quantisation of the down input, where another order of 32-bit sums flips single codes by one step."""
    if case["kind"] == "dense":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 4e-3, "max": 0.2, "differ": 0.02}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------

def _codes(tiles, bits):
    """Codes [R, K] and scales, zeros [R, K / 128] of one packed matrix [R / 16, K / 128, tile bytes]. In a tile, byte b
    of register r of lane p in step j holds row p / 4 + 8 (r % 2), column 32 j + 16 (r / 2) + 4 (p % 4) + b."""
    ns, nt = tiles.shape[:2]
    row, col = torch.meshgrid(torch.arange(16, device="cuda"), torch.arange(GROUP, device="cuda"), indexing="ij")
    j, r = col // 32, 2 * (col // 16 % 2) + row // 8
    p, b = 4 * (row % 8) + col // 4 % 4, col % 4

    def pick(byte, shift, mask):
        return (tiles[:, :, byte.reshape(-1)].int() >> shift.reshape(-1)) & mask

    if bits == 8:
        c = pick(((j * 32 + p) * 4 + r) * 4 + b, 0 * r, 255)
    elif bits == 4:
        wd = 2 * j + r // 2
        c = pick(((wd // 4 * 32 + p) * 4 + wd % 4) * 4 + b, 4 * (r % 2), 15)
    else:
        c = pick((p * 4 + j) * 4 + b, 2 * r, 3)
        if bits == 3:
            c = c | (pick(512 + (p * 2 + j // 2) * 4 + b, 4 * (j % 2) + r, 1) << 2)
    c = c.reshape(ns, nt, 16, GROUP).transpose(1, 2).reshape(ns * 16, nt * GROUP)
    wb = CODE_BYTES[bits]
    s = tiles[:, :, wb:wb + 32].contiguous().view(torch.float16).transpose(1, 2).reshape(ns * 16, nt)
    z = tiles[:, :, wb + 32:].transpose(1, 2).reshape(ns * 16, nt)
    return c, s, z


def _dequant(blob, off, R, K, bits):
    n = R // 16 * (K // GROUP) * (CODE_BYTES[bits] + 48)
    c, s, z = _codes(blob[off:off + n].reshape(R // 16, K // GROUP, -1), bits)
    w = (c.double().reshape(R, K // GROUP, GROUP) - z.double()[..., None]) * s.double()[..., None]
    return w.reshape(R, K)


def _a8(v):
    """(codes, scales, code sums) of rows quantised to 8 bits per 128-group."""
    g = v.reshape(v.shape[0], -1, GROUP)
    s = (g.abs().amax(2) / 127).clamp_min(1e-30)
    q = (g / s[..., None]).round().clamp(-127, 127)
    return q, s, q.sum(2)


def _deq(qs, shape):
    return (qs[0] * qs[1][..., None]).reshape(shape)


def _hadamard(n):
    m = torch.ones((1, 1), dtype=torch.float64, device="cuda")
    while m.shape[0] < n:
        m = torch.cat([torch.cat([m, m], 1), torch.cat([m, -m], 1)], 0)
    return m / math.sqrt(n)


def _exact_route(case, logits, bias):
    sig = torch.sigmoid(logits)
    s = sig + bias.double()
    T, E, K, C = case["T"], case["E"], case["K"], case["pool"]
    if C < E:
        for b in range(0, T, BLOCK):
            out = torch.ones(E, dtype=torch.bool, device="cuda")
            out[s[b:b + BLOCK].amax(0).topk(C).indices] = False
            s[b:b + BLOCK].masked_fill_(out, -math.inf)
    topk = s.topk(K, 1).indices
    w = sig.gather(1, topk)
    return topk, w / (w.sum(1, keepdim=True) + 1e-20) * SCALE


def _exact_layer(case, seed, li, x, xd):
    w = _weights(case, seed, li)
    r = _routing(case, seed, li)
    if case["entry"] == "external":
        topk, topw = r[0].long(), r[1].double()
    else:
        topk, topw = _exact_route(case, x.double() @ w["router"].double() if r is None else r.double(), w["bias"])
    h512 = _hadamard(I)
    out = torch.zeros((case["T"], H), dtype=torch.float64, device="cuda")
    for e, b in enumerate(w["bits"]):
        if e < case["E"]:
            rows, k = (topk == e).nonzero(as_tuple=True)
            if rows.numel() == 0:
                continue
            wt = topw[rows, k]
        else:
            rows, wt = torch.arange(case["T"], device="cuda"), torch.ones(case["T"], dtype=torch.float64, device="cuda")
        # strips of 16 rows: 8 gate rows, then the same channels' up rows
        gu = (xd[rows] @ _dequant(w["blob"], w["gu_off"][e], 2 * I, H, b).T).reshape(-1, I // 8, 2, 8)
        gate, up = gu[:, :, 0].reshape(-1, I), gu[:, :, 1].reshape(-1, I)
        z = (gate * torch.sigmoid(gate) * up).half().double()
        zd = _deq(_a8(z @ h512), z.shape)
        y = (zd @ _dequant(w["blob"], w["d_off"][e], H, I, b).T) * wt[:, None]
        out.index_add_(0, rows, y)
    return out


def exact(case, seed):
    x = _x(case, seed)
    xd = _deq(_a8(x.double()), x.shape)
    if case["kind"] == "dense":
        y = []
        for li in range(case["layers"]):
            m = _tiles(_gen(seed, 1, li), 1, case["rows"], H, case["bits"], case["bits"] == 8).reshape(-1)
            y.append(xd @ _dequant(m, 0, case["rows"], H, case["bits"]).T)
        return {"h": _residual(case, seed)[0].double() + sum(y)} if case["accumulate"] else {"y": y}
    outs = [_exact_layer(case, seed, li, x, xd) for li in range(case["layers"])]
    if case["entry"] != "norm":
        return {"out": outs}
    h, signs = _residual(case, seed)
    h, signs, rot = h.double(), signs.double(), _hadamard(H)
    res = {"h": None, "q": [], "s": [], "sum": []}
    for o in outs:
        h = h + (o @ rot) * signs
        v = (h / (h.square().mean(1, keepdim=True) + EPS).sqrt() * signs) @ rot
        q, s, t = _a8(v)
        res["q"].append(q.reshape(v.shape))
        res["s"].append(s)
        res["sum"].append(t)
    res["h"] = h
    return res
