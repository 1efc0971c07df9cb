"""What a user of this library has it do, as cases that can be timed and checked.

The library is one MoE expert layer over raw GGUF blocks, so the cases are its
calls: decode steps (one token at a time, one layer or a chain of layers),
prompt batches of a few to a few thousand tokens, and the single products a
caller runs outside a layer (one quantised matrix, one expert).  Weights are
N(0, 0.02) through the library's block quantisers, router rows N(0, 0.02),
tokens N(0, 1), as a trained layer's normalised input and weights look.
"""
import numpy as np
import torch

from winmoe_amd import moe

Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K = 8, 10, 11, 12, 13, 14
BYTES = {Q8_0: 34, Q2_K: 84, Q3_K: 110, Q4_K: 144, Q5_K: 176, Q6_K: 210}
ELEMS = {Q8_0: 32, Q2_K: 256, Q3_K: 256, Q4_K: 256, Q5_K: 256, Q6_K: 256}
TYPE = {"q8_0": Q8_0, "q2_k": Q2_K, "q3_k": Q3_K, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}

#: Distinct experts quantised per tensor; the others are these with their rows
#: moved round, so that every expert differs and the inputs are made quickly.
BANK = 32


def _layer(do, name, E, K, H, I, gu, down, tokens, shared="", layers=1, routed="router"):
    return {"name": name, "do": do, "E": E, "K": K, "H": H, "I": I, "gu": gu, "down": down, "shared": shared,
            "tokens": tokens, "layers": layers, "routed": routed}


def listed():
    return [
        # one token through a small layer: the shortest call there is, all latency
        _layer("decode", "decode_small_q8_0", 64, 4, 2048, 512, "q8_0", "q8_0", 1),
        # generation, 8-bit experts with a shared expert: 8 tokens one after another
        _layer("decode", "decode_top10_q8_0", 512, 10, 4096, 1024, "q8_0", "q8_0", 8, shared="q8_0"),
        # generation, the usual 4-bit mix (Q4_K gate/up, Q6_K down, 8-bit shared expert)
        _layer("decode", "decode_top3_q4_k", 512, 3, 4096, 1024, "q4_k", "q6_k", 8, shared="q8_0"),
        # generation through a chain of 2/3-bit layers (norm and residual inside), routed by the caller
        _layer("stack", "decode_stack_q2_k", 512, 3, 4096, 1024, "q2_k", "q3_k", 4, layers=8, routed="caller"),
        # a short prompt (or a few requests decoded together): few pairs per expert
        _layer("prefill", "prefill_23_q4_k", 512, 3, 4096, 1024, "q4_k", "q6_k", 23, shared="q8_0"),
        # a small layer under an odd prompt length
        _layer("prefill", "prefill_1001_small_q8_0", 64, 4, 2048, 512, "q8_0", "q8_0", 1001),
        # an ordinary prompt chunk, 8-bit experts, routed by the layer's router
        _layer("prefill", "prefill_512_q8_0", 512, 10, 4096, 1024, "q8_0", "q8_0", 512),
        # the same chunk through the 4-bit mix, skewed routing from the caller
        _layer("prefill", "prefill_512_q4_k", 512, 3, 4096, 1024, "q4_k", "q6_k", 512, shared="q8_0", routed="caller"),
        # a long prompt through the 4-bit mix
        _layer("prefill", "prefill_2000_q4_k", 512, 3, 4096, 1024, "q4_k", "q6_k", 2000, shared="q8_0"),
        # a long prompt in one call, 8-bit experts: the largest
        _layer("prefill", "prefill_4096_q8_0", 512, 10, 4096, 1024, "q8_0", "q8_0", 4096, routed="caller"),
        # one large quantised matrix times a vector (an output head)
        {"name": "matvec_64k_q4_k", "do": "matvec", "rows": 65536, "H": 4096, "gu": "q4_k"},
        # one expert on its own, as the engine's slot cache calls it
        {"name": "expert_q4_k", "do": "expert", "H": 4096, "I": 1024, "gu": "q4_k", "down": "q6_k"},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    types = list(TYPE)
    do = rng.choice(["decode", "decode", "stack", "prefill", "prefill", "prefill", "prefill", "matvec", "expert"])
    if do == "matvec":
        return {"do": do, "rows": _log(rng, 1000, 65536), "H": rng.choice([1024, 2048, 4096]), "gu": rng.choice(types)}
    if do == "expert":
        return {"do": do, "H": rng.choice([1024, 2048, 4096]), "I": rng.choice([512, 1024, 2048]),
                "gu": rng.choice(types), "down": rng.choice(types)}
    H, I = rng.choice([(2048, 512), (2048, 1024), (4096, 512), (4096, 1024)])
    E = rng.choice([64, 96, 128, 256, 512])
    # the format pairs that the decode step and its chained form are built for
    gu, down = rng.choice([("q8_0", "q8_0"), ("q8_0", "q8_0"), ("q4_k", "q6_k"), ("q4_k", "q6_k"), ("q2_k", "q3_k"),
                           ("q4_k", "q5_k")])
    c = _layer(do, "", E, rng.randint(2, 10), H, I, gu, down, 1, routed=rng.choice(["router", "caller"]))
    del c["name"]
    if do == "prefill":
        if rng.random() < 0.4:
            c["gu"], c["down"] = rng.choice(types), rng.choice(types)
        c["shared"] = rng.choice(["", "q8_0", c["gu"]])
        c["tokens"] = _log(rng, 2, 4096)
    elif do == "decode":
        c["shared"] = rng.choice(["", "q8_0"]) if gu != "q2_k" else ""
        c["tokens"] = rng.randint(1, 8)
    else:
        c.update(gu="q2_k", down="q3_k", K=rng.randint(2, 4), layers=rng.randint(2, 8), tokens=rng.randint(1, 4),
                 routed="caller", E=rng.choice([64, 128, 256]))
    return c


# ------------------------------------------------------------------ inputs


def _matrices(qt, n, rows, cols, g):
    """n quantised matrices [rows][cols], stacked: BANK of their own, the rest with the rows moved round."""
    per = rows * (cols // ELEMS[qt]) * BYTES[qt]
    nb = min(n, BANK)
    bank = torch.empty(nb, per, dtype=torch.uint8, device="cuda")
    for m in range(0, nb, 8):
        x = torch.randn(min(8, nb - m) * rows * cols, generator=g, device="cuda").mul_(0.02)
        bank[m:m + 8] = moe.quantize(x, qt).view(-1, per)
    if n <= BANK:
        return bank.view(-1)
    out = torch.empty(n, per, dtype=torch.uint8, device="cuda")
    b3 = bank.view(nb, rows, per // rows)
    for k, m in enumerate(range(0, n, nb)):
        out[m:m + nb] = torch.roll(b3, 29 * k, 1).view(nb, per)[:n - m]
    return out.view(-1)


def _caller_routes(case, rng):
    """Skewed routing (popularity r^-0.456 over a random order of the experts) without repeats, softmax weights."""
    T, E, K = case["tokens"], case["E"], case["K"]
    p = np.arange(1, E + 1) ** -0.456
    keys = np.log(p)[rng.permutation(E)] + rng.gumbel(size=(T, E))
    ids = np.argsort(-keys, axis=1)[:, :K].astype(np.int32)
    s = np.exp(rng.standard_normal((T, K)))
    return (torch.from_numpy(ids).cuda(), torch.from_numpy((s / s.sum(1, keepdims=True)).astype(np.float32)).cuda())


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    do, H = case["do"], case["H"]
    gu = TYPE[case["gu"]]
    if do == "matvec":
        return {"W": _matrices(gu, 1, case["rows"], H, g), "x": torch.randn(H, generator=g, device="cuda")}
    I, dn = case["I"], TYPE[case["down"]]
    if do == "expert":
        return {"gate": _matrices(gu, 1, I, H, g), "up": _matrices(gu, 1, I, H, g), "down": _matrices(dn, 1, H, I, g),
                "x": torch.randn(H, generator=g, device="cuda")}
    E, T, NL = case["E"], case["tokens"], case["layers"]
    rng = np.random.default_rng(seed)
    x = torch.randn(T, H, generator=g, device="cuda")
    d = {"x": x.to(torch.bfloat16) if do == "prefill" else x, "layers": []}
    for _ in range(NL):
        m = {"gate": _matrices(gu, E, I, H, g), "up": _matrices(gu, E, I, H, g), "down": _matrices(dn, E, H, I, g),
             "router": None, "routes": None, "shared": None, "norm": None}
        if case["routed"] == "router":
            m["router"] = torch.randn(E, H, generator=g, device="cuda").mul_(0.02)
        else:
            m["routes"] = _caller_routes(case, rng)
        if case["shared"]:
            st = TYPE[case["shared"]]
            m["shared"] = (_matrices(st, 1, I, H, g), _matrices(st, 1, I, H, g), _matrices(st, 1, H, I, g),
                           torch.randn(H, generator=g, device="cuda").mul_(0.02))
        if do == "stack":
            m["norm"] = 1.0 + 0.1 * torch.randn(H, generator=g, device="cuda")
        d["layers"].append(m)
    return d


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["do"] in ("matvec", "expert"):
        return s
    gu, dn = TYPE[case["gu"]], TYPE[case["down"]]
    s["moe"] = []
    for m in s["layers"]:
        sh = None
        if m["shared"]:
            st = TYPE[case["shared"]]
            sh = moe.SharedExpert(*m["shared"][:3], (st, st, st), m["shared"][3], case["I"])
        s["moe"].append(moe.MoELayer(case["H"], case["I"], case["E"], case["K"], m["router"], m["gate"], m["up"],
                                     m["down"], (gu, gu, dn), shared=sh, max_tokens=case["tokens"],
                                     norm_w=m["norm"], add_residual=m["norm"] is not None))
    T, H, NL = case["tokens"], case["H"], case["layers"]
    s["out"] = torch.empty((T, NL, H) if case["do"] == "stack" else (T, H), device="cuda")
    if case["do"] == "prefill":
        s["moe"][0]._prefill_ws(T)        # the workspace a program allocates once
    elif m["routes"]:
        # each token's routing as its own device vectors
        s["steps"] = [[(m["routes"][0][t].clone(), m["routes"][1][t].clone()) for m in s["layers"]] for t in range(T)]
    return s


def run(s):
    c, do = s["case"], s["case"]["do"]
    if do == "matvec":
        return moe.quant_matvec(s["W"], s["x"], c["rows"], c["H"], TYPE[c["gu"]])
    if do == "expert":
        gu, dn = TYPE[c["gu"]], TYPE[c["down"]]
        return moe.expert_ffn(s["gate"], s["up"], s["down"], s["x"], c["H"], c["I"], (gu, gu, dn))
    L, x, out = s["moe"][0], s["x"], s["out"]
    if do == "prefill":
        if c["routed"] == "router":
            return L.prefill(x, out=out)
        return L.prefill_forced(x, *s["layers"][0]["routes"], out=out)
    for t in range(c["tokens"]):
        if do == "stack":
            moe.decode_stack(s["moe"], x[t], out=out[t], routes=s["steps"][t], step=t)
        elif c["routed"] == "router":
            L.decode(x[t], out=out[t], step=t)
        else:
            L.decode_forced(x[t], *s["steps"][t][0], out=out[t], step=t)
    return out


# ------------------------------------------------------------------ what a pass needs


def _matrix(t, rows, cols):
    return rows * (cols // ELEMS[t]) * BYTES[t]


def work(case):
    do, H, gu = case["do"], case["H"], TYPE[case["gu"]]
    if do == "matvec":
        return {"bytes": _matrix(gu, case["rows"], H) + 4 * (H + case["rows"]), "flops": 2 * case["rows"] * H}
    I, dn = case["I"], TYPE[case["down"]]
    expert = 2 * _matrix(gu, I, H) + _matrix(dn, H, I)
    if do == "expert":
        return {"bytes": expert + 8 * H, "flops": 6 * H * I}
    T, E, K, NL = case["tokens"], case["E"], case["K"], case["layers"]
    st = TYPE[case["shared"]] if case["shared"] else None
    sh = 2 * _matrix(st, I, H) + _matrix(st, H, I) + 4 * H if st else 0
    router = 4 * E * H if case["routed"] == "router" else 0
    if do == "prefill":
        # experts that the batch uses, each once
        if case["routed"] == "router":
            used = E * (1.0 - (1.0 - K / E) ** T)
        else:
            p = np.arange(1, E + 1) ** -0.456
            used = float(np.sum(1.0 - (1.0 - np.minimum(1.0, K * p / p.sum())) ** T))
        b = used * expert + sh + router + T * H * 6
    else:
        # a token's weights are read again by the next one, as the chip's caches cannot hold a model's layers
        b = T * NL * (K * expert + sh + router + 8 * H)
    flops = T * NL * 6 * H * I * (K + (1 if st else 0)) + (2 * T * NL * E * H if router else 0)
    return {"bytes": int(b), "flops": int(flops)}


def tolerance(case):
    # decode, matvec, expert: activations as two int8 digits (15 bits per 64 values), sums in
    # integers and fp32 (2.3e-5 to 5.8e-5 from the 64-bit result); prefill: exact fp16 products, fp32
    # sums, the SwiGLU output in 22 bits (2e-7 to 5e-7 from it)
    if case["do"] == "prefill":
        return {"rel": 2.5e-6}
    return {"rel": 1e-4 if case["do"] == "matvec" else 2.2e-4}


# ------------------------------------------------------------------ the same in 64 bits


def _f16(raw):
    return raw.contiguous().view(torch.float16).to(torch.float64)


def dequant64(qt, raw, rows, cols):
    """fp64 [rows][cols] of raw blocks, from the public block layouts."""
    b = raw.reshape(-1, BYTES[qt])
    if qt == Q8_0:
        return (b[:, 2:].contiguous().view(torch.int8).double() * _f16(b[:, :2])).view(rows, cols)
    f = lambda t: t.to(torch.int32)
    n = b.shape[0]
    if qt in (Q4_K, Q5_K):
        d, dm, s = _f16(b[:, 0:2]), _f16(b[:, 2:4]), f(b[:, 4:16])
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = f(b[:, 16 if qt == Q4_K else 48:]).view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32)
        if qt == Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 8, 1)
            q = q + (((f(b[:, 16:48]).view(n, 1, 32) >> bit) & 1) << 4)
        w = (d * sc).unsqueeze(2) * q - (dm * mn).unsqueeze(2)
        return w.view(rows, cols)
    sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int32).view(1, 1, 4, 1)
    if qt == Q6_K:
        ql, qh = f(b[:, :128]).view(n, 2, 2, 32), f(b[:, 128:192]).view(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)                       # n, half, 4, 32
        q = (lo | (((qh >> sh) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b[:, 208:210])
        return (q.reshape(n, 16, 16) * sc.unsqueeze(2)).view(rows, cols)
    if qt == Q2_K:
        qs, s = f(b[:, 16:80]).view(n, 2, 1, 32), f(b[:, :16])
        q = ((qs >> sh) & 3).reshape(n, 16, 16)
        d, dm = _f16(b[:, 80:82]), _f16(b[:, 82:84])
        return ((d * (s & 15)).unsqueeze(2) * q - (dm * (s >> 4)).unsqueeze(2)).view(rows, cols)
    hm, qs, s, d = f(b[:, :32]).view(n, 1, 1, 32), f(b[:, 32:96]).view(n, 2, 1, 32), f(b[:, 96:108]), _f16(b[:, 108:110])
    bit = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 2, 4, 1)
    q = ((qs >> sh) & 3) - 4 * (1 - ((hm >> bit) & 1))
    low = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
    k = torch.arange(16, device=b.device)
    sc = (low | (((s[:, 8:][:, k % 4] >> (2 * (k // 4)).int()) & 3) << 4)) - 32
    return (q.reshape(n, 16, 16) * (d * sc).unsqueeze(2)).view(rows, cols)


def _ffn64(x, gate, up, down, gu, dn, H, I):
    """[n][H] of one expert for x fp64 [n][H]."""
    g, u = x @ dequant64(gu, gate, I, H).T, x @ dequant64(gu, up, I, H).T
    return (g * torch.sigmoid(g) * u) @ dequant64(dn, down, H, I).T


def _layer64(case, m, x, ids, w):
    """moe_out fp64 [T][H] of one layer; ids / w [T][K]."""
    H, I, E, gu, dn = case["H"], case["I"], case["E"], TYPE[case["gu"]], TYPE[case["down"]]
    out = torch.zeros_like(x)
    flat = ids.reshape(-1).long()
    order = torch.argsort(flat, stable=True)
    count = torch.bincount(flat, minlength=E).tolist()
    pg, pd = m["gate"].numel() // E, m["down"].numel() // E
    at = 0
    for e in range(E):
        if not count[e]:
            continue
        p = order[at:at + count[e]]
        at += count[e]
        t = p // ids.shape[1]
        y = _ffn64(x[t], m["gate"][e * pg:(e + 1) * pg], m["up"][e * pg:(e + 1) * pg],
                   m["down"][e * pd:(e + 1) * pd], gu, dn, H, I)
        out.index_add_(0, t, y * w.reshape(-1)[p].unsqueeze(1))
    if m["shared"]:
        st = TYPE[case["shared"]]
        gate = torch.sigmoid(x @ m["shared"][3].double())
        out += gate.unsqueeze(1) * _ffn64(x, *m["shared"][:3], st, st, H, I)
    return out


def _routes64(case, m, x):
    if m["routes"]:
        return m["routes"][0], m["routes"][1].double()
    v, ids = torch.topk(x @ m["router"].double().T, case["K"], dim=1)
    return ids, torch.softmax(v, 1)


def exact(case, seed):
    s = _inputs(case, seed)
    do, H, gu = case["do"], case["H"], TYPE[case["gu"]]
    x = s["x"].double()
    if do == "matvec":
        return dequant64(gu, s["W"], case["rows"], H) @ x
    if do == "expert":
        return _ffn64(x.view(1, H), s["gate"], s["up"], s["down"], gu, TYPE[case["down"]], H, case["I"]).view(H)
    if do != "stack":
        m = s["layers"][0]
        return _layer64(case, m, x, *_routes64(case, m, x))
    h, outs = x, []
    for m in s["layers"]:
        n = h / torch.sqrt((h * h).mean(1, keepdim=True) + 1e-6) * m["norm"].double()
        h = h + _layer64(case, m, n, *_routes64(case, m, n))
        outs.append(h)
    return torch.stack(outs, 1)
