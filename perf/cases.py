"""The work that a program has this framework do on one GPU, as measurable cases: one layer's calls of a GLM-style
mixture-of-experts decoder, each through the entry point such a program calls.

  decode     moe_decode, all-CB3 experts with the shared expert as one more group: one decode step of 1 .. 16 streams
  apply      ResidentFetch.apply, the routed experts in the formats of the quantised checkpoints: 1 .. 8 tokens take the
             decode kernels, more take the grouped (ragged) path: a larger decode batch, or a piece of a prompt
  prefill    moe_prefill, all-CB3 experts with the shared expert: a piece of a prompt
  int8       int8_project_many: the attention's Q, K and V projections of a decode batch
  mlp        mlp_partial: the shared expert (or a dense layer's MLP), int8 or bf16 leaves, decode and prompt pieces
  route      moe_route: the router in front of every layer

Sizes are those of the benchmarked layer (hidden 6144, 64 experts, top-8, intermediate 2048) in the listed cases, with
smaller layers among the drawn ones.  Weights are random in the stored formats, with the spread of trained ones (about
0.02), activations bf16 N(0, 1), routing from N(0, 1) logits (softmax) or Zipf(1.1)-skewed, as in the benchmark.
"""
import math
import os
import types

import numpy as np
import torch

import __graft_entry__

LIMIT = 10.0                    # the SwiGLU clamp
STD = 0.02                      # spread of the weights
DEV = "cuda"
BLOCK_BYTES = {"IQ2_S": 82, "IQ3_S": 110, "IQ4_XS": 136, "Q2_K": 84, "Q3_K": 110}
LAYOUTS = {"cb3": ("CB3", "CB3"), "iq3s": ("IQ3_S", "IQ3_S"), "iq2s_iq3s": ("IQ2_S", "IQ3_S"),
           "iq2s_iq4xs": ("IQ2_S", "IQ4_XS"), "q2k_q3k": ("Q2_K", "Q3_K")}
_pkg = []


def pkg():
    if not _pkg:
        _pkg.append(__graft_entry__.load_package())
    return _pkg[0]


def layer(kind, tokens, layout="cb3", routing="softmax", D=6144, I=2048, E=64, k=8, **more):
    return dict(kind=kind, tokens=tokens, layout=layout, routing=routing, D=D, I=I, E=E, k=k, **more)


def listed():
    return [
        # the router of one decode step with three streams: the smallest call, all launch and latency
        dict(layer("route", 3), name="route_t3"),
        # one decode step of one stream: the headline layer
        dict(layer("decode", 1), name="decode_cb3_t1"),
        # one decode step of 16 streams, expert loads skewed
        dict(layer("decode", 16, routing="zipf"), name="decode_cb3_t16"),
        # single-stream decode of the production checkpoint's layers (IQ2_S gate / up, IQ4_XS down)
        dict(layer("apply", 1, "iq2s_iq4xs"), name="apply_iq2s_iq4xs_t1"),
        # eight streams, the most that the operator's decode path takes by default
        dict(layer("apply", 8, "iq3s", "zipf"), name="apply_iq3s_t8"),
        # a decode batch above that: the operator's grouped path with a few tokens per expert
        dict(layer("apply", 27, "iq2s_iq4xs"), name="apply_iq2s_iq4xs_t27"),
        # a whole prompt piece (512 tokens, the default piece) through the benchmarked layer
        dict(layer("prefill", 512), name="prefill_cb3_t512"),
        # the same piece through the production checkpoint's layers
        dict(layer("apply", 512, "iq2s_iq4xs"), name="apply_iq2s_iq4xs_t512"),
        # a long prompt in one piece, its length whatever the prompt had
        dict(layer("apply", 1999, "iq3s"), name="apply_iq3s_t1999"),
        # Q, K and V of a decode batch over int8 weights
        dict(layer("int8", 8, weights="tiled", n_out="6144 6144 6144"), name="int8_qkv_t8"),
        # the shared expert over a prompt piece, int8 leaves
        dict(layer("mlp", 512, weights="int8"), name="mlp_int8_t512"),
        # the shared expert of one decode step over the default bf16 leaves
        dict(layer("mlp", 1, weights="bf16"), name="mlp_bf16_t1"),
    ]


def _log(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    kind = rng.choice(["decode", "apply", "apply", "ragged", "ragged", "prefill", "int8", "mlp", "mlp", "route"])
    D, I, E, k = rng.choice([(6144, 2048, 64, 8)] * 4 + [(4096, 1536, 32, 6), (3072, 1280, 48, 8), (2048, 768, 96, 4)])
    size = dict(D=D, I=I, E=E, k=k)
    if kind == "decode":
        t = rng.randint(1, 16)
        return layer("decode", t, routing=rng.choice(["softmax", "zipf"]), **size)
    if kind == "apply":
        t = rng.randint(1, 8)
        return layer("apply", t, rng.choice(sorted(LAYOUTS)), rng.choice(["softmax", "zipf"]), **size)
    if kind == "ragged":
        return layer("apply", _log(rng, 64 // k + 1, 1500), rng.choice(sorted(LAYOUTS)),
                     rng.choice(["softmax", "softmax", "zipf"]), **size)
    if kind == "prefill":
        return layer("prefill", _log(rng, 16, 1500), **size)
    if kind == "int8":
        outs = rng.choice(["%d %d %d" % (D, D, D), "%d" % D, "%d %d" % (I, I), "%d %d %d" % (D, I // 2, I // 2)])
        return layer("int8", rng.randint(1, 32), weights=rng.choice(["rows", "tiled"]), n_out=outs, **size)
    if kind == "mlp":
        return layer("mlp", _log(rng, 1, 1500), weights=rng.choice(["int8", "int8_tiled", "bf16"]), **size)
    return layer("route", _log(rng, 1, 1500), **size)


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(0x5EED0000 + int(seed))
    return g


def _words(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int32, device=DEV, generator=g)


def _f16_pairs(g, rows, R, typical):
    """u32 words of two f16 block scales each, uniform in [typical / 2, 3 typical / 2]."""
    d = (torch.rand((rows, R, 2), device=DEV, generator=g) + 0.5) * typical
    b = d.to(torch.float16).view(torch.int16).to(torch.int32) & 0xFFFF
    return b[..., 0] | (b[..., 1] << 16)


def _planes(g, qt, E, R, K):
    """Random experts in the stored planes of format qt."""
    if qt == "CB3":
        CT, G = -(-K // 160), K // 128
        c = torch.sort(torch.randn((E, G, R, 8), device=DEV, generator=g) * STD, dim=-1).values
        c = c.to(torch.bfloat16).view(torch.int16).to(torch.int32) & 0xFFFF
        sh = torch.tensor([0, 8, 16, 24], device=DEV, dtype=torch.int32)
        cb = torch.stack([((h.unflatten(-1, (2, 4)) & 0xFF) << sh).sum(-1).to(torch.int32) for h in (c, c >> 8)], -2)
        return {"qs": _words(g, E, CT * (R // 16) * 256), "cb": cb.reshape(E, G * R * 4)}
    n = K // 256
    if qt == "IQ2_S":
        rows, typical = {"qs": 8 * n, "sg": 8 * n, "qh": 2 * n, "sc": 2 * n}, STD / 60
    elif qt == "IQ3_S":
        rows, typical = {"qs": 16 * n, "sg": 8 * n, "qh": 2 * n, "sc": n}, STD / 150
    elif qt == "IQ4_XS":
        rows, typical = {"qs": 32 * n, "sl": n, "sh": n}, STD / 1000
    elif qt == "Q2_K":
        rows, typical = {"qs": 16 * n, "sc": 4 * n}, STD / 16
    else:
        rows, typical = {"qs": 16 * n, "hm": 8 * n, "sc": 4 * n}, STD / 40
    p = {key: _words(g, E * m, R) for key, m in rows.items()}
    if qt == "IQ4_XS":
        p["sh"] &= 0xFFFF
    if qt == "Q3_K":
        p["sc"] &= 0x3F3F3F3F
    p["d"] = _f16_pairs(g, E * (n if qt in ("Q2_K", "Q3_K") else (n + 1) // 2), R, typical)
    if qt == "Q3_K":
        p["d"] &= 0xFFFF
    return p


def _routing(case, seed):
    """(idx int32 [T, k], w f32 [T, k]): softmax top-k of N(0, 1) logits, or Zipf(1.1)-skewed distinct experts."""
    rng = np.random.default_rng([int(seed), 77])
    T, E, k = case["tokens"], case["E"], case["k"]
    logits = rng.standard_normal((T, E))
    score = logits
    if case["routing"] == "zipf":
        score = (-1.1 * np.log(np.arange(1, E + 1)))[rng.permutation(E)] + rng.gumbel(size=(T, E))
    idx = np.argsort(-score, axis=-1)[:, :k].astype(np.int32)
    w = np.exp(np.take_along_axis(logits, idx, -1))
    return idx, (w / w.sum(-1, keepdims=True)).astype(np.float32)


def _x(g, T, D):
    return torch.randn((T, D), device=DEV, generator=g).to(torch.bfloat16)


def _inputs(case, seed):
    """The case's inputs as plain tensors, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    T, D, I, E = case["tokens"], case["D"], case["I"], case["E"]
    s = {"x": _x(g, T, D)}
    if kind == "route":
        s["router_w"] = torch.randn((D, E), device=DEV, generator=g) / math.sqrt(D)
        s["router_bias"] = torch.randn(E, device=DEV, generator=g) * 0.05
    elif kind == "int8":
        s["w"] = [_int8(g, int(n), D) for n in case["n_out"].split()]
    elif kind == "mlp":
        if case["weights"] == "bf16":
            s["w"] = [(torch.randn((a, b), device=DEV, generator=g) * STD).to(torch.bfloat16)
                      for a, b in ((D, I), (D, I), (I, D))]
        else:
            s["w"] = [_int8(g, a, b) for a, b in ((I, D), (I, D), (D, I))]
    else:
        n = E + (kind != "apply")                       # the shared expert last
        gu, dn = LAYOUTS[case["layout"]]
        s["planes"] = [_planes(g, gu, n, I, D), _planes(g, gu, n, I, D), _planes(g, dn, n, D, I)]
        idx, w = _routing(case, seed)
        s["idx"], s["weights"] = torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV)
    return s


def _int8(g, n_out, n_in):
    q = torch.randint(-127, 128, (n_out, n_in), dtype=torch.int8, device=DEV, generator=g)
    return q, (torch.rand(n_out, device=DEV, generator=g) + 0.5) * (STD / 73)


# ------------------------------------------------------------------------------------------------ the calls
def prepare(case, seed):
    s, P = _inputs(case, seed), pkg()
    kind, D, I = case["kind"], case["D"], case["I"]
    st = {"kind": kind, "x": s["x"]}
    if kind == "route":
        st["p"] = {"router_w": s["router_w"], "router_bias": s["router_bias"]}
        st["cfg"] = types.SimpleNamespace(topk=case["k"], norm_topk=True, scaling=2.5)
    elif kind == "int8":
        tile = P.int8_tile if case["weights"] == "tiled" else (lambda q: q)
        st["projections"] = [(tile(q), sc) for q, sc in s["w"]]
    elif kind == "mlp":
        if case["weights"] == "bf16":
            leaves = [P.bf16_leaf(w) for w in s["w"]]
        else:
            tile = P.int8_tile if case["weights"] == "int8_tiled" else (lambda q: q)
            leaves = [(tile(q), sc, P._lib.MI_I8_COL_SCALES) for q, sc in s["w"]]
        st["p"] = dict(zip(("gate", "up", "down"), leaves))
    else:
        gu, dn = LAYOUTS[case["layout"]]
        st["idx"], st["w"] = s["idx"], s["weights"]
        if kind == "apply":
            st["fetch"] = P.ResidentFetch([{"gate_q": gu, "up_q": gu, "down_q": dn}], D, I)
            st["p"] = dict(zip(("gate_q", "up_q", "down_q"), s["planes"]))
        else:
            shapes = ((gu, I, D), (gu, I, D), (dn, D, I))
            st["tables"] = [P.ExpertTable(qt, pl, R, K) for pl, (qt, R, K) in zip(s["planes"], shapes)]
            st["shared"] = case["E"]
    return st


def run(state):
    P, s = pkg(), state
    kind = s["kind"]
    if kind == "route":
        return P.moe_route(s["p"], s["x"], s["cfg"])
    if kind == "int8":
        return P.int8_project_many(s["x"], s["projections"])
    if kind == "mlp":
        return P.mlp_partial(s["p"], s["x"], LIMIT)
    if kind == "apply":
        return s["fetch"].apply(s["p"], s["x"], s["idx"], s["w"], 0, LIMIT)
    call = P.moe_decode if kind == "decode" else P.moe_prefill
    return call(*s["tables"], s["x"], s["idx"], s["w"], LIMIT, shared_expert=s["shared"])[0]


# ------------------------------------------------------------------------------------------------ what it takes
def _matrix_bytes(qt, R, K):
    if qt == "CB3":
        return R * (4 * -(-K // 10) + 16 * (K // 128))
    return R * (K // 256) * BLOCK_BYTES[qt]


def _distinct(case):
    """Experts that a call's tokens reach, on average."""
    return float(np.mean([len(np.unique(_routing(case, s)[0])) for s in range(16)]))


def work(case):
    kind, T, D, I, E, k = (case[n] for n in ("kind", "tokens", "D", "I", "E", "k"))
    if kind == "route":
        return {"bytes": 4 * D * E + 4 * E + 2 * T * D + 8 * T * k, "flops": 2 * T * D * E}
    if kind == "int8":
        n = sum(int(v) for v in case["n_out"].split())
        return {"bytes": n * D + 4 * n + 2 * T * (D + n), "flops": 2 * T * D * n}
    if kind == "mlp":
        size = 2 if case["weights"] == "bf16" else 1
        return {"bytes": 3 * D * I * size + (4 * (2 * I + D) if size == 1 else 0) + 4 * T * D, "flops": 6 * T * D * I}
    gu, dn = LAYOUTS[case["layout"]]
    shared = kind != "apply"
    experts = _distinct(case) + shared
    rows = T * (k + shared)
    return {"bytes": int(experts * (2 * _matrix_bytes(gu, I, D) + _matrix_bytes(dn, D, I))) + 6 * T * D + 8 * T * k,
            "flops": 6 * rows * D * I}


def tolerance(case):
    kind = case["kind"]
    if kind == "route":                  # f32 logits: sums in another order; a near-tie may order differently
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.002}
    if kind == "decode" or (kind == "apply" and case["tokens"] * case["k"] <= 64):
        return {"rel": 2e-5, "max": 1e-3}            # f32 sums; activations as two bf16 parts (16 bits): 5e-6 seen
    return {"rel": 1e-2, "max": 0.1}    # bf16 weights, h and y (or g, u, h and the result): 2.4e-3 .. 4.5e-3 seen


# ------------------------------------------------------------------------------------------------ in 64 bits
def _data(name):
    return torch.from_numpy(np.load(os.path.join("oracle", "data", name)).astype(np.int64)).to(DEV)


def _f16(bits):
    return bits.to(torch.int16).view(torch.float16).double()


def _dense(qt, planes, e, R, K, tabs):
    """Expert e of a table, decoded to float64 [R, K]."""
    if qt == "CB3":
        CT, G = -(-K // 160), K // 128
        w = planes["qs"][e].reshape(CT, R // 16, 64, 2, 2, 1)
        a, b = (((w[..., j, :] >> torch.arange(0, 32, 8, device=DEV, dtype=torch.int32)) & 255) for j in (0, 1))
        codes = torch.cat([a & 7, (a >> 3) & 7, b & 7, (b >> 3) & 7, (a >> 6) | ((b >> 6) & 1) << 2], -1)
        codes = codes.reshape(CT, R // 16, 4, 16, 5, 8).permute(1, 3, 0, 4, 2, 5).reshape(R, CT * 160)[:, :K]
        cb = planes["cb"][e].reshape(G, R, 2, 2, 1)
        by = (cb >> torch.arange(0, 32, 8, device=DEV, dtype=torch.int32)) & 255     # [G, R, lo / hi, half, byte]
        val = ((by[:, :, 0] | by[:, :, 1] << 8) << 16).view(torch.float32).reshape(G, R, 8).double()
        return torch.gather(val.transpose(0, 1), 2, codes.reshape(R, G, 128).long()).reshape(R, K)
    n = K // 256
    p = {key: a.reshape(-1, a.shape[-1]) for key, a in planes.items()}
    rows = {key: a.shape[0] // tabs["E"] for key, a in p.items()}
    p = {key: a[e * rows[key]:(e + 1) * rows[key]] for key, a in p.items()}
    bit = lambda a, idx, sh, mask: (a[idx] >> sh[:, None].to(torch.int32)) & mask
    ar = lambda m: torch.arange(m, device=DEV)
    if qt in ("IQ2_S", "IQ3_S"):
        W = p["qs"].shape[0]
        w = ar(W)
        per = W // n                                                    # words per block: 8 or 16
        d = _f16(bit(p["d"], w // (2 * per), 16 * ((w // per) % 2), 0xFFFF))
        out = torch.empty((W, K // W, R), dtype=torch.float64, device=DEV)
        for j in range(4):
            lo = (p["qs"] >> (8 * j)) & 255
            if qt == "IQ2_S":
                hi = (bit(p["qh"], w // 4, 8 * (w % 4), 255) >> (2 * j)) & 3
                sc = (bit(p["sc"], w // 4, 8 * (w % 4), 255) >> (4 * (j // 2))) & 15
                lv, scale, sg = tabs["iq2"][(lo | hi << 8).long()], d * (0.5 + sc.double()) * 0.25, p["sg"] >> (8 * j)
            else:
                hi = (bit(p["qh"], w // 8, 4 * (w % 8), 15) >> j) & 1
                sc = bit(p["sc"], w // 16, 4 * ((w // 2) % 8), 15)
                sg = bit(p["sg"], w // 2, 16 * (w % 2), 0xFFFF) >> (4 * j)
                lv, scale = tabs["iq3"][(lo | hi << 8).long()], d * (1 + 2 * sc.double())
            m = lv.shape[-1]
            for t in range(m):
                out[:, m * j + t] = scale * lv[..., t] * (1 - 2 * ((sg >> t) & 1))
        return out.reshape(K, R).T.contiguous()
    out = torch.empty((K, R), dtype=torch.float64, device=DEV)
    if qt == "IQ4_XS":
        w = ar(32 * n)
        sub = w // 4
        sc = bit(p["sl"], sub // 8, 4 * (sub % 8), 15) | bit(p["sh"], sub // 8, 2 * (sub % 8), 3) << 4
        scale = _f16(bit(p["d"], sub // 16, 16 * ((sub // 8) % 2), 0xFFFF)) * (sc.double() - 32)
        for j in range(4):
            for h in range(2):
                out[32 * sub + 4 * (w % 4) + 16 * h + j] = scale * tabs["kv"][((p["qs"] >> (8 * j + 4 * h)) & 15).long()]
        return out.T.contiguous()
    w = ar(16 * n)
    b, half, q = w // 16, (w % 16) // 8, w % 8
    d = _f16(p["d"][b] & 0xFFFF)
    for s in range(4):
        i = 8 * half + 2 * s + (q >= 4)
        sc = bit(p["sc"], 4 * b + i // 4, 8 * (i % 4), 255)
        for j in range(4):
            v = ((p["qs"] >> (8 * j + 2 * s)) & 3).double()
            if qt == "Q2_K":
                val = d * (sc & 15) * v - _f16((p["d"][b] >> 16) & 0xFFFF) * (sc >> 4)
            else:
                hb = (bit(p["hm"], 8 * b + q, 8 * j + 4 * half + s, 1)).double()
                val = d * (sc.double() - 32) * (v - 4 * (1 - hb))
            out[256 * b + 128 * half + 32 * s + 4 * q + j] = val
    return out.T.contiguous()


def _swiglu(g, u):
    g = g.clamp(max=LIMIT)
    return g / (1 + torch.exp(-g)) * u.clamp(-LIMIT, LIMIT)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    x = s["x"].double()
    if kind == "route":
        score = torch.sigmoid(x @ s["router_w"].double())
        idx = torch.topk(score + s["router_bias"].double(), case["k"], dim=-1).indices
        w = torch.gather(score, 1, idx)
        return idx.to(torch.int32), w / (w.sum(-1, keepdim=True) + 1e-20) * 2.5
    if kind == "int8":
        return [x @ (q.double() * sc.double()[:, None]).T for q, sc in s["w"]]
    if kind == "mlp":
        if case["weights"] == "bf16":
            g, u, d = [w.double() for w in s["w"]]
        else:
            g, u, d = [(q.double() * sc.double()[:, None]).T for q, sc in s["w"]]
        return _swiglu(x @ g, x @ u) @ d
    D, I, E = case["D"], case["I"], case["E"] + (kind != "apply")
    gu, dn = LAYOUTS[case["layout"]]
    tabs = {"E": E}
    if "IQ2_S" in (gu, dn):
        tabs["iq2"] = _data("iq2s_grid.npy").double().reshape(1024, 8)
    if "IQ3_S" in (gu, dn):
        tabs["iq3"] = _data("iq3s_grid.npy").double().reshape(512, 4)
    if "IQ4_XS" in (gu, dn):
        tabs["kv"] = _data("iq4nl_kvalues.npy").double()
    out = torch.zeros((case["tokens"], D), dtype=torch.float64, device=DEV)
    every = torch.arange(case["tokens"], device=DEV)
    for e in range(E):
        if e == case["E"]:
            tok, w = every, torch.ones(len(every), dtype=torch.float64, device=DEV)
        else:
            tok, col = torch.nonzero(s["idx"] == e, as_tuple=True)
            w = s["weights"][tok, col].double()
        if not len(tok):
            continue
        G, U = (_dense(gu, s["planes"][m], e, I, D, tabs) for m in (0, 1))
        h = _swiglu(x[tok] @ G.T, x[tok] @ U.T)
        out.index_add_(0, tok, (h @ _dense(dn, s["planes"][2], e, D, I, tabs).T) * w[:, None])
    return out
