"""The workloads by which this framework's speed is judged, and how their results are checked.

A case is one piece of work a serving program has the routed-expert path do: the MoE layers of a decode step,
a batch of sequences decoded together, a prefill chunk, the MUL_MAT_ID hook as ggml's graph calls it, and the
f32-activation projections of a dense FFN.  `listed()` names the standing cases, `draw()` gives further ones of the
same ranges; `prepare()` makes the inputs, `run()` is one pass through the public API, and `exact()` computes the
same outputs in 64 bits with plain torch.

Decode passes replay a HIP graph of several layers' calls, as a serving loop does (each layer has its own weights and
inputs: attention sits between them in a model); prefill and batch passes are plain calls.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import zeromoe_amd as Z

QK = 256
BYTES = {"q2_K": 84, "q3_K": 110, "q4_K": 144, "q5_K": 176, "q6_K": 210, "iq2_xxs": 66, "iq3_xxs": 98, "iq4_xs": 136}
TYPE = {"q2_K": 10, "q3_K": 11, "q4_K": 12, "q5_K": 13, "q6_K": 14, "iq2_xxs": 16, "iq3_xxs": 18, "iq4_xs": 23}
SIGMA = 0.02  # standard deviation of a weight


# ---------------------------------------------------------------- cases


def _layer(name, S, H, F, E, K, gate, down, layers=1, graph=False, skew=0.0, gating="softmax", slots=0, groups=0,
           groups_used=0, norm=False, scale=0.0, shared=0, shared_type="q4_K", router=False):
    """One or more routed MoE layers.  skew: sd of a per-expert logit bias (uneven expert loads); slots: experts
    resident behind a slot table (0: all); shared: FFN width of a shared expert; router: the fp32 router's logits
    are part of the layer."""
    c = dict(kind="layer", S=S, H=H, F=F, E=E, K=K, gate=gate, down=down, layers=layers, graph=graph, skew=skew,
             gating=gating, slots=slots, groups=groups, groups_used=groups_used, norm=norm, scale=scale,
             shared=shared, shared_type=shared_type, router=router)
    return dict(c, name=name) if name else c


def _hook(name, S, H, F, E, K, gate, down, graph=False, hot=1.0):
    """A layer's three MUL_MAT_ID ops and the SwiGLU between them, as a ggml graph issues them.  hot: share of the
    routes that are resident (the others have id -1, as in a hot/cold split)."""
    c = dict(kind="hook", S=S, H=H, F=F, E=E, K=K, gate=gate, down=down, graph=graph, hot=hot)
    return dict(c, name=name) if name else c


def _dense(name, S, H, F, gate, down, graph=False):
    """A dense FFN over f32 activations (no Q8_K step): gate and up projections, SwiGLU, down projection."""
    c = dict(kind="dense", S=S, H=H, F=F, gate=gate, down=down, graph=graph)
    return dict(c, name=name) if name else c


def listed():
    block = dict(gating="sigmoid", slots=96, groups=8, groups_used=4, norm=True, scale=2.5, shared=2048, router=True)
    return [
        # one token through the MoE layers of a small model: the shortest calls, where latency counts
        _layer("decode_q4k", 1, 2048, 768, 128, 8, "q4_K", "q4_K", layers=8, graph=True),
        # one token through mid-sized layers in low-bit weights, the benchmark's headline layer
        _layer("decode_q2k_q3k", 1, 4096, 1536, 128, 8, "q2_K", "q3_K", layers=4, graph=True),
        # four sequences decoded together (or a speculative draft checked), codebook weights
        _layer("decode_iq2xxs_s4", 4, 5120, 1536, 160, 8, "iq2_xxs", "iq2_xxs", layers=2, graph=True),
        # one token through full blocks: fp32 router, grouped sigmoid routing, 96 of 256 experts resident, shared expert
        _layer("decode_block", 1, 7168, 2048, 256, 8, "q2_K", "q2_K", layers=2, graph=True, **block),
        # continuous batching: two dozen sequences decoded in one step, a few tokens per expert
        _layer("batch24_q4k_q6k", 24, 4096, 1536, 128, 8, "q4_K", "q6_K"),
        # the full block for a batch of 64 sequences
        _layer("batch64_block", 64, 7168, 2048, 256, 8, "q2_K", "q2_K", **block),
        # a prefill chunk of 512 tokens with uneven expert loads
        _layer("prefill512_q4k", 512, 4096, 1536, 128, 8, "q4_K", "q4_K", skew=1.5),
        # the prompt of the headline layer: a ragged chunk, even loads
        _layer("prefill333_q2k_q3k", 333, 4096, 1536, 128, 8, "q2_K", "q3_K"),
        # a long prefill chunk through a small model's layer, mixed 5- and 6-bit weights
        _layer("prefill2048_q5k_q6k", 2048, 2048, 768, 128, 8, "q5_K", "q6_K", skew=1.0),
        # the op hook under a ggml decode graph
        _hook("hook_decode_iq4xs", 1, 4096, 1536, 128, 8, "iq4_xs", "iq4_xs", graph=True),
        # the op hook over a prompt whose experts are split between GPU and host
        _hook("hook_prefill_iq3xxs", 130, 4096, 1536, 128, 8, "iq3_xxs", "iq3_xxs", hot=0.75),
        # the f32-activation executor over the tokens of one expert
        _dense("dense_f32_q4k_q6k", 40, 4096, 1536, "q4_K", "q6_K"),
    ]


_PAIRS = [("q4_K", "q4_K"), ("q2_K", "q3_K"), ("q2_K", "q2_K"), ("iq2_xxs", "iq2_xxs"), ("q4_K", "q6_K"),
          ("q5_K", "q6_K"), ("iq4_xs", "iq4_xs"), ("iq3_xxs", "iq3_xxs"), ("q3_K", "q4_K"), ("iq3_xxs", "iq4_xs")]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    """A case of the listed ones' ranges: any weight types, widths, expert counts and batch sizes, none of it costing
    more than the largest listed case (1.2 GB of expert weights, 150 GFLOP)."""
    gate, down = rng.choice(_PAIRS)
    H = 256 * rng.choice([4, 8, 9, 10, 12, 16, 20, 22, 28])
    F = 256 * rng.choice([2, 3, 4, 5, 6, 7, 8])
    eb = _expert_bytes(gate, down, H, F)
    E = rng.choice([e for e in (32, 60, 64, 96, 128, 160) if e * eb <= 1.2e9])
    K = rng.choice([2, 4, 6, 8, 8, 10])
    most = int(150e9 / (6.0 * H * F * K))  # tokens
    kind = rng.choice(["decode", "decode", "batch", "prefill", "prefill", "block", "hook", "dense"])
    norm = rng.random() < 0.5
    if kind == "decode":
        S = rng.choice([1, 1, 2, 3, 4, 5, 8])
        return _layer(None, S, H, F, E, K, gate, down, layers=2 if S * K * eb < 5e8 else 1, graph=True, norm=norm)
    if kind == "batch":
        return _layer(None, _log_int(rng, 9, 127), H, F, E, K, gate, down, norm=norm)
    if kind == "prefill":
        S = _log_int(rng, 128, min(2048, most))
        return _layer(None, S, H, F, E, K, gate, down, skew=rng.choice([0.0, 1.0, 1.5]))
    if kind == "block":
        S = rng.choice([1, 2, 4, _log_int(rng, 9, 96)])
        return _layer(None, S, H, F, 256, 8, gate, down, graph=S <= 8, gating=rng.choice(["sigmoid", "sigmoid", "sqrt_softplus"]),
                      slots=rng.choice([n for n in (32, 48, 64, 96) if n * eb <= 1.1e9]), groups=8, groups_used=4,
                      norm=True, scale=2.5, shared=256 * rng.choice([4, 6, 8]),
                      shared_type=rng.choice(["q4_K", "q6_K"]), router=True)
    if kind == "hook":
        S = rng.choice([1, 1, _log_int(rng, 2, min(400, most))])
        return _hook(None, S, H, F, E, K, gate, down, graph=S <= 8, hot=rng.choice([1.0, 0.75]))
    S = _log_int(rng, 1, 96)
    return _dense(None, S, H, F, gate, down, graph=S <= 8)


# ---------------------------------------------------------------- inputs


def _blocks(t, rows, n, gen):
    """`rows` x `n` weights of type `t` as GGUF super-blocks: random quants and sub-block scales under f16 scales
    that give zero-mean weights of about SIGMA; uint8 [rows, bytes]."""
    nb, bb = n // QK, BYTES[t]
    raw = torch.randint(0, 1 << 31, ((rows * nb * bb + 3) // 4,), dtype=torch.int32, device="cuda", generator=gen)
    raw = raw.view(torch.uint8)[:rows * nb * bb].view(rows * nb, bb)
    # the f16 scales d (and dmin): offsets, and the size of d that gives SIGMA for random fields
    off, off_min, size, ratio = {
        "q2_K": (80, 82, 0.071, 1.5), "q3_K": (108, None, 0.024, 0), "q4_K": (0, 2, 0.0042, 7.5),
        "q5_K": (0, 2, 0.0021, 15.5), "q6_K": (208, None, 0.00074, 0), "iq2_xxs": (0, None, 0.0266, 0),
        "iq3_xxs": (0, None, 0.0075, 0), "iq4_xs": (0, None, 0.00085, 0)}[t]
    d = (torch.rand(rows * nb, device="cuda", generator=gen) + 0.5) * (size * SIGMA)
    raw[:, off:off + 2] = d.to(torch.float16).view(torch.uint8).view(-1, 2)
    if off_min is not None:
        m = d * ratio * (0.9 + 0.2 * torch.rand(rows * nb, device="cuda", generator=gen))
        raw[:, off_min:off_min + 2] = m.to(torch.float16).view(torch.uint8).view(-1, 2)
    return raw.view(rows, nb * bb)


def _weights(c, gen):
    n = c.get("slots") or c.get("E", 1)
    w = {"gate": _blocks(c["gate"], n * c["F"], c["H"], gen).view(n, c["F"], -1),
         "up": _blocks(c["gate"], n * c["F"], c["H"], gen).view(n, c["F"], -1),
         "down": _blocks(c["down"], n * c["H"], c["F"], gen).view(n, c["H"], -1)}
    if c.get("shared"):
        t, fs = c["shared_type"], c["shared"]
        w["s_gate"], w["s_up"] = _blocks(t, fs, c["H"], gen), _blocks(t, fs, c["H"], gen)
        w["s_down"] = _blocks(t, c["H"], fs, gen)
    return w


def _inputs(c, seed):
    """Weights and activations of every layer of the case, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rand = lambda *shape: torch.randn(shape, device="cuda", generator=gen)  # noqa: E731
    S, H = c["S"], c["H"]
    got = []
    for _ in range(c.get("layers", 1)):
        w = _weights(c, gen)
        w["x"] = rand(S, H)
        if c["kind"] == "layer":
            E = c["E"]
            if c["router"]:
                w["router"] = rand(E, H) * 0.02
            else:
                w["logits"] = rand(S, E)
            if c["skew"]:
                w["bias"] = rand(E) * c["skew"]
            if c["slots"]:
                perm = torch.randperm(E, device="cuda", generator=gen)
                w["map"] = torch.full((E,), -1, dtype=torch.int32, device="cuda")
                w["map"][perm[:c["slots"]]] = torch.arange(c["slots"], dtype=torch.int32, device="cuda")
        elif c["kind"] == "hook":
            ids = rand(S, c["E"]).topk(c["K"], dim=1).indices.to(torch.int32)
            cold = torch.rand((S, c["K"]), device="cuda", generator=gen) >= c["hot"]
            w["ids"] = torch.where(cold, torch.full_like(ids, -1), ids).contiguous()
        got.append(w)
    return got


def _make_layer(c, w):
    return Z.MoELayer(H=c["H"], F=c["F"], n_experts=c["E"], topk=c["K"], type_gate=TYPE[c["gate"]],
                      type_up=TYPE[c["gate"]], type_down=TYPE[c["down"]], w_gate=w["gate"], w_up=w["up"],
                      w_down=w["down"], gating=c["gating"], n_groups=c["groups"], n_groups_used=c["groups_used"],
                      weights_norm=c["norm"], weights_scale=c["scale"], router_w=w.get("router"),
                      logit_bias=w.get("bias"), route_map=w.get("map"), F_shared=c["shared"],
                      type_shared=TYPE[c["shared_type"]] if c["shared"] else 0, ws_gate=w.get("s_gate"),
                      ws_up=w.get("s_up"), ws_down=w.get("s_down"))


@functools.lru_cache(maxsize=None)
def _capture_stream():
    return torch.cuda.Stream()


def prepare(case, seed):
    Z.init()
    c = case
    w = _inputs(c, seed)
    state = {"case": c, "w": w, "graph": None}
    if c["kind"] == "layer":
        state["layers"] = [_make_layer(c, wl) for wl in w]
        for L, wl in zip(state["layers"], w):
            L.workspace(c["S"], wl["x"].device)
    if c.get("graph"):
        side = _capture_stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(state)  # binds the hook's workspace to the stream before the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            state["out"] = _pass(state)
        state["graph"] = graph
    return state


# ---------------------------------------------------------------- one pass


def _pass(state):
    c, out = state["case"], []
    if c["kind"] == "layer":
        for L, w in zip(state["layers"], state["w"]):
            out.append(L.forward(w["x"], w.get("logits")))
        return out
    w = state["w"][0]
    if c["kind"] == "hook":
        x = w["x"].view(c["S"], 1, c["H"])
        g = Z.mul_mat_id(w["gate"], TYPE[c["gate"]], c["H"], x, w["ids"])
        u = Z.mul_mat_id(w["up"], TYPE[c["gate"]], c["H"], x, w["ids"])
        return [Z.mul_mat_id(w["down"], TYPE[c["down"]], c["F"], Z.swiglu(g, u), w["ids"])]
    g = Z.f32_matmul(w["gate"][0], TYPE[c["gate"]], c["H"], w["x"])
    u = Z.f32_matmul(w["up"][0], TYPE[c["gate"]], c["H"], w["x"])
    return [g, u, Z.f32_matmul(w["down"][0], TYPE[c["down"]], c["F"], Z.swiglu(g, u))]


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return _pass(state)


# ---------------------------------------------------------------- the work a pass cannot do without


def _expert_bytes(gate, down, H, F):
    return (2 * F * (H // QK)) * BYTES[gate] + H * (F // QK) * BYTES[down]


def work(case):
    c = case
    S, H, F = c["S"], c["H"], c["F"]
    eb = _expert_bytes(c["gate"], c["down"], H, F)
    if c["kind"] == "dense":
        return {"bytes": eb + 4 * S * (2 * H + 2 * F), "flops": 6.0 * S * H * F}
    # experts and resident routes of a typical batch of this size
    rng = np.random.default_rng(7)
    lg = rng.standard_normal((S, c["E"])) + rng.standard_normal(c["E"]) * c.get("skew", 0.0)
    ids = np.argsort(-lg, axis=1)[:, :c["K"]]
    share = c["slots"] / c["E"] if c.get("slots") else c.get("hot", 1.0)
    if c.get("slots"):
        routes, experts = ids.size * share, len(np.unique(ids)) * share
    else:
        keep = rng.random(ids.shape) < share
        routes, experts = int(keep.sum()), len(np.unique(ids[keep]))
    n = c.get("layers", 1)
    out = S * c["K"] * H if c["kind"] == "hook" else S * H
    b = experts * eb + 4 * (S * H + out + 2 * S * c["K"])
    f = 6.0 * H * F * routes
    if c.get("router"):
        b += 4 * c["E"] * H
        f += 2.0 * S * c["E"] * H
    elif c["kind"] == "layer":
        b += 4 * S * c["E"]
    if c.get("shared"):
        b += _expert_bytes(c["shared_type"], c["shared_type"], H, c["shared"])
        f += 6.0 * S * H * c["shared"]
    return {"bytes": n * b, "flops": n * f}


def tolerance(case):
    # f32 activations: sums of f32 products in another order (1e-7 to 2e-7 off the 64-bit result).
    if case["kind"] == "dense":
        return {"rel": 5e-6}
    # Q8_K activations: the integer dots are exact and the f32 sums agree to ~1e-6, but the FFN's inner activation is
    # rounded to 8 bits again, where a value within f32 rounding of a half-way point goes either way (1e-7 off the
    # 64-bit result without such a value, up to 3e-4 with a batch of them; one of them moves an output by far more).
    # Routes: f32 router sums may break a tie of two experts the other way.
    t = {"rel": 2e-3, "max": 0.1}
    if case.get("router"):
        t["differ"] = 0.002
    return t


# ---------------------------------------------------------------- 64-bit results


def _grid_iq2():
    """256 x 8 grid: vectors of {1, 3, 5}^8 with an even sum of (v - 1) / 2, by norm, then lexicographically."""
    d = np.stack(np.unravel_index(np.arange(6561), (3,) * 8), 1)
    v = 1 + 2 * d
    ok = np.flatnonzero(d.sum(1) % 2 == 0)
    order = ok[np.lexsort((ok, (v[ok] ** 2).sum(1)))][:256]
    return np.array([8, 25, 43])[d[order]]


def _grid_iq3():
    """256 x 4 grid: digit vectors with d0 + 2 d1 + 4 d2 + 8 d3 = 0 mod 16, in base-8 order."""
    n = np.arange(4096)
    d = np.stack([(n >> (3 * i)) & 7 for i in range(4)], 1)
    d = d[(d @ np.array([1, 2, 4, 8])) % 16 == 0][:256]
    return np.array([4, 12, 20, 28, 36, 44, 52, 62])[d]


_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _dequant(t, raw, n):
    """uint8 [rows, bytes] of type t -> float64 [rows, n]."""
    rows = raw.shape[0]
    b = raw.reshape(-1, BYTES[t])
    f16 = lambda o: b[:, o:o + 2].contiguous().view(torch.float16).double()  # noqa: E731
    i = lambda o, m: b[:, o:o + m].to(torch.int32)  # noqa: E731
    dev = raw.device

    def signs(word):  # [blocks, 8 sub-blocks] -> +-1 [blocks, 8, 4, 8]: 7 sign bits per 8 weights, the 8th their parity
        s = (word[:, :, None] >> (7 * torch.arange(4, device=dev))) & 127
        bits = (s[..., None] >> torch.arange(7, device=dev)) & 1
        return 1.0 - 2.0 * torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1).double()

    def words(o, m):
        return b[:, o:o + 4 * m].contiguous().view(torch.int32).to(torch.int64) & 0xffffffff

    if t == "q2_K":
        sc, qs = i(0, 16), i(16, 64).view(-1, 2, 1, 32)
        q = ((qs >> (2 * torch.arange(4, device=dev)).view(1, 1, 4, 1)) & 3).reshape(-1, 16, 16).double()
        w = f16(80)[:, :, None] * (sc & 15)[..., None] * q - f16(82)[:, :, None] * (sc >> 4)[..., None]
    elif t == "q3_K":
        hm, qs, s = i(0, 32), i(32, 64).view(-1, 2, 1, 32), i(96, 12)
        q = ((qs >> (2 * torch.arange(4, device=dev)).view(1, 1, 4, 1)) & 3).reshape(-1, 8, 32)
        h = (hm[:, None, :] >> torch.arange(8, device=dev).view(1, 8, 1)) & 1
        q = (q - 4 * (1 - h)).reshape(-1, 16, 16).double()
        low = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        high = torch.cat([(s[:, 8:12] >> (2 * k)) & 3 for k in range(4)], 1)
        w = f16(108)[:, :, None] * ((low | (high << 4)) - 32)[..., None] * q
    elif t in ("q4_K", "q5_K"):
        s = i(4, 12)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = i(48 if t == "q5_K" else 16, 128).view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        if t == "q5_K":
            q = q + 16 * ((i(16, 32)[:, None, :] >> torch.arange(8, device=dev).view(1, 8, 1)) & 1)
        w = f16(0)[:, :, None] * sc[..., None] * q.double() - f16(2)[:, :, None] * mn[..., None]
    elif t == "q6_K":
        ql, qh, s = i(0, 128).view(-1, 2, 64), i(128, 64).view(-1, 2, 1, 32), i(192, 16)
        low = torch.stack([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], 2)
        high = (qh >> (2 * torch.arange(4, device=dev)).view(1, 1, 4, 1)) & 3
        q = ((low | (high << 4)) - 32).reshape(-1, 16, 16).double()
        w = f16(208)[:, :, None] * torch.where(s > 127, s - 256, s)[..., None] * q
    elif t == "iq4_xs":
        tab = torch.tensor(_IQ4, dtype=torch.float64, device=dev)
        sh = i(2, 2)
        sh = sh[:, :1] | (sh[:, 1:] << 8)
        sl = i(4, 4)
        k = torch.arange(8, device=dev)
        ls = ((sl[:, k // 2] >> (4 * (k % 2))) & 15) | (((sh >> (2 * k)) & 3) << 4)
        qs = i(8, 128).view(-1, 8, 16)
        q = tab[torch.cat([qs & 15, qs >> 4], 2).long()]
        w = f16(0)[:, :, None] * (ls - 32)[..., None] * q
    elif t == "iq2_xxs":
        g = torch.tensor(_grid_iq2(), dtype=torch.float64, device=dev)
        aux = words(2, 16).view(-1, 8, 2)
        idx = (aux[:, :, 0, None] >> (8 * torch.arange(4, device=dev))) & 255
        db = f16(0) * (0.5 + (aux[..., 1] >> 28).double()) * 0.25
        w = db[..., None, None] * g[idx] * signs(aux[..., 1])
    else:  # iq3_xxs
        g = torch.tensor(_grid_iq3(), dtype=torch.float64, device=dev)
        aux = words(66, 8)
        db = f16(0) * (0.5 + (aux >> 28).double()) * 0.5
        w = db[..., None, None] * g[i(2, 64).long()].view(-1, 8, 4, 8) * signs(aux)
    return w.reshape(rows, n)


def _q8(x):
    """What the 8-bit activation blocks of f32 rows stand for: per 256 values the (first) value of largest magnitude
    maps to -127, the others round to the nearest integer; float64."""
    v = x.float().reshape(-1, QK)
    top = v.gather(1, v.abs().argmax(1, keepdim=True))
    inv = torch.where(top == 0, torch.zeros_like(top), -127.0 / top)
    q = torch.round(inv * v).clamp(max=127).double()
    d = torch.where(top == 0, torch.zeros_like(top), 1.0 / inv).double()
    return (q * d).reshape(x.shape)


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def _routes(c, w):
    """Slot ids and weights [S][K] of a layer, in 64 bits."""
    if c["router"]:
        lg = w["x"].double() @ w["router"].double().T
    else:
        lg = w["logits"].double()
    if c["skew"]:
        lg = (lg.float() + w["bias"]).double()
    if c["gating"] == "softmax":
        p = torch.softmax(lg, 1)
    elif c["gating"] == "sigmoid":
        p = torch.sigmoid(lg)
    else:
        p = torch.sqrt(torch.nn.functional.softplus(lg))
    sel = p
    if c["groups"]:
        score = p.view(c["S"], c["groups"], -1).topk(2, dim=2).values.sum(2)
        keep = torch.zeros_like(score, dtype=torch.bool).scatter_(1, score.topk(c["groups_used"], dim=1).indices, True)
        sel = torch.where(keep.repeat_interleave(c["E"] // c["groups"], 1), p, torch.full_like(p, -math.inf))
    ids = sel.topk(c["K"], dim=1).indices
    wt = p.gather(1, ids)
    if c["norm"]:
        wt = wt / wt.sum(1, keepdim=True)
    if c["scale"]:
        wt = wt * c["scale"]
    if c["slots"]:
        ids = w["map"].long()[ids]
        wt = torch.where(ids >= 0, wt, torch.zeros_like(wt))
    return ids, wt


def _ffn(c, w, xq, ids):
    """Expert FFN rows [S][K][H] of the routes (zero where the id is negative), in 64 bits over 8-bit activations."""
    S, K = ids.shape
    y = torch.zeros((S, K, c["H"]), dtype=torch.float64, device=xq.device)
    for e in torch.unique(ids[ids >= 0]).tolist():
        s, k = torch.nonzero(ids == e, as_tuple=True)
        g = xq[s] @ _dequant(c["gate"], w["gate"][e], c["H"]).T
        u = xq[s] @ _dequant(c["gate"], w["up"][e], c["H"]).T
        y[s, k] = _q8(_silu_mul(g, u)) @ _dequant(c["down"], w["down"][e], c["F"]).T
    return y


def exact(case, seed):
    c = case
    out = []
    for w in _inputs(c, seed):
        if c["kind"] == "dense":
            x = w["x"].double()
            g = x @ _dequant(c["gate"], w["gate"][0], c["H"]).T
            u = x @ _dequant(c["gate"], w["up"][0], c["H"]).T
            return [g, u, _silu_mul(g, u) @ _dequant(c["down"], w["down"][0], c["F"]).T]
        xq = _q8(w["x"])
        if c["kind"] == "hook":
            out.append(_ffn(c, w, xq, w["ids"].long()))
            continue
        ids, wt = _routes(c, w)
        y = (_ffn(c, w, xq, ids) * wt[..., None]).sum(1)
        if c["shared"]:
            t, fs = c["shared_type"], c["shared"]
            g = xq @ _dequant(t, w["s_gate"], c["H"]).T
            u = xq @ _dequant(t, w["s_up"], c["H"]).T
            y = y + _q8(_silu_mul(g, u)) @ _dequant(t, w["s_down"], fs).T
        out.append([y, ids.to(torch.int32), wt])
    return out
