"""The work that programs have this library do, as cases that can be timed and
checked: the projections of decoder layers for one token, a few or a prompt,
attention over a held cache, a mixture-of-experts layer, and whole sessions.

A case is a dict of plain values.  Its "kind" says which entry points it calls:

    layer    the seven projections of decoder layers, `tokens` rows each
    matmul   one Weight.matmul_bt over a prompt's rows
    attend   GQA attention of one token, a call per layer's cache
    mla      absorbed latent attention of one token, a call per layer's cache
    moe      a mixture-of-experts layer over `tokens` rows
    prompt   a session reading a prompt: logits of the last token
    each     conversations advanced by a token together: logits of each

Device arrays come in and go out wherever the library takes them, as in a
program that keeps its activations on the GPU; a session's logits come back to
the host, as its entry points give them.
"""
import math

import numpy as np
import torch

import kvad_amd as K

DEV = "cuda:0"
PREC = {"q8": K.Q8, "q4": K.Q4, "q4k": K.Q4K, "f32": K.F32}
BLOCK = 32

_ctx = None


def context():
    """One context for the process: a device and a stream."""
    global _ctx
    if _ctx is None:
        _ctx = K.Context(0)
    return _ctx


# ---- the cases ---------------------------------------------------------------

def listed():
    small = {"n_embd": 896, "n_head": 14, "n_kv_head": 2, "head_dim": 64, "n_ff": 4864, "n_layer": 24,
             "vocab": 151936, "precision": "q8"}
    return [
        # One token through one layer of a half-billion-parameter decoder: four
        # launches of a few microseconds, what an embedded model's decode is
        # made of.
        {"name": "layer_q8_1tok", "kind": "layer", "precision": "q8", "hidden": 896, "kv": 128, "inter": 4864,
         "layers": 1, "tokens": 1},
        # One token through eight layers of an 8B decoder in Q4_K: distinct
        # weights past the last-level cache, the decode that HBM bounds.
        {"name": "layers_q4k_1tok", "kind": "layer", "precision": "q4k", "hidden": 4096, "kv": 1024, "inter": 14336,
         "layers": 8, "tokens": 1},
        # A layer of the same model for a dozen conversations decoded together
        # (or drafts verified): too many rows for the one-token kernels, far
        # too few for a prompt's.
        {"name": "layer_q4k_12tok", "kind": "layer", "precision": "q4k", "hidden": 4096, "kv": 1024, "inter": 14336,
         "layers": 1, "tokens": 12},
        # A prompt pass over the widest projection of that layer, a token count
        # that fills no tile evenly.
        {"name": "matmul_q4k_1000tok", "kind": "matmul", "precision": "q4k", "rows": 14336, "cols": 4096,
         "tokens": 1000, "bias": False},
        # Weights kept in f32 (models run unquantised, rows that do not block),
        # odd sizes in both directions.
        {"name": "matmul_f32_90tok", "kind": "matmul", "precision": "f32", "rows": 3000, "cols": 2052, "tokens": 90,
         "bias": True},
        # A token's attention over a chat-length cache, all layers of the small
        # decoder: launches and latency.
        {"name": "attend_short", "kind": "attend", "n_head": 14, "n_kv_head": 2, "head_dim": 64, "positions": 1000,
         "layers": 24},
        # The same over a long document at the 8B decoder's geometry.
        {"name": "attend_long", "kind": "attend", "n_head": 32, "n_kv_head": 8, "head_dim": 128, "positions": 20001,
         "layers": 2},
        # Latent attention over a few thousand positions.
        {"name": "mla", "kind": "mla", "n_head": 16, "positions": 6001, "layers": 8},
        # A token through a 64-expert layer: a router and six experts' GEMVs.
        {"name": "moe_1tok", "kind": "moe", "precision": "q8", "n_experts": 64, "top_k": 6, "hidden": 2048,
         "inter": 1408, "shared": 2816, "tokens": 1, "norm_topk": False},
        # A prompt pass through it: every expert is picked by some row.
        {"name": "moe_400tok", "kind": "moe", "precision": "q8", "n_experts": 64, "top_k": 6, "hidden": 2048,
         "inter": 1408, "shared": 2816, "tokens": 400, "norm_topk": False},
        # A document's prompt read by a session, several passes.
        dict(small, name="prompt_1500tok", kind="prompt", tokens=1500),
        # Twelve conversations of different lengths, a token for each.
        dict(small, name="each_12", kind="each", conversations=12, longest=900),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of lo .. hi."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


MODELS = [  # hidden, kv width, inter of one layer
    (896, 128, 4864), (1024, 256, 2816), (1536, 256, 8960), (2048, 512, 5632), (2560, 640, 6912), (3072, 1024, 8192),
    (4096, 1024, 14336), (4096, 4096, 11008),
]


def _fits(precision, *widths):
    return precision != "q4k" or all(w % 256 == 0 for w in widths)


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "matmul", "matmul", "matmul", "attend", "attend", "mla", "moe",
                       "moe", "prompt", "each"])
    if kind == "layer":
        while True:
            precision = rng.choice(["q8", "q4", "q4k"])
            hidden, kv, inter = rng.choice(MODELS)
            if _fits(precision, hidden, inter):
                break
        return {"kind": kind, "precision": precision, "hidden": hidden, "kv": kv, "inter": inter,
                "layers": rng.randint(1, 4), "tokens": _log(rng, 1, 32)}
    if kind == "matmul":
        precision = rng.choice(["q8", "q8", "q4", "q4k", "q4k", "f32"])
        unit = {"q4k": 256, "f32": 4}.get(precision, 32)
        cols = unit * max(1, _log(rng, 512, 14336) // unit)
        rows = _log(rng, 64, 14336)
        tokens = _log(rng, 2, 1000 if precision != "f32" else 300)
        return {"kind": kind, "precision": precision, "rows": rows, "cols": cols, "tokens": tokens,
                "bias": rng.random() < 0.5}
    if kind == "attend":
        n_head, n_kv_head, head_dim = rng.choice([(14, 2, 64), (32, 8, 128), (32, 8, 64), (16, 16, 128), (12, 2, 128)])
        positions = _log(rng, 16, 20000)
        return {"kind": kind, "n_head": n_head, "n_kv_head": n_kv_head, "head_dim": head_dim, "positions": positions,
                "layers": rng.randint(1, 24) if positions < 4000 else 2}
    if kind == "mla":
        positions = _log(rng, 16, 20000)
        return {"kind": kind, "n_head": rng.choice([16, 16, 32, 128]), "positions": positions,
                "layers": rng.randint(1, 8) if positions < 4000 else 2}
    if kind == "moe":
        n_experts, top_k, hidden, inter, shared = rng.choice(
            [(64, 6, 2048, 1408, 2816), (60, 4, 2048, 1408, 5632), (8, 2, 2048, 3584, 0), (128, 8, 2048, 768, 0)])
        precision = rng.choice(["q8", "q8", "q4", "q4k"])
        if not _fits(precision, hidden, inter, shared):
            precision = "q8"
        return {"kind": kind, "precision": precision, "n_experts": n_experts, "top_k": top_k, "hidden": hidden,
                "inter": inter, "shared": shared, "tokens": _log(rng, 1, 400), "norm_topk": rng.random() < 0.5}
    n_embd, n_head, n_kv_head, head_dim, n_ff = rng.choice(
        [(896, 14, 2, 64, 4864), (1024, 16, 8, 64, 2816), (2048, 32, 4, 64, 5632), (1536, 12, 2, 128, 8960)])
    model = {"n_embd": n_embd, "n_head": n_head, "n_kv_head": n_kv_head, "head_dim": head_dim, "n_ff": n_ff,
             "n_layer": rng.randint(3, 8), "vocab": _log(rng, 8000, 64000), "precision": rng.choice(["q8", "q8", "q4"])}
    if kind == "prompt":
        return dict(model, kind=kind, tokens=_log(rng, 2, 1500))
    return dict(model, kind=kind, conversations=_log(rng, 1, 32), longest=_log(rng, 40, 900))


# ---- inputs ------------------------------------------------------------------

class Maker:
    """Arrays on the GPU from a seed, the same ones for prepare and exact."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(1000003 * int(seed) + 12345)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, device=DEV, generator=self.g) * std

    def ints(self, lo, hi, *shape):
        """lo .. hi - 1"""
        return torch.randint(lo, hi, shape, device=DEV, generator=self.g, dtype=torch.int32)

    def hidden(self, rows, cols):
        """Hidden states: some channels several times the others."""
        return self.normal(rows, cols) * torch.exp(0.5 * self.normal(cols))

    def weight(self, precision, rows, cols, std=0.02):
        """A weight's data: f32 values that are quantised on the device, or a
        Q4_K weight's parts, whose blocks are made here."""
        if precision != "q4k":
            return self.normal(rows, cols, std=std)
        sup = cols // 256
        sc, mn = self.ints(20, 64, rows, sup, 8), self.ints(20, 64, rows, sup, 8)
        q = torch.clamp(torch.round(7.5 + 3.0 * self.normal(rows, sup, 8, 32)), 0, 15).to(torch.uint8)
        d = (std / 42 / 3 * torch.exp(0.2 * self.normal(rows, sup))).half()
        return {"d": d, "dmin": (7.5 * d.float()).half(), "sc": sc.to(torch.uint8), "mn": mn.to(torch.uint8), "q": q}


def q4k_blocks(p):
    """Q4_K parts as GGML lays a block of 256 out: d, dmin, 12 bytes of 6-bit
    scales and minimums, 128 bytes of codes, two sub-blocks to 32 bytes."""
    rows, sup = p["d"].shape
    out = torch.empty(rows, sup, 144, dtype=torch.uint8, device=DEV)
    out[:, :, 0:2] = p["d"].reshape(rows, sup, 1).view(torch.uint8)
    out[:, :, 2:4] = p["dmin"].reshape(rows, sup, 1).view(torch.uint8)
    sc, mn = p["sc"], p["mn"]
    out[:, :, 4:8] = sc[:, :, :4] | ((sc[:, :, 4:] >> 4) << 6)
    out[:, :, 8:12] = mn[:, :, :4] | ((mn[:, :, 4:] >> 4) << 6)
    out[:, :, 12:16] = (sc[:, :, 4:] & 15) | ((mn[:, :, 4:] & 15) << 4)
    out[:, :, 16:] = (p["q"][:, :, 0::2] | (p["q"][:, :, 1::2] << 4)).reshape(rows, sup, 128)
    return out


def device_weight(precision, rows, cols, data):
    """The device Weight of Maker.weight's data."""
    if precision == "q4k":
        return K.Weight.from_q4k(context(), rows, cols, q4k_blocks(data).reshape(-1).cpu().numpy())
    torch.cuda.synchronize()
    w = K.Weight.quantize_dev(context(), rows, cols, data.data_ptr(), PREC[precision])
    context().synchronize()
    return w


def layer_shapes(case):
    """(name, rows, cols, input) of a layer's seven projections, in order."""
    e, kv, ff = case["hidden"], case["kv"], case["inter"]
    return [("q", e, e, "x"), ("k", kv, e, "x"), ("v", kv, e, "x"), ("o", e, e, "a"), ("gate", ff, e, "h"),
            ("up", ff, e, "h"), ("down", e, ff, "s")]


def layer_data(case, seed):
    """Per layer: ({input: rows}, [(name, rows, cols, input, weight data)])."""
    mk, m = Maker(seed), case["tokens"]
    for _ in range(case["layers"]):
        xs = {"x": mk.hidden(m, case["hidden"]), "a": mk.hidden(m, case["hidden"]),
              "h": mk.hidden(m, case["hidden"]), "s": mk.hidden(m, case["inter"])}
        yield xs, [(n, r, c, i, mk.weight(case["precision"], r, c)) for n, r, c, i in layer_shapes(case)]


def matmul_data(case, seed):
    mk = Maker(seed)
    x = mk.hidden(case["tokens"], case["cols"])
    w = mk.weight(case["precision"], case["rows"], case["cols"])
    return x, w, mk.normal(case["rows"]) if case["bias"] else None


def attend_data(case, seed):
    """Per layer q, k, v.  Scores spread as trained heads' do (a standard
    deviation of 2), so that a long cache holds positions on either side of
    the 1e-8 under which the reference drops a weight."""
    mk, L, kvd = Maker(seed), case["positions"], case["n_kv_head"] * case["head_dim"]
    for _ in range(case["layers"]):
        yield 2.0 * mk.normal(case["n_head"] * case["head_dim"]), mk.normal(L, kvd), mk.normal(L, kvd)


LAT, ROPE = 512, 64


def mla_scale(case):
    return 1.0 / math.sqrt(192.0)


def mla_data(case, seed):
    mk, L, H = Maker(seed), case["positions"], case["n_head"]
    q_std = 2.0 * math.sqrt(192.0 / (LAT + ROPE))  # scores of standard deviation 2
    for _ in range(case["layers"]):
        yield (mk.normal(H, LAT, std=q_std), mk.normal(H, ROPE, std=q_std), mk.normal(L, LAT), mk.normal(L, ROPE))


def moe_data(case, seed):
    """Hidden rows, the router's weight, the experts' and the shared one's
    (gate, up, down)."""
    mk, e, ff, sh, p = Maker(seed), case["hidden"], case["inter"], case["shared"], case["precision"]
    x = mk.normal(case["tokens"], e)
    router = mk.normal(case["n_experts"], e, std=0.05)
    experts = [(mk.weight(p, ff, e), mk.weight(p, ff, e), mk.weight(p, e, ff)) for _ in range(case["n_experts"])]
    shared = (mk.weight(p, sh, e), mk.weight(p, sh, e), mk.weight(p, e, sh)) if sh else None
    return x, router, experts, shared


def model_shapes(case):
    e, qd, kvd, ff = (case["n_embd"], case["n_head"] * case["head_dim"], case["n_kv_head"] * case["head_dim"],
                      case["n_ff"])
    return [("q", qd, e), ("k", kvd, e), ("v", kvd, e), ("o", e, qd), ("gate", ff, e), ("up", ff, e), ("down", e, ff)]


CONTEXT = 2048
EPS = 1e-6


def model_data(case, mk):
    """Layers as (weights, norms, biases), then the embedding and final norm.
    The projections back into the residual are smaller by the root of their
    number, as initialised and trained decoders have them."""
    def norm(n):
        return 1.0 + mk.normal(n, std=0.1)

    back = 1.0 / math.sqrt(2 * case["n_layer"])
    for _ in range(case["n_layer"]):
        ws = {n: (r, c, mk.weight(case["precision"], r, c, std=(back if n in ("o", "down") else 1.0) / math.sqrt(c)))
              for n, r, c in model_shapes(case)}
        yield (ws, (norm(case["n_embd"]), norm(case["n_embd"])),
               {n: mk.normal(ws[n][0], std=0.1) for n in ("q", "k", "v")})
    yield mk.weight(case["precision"], case["vocab"], case["n_embd"], std=0.5), norm(case["n_embd"])


def rope_tables(case):
    half = case["head_dim"] // 2
    inv = 1.0 / (1e6 ** (np.arange(half, dtype=np.float64) * 2 / case["head_dim"]))
    ang = np.arange(CONTEXT, dtype=np.float64)[:, None] * inv[None, :]
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def make_model(case, mk):
    spec = {k: case[k] for k in ("n_embd", "n_head", "n_kv_head", "head_dim", "n_ff", "n_layer", "vocab")}
    m = K.Llm(context(), **spec, n_ctx=CONTEXT, eps=EPS, rope_interleaved=0)
    host = lambda t: t.cpu().numpy()  # noqa: E731
    l = 0
    for part in model_data(case, mk):
        if len(part) == 3:
            ws, norms, biases = part
            w = {n: device_weight(case["precision"], *ws[n]) for n in ws}
            m.set_layer(l, *[w[n] for n in ("q", "k", "v", "o", "gate", "up", "down")], host(norms[0]),
                        host(norms[1]), *[host(biases[n]) for n in ("q", "k", "v")])
            l += 1
        else:
            embed, final = part
            m.set_ends(device_weight(case["precision"], case["vocab"], case["n_embd"], embed), host(final))
    m.set_rope(*rope_tables(case), CONTEXT)
    return m


def conversations(case, seed):
    """The conversations' prompts: lengths from a third of `longest` up."""
    rng = np.random.default_rng(int(seed) + 77)
    n, top = case["conversations"], case["longest"]
    lens = [top] + [int(v) for v in rng.integers(max(1, top // 3), top + 1, n - 1)]
    return [rng.integers(0, case["vocab"], k).astype(np.int32) for k in lens], rng.integers(
        0, case["vocab"], n).astype(np.int32)


def prompt_tokens(case, seed):
    return np.random.default_rng(int(seed) + 78).integers(0, case["vocab"], case["tokens"]).astype(np.int32)


# ---- prepare -----------------------------------------------------------------

def prepare(case, seed):
    kind, ctx = case["kind"], context()
    s = {"case": case}
    if kind == "layer":
        s["layers"] = []
        for xs, ws in layer_data(case, seed):
            L = {"x": xs, "w": {}, "y": {}}
            for n, r, c, i, data in ws:
                L["w"][n] = device_weight(case["precision"], r, c, data)
                L["y"][n] = torch.empty(case["tokens"], r, device=DEV)
            s["layers"].append(L)
    elif kind == "matmul":
        s["x"], data, s["bias"] = matmul_data(case, seed)
        s["w"] = device_weight(case["precision"], case["rows"], case["cols"], data)
        s["y"] = torch.empty(case["tokens"], case["rows"], device=DEV)
    elif kind == "attend":
        s["spec"] = K.Spec(case["n_head"], case["n_kv_head"], case["head_dim"])
        s["layers"] = [d + (torch.empty_like(d[0]),) for d in attend_data(case, seed)]
    elif kind == "mla":
        s["layers"] = [d + (torch.empty_like(d[0]),) for d in mla_data(case, seed)]
    elif kind == "moe":
        x, router, experts, shared = moe_data(case, seed)
        e, ff, sh, p = case["hidden"], case["inter"], case["shared"], case["precision"]
        m = K.Moe(ctx, case["n_experts"], case["top_k"], e, ff, norm_topk=case["norm_topk"])
        m.set_router(device_weight("q8", case["n_experts"], e, router))
        for i, (g, u, d) in enumerate(experts):
            m.set_expert(i, device_weight(p, ff, e, g), device_weight(p, ff, e, u), device_weight(p, e, ff, d))
        if shared:
            g, u, d = shared
            m.set_shared(device_weight(p, sh, e, g), device_weight(p, sh, e, u), device_weight(p, e, sh, d))
        s["moe"], s["x"], s["y"] = m, x, torch.empty_like(x)
    elif kind == "prompt":
        s["model"] = make_model(case, Maker(seed))
        s["tokens"] = prompt_tokens(case, seed)
    else:
        m = s["model"] = make_model(case, Maker(seed))
        prompts, s["next"] = conversations(case, seed)
        s["held"] = []
        for p in prompts:
            m.forward_tokens(p, want_logits=False)
            s["held"].append(m.park())
        s["steps"], s["lens"] = 0, [len(p) for p in prompts]
    torch.cuda.synchronize()
    return s


# ---- run ---------------------------------------------------------------------

def _many(ctx, ws, x, ys):
    """quant::matvec_many over device arrays that share their input."""
    n = len(ws)
    arr = K.C.c_void_p * n
    K._check(K.lib.kh_matvec_many_dev(ctx.h, n, arr(*[w.h.value for w in ws]), arr(*([x.data_ptr()] * n)),
                                      arr(*[y.data_ptr() for y in ys])))


def run(s):
    case, ctx = s["case"], context()
    kind = case["kind"]
    if kind == "layer":
        m = case["tokens"]
        for L in s["layers"]:
            x, w, y = L["x"], L["w"], L["y"]
            if m == 1:
                _many(ctx, [w["q"], w["k"], w["v"]], x["x"], [y["q"], y["k"], y["v"]])
                w["o"].matvec_bt_dev(x["a"].data_ptr(), y["o"].data_ptr())
                _many(ctx, [w["gate"], w["up"]], x["h"], [y["gate"], y["up"]])
                w["down"].matvec_bt_dev(x["s"].data_ptr(), y["down"].data_ptr())
            else:
                for n, i in (("q", "x"), ("k", "x"), ("v", "x"), ("o", "a"), ("gate", "h"), ("up", "h"), ("down", "s")):
                    w[n].matmul_bt_dev(x[i].data_ptr(), m, y[n].data_ptr())
        return [[L["y"][n] for n in ("q", "k", "v", "o", "gate", "up", "down")] for L in s["layers"]]
    if kind == "matmul":
        b = s["bias"]
        s["w"].matmul_bt_dev(s["x"].data_ptr(), case["tokens"], s["y"].data_ptr(), None if b is None else b.data_ptr())
        return s["y"]
    if kind == "attend":
        for q, k, v, out in s["layers"]:
            K.attend_dev(ctx, s["spec"], q.data_ptr(), k.data_ptr(), v.data_ptr(), case["positions"], out.data_ptr())
        return [d[-1] for d in s["layers"]]
    if kind == "mla":
        for ql, qp, c, pe, out in s["layers"]:
            K.mla_attend_dev(ctx, case["n_head"], ql.data_ptr(), qp.data_ptr(), c.data_ptr(), pe.data_ptr(),
                             case["positions"], mla_scale(case), out.data_ptr())
        return [d[-1] for d in s["layers"]]
    if kind == "moe":
        s["moe"].run_dev(s["x"].data_ptr(), case["tokens"], s["y"].data_ptr())
        return s["y"]
    m = s["model"]
    if kind == "prompt":
        m.truncate(0)
        return m.forward_tokens(s["tokens"])[0]
    if s["steps"] == 64:  # the answers are given: back to the prompts
        for i, n in enumerate(s["lens"]):
            m.resume(s["held"][i])
            m.truncate(n)
            s["held"][i] = m.park()
        s["steps"] = 0
    s["steps"] += 1
    return m.forward_each(s["next"], s["held"])[0]


# ---- what a pass cannot do without ---------------------------------------------

def weight_bytes(precision, rows, cols):
    n = rows * cols
    return {"q8": n + n // 8, "q4": n // 2 + n // 8, "q4k": n // 256 * 144, "f32": 4 * n}[precision]


def work(case):
    kind = case["kind"]
    if kind == "layer":
        m, shapes = case["tokens"], layer_shapes(case)
        ins = 4 * m * (3 * case["hidden"] + case["inter"])
        return {"bytes": case["layers"] * (ins + sum(weight_bytes(case["precision"], r, c) + 4 * m * r
                                                     for _, r, c, _ in shapes)),
                "flops": case["layers"] * sum(2 * m * r * c for _, r, c, _ in shapes)}
    if kind == "matmul":
        r, c, m = case["rows"], case["cols"], case["tokens"]
        return {"bytes": weight_bytes(case["precision"], r, c) + 4 * m * (r + c) + (4 * r if case["bias"] else 0),
                "flops": 2 * m * r * c}
    if kind == "attend":
        L, qd, kvd = case["positions"], case["n_head"] * case["head_dim"], case["n_kv_head"] * case["head_dim"]
        return {"bytes": case["layers"] * (8 * L * kvd + 8 * qd), "flops": case["layers"] * 4 * L * qd}
    if kind == "mla":
        L, H = case["positions"], case["n_head"]
        return {"bytes": case["layers"] * 4 * (L * (LAT + ROPE) + H * (2 * LAT + ROPE)),
                "flops": case["layers"] * 2 * L * H * (2 * LAT + ROPE)}
    if kind == "moe":
        e, ff, sh, m, p = case["hidden"], case["inter"], case["shared"], case["tokens"], case["precision"]
        n, k = case["n_experts"], case["top_k"]
        picked = n * (1 - (1 - k / n) ** m)  # experts that some row picks
        each = 2 * weight_bytes(p, ff, e) + weight_bytes(p, e, ff)
        fused = 2 * weight_bytes(p, sh, e) + weight_bytes(p, e, sh) if sh else 0
        return {"bytes": weight_bytes("q8", n, e) + picked * each + fused + 8 * m * e,
                "flops": 2 * m * (n * e + 3 * k * ff * e + 3 * sh * e)}
    shapes = model_shapes(case)
    weights = case["n_layer"] * sum(weight_bytes(case["precision"], r, c) for _, r, c in shapes)
    head = weight_bytes(case["precision"], case["vocab"], case["n_embd"])
    kvd, qd = case["n_kv_head"] * case["head_dim"], case["n_head"] * case["head_dim"]
    per_row = case["n_layer"] * sum(2 * r * c for _, r, c in shapes)
    if kind == "prompt":
        n = case["tokens"]
        return {"bytes": weights + head + case["n_layer"] * 8 * n * kvd + 4 * case["vocab"],
                "flops": n * per_row + case["n_layer"] * 2 * n * n * qd + 2 * case["vocab"] * case["n_embd"]}
    n, held = case["conversations"], case["conversations"] * case["longest"] * 2 // 3
    return {"bytes": weights + head + case["n_layer"] * 8 * held * kvd + 4 * n * case["vocab"],
            "flops": n * (per_row + 2 * case["vocab"] * case["n_embd"]) + case["n_layer"] * 4 * held * qd}


def tolerance(case):
    kind = case["kind"]
    if kind in ("layer", "matmul"):
        # 32-bit sums over exact integer block dots, or of f32 products: 0.7e-7
        # to 6e-7 off 64 bits over these widths, an order of summing to another
        return {"rel": 4e-6, "max": 4e-5}
    if kind in ("attend", "mla"):
        # 32-bit scores, exponentials and sums: 0.5e-6 to 2.6e-6 off 64 bits
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "moe":
        # an ulp in a hidden value now and then moves its 8-bit code by one:
        # 3e-4 of a lone token's output where one of its codes moves
        return {"rel": 1.5e-3, "max": 2e-2}
    # The same at every layer of a model: a code that moves makes the next
    # layer's move, and after a few layers two orders of summing differ as two
    # draws of the 8-bit rounding do.
    return {"rel": 2.8e-2, "max": 0.25}


# ---- the same in 64 bits ---------------------------------------------------------

def codes(x):
    """QActivation::new's codes times their scales, in 64 bits: per block of 32
    amax / 127 in f32, x / scale rounded half away from zero."""
    shape = x.shape
    b = x.float().reshape(-1, BLOCK)
    scale = b.abs().amax(1, keepdim=True)
    scale = scale / torch.full_like(scale, 127.0)  # by a tensor: a quotient, not a product with 1 / 127
    inv = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
    t = (b * inv).double()
    q = torch.clamp(torch.sign(t) * torch.floor(t.abs() + 0.5), -127, 127)
    return (q * scale.double()).reshape(shape)


def values(precision, data):
    """A weight's values as its precision holds them, in 64 bits."""
    if precision == "f32":
        return data.double()
    if precision == "q4k":
        rows, sup = data["d"].shape
        d, dmin = data["d"].double()[:, :, None], data["dmin"].double()[:, :, None]
        w = (d * data["sc"].double())[..., None] * data["q"].double() - (dmin * data["mn"].double())[..., None]
        return w.reshape(rows, sup * 256)
    if precision == "q8":
        return codes(data)
    b = data.reshape(-1, BLOCK)
    ext = b.gather(1, b.abs().argmax(1, keepdim=True))
    scale = ext / -8.0
    inv = torch.where(scale != 0, 1.0 / scale, torch.zeros_like(scale))
    q = torch.clamp(torch.floor((b * inv + 8.5).double()), 0, 15) - 8
    return (q * scale.double()).reshape(data.shape)


def times(x, precision, w64):
    return (x.double() if precision == "f32" else codes(x)) @ w64.T


def silu_mul(g, u):
    return (g / (1 + torch.exp(-g)) * u).float()


def exact_softmax(s):
    """The reference's weights: softmax, those under 1e-8 dropped."""
    p = torch.softmax(s, -1)
    return torch.where(p < 1e-8, torch.zeros_like(p), p)


def exact_moe(case, seed):
    x, router, experts, shared = moe_data(case, seed)
    p = case["precision"]

    def ffn(rows, w):
        g, u, d = w
        h = silu_mul(times(rows, p, values(p, g)), times(rows, p, values(p, u)))
        return times(h, p, values(p, d))

    prob = torch.softmax(times(x, "q8", values("q8", router)), -1)
    pw, pe = torch.topk(prob, case["top_k"], -1)
    if case["norm_topk"]:
        pw = pw / pw.sum(-1, keepdim=True)
    out = ffn(x, shared) if shared else torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    for i, w in enumerate(experts):
        t, slot = torch.nonzero(pe == i, as_tuple=True)
        if t.numel():
            out[t] += pw[t, slot][:, None] * ffn(x[t], w)
    return out


def exact_model(case, mk, sequences):
    """The logits of each sequence's last token."""
    p, hd = case["precision"], case["head_dim"]
    nh, nkv, half = case["n_head"], case["n_kv_head"], case["head_dim"] // 2
    cos, sin = (torch.from_numpy(t).to(DEV).double() for t in rope_tables(case))
    parts = list(model_data(case, mk))
    embed, final = parts[-1]
    head = values(p, embed)
    lens = [len(t) for t in sequences]
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    at = np.cumsum([0] + lens)
    x = head[torch.from_numpy(np.concatenate(sequences)).to(DEV).long()]

    def norm(v, w):
        return (v / torch.sqrt((v * v).mean(-1, keepdim=True) + EPS) * w.double()).float()

    def rotate(v, n):
        v = v.reshape(-1, n, hd)
        a, b, c, s = v[..., :half], v[..., half:], cos[pos][:, None], sin[pos][:, None]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    for ws, norms, biases in parts[:-1]:
        w = {n: values(p, ws[n][2]) for n in ws}
        h = norm(x, norms[0])
        q, k, v = (times(h, p, w[n]) + biases[n].double() for n in ("q", "k", "v"))
        q, k, v = rotate(q, nh), rotate(k, nkv), v.reshape(-1, nkv, hd)
        att = torch.empty(x.shape[0], nh, hd, dtype=torch.float64, device=DEV)
        for a, b in zip(at[:-1], at[1:]):
            n = int(b - a)
            mask = torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1)
            for j in range(nh):
                g = j // (nh // nkv)
                sc = (q[a:b, j] @ k[a:b, g].T.contiguous() / math.sqrt(hd)).masked_fill(mask, -math.inf)
                att[a:b, j] = exact_softmax(sc) @ v[a:b, g]
        x = x + times(att.reshape(-1, nh * hd).float(), p, w["o"])
        h = norm(x, norms[1])
        x = x + times(silu_mul(times(h, p, w["gate"]), times(h, p, w["up"])), p, w["down"])
    return times(norm(x[torch.from_numpy(at[1:] - 1).to(DEV)], final), p, head)


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        p = case["precision"]
        return [[times(xs[i], p, values(p, data)) for _, _, _, i, data in ws] for xs, ws in layer_data(case, seed)]
    if kind == "matmul":
        x, w, b = matmul_data(case, seed)
        y = times(x, case["precision"], values(case["precision"], w))
        return y if b is None else y + b.double()
    if kind == "attend":
        hd, out = case["head_dim"], []
        for q, k, v in attend_data(case, seed):
            q, k, v = (t.double().reshape(-1, n, hd) for t, n in
                       ((q, case["n_head"]), (k, case["n_kv_head"]), (v, case["n_kv_head"])))
            g = case["n_head"] // case["n_kv_head"]
            out.append(torch.cat([exact_softmax(q[0, j:j + 1] @ k[:, j // g].T.contiguous() / math.sqrt(hd)) @ v[:, j // g]
                                  for j in range(case["n_head"])]).reshape(-1))
        return out
    if kind == "mla":
        out = []
        for ql, qp, c, pe in mla_data(case, seed):
            s = (ql.double() @ c.double().T + qp.double() @ pe.double().T) * mla_scale(case)
            out.append(exact_softmax(s) @ c.double())
        return out
    if kind == "moe":
        return exact_moe(case, seed)
    mk = Maker(seed)
    if kind == "prompt":
        return exact_model(case, mk, [prompt_tokens(case, seed)])[0]
    prompts, nxt = conversations(case, seed)
    return exact_model(case, mk, [np.append(p, t) for p, t in zip(prompts, nxt)])
