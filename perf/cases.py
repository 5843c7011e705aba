"""The calls this framework is used for, as measurable cases.

A case is one forward call through the package's modules: a coded linear, the
projections of an attention block, a coded MLP, the routed experts of an MoE
layer, a whole MoE block, an int8 (w8a16) linear such as the vocabulary head, or
a call over many independent token-layers.  The engine runs inference only: its
two directions are decode (one row to a few tens) and prefill (up to thousands of
rows).  Every size is one of the workloads the benchmark names (hidden 2048 /
256 experts / top-8 / intermediate 512, and hidden 5120 / 17408), or a generic
one of the same range.

Codes are uniform random bits (every bitstream is a valid trellis path), sign
vectors are random +-1, per-row scales U[0.5, 1.5] times a constant, activations
N(0, 1), as the benchmark's own inputs.
"""
import math
import os

import torch

from escha_mlx_amd import dense, moe, ops, quant

DEV = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
RS = 0.088388347648  # 1/sqrt(128) as the codec pins it


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one decode row through the smallest benchmarked projection: launch
        # latency and the host path
        {"name": "linear-1-row", "kind": "linear", "rows": 1, "ic": 2048, "oc": 2048, "K": 2,
         "dtype": "f16", "lut": False},
        # q, k and v of a dense decoder layer for four rows (speculative verify)
        {"name": "qkv-4-rows", "kind": "qkv", "rows": 4, "ic": 5120, "ocs": "5120,5120,5120",
         "K": 2, "dtype": "f16", "lut": True},
        # the dense decoder layer's MLP for one decode row, table decode
        {"name": "mlp-1-row", "kind": "mlp", "rows": 1, "hidden": 5120, "inter": 17408, "K": 3,
         "dtype": "f16", "lut": True},
        # the MLP's down projection for a decode batch, bf16 activations
        {"name": "linear-40-rows-bf16", "kind": "linear", "rows": 40, "ic": 17408, "oc": 5120,
         "K": 3, "dtype": "bf16", "lut": False},
        # the dense decoder layer's MLP over a 2048-token prompt
        {"name": "mlp-2048-rows", "kind": "mlp", "rows": 2048, "hidden": 5120, "inter": 17408,
         "K": 3, "dtype": "f16", "lut": False},
        # routed experts under continuous batching, table decode
        {"name": "experts-32-tokens", "kind": "experts", "tokens": 32, "experts": 256, "top_k": 8,
         "hidden": 2048, "inter": 512, "K_gu": 2, "K_dn": 2, "dtype": "f16", "lut": True},
        # routed experts over a 2048-token prompt
        {"name": "experts-2048-tokens", "kind": "experts", "tokens": 2048, "experts": 256,
         "top_k": 8, "hidden": 2048, "inter": 512, "K_gu": 2, "K_dn": 2, "dtype": "f16",
         "lut": False},
        # a whole MoE block for one decode token
        {"name": "block-1-token", "kind": "block", "tokens": 1, "experts": 256, "top_k": 8,
         "hidden": 2048, "inter": 512, "shared": 512, "K_gu": 2, "K_dn": 3, "dtype": "f16",
         "lut": False},
        # a whole MoE block over a short prompt of odd length, bf16 activations
        {"name": "block-203-tokens-bf16", "kind": "block", "tokens": 203, "experts": 256,
         "top_k": 8, "hidden": 2048, "inter": 512, "shared": 512, "K_gu": 2, "K_dn": 3,
         "dtype": "bf16", "lut": False},
        # the int8 vocabulary head on the last position
        {"name": "head-1-row", "kind": "q8", "rows": 1, "ic": 2048, "oc": 248320, "dtype": "f16"},
        # an int8 projection over a prompt
        {"name": "q8-1000-rows", "kind": "q8", "rows": 1000, "ic": 2048, "oc": 4096,
         "dtype": "f16"},
        # forty independent token-layers of routed experts in one call
        {"name": "layers-40", "kind": "layers", "layers": 40, "tokens": 1, "experts": 256,
         "top_k": 8, "hidden": 2048, "inter": 512},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _log_128(rng, lo, hi):
    """A multiple of 128 (the codec's granularity), spread over the logarithm."""
    return 128 * _log_int(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choice(["linear", "linear", "qkv", "mlp", "experts", "experts", "block", "q8",
                       "layers"])
    dtype = rng.choice(["f16", "f16", "bf16"])
    lut = rng.random() < 0.3
    K = rng.choice([2, 3])
    if kind in ("linear", "qkv"):
        rows = _log_int(rng, 1, 2048) if kind == "linear" else _log_int(rng, 1, 64)
        ic = _log_128(rng, 1024, 17408)
        oc = _log_128(rng, 1024, min(17408, 5120 * 17408 // ic))
        if kind == "linear":
            return {"kind": kind, "rows": rows, "ic": ic, "oc": oc, "K": K, "dtype": dtype,
                    "lut": lut}
        kv = 128 * max(2, oc // 128 // rng.choice([1, 2, 4, 8]))
        return {"kind": kind, "rows": rows, "ic": ic, "ocs": f"{oc},{kv},{kv}", "K": K,
                "dtype": dtype, "lut": lut}
    if kind == "mlp":
        hidden = _log_128(rng, 1024, 5120)
        return {"kind": kind, "rows": _log_int(rng, 1, 2048), "hidden": hidden,
                "inter": _log_128(rng, hidden, 17408), "K": K, "dtype": dtype, "lut": lut}
    if kind in ("experts", "block"):
        c = {"kind": kind, "tokens": _log_int(rng, 1, 2048 if kind == "experts" else 512),
             "experts": rng.choice([64, 128, 160, 256]), "top_k": rng.choice([2, 4, 6, 8]),
             "hidden": _log_128(rng, 1024, 2048), "inter": _log_128(rng, 256, 512), "K_gu": 2,
             "K_dn": K, "dtype": dtype, "lut": lut}
        if kind == "block":
            c["shared"] = _log_128(rng, 256, 1024)
        return c
    if kind == "q8":
        ic = 64 * _log_int(rng, 16, 80)
        oc = _log_int(rng, 512, 248320)
        rows = _log_int(rng, 1, max(1, min(2048, 2048 * 5120 * 17408 // (ic * oc))))
        return {"kind": kind, "rows": rows, "ic": ic, "oc": oc, "dtype": dtype}
    return {"kind": kind, "layers": rng.randint(2, 40), "tokens": rng.choice([1, 1, 2, 3]),
            "experts": rng.choice([64, 128, 256]), "top_k": rng.choice([4, 6, 8]),
            "hidden": 512 * rng.randint(2, 4), "inter": rng.choice([256, 512])}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _code(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, generator=g, device=DEV, dtype=torch.int32)


def _sign(g, *shape):
    return torch.randint(0, 2, shape, generator=g, device=DEV).float() * 2 - 1


def _scale(g, by, *shape):
    return _sign(g, *shape) * (0.5 + torch.rand(*shape, generator=g, device=DEV)) * by


def _lin_inputs(g, ic, oc, K):
    return {"code": _code(g, ic // 16, oc // 16, 8 * K), "rin": _sign(g, ic),
            "rout": _scale(g, 1e-2, oc), "K": K, "ic": ic, "oc": oc}


def _experts_inputs(g, c):
    e, h, i = c["experts"], c["hidden"], c["inter"]
    kg, kd = c.get("K_gu", 2), c.get("K_dn", 2)
    return {"gu": {"code": _code(g, e, h // 16, 2 * i // 16, 8 * kg), "rin": _sign(g, e, h),
                   "rout": _scale(g, 4e-2, e, 2 * i), "K": kg, "ic": h, "oc": 2 * i},
            "dn": {"code": _code(g, e, i // 16, h // 16, 8 * kd), "rin": _sign(g, e, i),
                   "rout": _scale(g, 4e-2, e, h), "K": kd, "ic": i, "oc": h}}


def _q8_inputs(g, ic, oc):
    return {"w8": torch.randint(-127, 128, (oc, ic), generator=g, device=DEV, dtype=torch.int8),
            "scale": (0.5 + torch.rand(oc, generator=g, device=DEV)) * (0.013 / math.sqrt(ic))}


def _route(logits, k):
    """Descending top-k, ties to the lower id, softmax over the k values."""
    v, i = torch.sort(logits, dim=1, descending=True, stable=True)
    return i[:, :k], v[:, :k]


def _block_rows(g, tokens, hidden, gate, k, dtype):
    """Rows whose k-th and (k+1)-th router logits differ by more than a few f16
    roundings: a row with a tie there has two correct answers, so it is drawn
    again."""
    x = torch.randn(tokens, hidden, generator=g, device=DEV).to(dtype)
    for _ in range(8):
        lg = torch.sort(x.half().double() @ gate.double().t(), dim=1, descending=True).values
        close = (lg[:, k - 1] - lg[:, k]).abs() < 4 * 2.0 ** -10 * lg[:, k - 1].abs()
        fresh = torch.randn(tokens, hidden, generator=g, device=DEV).to(dtype)
        x = torch.where(close[:, None], fresh, x)
    return x.contiguous()


def _inputs(case, seed):
    """Everything that is random, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    dtype = DTYPES[case.get("dtype", "f16")]
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    if kind == "linear":
        return {"lin": [_lin_inputs(g, case["ic"], case["oc"], case["K"])],
                "x": rnd(case["rows"], case["ic"])}
    if kind == "qkv":
        return {"lin": [_lin_inputs(g, case["ic"], int(o), case["K"])
                        for o in case["ocs"].split(",")], "x": rnd(case["rows"], case["ic"])}
    if kind == "mlp":
        h, i, K = case["hidden"], case["inter"], case["K"]
        return {"lin": [_lin_inputs(g, h, i, K), _lin_inputs(g, h, i, K), _lin_inputs(g, i, h, K)],
                "x": rnd(case["rows"], h)}
    if kind == "experts":
        s = _experts_inputs(g, case)
        s["x"] = rnd(case["tokens"], case["hidden"])
        s["logits"] = torch.randn(case["tokens"], case["experts"], generator=g, device=DEV)
        return s
    if kind == "block":
        s = _experts_inputs(g, case)
        h, sh = case["hidden"], case["shared"]
        s["gate"] = (torch.randn(case["experts"], h, generator=g, device=DEV) / math.sqrt(h)).half()
        s["shg"] = (torch.randn(1, h, generator=g, device=DEV) / math.sqrt(h)).half()
        s["sh_gate"], s["sh_up"] = _q8_inputs(g, h, sh), _q8_inputs(g, h, sh)
        s["sh_down"] = _q8_inputs(g, sh, h)
        s["x"] = _block_rows(g, case["tokens"], h, s["gate"], case["top_k"], dtype)
        return s
    if kind == "q8":
        return {"q8": _q8_inputs(g, case["ic"], case["oc"]), "x": rnd(case["rows"], case["ic"])}
    lays = []
    for _ in range(case["layers"]):
        s = _experts_inputs(g, case)
        s["x"] = rnd(case["tokens"], case["hidden"])
        s["logits"] = torch.randn(case["tokens"], case["experts"], generator=g, device=DEV)
        lays.append(s)
    return {"layers": lays}


# ------------------------------------------------------------------ the program

def _with_lut(case, make):
    """The decode option is an environment knob that modules latch when built."""
    old = os.environ.get("ESCHA_MLX_LUT")
    os.environ["ESCHA_MLX_LUT"] = "1" if case.get("lut") else "0"
    try:
        return make()
    finally:
        if old is None:
            del os.environ["ESCHA_MLX_LUT"]
        else:
            os.environ["ESCHA_MLX_LUT"] = old


def _linear(p):
    return dense.EschaLinear(dense.EschaWeight(p["code"], p["rin"].cpu().numpy(),
                                               p["rout"].cpu().numpy(), device=DEV))


def _experts(s):
    return [moe.EschaExperts.from_device(p["code"], p["rin"], p["rout"], p["K"])
            for p in (s["gu"], s["dn"])]


@torch.no_grad()
def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind in ("linear", "qkv"):
        lins = _with_lut(case, lambda: [_linear(p) for p in s["lin"]])
        return {"kind": kind, "lins": lins, "x": s["x"]}
    if kind == "mlp":
        lins = _with_lut(case, lambda: [_linear(p) for p in s["lin"]])
        return {"kind": kind, "module": dense.EschaMLP(*lins), "x": s["x"]}
    if kind == "experts":
        gu, dn = _experts(s)
        m = _with_lut(case, lambda: moe.EschaMoEExperts(gu, dn, case["experts"], case["top_k"]))
        return {"kind": kind, "module": m, "x": s["x"], "logits": s["logits"],
                "top_k": case["top_k"]}
    if kind == "block":
        gu, dn = _experts(s)
        shared = {}
        for n in ("gate", "up", "down"):
            shared[f"{n}_w8"], shared[f"{n}_scale"] = s[f"sh_{n}"]["w8"], s[f"sh_{n}"]["scale"]
        m = _with_lut(case, lambda: moe.EschaSparseMoeBlock(
            case["hidden"], case["experts"], case["top_k"], gu, dn, s["gate"], s["shg"], shared))
        return {"kind": kind, "module": m, "x": s["x"]}
    if kind == "q8":
        return {"kind": kind, "module": quant.EschaQ8Head(s["q8"]["w8"], s["q8"]["scale"]),
                "x": s["x"]}
    lays = []
    for p in s["layers"]:
        ids, scores = moe.route(p["logits"], case["top_k"])
        lays.append({"x": p["x"], "ids": ids, "scores": scores, "y": torch.empty_like(p["x"]),
                     **{f"{leg}_{f}": p[leg][f] for leg in ("gu", "dn")
                        for f in ("code", "rin", "rout")}})
    t, k, e, h, i = (case[n] for n in ("tokens", "top_k", "experts", "hidden", "inter"))
    ws = torch.zeros(max(4, ops.moe_layers_workspace(len(lays), t, k, h, i)), dtype=torch.uint8,
                     device=DEV)
    return {"kind": kind, "layers": lays, "table": ops.moe_layers_table(lays, DEV), "ws": ws,
            "shape": (t, k, e, h, i)}


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["lins"][0](state["x"])
    if kind == "qkv":
        return dense.project_many(state["lins"], state["x"])
    if kind == "experts":
        ids, scores = moe.route(state["logits"], state["top_k"])
        return state["module"](state["x"], ids, scores)
    if kind == "layers":
        t, k, e, h, i = state["shape"]
        ops.moe_expert_path_layers(state["table"], t, k, e, h, i, 2, 2, ws=state["ws"])
        return [lay["y"] for lay in state["layers"]]
    return state["module"](state["x"])


# ------------------------------------------------------------------ what it costs

def work(case):
    kind = case["kind"]
    el = 2  # activations are 16-bit
    lin = lambda m, ic, oc, K: (ic * oc * K / 8 + 4 * (ic + oc), 2.0 * m * ic * oc)
    if kind == "linear":
        b, f = lin(case["rows"], case["ic"], case["oc"], case["K"])
        return {"bytes": b + el * case["rows"] * (case["ic"] + case["oc"]), "flops": f}
    if kind == "qkv":
        ocs = [int(o) for o in case["ocs"].split(",")]
        b, f = zip(*(lin(case["rows"], case["ic"], o, case["K"]) for o in ocs))
        return {"bytes": sum(b) + el * case["rows"] * (case["ic"] + sum(ocs)), "flops": sum(f)}
    if kind == "mlp":
        b, f = lin(case["rows"], case["hidden"], case["inter"], case["K"])
        return {"bytes": 3 * b + 2 * el * case["rows"] * case["hidden"], "flops": 3 * f}
    if kind == "q8":
        m, ic, oc = case["rows"], case["ic"], case["oc"]
        return {"bytes": oc * (ic + 4) + el * m * (ic + oc), "flops": 2.0 * m * ic * oc}
    t, k, e, h, i = (case[n] for n in ("tokens", "top_k", "experts", "hidden", "inter"))
    kg, kd = case.get("K_gu", 2), case.get("K_dn", 2)
    distinct = e * (1 - (1 - k / e) ** t)  # experts that are routed to, on average
    b = distinct * (2 * h * i * kg / 8 + h * i * kd / 8 + 4 * 3 * (h + i)) + 2 * el * t * h
    f = 2.0 * t * k * 3 * h * i
    if kind == "block":
        sh = case["shared"]
        b += 2 * e * h + 2 * h + 3 * h * sh + 4 * (2 * sh + h)
        f += 2.0 * t * (e * h + h + 3 * h * sh)
    elif kind == "experts":
        b += 4 * t * e
    n = case.get("layers", 1)
    return {"bytes": b * n, "flops": f * n}


def tolerance(case):
    """About four times the distance from the 64-bit result: one f16 rounding of
    the output for a linear, a few f16 roundings in a row for the MLP and the
    experts, one bf16 rounding where the output is bf16."""
    if case.get("dtype") == "bf16":
        return {"rel": 7e-3}
    return {"rel": 1e-3 if case["kind"] in ("linear", "qkv", "q8") else 2e-3}


# ------------------------------------------------------------------ in 64 bits

def _decode(code, K, ic, oc):
    """Bare weights f64 [ic, oc] of one packed stream: a tile's 8K words are one
    circular bitstream, step t's state the 16 bits that end at bit K(t+1), the
    value the f16 sum of a multiplicative hash's two halves."""
    tk, tn = ic // 16, oc // 16
    t = torch.arange(256, device=code.device)
    start = (K * (t + 1) - 16) % (256 * K)
    lane, j = t >> 3, t & 7
    row = 2 * (lane & 3) + (j & 1) + 8 * ((j >> 1) & 1)
    col = 2 * ((lane >> 3) + 4 * (j >= 4).long()) + ((lane >> 2) & 1)
    s = torch.arange(65536, device=code.device)
    r = ((s * 0xCBAC1FED) & 0x8FFF8FFF) ^ 0x3B603B60
    half = lambda v: v.to(torch.int16).view(torch.float16).double()
    lo, hi = r & 0xFFFF, r >> 16
    signed = lambda v: torch.where(v >= 32768, v - 65536, v)
    table = (half(signed(lo)) + half(signed(hi))).half().double()
    w = torch.empty(ic, oc, dtype=torch.float64, device=code.device)
    for k0 in range(0, tk, 64):
        words = code[k0:k0 + 64].long() & 0xFFFFFFFF
        a, off = start >> 5, start & 31
        pair = words[..., a] << 16 | words[..., (a + 1) % (8 * K)] >> 16  # 48 bits are enough
        state = (pair >> (32 - off)) & 0xFFFF
        tiles = torch.empty(words.shape[0], tn, 16, 16, dtype=torch.float64, device=code.device)
        tiles[:, :, row, col] = table[state]
        w[16 * k0:16 * (k0 + words.shape[0])] = tiles.permute(0, 2, 1, 3).reshape(-1, oc)
    return w


def _h128(v):
    """The unnormalised 128-point Walsh-Hadamard transform of each 128-block."""
    n = torch.arange(128, device=v.device)
    bits = n[:, None] & n[None, :]
    par = torch.zeros_like(bits)
    for b in range(7):
        par ^= (bits >> b) & 1
    h = (1 - 2 * par).double()
    return (v.reshape(-1, 128) @ h).reshape(v.shape)


def _r16(v):
    return v.half().double()


def _exact_linear(x, p, e=None):
    """The codec's linear with its f16 rounding points, sums in 64 bits."""
    pick = (lambda t: t) if e is None else (lambda t: t[e])
    xh = _r16(_h128(x.double() * pick(p["rin"]).double()) * RS)
    mid = xh @ _decode(pick(p["code"]), p["K"], p["ic"], p["oc"])
    return _h128(mid) * RS * pick(p["rout"]).double()


def _silu(v):
    return v / (1 + torch.exp(-v))


def _exact_experts(x, ids, scores, s, k):
    """f64 [T, H]: the experts' outputs (f16) times the f16 score, summed."""
    t = x.shape[0]
    flat, d = ids.reshape(-1), torch.zeros(ids.numel(), x.shape[1], dtype=torch.float64, device=DEV)
    i = s["dn"]["ic"]
    for e in torch.unique(flat).tolist():
        rows = (flat == e).nonzero()[:, 0]
        gu = _r16(_exact_linear(x[rows // k], s["gu"], e))
        h = _r16(_r16(_silu(gu[:, :i])) * gu[:, i:])
        d[rows] = _r16(_exact_linear(h, s["dn"], e))
    return (d.reshape(t, k, -1) * _r16(scores)[..., None]).sum(1)


def _exact_q8(x, p):
    wf = (p["w8"].float() * p["scale"].float()[:, None]).half()
    y = torch.empty(x.shape[0], wf.shape[0], dtype=torch.float64, device=DEV)
    for o in range(0, wf.shape[0], 8192):
        y[:, o:o + 8192] = x.double() @ wf[o:o + 8192].double().t()
    return y


@torch.no_grad()
def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return _exact_linear(s["x"], s["lin"][0])
    if kind == "qkv":
        return [_exact_linear(s["x"], p) for p in s["lin"]]
    if kind == "mlp":
        # the projections' outputs take x's type, the activation is f16
        g, u = (_r16(_r16(_exact_linear(s["x"], p)).to(s["x"].dtype).double())
                for p in s["lin"][:2])
        return _exact_linear(_r16(_silu(g) * u), s["lin"][2])
    if kind == "q8":
        return _exact_q8(s["x"].half(), s["q8"])

    def routed(p, x, logits):
        ids, top = _route(logits, case["top_k"])
        return _exact_experts(x, ids, torch.softmax(top.double(), dim=1), p, case["top_k"])

    if kind == "experts":
        return routed(s, s["x"], s["logits"])
    if kind == "layers":
        return [routed(p, p["x"], p["logits"]) for p in s["layers"]]
    xf = s["x"].half()
    y = _r16(routed(s, s["x"], _r16(xf.double() @ s["gate"].double().t())))
    hh = _r16(_silu(_r16(_exact_q8(xf, s["sh_gate"]))) * _r16(_exact_q8(xf, s["sh_up"])))
    sh = _r16(_exact_q8(hh, s["sh_down"]))
    return y + sh * torch.sigmoid(_r16(xf.double() @ s["shg"].double().t()))
