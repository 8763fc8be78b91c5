"""Timed cases of the full-attention path: what they run, on which inputs, and what the results should be.

Every case goes through the library's entry points with the argument structs built beforehand, as a compiled runtime
holds them. Kinds:
  ragged   bn_attn_decode_ragged: one new token for each of a batch of sequences (append, attention, gate)
  attn     bn_attn_forward: several rows of one sequence over its cached prefix (append, attention, gate)
  layer    bn_attn_layer: the attention arm from the raw projections (norms, rotary embedding, append, attention,
           gate, Hadamard rotation): one row is a decode step, 2..16 rows are speculative drafts, more are a prefill
  ternary  bn_ternary_matmul: the q/k/v projections in one call, or o_proj added into the hidden rows
  block    a whole attention layer: bn_norm_rotate, q/k/v, bn_attn_layer, o_proj
Head counts and widths are the two model sizes of the runtime: 8 query / 2 kv heads with hidden width 2048, and 16 / 4
with 2560.
"""
import importlib.util
import math
import os
import random
import sys

import torch

D = 256
SIZES = {"2b": (2048, 8, 2), "4b": (2560, 16, 4)}  # hidden width, query heads, kv heads


def _package():
    if "glimpse_language_amd" not in sys.modules:
        folder = os.path.join(os.getcwd(), "glimpse-language_amd")
        spec = importlib.util.spec_from_file_location("glimpse_language_amd", os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["glimpse_language_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["glimpse_language_amd"].bonsai_attn


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = _package().Context(0)
    return _ctx


# ---- the cases ----------------------------------------------------------------------------------------------------
def listed():
    return [
        # a decode server's step: 32 conversations at 8K cached rows each
        dict(name="decode_8k_batch32", kind="ragged", size="4b", nseq=32, lo=8192, hi=8192, lens_seed=0, rotate=False),
        # the same with the lengths that conversations really have, the output rotated for o_proj
        dict(name="decode_ragged_21", kind="ragged", size="4b", nseq=21, lo=75, hi=16384, lens_seed=7, rotate=True),
        # one decode step of a short conversation: latency
        dict(name="layer_decode_1k", kind="layer", size="2b", T=1, off=1023, q_f16=False),
        # 8 speculative draft rows over a long conversation
        dict(name="layer_verify_8_8k", kind="layer", size="4b", T=8, off=8184, q_f16=False),
        # a user turn over a cached 512-row system prefix
        dict(name="prefill_256_over_512", kind="attn", size="2b", T=256, off=512, q_f16=False),
        # a longer user turn, ragged in both sizes, at the runtime's default precision (fp32 q)
        dict(name="layer_prefill_777", kind="layer", size="4b", T=777, off=1031, q_f16=False),
        # a long prompt at the runtime's default precision
        dict(name="layer_prefill_4k", kind="layer", size="4b", T=4096, off=0, q_f16=False),
        # a long prompt with fp16 query rows
        dict(name="prefill_4k_f16q", kind="attn", size="4b", T=4096, off=0, q_f16=True),
        # the q/k/v projections of 8 draft rows
        dict(name="qkv_verify_8", kind="ternary", size="4b", proj="qkv", T=8),
        # the q/k/v projections of a long prompt
        dict(name="qkv_prefill_4k", kind="ternary", size="4b", proj="qkv", T=4096),
        # a decode step's whole attention layer
        dict(name="block_decode_8k", kind="block", size="4b", T=1, off=8191, lora=0),
        # a prompt chunk's whole attention layer over a cached prefix
        dict(name="block_prefill_500", kind="block", size="2b", T=500, off=517, lora=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng, kind):
    """Rows and cached rows of a single-sequence call: a decode step, drafts, or a prefill."""
    how = rng.random()
    if kind != "attn" and how < 0.25:
        return 1, _log(rng, 16, 32767)
    if how < 0.5:
        return rng.randint(2, 16), _log(rng, 16, 16384)
    T = _log(rng, 17, 3500)
    return T, 0 if rng.random() < 0.3 else _log(rng, 7, min(8192, 8400000 // T - T // 2))


def draw(rng):
    """One more case over the same ranges: any kind, both model sizes, sizes spread over their logarithm."""
    kind = rng.choice(("ragged", "attn", "layer", "layer", "ternary", "block"))
    size = rng.choice(tuple(SIZES))
    if kind == "ragged":
        nseq = _log(rng, 1, 40)
        hi = _log(rng, 200, min(32768, 250000 // nseq))
        return dict(kind=kind, size=size, nseq=nseq, lo=min(hi, _log(rng, 20, 8192)), hi=hi,
                    lens_seed=rng.randrange(1 << 20), rotate=rng.random() < 0.5)
    if kind == "ternary":
        return dict(kind=kind, size=size, proj=rng.choice(("qkv", "o")), T=_log(rng, 5, 4000))
    T, off = _rows(rng, kind)
    if kind == "block":
        T = min(T, 1500)
        return dict(kind=kind, size=size, T=T, off=off, lora=rng.choice((0, 0, 8, 16)))
    return dict(kind=kind, size=size, T=T, off=off, q_f16=T > 16 and rng.random() < 0.5)


def _lens(case):
    rng = random.Random(case["lens_seed"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["nseq"])]


def _projections(case):
    """Rows of each matrix and their width."""
    hid, H, KV = SIZES[case["size"]]
    return ((2 * H * D, KV * D, KV * D), hid) if case["proj"] == "qkv" else ((hid,), H * D)


# ---- inputs -------------------------------------------------------------------------------------------------------
def _rms(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)


class _Draw:
    """Seeded inputs on the GPU: cache and query rows as the norms leave them, projections and gate logits N(0, 1)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(*shape, device="cuda", generator=self.g)

    def unit(self, *shape):
        return _rms(self.normal(*shape))

    def signs(self, n):
        return torch.randint(0, 2, (n,), device="cuda", generator=self.g).float() * 2 - 1

    def weight(self, n):
        return 1 + 0.1 * self.normal(n)

    def lin(self, o, k):
        """Packed ternary rows (codes 0, 1, 2; 16 to a word) and their fp16 scales."""
        codes = torch.randint(0, 3, (o, k // 16, 16), device="cuda", generator=self.g)
        w = (codes << (2 * torch.arange(16, device="cuda"))).sum(-1)
        w = torch.where(w >= 2 ** 31, w - 2 ** 32, w).to(torch.int32)
        s = (self.normal(o, k // 128).abs() * 0.02 + 0.005).half()
        return w, s


def _cache(d, rows, KV):
    return d.unit(rows, KV, D).half(), d.normal(rows, KV, D).half()


def _positions(off, T):
    p = torch.arange(off, off + T, device="cuda", dtype=torch.int32)
    return torch.stack([p, p, p]).contiguous()


def _inputs(case, seed):
    d, kind = _Draw(seed), case["kind"]
    hid, H, KV = SIZES[case["size"]]
    x = {}
    if kind == "ragged":
        lens = _lens(case)
        n = len(lens)
        x["kc"], x["vc"] = _cache(d, sum(lens), KV)
        x["kv_off"] = torch.tensor([sum(lens[:i]) for i in range(n)], device="cuda", dtype=torch.int64)
        x["kv_len"] = torch.tensor(lens, device="cuda", dtype=torch.int32)
        x["q"], x["k_new"], x["v_new"] = d.unit(n, H, D), d.unit(n, KV, D), d.normal(n, KV, D)
        x["gate"] = d.normal(n, H, D)
        x["signs"] = d.signs(H * D) if case["rotate"] else None
        return x
    T = case["T"]
    if kind == "ternary":
        os_, k = _projections(case)
        x["x"] = d.normal(T, k)
        x["mats"] = [d.lin(o, k) for o in os_]
        x["y"] = [d.normal(T, o) for o in os_]
        return x
    off = case["off"]
    x["kc"], x["vc"] = _cache(d, off + T, KV)
    if kind == "attn":
        x["q"] = d.unit(T, H, D)
        if case["q_f16"]:
            x["q"] = x["q"].half()
        x["k_new"], x["v_new"], x["gate"] = d.unit(T, KV, D), d.normal(T, KV, D), d.normal(T, H, D)
        return x
    x["qn"], x["kn"] = d.weight(D), d.weight(D)
    x["pos"] = _positions(off, T)
    x["inv"] = 1.0 / (1e7 ** (torch.arange(32, device="cuda", dtype=torch.float32) * 2 / 64))
    x["signs"] = d.signs(H * D)
    if kind == "layer":
        x["qp"], x["kp"], x["vp"] = d.normal(T, H, 2 * D), d.normal(T, KV, D), d.normal(T, KV, D)
        return x
    x["h"], x["in_w"], x["in_signs"] = d.normal(T, hid), d.weight(hid), d.signs(hid)
    x["lin"] = {"q": d.lin(2 * H * D, hid), "k": d.lin(KV * D, hid), "v": d.lin(KV * D, hid), "o": d.lin(hid, H * D)}
    r = case["lora"]
    if r:
        half = lambda *shape: (d.normal(*shape) * 0.05).half()  # noqa: E731
        x["A_in"], x["A_o"] = half(3 * r, hid), half(r, H * D)
        x["B"] = {"q": half(2 * H * D, r), "k": half(KV * D, r), "v": half(KV * D, r), "o": half(hid, r)}
    return x


def prepare(case, seed):
    ba, ctx = _package(), _context()
    x = _inputs(case, seed)
    _, H, KV = SIZES[case["size"]]
    ws = ba.Workspace(ctx, "cuda")
    s = dict(x=x, ws=ws)
    if case["kind"] == "ragged":
        a, out = ba.decode_ragged_args(ctx, ws, x["q"], x["kc"], x["vc"], x["kv_off"], x["kv_len"], max(_lens(case)),
                                       k_new=x["k_new"], v_new=x["v_new"], gate=x["gate"], signs=x["signs"])
        s["calls"] = [ba.bind(ctx, "bn_attn_decode_ragged", a)]
        s["out"] = dict(out=out, kc=x["kc"], vc=x["vc"])
        return s
    T = case["T"]
    if case["kind"] == "ternary":
        work = s["work"] = ba.ternary_workspace(x["x"])
        mats = [(w, sc, y) for (w, sc), y in zip(x["mats"], x["y"])]
        s["calls"] = [ba.bind(ctx, "bn_ternary_matmul",
                              ba.ternary_args(x["x"], mats, add=case["proj"] == "o", work=work))]
        s["out"] = dict(y=x["y"])
        return s
    if case["kind"] == "attn":
        a, out = ba.attention_args(ctx, ws, x["q"], x["kc"], x["vc"], case["off"], k_new=x["k_new"], v_new=x["v_new"],
                                   gate=x["gate"])
        s["calls"] = [ba.bind(ctx, "bn_attn_forward", a)]
        s["out"] = dict(out=out, kc=x["kc"], vc=x["vc"])
        return s
    block = case["kind"] == "block"
    if block:
        hid = x["h"].shape[1]
        x["qp"] = torch.empty(T, H, 2 * D, device="cuda")
        x["kp"], x["vp"] = (torch.empty(T, KV, D, device="cuda") for _ in range(2))
    f16 = not block and case["q_f16"]
    q = torch.empty(T, H, D, device="cuda", dtype=torch.float16 if f16 else torch.float32) if T > ba.VERIFY_MAX else None
    pa, la, out = ba.attention_layer_args(ctx, ws, x["qp"], x["kp"], x["vp"], x["qn"], x["kn"], x["pos"], x["inv"],
                                          x["kc"], x["vc"], case["off"], gate=x["qp"][:, :, D:], signs=x["signs"], q=q)
    s["keep"] = [q, out]
    if not block:
        s["calls"] = [ba.bind(ctx, "bn_attn_layer", pa, la)]
        s["out"] = dict(out=out, kc=x["kc"], vc=x["vc"])
        return s
    r, lin = case["lora"], x["lin"]
    xr = torch.empty(T, hid, device="cuda")
    xo = out.view(T, H * D)
    u = torch.empty(T, 3 * r, device="cuda") if r else None
    uo = torch.empty(T, r, device="cuda") if r else None
    ba.set_lora(la, (x["A_o"], uo) if r else None)
    up = lambda m: (x["B"][m],) if r else ()  # noqa: E731
    work, work_o = ba.ternary_workspace(xr), ba.ternary_workspace(xo)
    s["keep"] += [xr, u, uo, work, work_o]
    qkv = [(*lin[m], y.view(T, -1), *up(m)) for m, y in (("q", x["qp"]), ("k", x["kp"]), ("v", x["vp"]))]
    s["calls"] = [
        ba.bind(ctx, "bn_norm_rotate", ba.norm_args(x["h"], x["in_w"], x["in_signs"], xr,
                                                    lora=(x["A_in"], u) if r else None)),
        ba.bind(ctx, "bn_ternary_matmul", ba.ternary_args(xr, qkv, lora_u=u, lora_r=r, work=work)),
        ba.bind(ctx, "bn_attn_layer", pa, la),
        ba.bind(ctx, "bn_ternary_matmul", ba.ternary_args(xo, [(*lin["o"], x["h"], *up("o"))], add=True, lora_u=uo,
                                                          lora_r=r, work=work_o)),
    ]
    s["out"] = dict(h=x["h"], attn=xo, kc=x["kc"], vc=x["vc"])
    return s


def run(state):
    for call in state["calls"]:
        call()
    return state["out"]


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def _attn_work(T, off, H, KV, q_bytes):
    """Cached K/V rows, q, gate and output once, the new K/V rows read in fp32 and written in fp16."""
    rows = T * off + T * (T + 1) // 2  # (query row, key) pairs
    return (4 * KV * D * off + T * H * D * (q_bytes + 8) + T * KV * D * (8 + 4), 4 * H * D * rows)


def _lin_work(T, o, k):
    return o * k // 4 + o * (k // 128) * 2, 2 * T * o * k


def work(case):
    hid, H, KV = SIZES[case["size"]]
    if case["kind"] == "ragged":
        each = [_attn_work(1, n - 1, H, KV, 4) for n in _lens(case)]
        return dict(bytes=sum(b for b, _ in each), flops=sum(f for _, f in each))
    T = case["T"]
    if case["kind"] == "ternary":
        os_, k = _projections(case)
        each = [_lin_work(T, o, k) for o in os_]
        y = 4 * T * sum(os_) * (2 if case["proj"] == "o" else 1)
        return dict(bytes=sum(b for b, _ in each) + 4 * T * k + y, flops=sum(f for _, f in each))
    b, f = _attn_work(T, case["off"], H, KV, 4)
    if case["kind"] == "attn":
        return dict(bytes=_attn_work(T, case["off"], H, KV, 2 if case["q_f16"] else 4)[0], flops=f)
    if case["kind"] == "layer":
        return dict(bytes=b + 4 * H * D, flops=f)
    # a whole layer: the weights and the hidden rows instead of q, gate, output and new rows
    each = [_lin_work(T, 2 * H * D + 2 * KV * D, hid), _lin_work(T, hid, H * D)]
    return dict(bytes=4 * KV * D * case["off"] + 4 * KV * D * T + 8 * T * hid + sum(x for x, _ in each),
                flops=f + sum(x for _, x in each))


# ---- what the results should be -----------------------------------------------------------------------------------
def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times the distance from exact() that was measured: decodes and projections are 32-bit sums (3e-7 to 4e-7),
# several rows of one sequence multiply fp16 probabilities (1.5e-4 to 2.5e-4), and a block carries those on
TOLERANCE = {"ragged": {"rel": 2e-6}, "ternary": {"rel": 2e-6}, "attn": {"rel": 1e-3}, "layer": {"rel": 1e-3},
             "block": {"rel": 1e-3}}


def _attend(q, kc, vc, off, gate):
    """Causal attention of rows q [T, H, D] at positions off.. over a cache, in float64, gated."""
    T, H = q.shape[:2]
    mask = torch.arange(off + T, device="cuda")[None, :] > off + torch.arange(T, device="cuda")[:, None]
    out = torch.empty(T, H, D, device="cuda", dtype=torch.float64)
    for h in range(H):
        k, v = kc[:off + T, h // 4].double(), vc[:off + T, h // 4].double()
        p = torch.softmax((q[:, h].double() @ k.T / 16).masked_fill_(mask, -math.inf), -1)
        out[:, h] = p @ v
    return out * torch.sigmoid(gate.double())


def _rotate(x, signs):
    """H_512 (x * signs) / sqrt(512) per block of 512 columns."""
    m = torch.ones(1, 1, device="cuda", dtype=torch.float64)
    while m.shape[0] < 512:
        m = torch.cat([torch.cat([m, m], 1), torch.cat([m, -m], 1)], 0)
    T = x.shape[0]
    return ((x.reshape(T, -1) * signs.double()).reshape(T, -1, 512) @ m / math.sqrt(512)).reshape(T, -1)


def _norm(x, w):
    return x / ((x * x).mean(-1, keepdim=True) + 1e-6).sqrt() * w.double()


def _rope(x, pos, inv):
    """Rotate-half embedding on the first 64 dims (the three position rows are equal)."""
    a = (pos[0].double()[:, None] * inv.double()[None, :])[:, None, :]
    lo, hi = x[..., :32], x[..., 32:64]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin(), x[..., 64:]], -1)


def _matmul(x, lin):
    w, s = lin
    codes = (w[:, :, None] >> (2 * torch.arange(16, device="cuda", dtype=torch.int32))) & 3
    full = (codes.reshape(w.shape[0], -1) - 1).double() * s.double().repeat_interleave(128, 1)
    return x.double() @ full.T


def _layer(x, qp, kp, vp, off):
    """norms, rotary embedding, append (into x's caches), attention, gate, rotation."""
    T = qp.shape[0]
    q = _rope(_norm(qp[..., :D], x["qn"]), x["pos"], x["inv"])
    x["kc"][off:off + T] = _rope(_norm(kp, x["kn"]), x["pos"], x["inv"]).half()
    x["vc"][off:off + T] = vp.half()
    gated = _attend(q, x["kc"], x["vc"], off, qp[..., D:])
    return gated, _rotate(gated, x["signs"])


def exact(case, seed):
    x = _inputs(case, seed)
    _, H, KV = SIZES[case["size"]]
    if case["kind"] == "ragged":
        outs, at = [], 0
        for i, n in enumerate(_lens(case)):
            x["kc"][at + n - 1], x["vc"][at + n - 1] = x["k_new"][i].half(), x["v_new"][i].half()
            outs.append(_attend(x["q"][i:i + 1], x["kc"][at:at + n], x["vc"][at:at + n], n - 1, x["gate"][i:i + 1]))
            at += n
        out = torch.cat(outs)
        if case["rotate"]:
            out = _rotate(out, x["signs"]).view_as(out)
        return dict(out=out, kc=x["kc"], vc=x["vc"])
    T = case["T"]
    if case["kind"] == "ternary":
        add = case["proj"] == "o"
        return dict(y=[_matmul(x["x"], m) + (y.double() if add else 0) for m, y in zip(x["mats"], x["y"])])
    off = case["off"]
    if case["kind"] == "attn":
        x["kc"][off:], x["vc"][off:] = x["k_new"].half(), x["v_new"].half()
        return dict(out=_attend(x["q"], x["kc"], x["vc"], off, x["gate"]), kc=x["kc"], vc=x["vc"])
    if case["kind"] == "layer":
        _, out = _layer(x, x["qp"].double(), x["kp"].double(), x["vp"].double(), off)
        return dict(out=out.view(T, H, D), kc=x["kc"], vc=x["vc"])
    r, lin = case["lora"], x["lin"]
    xn = _norm(x["h"].double(), x["in_w"])
    xr = _rotate(xn, x["in_signs"])
    p = {m: _matmul(xr, lin[m]) for m in "qkv"}
    if r:
        u = xn @ x["A_in"].double().T
        for i, m in enumerate("qkv"):
            p[m] += u[:, i * r:(i + 1) * r] @ x["B"][m].double().T
    gated, out = _layer(x, p["q"].view(T, H, 2 * D), p["k"].view(T, KV, D), p["v"].view(T, KV, D), off)
    h = x["h"].double() + _matmul(out, lin["o"])
    if r:
        h += gated.reshape(T, -1) @ x["A_o"].double().T @ x["B"]["o"].double().T
    return dict(h=h, attn=out, kc=x["kc"], vc=x["vc"])
