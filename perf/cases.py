"""The work that a user of mdx has it do, as cases to be measured: the W4A8 linear, the layers' blocks (MLP, attention,
Gated-DeltaNet layer), the heads (int8 lm_head with its top-k, two-stage draft head), a whole decode step and a prefill.

Every case goes through the package's public operators (mdx._C) or its model (mdx.hybrid.HybridModel). A decode program
replays captured graphs, so the block cases capture the calls of several layers (distinct weights and caches, as the
layers of a model) once and a pass replays them; the linear is called eagerly, as a host's linear hook calls it, and the
prefill as a program starts a sequence. The float64 references restate the operator contracts: where the contract rounds
(bf16 rows between operators, int8 activations) they round too, everything between is float64.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "comfy-mono-decode-xpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from mdx import _C, _lib, hybrid, layout  # noqa: E402

DEV = "cuda"
HID = 4096
EPS = 1e-6
BF = torch.bfloat16
F64 = torch.float64
HEADS = ((32, 8, 128), (16, 4, 256), (16, 8, 64), (32, 4, 128))  # q heads, kv heads, head_dim of the configurations and tests


# ---- the cases -------------------------------------------------------------------------------------
def listed():
    return [
        # a host's W4A8 linear hook on one token: row-major checkpoint codes, fp16 group scales, one eager call
        dict(name="linear_r1", kind="linear", rows=1, n=4096, k=4096, form="fp16", tiled=False),
        # the MLP blocks of a plain decode step: GPTQ weights, one row
        dict(name="mlp_r1", kind="mlp", rows=1, inter=12288, form="fp16", rot=False, layers=4),
        # the MLP blocks of a tree verify on a comfy-kitchen W4A8 checkpoint: fp8 group-16 scales, H256 rotation, 8 rows
        dict(name="mlp_r8_fp8_rot", kind="mlp", rows=8, inter=12288, form="fp8", rot=True, layers=4),
        # the MLP blocks of a wide tree: an odd count of rows above eight
        dict(name="mlp_r13", kind="mlp", rows=13, inter=12288, form="fp16", rot=False, layers=4),
        # attention blocks of a 16-row verify in the hybrid stack's shape, context 2048
        dict(name="attn_r16_2k", kind="attn", rows=16, heads=32, kv_heads=8, dim=128, ctx=2048, layers=8),
        # attention blocks of an 8-row verify in the reference model's shape (head_dim 256), a long ragged context
        dict(name="attn_r8_d256_8k", kind="attn", rows=8, heads=16, kv_heads=4, dim=256, ctx=8191, layers=8),
        # Gated-DeltaNet layers of a plain decode step (one pending row to replay)
        dict(name="gdn_r1", kind="gdn", rows=1, form="fp16", rot=False, tiled=True, pending=1, layers=4),
        # Gated-DeltaNet layers of a tree verify through the host hooks: comfy-kitchen weights in checkpoint layout
        dict(name="gdn_r8_fp8_rot", kind="gdn", rows=8, form="fp8", rot=True, tiled=False, pending=3, layers=4),
        # the verify's head on an int8 ConvRot lm_head: final norm, rotation, logits, exact top-20 of 8 rows
        dict(name="int8_head_r8", kind="int8_head", rows=8, vocab=151936, k=20),
        # a draft's head: int4 scores of the vocabulary, then the exact logits of the candidates
        dict(name="draft_head", kind="draft_head", vocab=151936, nout=4),
        # a whole decode step: a chain of 7 drafts that are accepted, the verify of 8 rows, sampling, accept
        dict(name="decode_step", kind="step", layers=8, drafts=7, prompt=200),
        # the prompt of a new sequence
        dict(name="prefill_1k", kind="prefill", layers=8, tokens=1001),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("linear", "linear", "mlp", "mlp", "attn", "attn", "gdn", "gdn", "int8_head", "draft_head", "step", "prefill"))
    if kind == "linear":
        n, k = rng.choice(((4096, 4096), (1024, 4096), (12288, 4096), (4096, 12288), (8192, 4096), (log_int(1, 768) * 16, log_int(2, 96) * 128)))
        return dict(kind=kind, rows=rng.randint(1, 16 if k <= 8192 else 8), n=n, k=k, form=rng.choice(("fp16", "fp8", "f32")),
                    tiled=rng.random() < 0.5)
    if kind == "mlp":
        form = rng.choice(("fp16", "fp8"))
        return dict(kind=kind, rows=rng.randint(1, 16), inter=rng.choice((12288, 12288, log_int(2, 64) * 256)), form=form,
                    rot=form == "fp8" or rng.random() < 0.25, layers=4)
    if kind == "attn":
        heads, kv_heads, dim = rng.choice(HEADS)
        return dict(kind=kind, rows=rng.randint(1, min(16, 64 * kv_heads // heads)), heads=heads, kv_heads=kv_heads, dim=dim,
                    ctx=log_int(1, 16384), layers=8)
    if kind == "gdn":
        form = rng.choice(("fp16", "fp8"))
        return dict(kind=kind, rows=rng.randint(1, 16), form=form, rot=form == "fp8", tiled=rng.random() < 0.5,
                    pending=rng.randint(0, 8), layers=4)
    if kind == "int8_head":
        return dict(kind=kind, rows=rng.randint(1, 16), vocab=log_int(2048, 9496) * 16, k=rng.choice((1, 20, 50)))
    if kind == "draft_head":
        return dict(kind=kind, vocab=log_int(2048, 9496) * 16, nout=rng.randint(1, 8))
    if kind == "step":
        return dict(kind=kind, layers=rng.choice((4, 8)), drafts=rng.randint(1, 7), prompt=log_int(20, 1000))
    return dict(kind=kind, layers=rng.choice((4, 8)), tokens=log_int(4, 1000))


# ---- inputs ----------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _bf(gen, *shape, scale=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV) * scale).to(BF)


def _norm_w(gen, n):
    return (1 + 0.1 * torch.randn(n, generator=gen, device=DEV)).to(BF)


def _raw_w4(gen, n, k, form):
    """Codes uint8 [n, k], relative group scales and channel scales of one linear: GPTQ fp16 ratios per 128, comfy-kitchen
    fp8 e4m3 per 16, or f32 per 32; weights of about 0.02."""
    codes = (torch.randn(n, k, generator=gen, device=DEV) * 2.5).round_().clamp_(-8, 7).add_(8).to(torch.uint8)
    group, dt = {"fp16": (128, torch.float16), "fp8": (16, torch.float8_e4m3fn), "f32": (32, torch.float32)}[form]
    s = ((0.25 + 0.75 * torch.rand(n, k // group, generator=gen, device=DEV)) * 15.5).to(dt)
    sc = (0.8 + 0.4 * torch.rand(n, generator=gen, device=DEV)) * 8e-4
    return codes, s, sc


def _handle(raw, tiled):
    codes, s, sc = raw
    q = layout.pack_codes(codes)
    if tiled:
        return layout.W4(layout.tile_major_codes(q), s, sc, None, _lib.LAYOUT_TILE)
    return layout.W4(q, s, sc, None, _lib.LAYOUT_ROW)


def _mlp_raw(gen, c):
    return dict(g=_raw_w4(gen, c["inter"], HID, c["form"]), u=_raw_w4(gen, c["inter"], HID, c["form"]),
                d=_raw_w4(gen, HID, c["inter"], c["form"]), nw=_norm_w(gen, HID), x=_bf(gen, c["rows"], HID))


def _attn_raw(gen, c):
    S, H, Hk, D, L = c["rows"], c["heads"], c["kv_heads"], c["dim"], c["ctx"]
    kv = [torch.zeros(1, Hk, L + 64, D, dtype=BF, device=DEV) for _ in range(2)]
    for t in kv:
        t[:, :, :L] = _bf(gen, 1, Hk, L, D)
    return dict(q=_bf(gen, 1, S, H, D, scale=2.0), k=_bf(gen, 1, S, Hk, D), v=_bf(gen, 1, S, Hk, D), wq=_norm_w(gen, D),
                wk=_norm_w(gen, D), key=kv[0], value=kv[1])


def _attn_common(c):
    """RoPE rows (partial, theta 1e7), positions, prefix length and ancestor masks of a chain of rows after the prefix."""
    S, L = c["rows"], c["ctx"]
    rd = 64
    inv = 1e7 ** (-torch.arange(rd // 2, dtype=F64) * 2 / rd)
    ang = torch.arange(L, L + S, dtype=F64)[:, None] * inv[None]
    co, si = torch.cos(ang), torch.sin(ang)
    freqs = torch.stack([torch.stack([co, -si], -1), torch.stack([si, co], -1)], -2).float().contiguous().to(DEV)
    return dict(rd=rd, freqs=freqs, pos=torch.arange(L, L + S, dtype=torch.int64, device=DEV),
                seq=torch.tensor([L], dtype=torch.int32, device=DEV),
                mask=torch.tensor([(1 << (r + 1)) - 1 for r in range(S)], dtype=torch.int32, device=DEV))


HK, HV, DH = 16, 32, 128  # Gated-DeltaNet heads
CH = 2 * HK * DH + HV * DH


def _gdn_raw(gen, c):
    S = _slots(c)
    d = {r: _raw_w4(gen, n, k, c["form"]) for r, n, k in (("qkv", CH, HID), ("z", HV * DH, HID), ("o", HID, HV * DH),
                                                          ("g", 12288, HID), ("u", 12288, HID), ("d", HID, 12288))}
    d.update(nin=_norm_w(gen, HID), npost=_norm_w(gen, HID), gn=_norm_w(gen, DH), wa=_bf(gen, HV, HID, scale=0.02),
             wb=_bf(gen, HV, HID, scale=0.02), cw=_bf(gen, CH, 4, scale=0.5), conv=_bf(gen, CH, 3),
             pb=_bf(gen, 2, S, CH), qb=torch.nn.functional.silu(_bf(gen, 2, S, CH)),
             dt=torch.rand(HV, generator=gen, device=DEV) * 2 - 1,
             gd=-torch.exp(torch.rand(HV, generator=gen, device=DEV) * 1.5 - 1),
             rec=torch.randn(HV, DH, DH, generator=gen, device=DEV) * 0.1,
             gates=torch.rand(2, S, HV, 2, generator=gen, device=DEV) * 0.3 + 0.7, x=_bf(gen, c["rows"], HID))
    return d


def _slots(c):
    return 8 if c["rows"] <= 8 else 16


def _gdn_ctl(c):
    """`pending` accepted rows to replay, then a chain of rows that all commit."""
    S, R = _slots(c), c["rows"]
    return ([c["pending"], 0] + list(range(S)) + [r - 1 for r in range(R)] + [-1] * (S - R) + [r | 32 for r in range(R)]
            + [0] * (S - R))


def _head_raw(gen, c, rows):
    return dict(w=_bf(gen, c["vocab"], HID, scale=0.02), nw=_norm_w(gen, HID), x=_bf(gen, rows, HID))


def _graph(call):
    """`call` captured after a warm-up on a side stream (workspaces reach their sizes), and its outputs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = call()
    return g, out


# ---- prepare ---------------------------------------------------------------------------------------
def prepare(case, seed):
    with torch.no_grad():
        return globals()["_prepare_" + case["kind"]](case, _gen(seed), int(seed))


def _prepare_linear(c, gen, seed):
    w = _handle(_raw_w4(gen, c["n"], c["k"], c["form"]), c["tiled"])
    x = torch.randint(-127, 128, (c["rows"], c["k"]), generator=gen, device=DEV, dtype=torch.int8)
    xs = torch.rand(c["rows"], generator=gen, device=DEV) * 0.02 + 0.01
    out = torch.empty(c["rows"], c["n"], dtype=BF, device=DEV)
    return dict(kind="linear", w=w, x=x, xs=xs, out=out, group=w.group_size)


def _prepare_mlp(c, gen, seed):
    silu, h = layout.silu_lut(DEV), layout.regular_hadamard(DEV)
    rot, hm = (_lib.ROT_H256, h) if c["rot"] else (_lib.ROT_NONE, None)
    layers = []
    for _ in range(c["layers"]):
        r = _mlp_raw(gen, c)
        layers.append(dict(g=_handle(r["g"], True), u=_handle(r["u"], True), d=_handle(r["d"], True), nw=r["nw"], x=r["x"],
                           out=torch.empty_like(r["x"])))

    def call():
        return [_C.mono_mlp_w4(w["x"], rot, hm, silu, w["g"], w["u"], w["d"], norm_w=w["nw"], eps=EPS, out=w["out"],
                               residual=w["x"]) for w in layers]
    g, out = _graph(call)
    return dict(kind="graph", graph=g, out=out, keep=(layers, silu, h))


def _prepare_attn(c, gen, seed):
    S, H, Hk, D = c["rows"], c["heads"], c["kv_heads"], c["dim"]
    m = _attn_common(c)
    layers = [_attn_raw(gen, c) for _ in range(c["layers"])]
    fused = _C.rope_attn_fits(H, Hk, S, D, m["rd"])

    def call():
        out = []
        for w in layers:
            if fused:
                ko = torch.empty(1, Hk, S, D, dtype=BF, device=DEV)
                y = _C.qk_norm_rope_attn(w["q"], w["k"], w["v"], w["wq"], w["wk"], m["freqs"], w["key"], w["value"], m["pos"],
                                         EPS, EPS, m["rd"], m["seq"], m["mask"], ko)
            else:
                q, ko = _C.qk_norm_rope_kv(w["q"], w["k"], w["v"], w["wq"], w["wk"], m["freqs"], w["key"], w["value"],
                                           m["pos"], EPS, EPS, m["rd"])
                y = _C.attn_dpas(q, w["key"], w["value"], m["seq"], ko, w["v"].transpose(1, 2), m["mask"], 0)
            out.append([y, ko])
        return out
    g, out = _graph(call)
    return dict(kind="graph", graph=g, out=out, keep=(layers, m))


def _prepare_gdn(c, gen, seed):
    silu = layout.silu_lut(DEV)
    h = layout.regular_hadamard(DEV) if c["rot"] else None
    ctl = torch.tensor(_gdn_ctl(c), dtype=torch.int32, device=DEV)
    sums = torch.zeros(2, _slots(c), HK, 2, device=DEV)
    layers = []
    for _ in range(c["layers"]):
        r = _gdn_raw(gen, c)
        w4 = []
        for name in ("qkv", "z", "o", "g", "u", "d"):
            w = _handle(r.pop(name), c["tiled"])
            w4 += [w.q, w.s, w.sc, None]
        layers.append(dict(r, w4=w4, row=torch.empty_like(r["x"])))

    def call():
        out = []
        for w in layers:
            w["row"].copy_(w["x"])  # the rows that the layer before left
            _C.layer_gdn(w["row"], w["nin"], EPS, h, w["w4"], w["wa"], w["wb"], w["cw"], w["conv"], w["pb"], w["qb"], ctl,
                         w["dt"], w["gd"], w["rec"], w["gates"], sums, w["gn"], EPS, DH ** -0.5, HK, w["npost"], EPS, silu,
                         0, 11, c["tiled"])
            out.append([w["row"], w["rec"], w["conv"]])
        return out
    kept = [(w[k], w[k].clone()) for w in layers for k in ("conv", "pb", "qb", "rec", "gates")]
    g, out = _graph(call)
    for t, was in kept:  # the warm-up was a step of its own
        t.copy_(was)
    return dict(kind="graph", graph=g, out=out, keep=(layers, ctl, sums, silu, h))


def _prepare_int8_head(c, gen, seed):
    r = _head_raw(gen, c, c["rows"])
    q8, s8 = layout.int8_convrot_head(r["w"])
    w8 = layout.tile_major_i8(q8)
    h = layout.regular_hadamard(DEV)

    def call():
        q, s = _C.rms_rot_quant(r["x"], r["nw"], EPS, _lib.ROT_H256, h)
        logits = _C.int8_linear_prequantized(q, s, w8, s8, tiled=True)
        return [logits] + _C.topk_rows(logits, c["k"])
    g, out = _graph(call)
    return dict(kind="graph", graph=g, out=out, keep=(r["x"], r["nw"], w8, s8, h))


def _prepare_draft_head(c, gen, seed):
    r = _head_raw(gen, c, 1)
    lm4, x = layout.int4_scoring_copy(r["w"]), r["x"]
    i64 = dict(dtype=torch.int64, device=DEV)
    top, tok, vtok = torch.zeros(8, **i64), torch.zeros(1, **i64), torch.zeros(16, **i64)
    vals = torch.zeros(8, dtype=BF, device=DEV)
    scores = torch.empty(1, c["vocab"], dtype=BF, device=DEV)

    def call():
        q, s = _C.quant_rows(x)
        _C.stream_gemv(q, s.view(-1), [lm4], [scores])
        _C.draft_pick_bf16(scores.view(-1), x.view(-1), r["w"], c["nout"], False, top, vals, tok, vtok,
                           list(range(1, 1 + c["nout"])), tiled=False)
        return [scores, vals[:c["nout"]], top[:c["nout"]]]
    g, out = _graph(call)
    return dict(kind="graph", graph=g, out=out, keep=(r, lm4, x, top, tok, vtok, vals))


def _prepare_step(c, gen, seed):
    cfg = hybrid.HybridConfig(layers=c["layers"], widths=(1,) * c["drafts"], two_stage=True, predictable=True, cap=2048)
    m = hybrid.HybridModel(cfg, DEV, seed=seed)
    m.prefill(torch.randint(0, cfg.vocab, (c["prompt"],), generator=torch.Generator().manual_seed(seed)))
    m.capture()
    # the sequence's position, control words, next token and hidden row after the steps of the warm-up
    rewind = [(t, t.clone()) for t in (m.st, m.ctl, m.nt, m.hbuf)]
    out = [m.logits, m.x, m.toks, m.hbuf] + [t for kv in m.kv if kv is not None for t in kv] + [g["rec"] for g in m.gdn if g is not None]
    return dict(kind="step", m=m, rewind=rewind, pos=m.pos_bound, out=out)


def _prepare_prefill(c, gen, seed):
    cfg = hybrid.HybridConfig(layers=c["layers"], vocab=32768, cap=2048)
    m = hybrid.HybridModel(cfg, DEV, seed=seed)
    prompt = torch.randint(0, cfg.vocab, (c["tokens"],), generator=torch.Generator().manual_seed(seed))
    n = c["tokens"] - 1
    out = [m.hbuf, m.nt] + [t[:, :, :n] for kv in m.kv + [m.mkv] if kv is not None for t in kv] + [
        g[k] for g in m.gdn if g is not None for k in ("rec", "conv")]
    fresh = [m.st, m.ctl] + [g[k] for g in m.gdn if g is not None for k in ("rec", "conv")]
    return dict(kind="prefill", m=m, prompt=prompt, out=out, fresh=fresh)


# ---- run -------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "graph":
        state["graph"].replay()
    elif kind == "linear":
        w = state["w"]
        if w.layout == _lib.LAYOUT_ROW:
            return _C.w4a8_decode_linear(state["x"], state["xs"], w.q, w.s, w.sc, None, None, state["group"])
        _C.stream_gemv(state["x"], state["xs"], [w], [state["out"]])
    elif kind == "step":
        m = state["m"]
        for t, was in state["rewind"]:  # the same step again
            t.copy_(was)
        m.pos_bound = state["pos"]
        m.replay(1)
    else:
        for t in state["fresh"]:  # a new sequence
            t.zero_()
        state["m"].prefill(state["prompt"])
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------
def _w4_bytes(n, k, form):
    return n * k // 2 + n * (k // {"fp16": 128, "fp8": 16, "f32": 32}[form]) * {"fp16": 2, "fp8": 1, "f32": 4}[form] + 4 * n


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        return dict(bytes=_w4_bytes(c["n"], c["k"], c["form"]) + c["rows"] * (c["k"] + 4 + 2 * c["n"]),
                    flops=2 * c["rows"] * c["n"] * c["k"])
    if kind == "mlp":
        I, R = c["inter"], c["rows"]
        return dict(bytes=c["layers"] * (2 * _w4_bytes(I, HID, c["form"]) + _w4_bytes(HID, I, c["form"]) + 4 * R * HID + 2 * HID),
                    flops=c["layers"] * 6 * R * I * HID)
    if kind == "attn":
        S, H, Hk, D, L = c["rows"], c["heads"], c["kv_heads"], c["dim"], c["ctx"]
        return dict(bytes=c["layers"] * (4 * Hk * L * D + S * D * (4 * H + 10 * Hk)), flops=c["layers"] * 4 * S * H * D * (L + S // 2))
    if kind == "gdn":
        R, S = c["rows"], _slots(c)
        shapes = ((CH, HID), (HV * DH, HID), (HID, HV * DH), (12288, HID), (12288, HID), (HID, 12288))
        per = sum(_w4_bytes(n, k, c["form"]) for n, k in shapes) + 4 * HV * HID + 2 * CH * (4 + 6 + 2 * c["pending"] + 2 * R)
        return dict(bytes=c["layers"] * (per + 8 * HV * DH * DH + 4 * R * HID),
                    flops=c["layers"] * (2 * R * sum(n * k for n, k in shapes) + 8 * (R + c["pending"]) * HV * DH * DH))
    if kind == "int8_head":
        V, R = c["vocab"], c["rows"]
        return dict(bytes=V * HID + 4 * V + R * (2 * HID + 2 * V + 12 * c["k"]), flops=2 * R * V * HID)
    if kind == "draft_head":
        return dict(bytes=_w4_bytes(c["vocab"], HID, "fp16") + 2 * c["vocab"] + 2 * HID * (1 + c["nout"]), flops=2 * c["vocab"] * HID)
    n_attn = c["layers"] // 4
    mlp = 2 * _w4_bytes(12288, HID, "fp16") + _w4_bytes(HID, 12288, "fp16")
    gdn = _w4_bytes(CH, HID, "fp16") + 2 * _w4_bytes(HID, HID, "fp16") + 4 * HV * HID + 8 * HV * DH * DH
    attn = 2 * _w4_bytes(HID, HID, "fp16") + 2 * _w4_bytes(1024, HID, "fp16")
    layers = c["layers"] * mlp + (c["layers"] - n_attn) * gdn + n_attn * attn
    elems = c["layers"] * 3 * 12288 * HID + (c["layers"] - n_attn) * (CH + 2 * HID) * HID + n_attn * (2 * HID + 2048) * HID
    if kind == "step":
        V, R, L = 151936, 1 + c["drafts"], c["prompt"] + 2 * (1 + c["drafts"])
        block = 2 * HID * (2 * HID + 10240 + HID + 3 * 12288)  # the bf16 draft block: fc, q | gate | k | v, o, MLP
        return dict(bytes=layers + n_attn * 4096 * L + 2 * V * HID + 2 * R * V + c["drafts"] * (block + 4096 * L + _w4_bytes(V, HID, "fp16")),
                    flops=2 * R * (elems + V * HID) + n_attn * 4 * R * HID * L + c["drafts"] * (block + 2 * V * HID + 4 * HID * L))
    n = c["tokens"] - 1  # the prefill's caches: the layers' and the draft block's (its fc and k / v projections fill it)
    return dict(bytes=layers + n * (2 * HID + 4096 * (n_attn + 1)) + 2 * HID * (2 * HID + 2048),
                flops=2 * n * elems + n_attn * 2 * HID * n * n + 2 * n * HID * (2 * HID + 2048))


def tolerance(case):
    # about four times the error that the float64 references (or, for the whole calls, the exact attention's order of sums)
    # show; one int8 code that moves by a rounding shifts a whole row of the MLP and Gated-DeltaNet blocks
    return {
        "linear": {"rel": 5e-3},                  # exact int32 sums, one bf16 rounding
        "mlp": {"rel": 1.5e-2},                   # bf16 rows and int8 codes between the three products
        "attn": {"rel": 1e-2},                    # bf16 q / k / probabilities, fp32 sums
        "gdn": {"rel": 3e-2},                     # as the MLP, with the fp32 delta rule between
        "int8_head": {"rel": 5e-3, "differ": 0.1},  # exact sums; equal bf16 logits may change places
        "draft_head": {"rel": 1e-2, "differ": 0.5},
        "step": {"rel": 1e-2, "differ": 0.1},     # whole calls: roundings travel through the layers
        "prefill": {"rel": 2e-3, "differ": 0.1},
    }[case["kind"]]


# ---- float64 references ----------------------------------------------------------------------------
def exact(case, seed):
    f = globals().get("_exact_" + case["kind"])  # whole calls (step, prefill) have none: their roundings compound
    if f is None:
        return None
    with torch.no_grad():
        return f(case, _gen(seed))


def _w8(raw):
    codes, s, sc = raw
    n, k = codes.shape
    sr = s.to(F64).repeat_interleave(k // s.shape[1], dim=1)
    return torch.round((codes.to(F64) - 8) * sr).clamp_(-127, 127).mul_(sc.to(F64)[:, None])


def _r(x):
    return x.to(torch.float32).to(BF).to(F64)


def _rms(x, w, eps=EPS):
    return _r(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64))


def _h256():
    h4 = torch.tensor(((1, 1, 1, -1), (1, 1, -1, 1), (1, -1, 1, 1), (-1, 1, 1, 1)), dtype=F64, device=DEV)
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    return h / 16


def _quant(x, rot):
    """Per-row int8 codes times their scale, as float64 (codes of bf16(x / bf16(scale)))."""
    if rot:
        x = _r((x.reshape(-1, 256) @ _h256()).reshape(x.shape))
    s = (x.abs().amax(-1, keepdim=True).float() / 127.0).clamp_min(1e-30)
    return torch.round(_r(x / _r(s.to(F64)))).clamp(-128, 127) * s.to(F64)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _mlp64(x, g, u, d, nw, rot):
    q = _quant(_rms(x, nw), rot)
    act = _r(_silu(_r(q @ _w8(g).T)))
    h = _r(act * _r(q @ _w8(u).T))
    return x + _quant(h, rot) @ _w8(d).T


def _exact_linear(c, gen):
    w = _w8(_raw_w4(gen, c["n"], c["k"], c["form"]))
    x = torch.randint(-127, 128, (c["rows"], c["k"]), generator=gen, device=DEV, dtype=torch.int8)
    xs = torch.rand(c["rows"], generator=gen, device=DEV) * 0.02 + 0.01
    return (x.to(F64) @ w.T) * xs.to(F64)[:, None]


def _exact_mlp(c, gen):
    out = []
    for _ in range(c["layers"]):
        r = _mlp_raw(gen, c)
        out.append(_mlp64(r["x"].to(F64), r["g"], r["u"], r["d"], r["nw"], c["rot"]))
    return out


def _exact_attn(c, gen):
    S, H, Hk, D, L = c["rows"], c["heads"], c["kv_heads"], c["dim"], c["ctx"]
    m = _attn_common(c)
    f = m["freqs"].to(F64)[:, None]  # [S, 1, rd / 2, 2, 2]
    hf = m["rd"] // 2

    def rope(t):
        lo, hi, rest = t[..., :hf], t[..., hf:2 * hf], t[..., 2 * hf:]
        return _r(torch.cat([lo * f[..., 0, 0] + hi * f[..., 0, 1], hi * f[..., 1, 1] + lo * f[..., 1, 0], rest], -1))
    causal = torch.ones(S, S, dtype=torch.bool, device=DEV).tril()
    keep = torch.cat([torch.ones(S, L, dtype=torch.bool, device=DEV), causal], 1).repeat(H // Hk, 1)
    out = []
    for _ in range(c["layers"]):
        r = _attn_raw(gen, c)
        q, k = rope(_rms(r["q"][0].to(F64), r["wq"])), rope(_rms(r["k"][0].to(F64), r["wk"]))
        y = torch.empty(S, H, D, dtype=F64, device=DEV)
        for h in range(Hk):
            keys = torch.cat([r["key"][0, h, :L].to(F64), k[:, h]])
            vals = torch.cat([r["value"][0, h, :L].to(F64), r["v"][0, :, h].to(F64)])
            qh = q[:, h * (H // Hk):(h + 1) * (H // Hk)].transpose(0, 1).reshape(-1, D)  # [group * S, D]
            p = torch.softmax((qh @ keys.T / math.sqrt(D)).masked_fill(~keep, -math.inf), -1)
            y[:, h * (H // Hk):(h + 1) * (H // Hk)] = (p @ vals).reshape(H // Hk, S, D).transpose(0, 1)
        out.append([y.reshape(1, S, H * D), k.transpose(0, 1).unsqueeze(0)])
    return out


def _exact_gdn(c, gen):
    R, P = c["rows"], c["pending"]
    out = []
    for _ in range(c["layers"]):
        r = _gdn_raw(gen, c)
        x = r["x"].to(F64)
        xn = _rms(x, r["nin"])
        q = _quant(xn, c["rot"])
        proj, z = _r(q @ _w8(r["qkv"]).T), _r(q @ _w8(r["z"]).T)
        # the conv over the history, the replayed rows and this step's chain
        hist = torch.cat([r["conv"].to(F64).T, r["pb"][1, :P].to(F64)])[-3:]
        taps = torch.cat([hist, proj])
        y = _r(sum(taps[d:d + R] * r["cw"].to(F64)[:, d] for d in range(4)))
        qkv = _r(_silu(y))
        a, b = _r(xn @ r["wa"].to(F64).T), _r(xn @ r["wb"].to(F64).T)
        decay = torch.exp(r["gd"].to(F64) * torch.nn.functional.softplus(a + r["dt"].to(F64)))
        beta = _r(torch.sigmoid(b))
        rows = torch.cat([r["qb"][1, :P].to(F64), qkv])
        decay = torch.cat([r["gates"][1, :P, :, 0].to(F64), decay])
        beta = torch.cat([r["gates"][1, :P, :, 1].to(F64), beta])
        kd = HK * DH
        qn = torch.nn.functional.normalize(rows[:, :kd].reshape(-1, HK, DH), dim=-1) * DH ** -0.5
        kn = torch.nn.functional.normalize(rows[:, kd:2 * kd].reshape(-1, HK, DH), dim=-1)
        qn, kn = (t.repeat_interleave(HV // HK, dim=1) for t in (qn, kn))
        v = rows[:, 2 * kd:].reshape(-1, HV, DH)
        state = r["rec"].to(F64).clone()
        rec, core = state.clone(), []
        for e in range(P + R):
            state = state * decay[e][:, None, None]
            delta = (v[e] - torch.einsum("hk,hkv->hv", kn[e], state)) * beta[e][:, None]
            state = state + kn[e][:, :, None] * delta[:, None, :]
            if e < P:
                rec = state.clone()
            else:
                core.append(torch.einsum("hk,hkv->hv", qn[e], state))
        core = _r(torch.stack(core))
        core = _r(_rms(core, r["gn"]) * _r(_silu(z)).reshape(R, HV, DH)).reshape(R, HV * DH)
        x1 = _r(x + _r(_quant(core, c["rot"]) @ _w8(r["o"]).T))
        out.append([_mlp64(x1, r["g"], r["u"], r["d"], r["npost"], c["rot"]), rec, hist.T])
    return out


def _blocks(w, f, rows=8192):
    return torch.cat([f(w[i:i + rows]) for i in range(0, w.shape[0], rows)], -1)


def _exact_int8_head(c, gen):
    r = _head_raw(gen, c, c["rows"])
    q = _quant(_rms(r["x"].to(F64), r["nw"]), True)
    h = _h256()

    def part(w):
        rot = (w.to(F64).reshape(-1, 256) @ h).reshape(w.shape).float()
        s = (rot.abs().amax(1, keepdim=True) / 127.0).clamp_min(1e-30)
        return q @ (torch.round(rot / s).clamp(-127, 127).to(F64) * s.to(F64)).T
    logits = _blocks(r["w"], part)
    return [logits, _r(logits).topk(c["k"], dim=-1).values, None]


def _exact_draft_head(c, gen):
    r = _head_raw(gen, c, 1)
    x = r["x"].to(F64)
    q = _quant(x, False)

    def part(w):  # the int4 scoring copy: symmetric codes per 128, scales as 1..15 fifteenths of the row's largest
        b = w.float().view(-1, HID // 128, 128)
        s = (b.abs().amax(-1) / 7.0).clamp_min(1e-30)
        codes = (b / s[..., None]).round().clamp(-8, 7)
        s = s.to(torch.float16).float()
        sch = s.amax(1, keepdim=True) / 15.0
        rel = torch.round(s / sch).clamp(1, 15)
        return q @ (codes * rel[..., None]).reshape(-1, HID).to(F64).mul(sch.to(F64)).T
    logits = _blocks(r["w"], lambda w: x @ w.to(F64).T)
    return [_blocks(r["w"], part), logits[0].topk(c["nout"]).values, None]
