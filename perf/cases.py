"""The workloads the framework's speed is measured on.

A case is one call (or one short sequence of calls) that a program using this
library makes: a windowed attention layer, a DiT block, the whole 32-block DiT
forward of one Euler step, and the sampler's latent updates around it.  Sizes
are the library's own: clips from 480x256x5 (token grid 2x16x30) to
1280x720x21 (6x45x80), hidden size 2560, 20 heads of 128, MLP 6912, 58 or 64
text tokens (the two bundled embeddings), window extents of the adaptive rule
(0, 0, 0) or fixed ones.

  listed()            the named cases
  draw(rng)           one more case from the same ranges
  prepare(case, seed) inputs, weights and handles on the GPU
  run(state)          one pass through the public entry points
  work(case)          the bytes and operations the pass cannot do without
  tolerance(case)     how far another correct implementation may be off
  exact(case, seed)   the same outputs in float64 from plain torch
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "seedvr2-ncnn-valkan_amd"))
import sv2hip  # noqa: E402

HEADS, HD, DIM, FFN = 20, 128, 2560, 6912
BLOCKS, FIRST_SHARED = 32, 10
LATENT_C, OUT_C, TEXT_C, SINUSOID = 33, 16, 5120, 256
EPS = 1e-5
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ROPES = {"reference": sv2hip.ROPE_REFERENCE, "absolute": sv2hip.ROPE_ABSOLUTE, "none": sv2hip.ROPE_NONE}
MATRICES = ("w_qkv", "w_proj", "w_gate", "w_in", "w_out")


# ---------------------------------------------------------------- the cases


def _attention(T, H, W, win, shifted, text, dtype, rope="reference", **more):
    return dict(kind="attention", T=T, H=H, W=W, wt=win[0], wh=win[1], ww=win[2], shifted=shifted, text=text,
                dtype=dtype, rope=rope, **more)


def _block(T, H, W, win, shifted, text, dtype, shared, **more):
    return dict(kind="block", T=T, H=H, W=W, wt=win[0], wh=win[1], ww=win[2], shifted=shifted, text=text,
                dtype=dtype, shared=shared, **more)


def _dit(T, H, W, win, text, **more):
    return dict(kind="dit", T=T, H=H, W=W, wt=win[0], wh=win[1], ww=win[2], text=text, **more)


def _sampler(T, H, W, rescale, **more):
    return dict(kind="sampler", T=T, H=H, W=W, rescale=rescale, **more)


def listed():
    adaptive = (0, 0, 0)
    return [
        # one sampler step (DiT input, guidance with rescale, Euler update) on
        # the smallest clip: launch-bound, once per Euler step
        _sampler(2, 16, 30, 0.7, name="sampler_480x256x5"),
        # the same on the largest clip, guidance without the rescale
        _sampler(6, 45, 80, 0.0, name="sampler_720p"),
        # a single attention layer of the smallest clip: fixed 2x8x10 windows
        # shifted by half a window, so the edge windows are ragged
        _attention(2, 16, 30, (2, 8, 10), True, 58, "f16", name="attn_480x256x5_f16"),
        # the fp32-input layer without norm and RoPE: the plainest form
        _attention(2, 16, 30, (2, 8, 10), False, 58, "f32", rope="none", name="attn_480x256x5_f32"),
        # an ordinary clip (960x544, 17 frames) in bf16 with the other text
        # length, adaptive windows shifted: every window ragged
        _attention(5, 34, 60, adaptive, True, 64, "bf16", name="attn_960x544x17_bf16"),
        # the 720p layer on 2x9x16 windows, shifted: many short windows
        _attention(6, 45, 80, (2, 9, 16), True, 58, "f16", name="attn_720p_2x9x16_f16"),
        # the 720p layer as the model runs it: adaptive 2x15x27 windows
        _attention(6, 45, 80, adaptive, False, 58, "f16", name="attn_720p_f16"),
        # one early block (text rows with weights of their own) on the
        # smallest clip: few rows, so the weights are most of the bytes
        _block(2, 16, 30, adaptive, False, 58, "f16", False, name="block_480x256x5_f16"),
        # the fp32 parity mode a loader gets unless it asks for fp16
        _block(2, 16, 30, adaptive, True, 58, "f32", True, name="block_480x256x5_f32"),
        # one late block (shared weights) of the 720p clip, shifted
        _block(6, 45, 80, adaptive, True, 58, "f16", True, name="block_720p_f16"),
        # whole DiT forwards: the smallest clip and the largest
        _dit(2, 16, 30, adaptive, 58, name="dit_480x256x5"),
        _dit(6, 45, 80, adaptive, 58, name="dit_720p"),
    ]


# Row counts for which the fp16 blocks find no library product without a
# workspace and refuse the forward (out of 1 to 21760): nothing to measure.
REFUSED_ROWS = ((7201, 7280), (10881, 10976), (11777, 11872), (14401, 14784), (16385, 16640), (16897, 17040))


def _refused(case):
    if case["kind"] not in ("block", "dit") or case.get("dtype") == "f32":
        return False
    counts = (_rows(case), _rows(case) + case["text"])
    return any(lo <= n <= hi for n in counts for lo, hi in REFUSED_ROWS)


def draw(rng):
    while True:
        case = _draw(rng)
        if not _refused(case):
            return case


def _draw(rng):
    # token grids between the two clip sizes: 480 to 3600 cells a frame spread
    # over the logarithm, landscape, square and portrait, any parity
    T = rng.randint(1, 6)
    cells = math.exp(rng.uniform(math.log(480), math.log(3600)))
    aspect = rng.choice((16 / 9, 30 / 16, 4 / 3, 1.0, 9 / 16)) * rng.uniform(0.95, 1.05)
    W = max(16, round(math.sqrt(cells * aspect)))
    H = max(16, min(round(cells / W), 3600 // W))
    text = rng.choice((58, 64, rng.randint(1, 128)))
    win = rng.choice(((0, 0, 0), (0, 0, 0), (2, 8, 10), (2, 9, 16), (rng.randint(1, 3), rng.randint(5, 15),
                                                                     rng.randint(5, 24))))
    shifted = rng.random() < 0.5
    kind = rng.choices(("attention", "block", "dit", "sampler"), (5, 3, 1, 1))[0]
    if kind == "sampler":
        return _sampler(T, H, W, rng.choice((0.0, 0.7)))
    if kind == "dit":
        return _dit(T, H, W, win, text)
    if kind == "block":
        # the parity mode sums in double: small clips only
        dtype = "f32" if T * H * W <= 1500 and rng.random() < 0.5 else "f16"
        return _block(T, H, W, win, shifted, text, dtype, rng.random() < 0.6)
    return _attention(T, H, W, win, shifted, text, rng.choice(("f16", "f16", "f16", "bf16", "f32")),
                      rng.choice(("reference", "reference", "reference", "absolute", "none")))


# ---------------------------------------------------------------- inputs


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, shape, dtype, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _gamma(g, n=HD):
    return torch.rand(n, generator=g, device="cuda") + 0.5


def _freqs():
    return (1.0 / (10000.0 ** (np.arange(0, 42, 2, dtype=np.float64) / 42.0))).astype(np.float32)


def _branch(g, dtype):
    shapes = {"attn_shift": (DIM,), "attn_scale": (DIM,), "attn_gate": (DIM,), "mlp_shift": (DIM,),
              "mlp_scale": (DIM,), "mlp_gate": (DIM,), "w_qkv": (3 * DIM, DIM), "w_proj": (DIM, DIM),
              "b_proj": (DIM,), "w_gate": (FFN, DIM), "w_in": (FFN, DIM), "w_out": (DIM, FFN)}
    out = {k: _randn(g, s, dtype if k in MATRICES else torch.float32, 0.02) for k, s in shapes.items()}
    out["norm_q"], out["norm_k"] = _gamma(g), _gamma(g)
    return out


def _block_weights(g, dtype, shared):
    w = {"vid": _branch(g, dtype), "freqs": _freqs()}
    if not shared:
        w["txt"] = _branch(g, dtype)
    return w


def _win(case):
    return case["wt"], case["wh"], case["ww"]


def _rows(case):
    return case["T"] * case["H"] * case["W"]


def _attention_inputs(case, seed):
    g = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    # random-init q, k and v are N(0, 1) after the qkv product
    vid = _randn(g, (_rows(case), 3 * DIM), dtype)
    txt = _randn(g, (case["text"], 3 * DIM), dtype)
    if case["rope"] == "none":
        # no norm: q and k are scaled so that scores stay of order one
        vid[:, :2 * DIM] *= HD ** -0.25
        txt[:, :2 * DIM] *= HD ** -0.25
        return vid, txt, None
    return vid, txt, [_gamma(g) for _ in range(4)]


def _block_inputs(case, seed):
    g = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    w = _block_weights(g, dtype, case["shared"])
    # the DiT keeps the text rows right after the video rows
    x = _randn(g, (_rows(case) + case["text"], DIM), dtype)
    emb = _randn(g, (6 * DIM,), torch.float32)
    return w, x, emb


def _dit_flags(i):
    return dict(block_index=i, shared_weights=int(i >= FIRST_SHARED), last_layer=int(i == BLOCKS - 1),
                shifted_window=i % 2)


def _dit_heads(g):
    f16, f32 = torch.float16, torch.float32
    wi = {"w_vid": _randn(g, (DIM, 4 * LATENT_C), f16, 0.02), "b_vid": _randn(g, (DIM,), f32, 0.02),
          "w_txt": _randn(g, (DIM, TEXT_C), f16, 0.02), "b_txt": _randn(g, (DIM,), f32, 0.02),
          "w_time_in": _randn(g, (DIM, SINUSOID), f32, 0.02), "b_time_in": _randn(g, (DIM,), f32, 0.02),
          "w_time_hid": _randn(g, (DIM, DIM), f32, 0.02), "b_time_hid": _randn(g, (DIM,), f32, 0.02),
          "w_time_out": _randn(g, (6 * DIM, DIM), f32, 0.02), "b_time_out": _randn(g, (6 * DIM,), f32, 0.02)}
    wo = {"norm_weight": _gamma(g, DIM), "shift": _randn(g, (DIM,), f32, 0.02),
          "scale": _randn(g, (DIM,), f32, 0.02), "w_proj": _randn(g, (4 * OUT_C, DIM), f16, 0.02),
          "b_proj": _randn(g, (4 * OUT_C,), f32, 0.02)}
    return wi, wo


def _dit_latent(g, case):
    latent = torch.randn((LATENT_C, case["T"], 2 * case["H"], 2 * case["W"]), generator=g, device="cuda")
    latent[LATENT_C - 1].fill_(1.0)
    return latent, torch.randn((case["text"], TEXT_C), generator=g, device="cuda")


def _sampler_inputs(case, seed):
    g = _generator(seed)
    shape = (OUT_C, case["T"], 2 * case["H"], 2 * case["W"])
    return [torch.randn(shape, generator=g, device="cuda") for _ in range(4)]


# ---------------------------------------------------------------- prepare, run


def prepare(case, seed):
    return {"attention": _prepare_attention, "block": _prepare_block, "dit": _prepare_dit,
            "sampler": _prepare_sampler}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_attention(case, seed):
    vid, txt, gammas = _attention_inputs(case, seed)
    rule = sv2hip.rule(case["T"], case["H"], case["W"], case["shifted"], *_win(case))
    layer = sv2hip.WindowAttention(rule, HEADS, case["text"], eps=EPS, qk_norm=gammas is not None,
                                   rope_mode=ROPES[case["rope"]], freqs=_freqs())
    out_v = torch.empty((vid.shape[0], DIM), dtype=vid.dtype, device="cuda")
    out_t = torch.empty((txt.shape[0], DIM), dtype=vid.dtype, device="cuda")
    return dict(run=_run_attention, layer=layer, vid=vid, txt=txt, gammas=gammas, out_v=out_v, out_t=out_t)


def _run_attention(s):
    s["layer"](s["vid"], s["txt"], s["gammas"], s["out_v"], s["out_t"])
    return s["out_v"], s["out_t"]


def _prepare_block(case, seed):
    w, x, emb = _block_inputs(case, seed)
    code = sv2hip.F16 if case["dtype"] == "f16" else sv2hip.F32
    wt, wh, ww = _win(case)
    cfg = sv2hip.block_config(block_index=FIRST_SHARED if case["shared"] else 0, shared_weights=int(case["shared"]),
                              shifted_window=int(case["shifted"]), window_t=wt, window_h=wh, window_w=ww)
    block = sv2hip.DitBlock.from_device(cfg, w, code)
    block.set_runtime_shape(case["T"], case["H"], case["W"])
    ws = torch.empty(block.workspace_size(case["text"]), dtype=torch.uint8, device="cuda")
    return dict(run=_run_block, block=block, x=x, out=torch.empty_like(x), rows=_rows(case), emb=emb, ws=ws)


def _run_block(s):
    n, x, out = s["rows"], s["x"], s["out"]
    s["block"].forward(x[:n], x[n:], s["emb"], out[:n], out[n:], workspace=s["ws"])
    return out[:n], out[n:]


def _prepare_dit(case, seed):
    g = _generator(seed)
    wt, wh, ww = _win(case)
    blocks = []
    for i in range(BLOCKS):
        w = _block_weights(g, torch.float16, i >= FIRST_SHARED)
        cfg = sv2hip.block_config(window_t=wt, window_h=wh, window_w=ww, **_dit_flags(i))
        blocks.append(sv2hip.DitBlock.from_device(cfg, w, sv2hip.F16))
    wi, wo = _dit_heads(g)
    dit = sv2hip.Dit.create(sv2hip.DitInput.create(wi, sv2hip.F16, on_device=True), blocks,
                            sv2hip.DitOutput.create(wo, sv2hip.F16, on_device=True))
    latent, text = _dit_latent(g, case)
    out = torch.empty((OUT_C,) + tuple(latent.shape[1:]), device="cuda")
    need = dit.workspace_size(case["T"], 2 * case["H"], 2 * case["W"], case["text"])
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    return dict(run=_run_dit, dit=dit, latent=latent, text=text, out=out, ws=ws)


def _run_dit(s):
    s["dit"].forward(s["latent"], s["text"], 1000.0, s["out"], workspace=s["ws"])
    return s["out"]


def _prepare_sampler(case, seed):
    latent, condition, positive, negative = _sampler_inputs(case, seed)
    return dict(run=_run_sampler, sampler=sv2hip.EulerSampler(50), latent=latent, condition=condition,
                positive=positive, negative=negative, rescale=case["rescale"],
                dit_in=torch.empty((LATENT_C,) + tuple(latent.shape[1:]), device="cuda"),
                guided=torch.empty_like(latent), after=torch.empty_like(latent))


def _run_sampler(s):
    e = s["sampler"]
    e.make_dit_input(s["latent"], s["condition"], output=s["dit_in"])
    e.apply_cfg(s["positive"], s["negative"], 6.5, s["rescale"], output=s["guided"])
    e.step_to(s["guided"], s["latent"], 980.0, 960.0, output=s["after"])
    return s["dit_in"], s["guided"], s["after"]


# ---------------------------------------------------------------- work, tolerance


def _adaptive(T, H, W):
    s = math.sqrt(3600.0 / (H * W))
    return -(-min(T, 30) // 4), -(-round(H * s) // 3), -(-round(W * s) // 3)


def _axis(extent, window, shifted):
    shift = 0.5 if shifted and window < extent else 0.0
    count = -(-extent // window) if not shifted else (math.ceil((extent - shift) / window) + 1 if shift else 1)
    cuts = [(max(int((i - shift) * window), 0), min(int((i - shift + 1) * window), extent)) for i in range(count)]
    return [c for c in cuts if c[1] > c[0]]


def _windows(case, shifted):
    T, H, W = case["T"], case["H"], case["W"]
    wt, wh, ww = (a or b for a, b in zip(_win(case), _adaptive(T, H, W)))
    return [t + h + w for w in _axis(W, ww, shifted) for h in _axis(H, wh, shifted) for t in _axis(T, wt, shifted)]


def _attention_flops(case, shifted):
    sizes = [(t1 - t0) * (h1 - h0) * (w1 - w0) + case["text"] for t0, t1, h0, h1, w0, w1 in _windows(case, shifted)]
    return sum(4.0 * s * s * HD * HEADS for s in sizes)


def work(case):
    rows, text = _rows(case), case.get("text", 0)
    size = {"f16": 2, "bf16": 2, "f32": 4}[case.get("dtype", "f16")]
    params = DIM * (3 * DIM + DIM + 3 * FFN)
    if case["kind"] == "sampler":
        n = OUT_C * 4 * rows
        # sources read: latent (shared by two calls), condition, both
        # predictions; written: 33 channels, guided, updated latent
        return {"bytes": 4 * (n * (4 + 2) + n // OUT_C * LATENT_C), "flops": 10 * n}
    if case["kind"] == "attention":
        return {"bytes": (rows + text) * 4 * DIM * size, "flops": _attention_flops(case, case["shifted"])}
    if case["kind"] == "block":
        return {"bytes": size * (params * (1 if case["shared"] else 2) + 2 * (rows + text) * DIM),
                "flops": 2.0 * (rows + text) * params + _attention_flops(case, case["shifted"])}
    # the last block's text rows have no MLP
    text_rows = text * (BLOCKS - 3 * FFN / (3 * DIM + DIM + 3 * FFN))
    products = 2.0 * params * (rows * BLOCKS + text_rows)
    heads = 2.0 * DIM * (rows * 4 * LATENT_C + text * TEXT_C + rows * 4 * OUT_C + SINUSOID + 7 * DIM)
    attention = BLOCKS / 2 * (_attention_flops(case, False) + _attention_flops(case, True))
    weights = 2 * params * (BLOCKS + FIRST_SHARED + 1) + 4 * DIM * 7 * DIM + 2 * DIM * TEXT_C
    return {"bytes": weights + 4 * 4 * rows * (LATENT_C + OUT_C) + 4 * text * TEXT_C,
            "flops": products + heads + attention}


def tolerance(case):
    """About four times the distance of the present code from exact()."""
    if case["kind"] == "sampler":
        return {"rel": 1.5e-6, "max": 3e-5}  # fp32, one factor from sums in double (3.4e-7)
    if case["kind"] == "attention":
        # every output is a bf16 value: a change of the order of a sum moves
        # some of them by one bf16 step (2^-8 of the value); 1.7e-3 in all is
        # the rounding alone
        return {"rel": 4e-3 if case["dtype"] == "f16" else 2e-3, "max": 0.03}
    if case["kind"] == "dit":
        return {"rel": 5e-3, "max": 0.05}  # fp16 activations through 32 blocks (1.2e-3)
    if case["dtype"] == "f32":
        # fp32 around bf16-rounded q, k, v and attention outputs (4.5e-5: a
        # few of them fall on the other side of a rounding boundary)
        return {"rel": 2e-4, "max": 0.01}
    return {"rel": 4e-3, "max": 0.05}  # fp16 activations and products (9e-4)


# ---------------------------------------------------------------- float64


def _bf16(x):
    return x.to(torch.float32).to(torch.bfloat16).to(torch.float64)


def _rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rotate(x, pos, case_rope):
    """x [rows, heads, 128], pos [rows, 3]: adjacent pairs rotated per axis,
    21 pairs an axis (reference) or 16 / 24 / 24 (absolute)."""
    pairs = (21, 21, 21) if case_rope == "reference" else (16, 24, 24)
    y = x.clone()
    at = 0
    for a, n in enumerate(pairs):
        if case_rope == "reference":
            f = torch.from_numpy(_freqs().astype(np.float64)).cuda()
        else:
            f = 10000.0 ** (-torch.arange(n, dtype=torch.float64, device="cuda") / n)
        ang = (pos[:, a, None] * f)[:, None, :]
        c, s = torch.cos(ang), torch.sin(ang)
        p, q = x[..., at:at + 2 * n:2], x[..., at + 1:at + 2 * n:2]
        y[..., at:at + 2 * n:2] = p * c - q * s
        y[..., at + 1:at + 2 * n:2] = q * c + p * s
        at += 2 * n
    return y


def _exact_attention(case, shifted, vid, txt, gammas, rope, round_out):
    """Joint window attention in float64, q, k and v rounded to bf16 where
    the layer is defined to round them; `round_out`: its outputs too."""
    T, H, W, L = case["T"], case["H"], case["W"], txt.shape[0]
    vid, txt = vid.double().view(-1, 3, HEADS, HD), txt.double().view(-1, 3, HEADS, HD)
    out_v = torch.empty((vid.shape[0], HEADS, HD), dtype=torch.float64, device="cuda")
    out_t = torch.zeros((L, HEADS, HD), dtype=torch.float64, device="cuda")
    grid = torch.arange(T * H * W, device="cuda").view(T, H, W)
    text_pos = torch.arange(L, dtype=torch.float64, device="cuda")[:, None].expand(L, 3)
    wins = _windows(case, shifted)

    def qk(x, gamma, pos):
        if gamma is not None:
            x = _rms(x) * gamma.double()
        return x if rope == "none" or pos is None else _rotate(x, pos, rope)

    for t0, t1, h0, h1, w0, w1 in wins:
        rows = grid[t0:t1, h0:h1, w0:w1].reshape(-1)
        t, y, x = rows // (H * W), rows // W % H, rows % W
        if rope == "reference":
            pos, tpos = torch.stack([L + t - t0, y - h0, x - w0], 1).double(), text_pos
        else:
            pos, tpos = torch.stack([t, y, x], 1).double(), None
        parts = []
        for i in range(2):
            gv, gt = (gammas[i], gammas[2 + i]) if gammas is not None else (None, None)
            parts.append(torch.cat([qk(vid[rows, i], gv, pos), qk(txt[:, i], gt, tpos)]))
        q, k, v = (_bf16(p).transpose(0, 1).contiguous() for p in (*parts, torch.cat([vid[rows, 2], txt[:, 2]])))
        s = torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(HD)
        o = torch.bmm(torch.softmax(s, -1), v).transpose(0, 1)
        if round_out:
            o = _bf16(o)
        out_v[rows] = o[:len(rows)]
        # the text rows' outputs are rounded per window, then averaged
        out_t += _bf16(o[len(rows):])
    return out_v.view(-1, DIM), (out_t / len(wins)).view(-1, DIM)


def _exact_block(case, shifted, last, w, vid, txt, emb):
    e = emb.double().view(DIM, 6)
    vb, tb = w["vid"], w.get("txt", w["vid"])

    def ada(x, b, kind):
        base = 0 if kind == "attn" else 3
        return _rms(x) * (e[:, base + 1] + b[kind + "_scale"].double()) + e[:, base] + b[kind + "_shift"].double()

    def mm(x, m):
        return x @ m.double().T.contiguous()

    xt = _rms(txt) if last else ada(txt, tb, "attn")
    gammas = [vb["norm_q"], vb["norm_k"], tb["norm_q"], tb["norm_k"]]
    av, at = _exact_attention(case, shifted, mm(ada(vid, vb, "attn"), vb["w_qkv"]), mm(xt, tb["w_qkv"]), gammas,
                              "reference", True)

    def proj(a, b, x, gated):
        p = mm(a, b["w_proj"]) + b["b_proj"].double()
        return p * (e[:, 2] + b["attn_gate"].double()) + x if gated else p + x

    def mlp(x, b):
        m = ada(x, b, "mlp")
        h = torch.nn.functional.silu(mm(m, b["w_gate"])) * mm(m, b["w_in"])
        return mm(h, b["w_out"]) * (e[:, 5] + b["mlp_gate"].double()) + x

    pv, pt = proj(av, vb, vid, True), proj(at, tb, txt, not last)
    return mlp(pv, vb), 2.0 * pt if last else mlp(pt, tb)


def _exact_dit(case, seed):
    g = _generator(seed)
    weights = [_block_weights(g, torch.float16, i >= FIRST_SHARED) for i in range(BLOCKS)]
    wi, wo = _dit_heads(g)
    latent, text = _dit_latent(g, case)
    T, H, W = case["T"], case["H"], case["W"]
    wi, wo = ({k: v.double() for k, v in d.items()} for d in (wi, wo))
    x = latent.double().view(LATENT_C, T, H, 2, W, 2).permute(1, 2, 4, 3, 5, 0).reshape(-1, 4 * LATENT_C)
    vid = x @ wi["w_vid"].T + wi["b_vid"]
    txt = text.double() @ wi["w_txt"].T + wi["b_txt"]
    f = 10000.0 ** (-torch.arange(SINUSOID // 2, dtype=torch.float64, device="cuda") / (SINUSOID // 2))
    emb = torch.cat([torch.sin(1000.0 * f), torch.cos(1000.0 * f)])
    silu = torch.nn.functional.silu
    emb = silu(wi["w_time_in"] @ emb + wi["b_time_in"])
    emb = wi["w_time_out"] @ silu(wi["w_time_hid"] @ emb + wi["b_time_hid"]) + wi["b_time_out"]
    for i, w in enumerate(weights):
        vid, txt = _exact_block(case, i % 2 == 1, i == BLOCKS - 1, w, vid, txt, emb)
    e = emb.view(DIM, 6)
    n = _rms(vid) * wo["norm_weight"] * (e[:, 1] + wo["scale"]) + e[:, 0] + wo["shift"]
    p = n @ wo["w_proj"].T + wo["b_proj"]
    return p.view(T, H, W, 2, 2, OUT_C).permute(5, 0, 1, 3, 2, 4).reshape(OUT_C, T, 2 * H, 2 * W).contiguous()


def exact(case, seed):
    if case["kind"] == "attention":
        vid, txt, gammas = _attention_inputs(case, seed)
        return _exact_attention(case, case["shifted"], vid, txt, gammas, case["rope"], False)
    if case["kind"] == "block":
        w, x, emb = _block_inputs(case, seed)
        n = _rows(case)
        return _exact_block(case, case["shifted"], False, w, x[:n].double(), x[n:].double(), emb)
    if case["kind"] == "dit":
        return _exact_dit(case, seed)
    latent, condition, pos, neg = (x.double() for x in _sampler_inputs(case, seed))
    guided = neg + 6.5 * (pos - neg)
    if case["rescale"]:
        guided = guided * (case["rescale"] * pos.std() / guided.std() + 1.0 - case["rescale"])
    a, b = 1.0 - 980.0 / 1000.0, 1.0 - 960.0 / 1000.0
    after = b * (latent - 0.98 * guided) + 0.96 * (latent + a * guided)
    return torch.cat([latent, condition, torch.ones_like(latent[:1])]), guided, after
