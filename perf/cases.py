"""The work this framework is used for, as cases that can be timed and checked.

A case is one pass through the public op surface (``HipContext`` and the
block and trunk drivers built on it): whole pre-norm blocks as the DINO
stage, the trunk and the camera head run them, the attention and linear
layers inside them, the per-layer ops between them, and the whole trunk.
Sizes come from this repository's configurations: 1 to 32 frames of a 37x37
or 21x37 patch grid, 17 prefix tokens per frame in the trunk and 5 in DINO,
width 1024 with 16 heads of 64, MLP 4096; the camera head runs f32 blocks of
width 2048 (16 heads of 128) over one token per frame.

Inputs are synthetic: unit-variance activations, weights ~N(0, 1/fan_in),
LayerNorm weights around 1, LayerScale of about 0.1, biases of about 0.02.
"""
from __future__ import annotations

import math

import torch

from headshot_amd.aggregator import BlockIO, BlockParams, BlockWeights, block_forward, run_block_ops
from headshot_amd.context import HipContext
from headshot_amd.trunk import CACHED_LAYERS, REGISTER_ATTENTION_LAYERS, Trunk

DEVICE = "cuda:0"
TRUNK_PREFIX, DINO_PREFIX = 17, 5
EPS = 1e-5

# ---------------------------------------------------------------------------
# the cases

# kind "block": one block_forward. "seqs" sequences of "tokens" tokens; a
#   grid (gh x gw, RoPE over tokens - prefix patch tokens) for frame blocks,
#   none (gh = 0) for blocks over one joint sequence.
# kind "attention": attention_merged on head-major q, k, v.
# kind "mlp": linear_gelu then linear_ls_residual (fc1, fc2).
# kind "qkv": linear_qkv_heads with RoPE (and QK-norm in the trunk).
# kind "pass_ops": token assembly, one frame block's per-layer ops around
#   given products, and the head-input cache of the result.
# kind "trunk": Trunk.forward, all 24 block pairs.


def _block(name, dtype, seqs, tokens, prefix=0, gh=0, gw=0, dim=1024, heads=16, qk_norm=True,
           fuse_ln=False):
    return {"name": name, "kind": "block", "dtype": dtype, "seqs": seqs, "tokens": tokens,
            "prefix": prefix, "gh": gh, "gw": gw, "dim": dim, "heads": heads, "qk_norm": qk_norm,
            "fuse_ln": fuse_ln}


def listed() -> list:
    t37, t21 = 37 * 37 + TRUNK_PREFIX, 21 * 37 + TRUNK_PREFIX
    d37 = 37 * 37 + DINO_PREFIX
    return [
        # a register-attention layer of an 8-frame scene: 17 tokens a frame,
        # the smallest calls of the trunk, five of its 24 inter-frame blocks
        _block("register_block_f16_n8", "f16", 1, 8 * TRUNK_PREFIX),
        # a camera-head block of an 8-frame scene: one token a frame against
        # f32 weights of width 2048 (latency and weight traffic)
        _block("camera_block_f32_n8", "f32", 1, 8, dim=2048, qk_norm=False),
        # a frame block of a two-image reconstruction
        _block("frame_block_f16_n2", "f16", 2, t37, TRUNK_PREFIX, 37, 37),
        # an inter-frame block of an 8-frame scene, all tokens one sequence
        _block("global_block_f16_n8", "f16", 1, 8 * t37),
        # a frame block on the wide 21x37 grid with each LayerNorm run as the
        # prologue of the product after it (block_forward's fuse_ln option)
        _block("frame_block_f16_n16_wide_lnfused", "f16", 16, t21, TRUNK_PREFIX, 21, 37, fuse_ln=True),
        # a DINO block: f32 whatever the trunk's precision, per frame, no QK-norm
        _block("dino_block_f32_n8", "f32", 8, d37, DINO_PREFIX, 37, 37, qk_norm=False),
        # the f32 attention layer alone, two frames
        {"name": "dino_attention_f32_n2", "kind": "attention", "dtype": "f32", "seqs": 2,
         "tokens": d37, "heads": 16},
        # the f32 q|k|v projection with head split and RoPE, two frames
        {"name": "dino_qkv_f32_n2", "kind": "qkv", "dtype": "f32", "seqs": 2, "tokens": d37,
         "prefix": DINO_PREFIX, "gh": 37, "gw": 37, "qk_norm": False},
        # joint attention over a 32-frame scene, the largest single layer
        {"name": "global_attention_f16_n32", "kind": "attention", "dtype": "f16", "seqs": 1,
         "tokens": 32 * t37, "heads": 16},
        # the MLP's two products over a 32-frame scene
        {"name": "mlp_f16_n32", "kind": "mlp", "dtype": "f16", "rows": 32 * t37},
        # the memory-bound ops of one frame block of a 32-frame scene, with
        # the trunk's token assembly and head-input cache around them
        {"name": "pass_ops_f16_n32", "kind": "pass_ops", "dtype": "f16", "frames": 32,
         "prefix": TRUNK_PREFIX, "gh": 37, "gw": 37},
        # the whole trunk on a two-image reconstruction: one call of a session
        {"name": "trunk_f16_n2", "kind": "trunk", "dtype": "f16", "frames": 2, "gh": 37, "gw": 37},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng) -> dict:
    gh, gw = rng.randint(13, 37), rng.randint(13, 37)
    trunk_t, dino_t = gh * gw + TRUNK_PREFIX, gh * gw + DINO_PREFIX
    frames = _log_int(rng, 1, 32)
    kind = rng.choice(["register", "camera", "frame", "global", "dino", "attention_f16",
                       "attention_f32", "qkv_f16", "qkv_f32", "mlp_f16", "mlp_f32", "pass_ops",
                       "trunk"])
    if kind == "register":
        c = _block("", "f16", 1, TRUNK_PREFIX * _log_int(rng, 1, 200))
    elif kind == "camera":
        c = _block("", "f32", 1, _log_int(rng, 1, 200), dim=2048, qk_norm=False)
    elif kind == "frame":
        c = _block("", "f16", frames, trunk_t, TRUNK_PREFIX, gh, gw, fuse_ln=rng.random() < 0.3)
    elif kind == "global":
        c = _block("", "f16", 1, trunk_t * _log_int(rng, 1, 12))
    elif kind == "dino":
        c = _block("", "f32", _log_int(rng, 1, 12), dino_t, DINO_PREFIX, gh, gw, qk_norm=False)
    elif kind == "attention_f16":
        joint = rng.random() < 0.5
        c = {"kind": "attention", "dtype": "f16", "seqs": 1 if joint else frames,
             "tokens": trunk_t * frames if joint else trunk_t, "heads": 16}
    elif kind == "attention_f32":
        c = {"kind": "attention", "dtype": "f32", "seqs": _log_int(rng, 1, 12), "tokens": dino_t,
             "heads": 16}
    elif kind in ("qkv_f16", "qkv_f32"):
        f16 = kind == "qkv_f16"
        c = {"kind": "qkv", "dtype": "f16" if f16 else "f32",
             "seqs": frames if f16 else _log_int(rng, 1, 12), "tokens": trunk_t if f16 else dino_t,
             "prefix": TRUNK_PREFIX if f16 else DINO_PREFIX, "gh": gh, "gw": gw, "qk_norm": f16}
    elif kind in ("mlp_f16", "mlp_f32"):
        f16 = kind == "mlp_f16"
        c = {"kind": "mlp", "dtype": "f16" if f16 else "f32",
             "rows": _log_int(rng, TRUNK_PREFIX, 32 * 1386 if f16 else 12 * 1374)}
    elif kind == "pass_ops":
        c = {"kind": "pass_ops", "dtype": "f16", "frames": frames, "prefix": TRUNK_PREFIX, "gh": gh,
             "gw": gw}
    else:
        c = {"kind": "trunk", "dtype": "f16", "frames": rng.randint(1, 2), "gh": gh, "gw": gw}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# inputs


def _dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.float32


class _Draws:
    """Seeded normal values on the device."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(seed)

    def __call__(self, shape, mean=0.0, std=1.0, dtype=torch.float32):
        v = torch.randn(shape, generator=self.g, device=DEVICE)
        return (v.mul_(std).add_(mean)).to(dtype)


def _norm(n, width):
    return n((width,), 1.0, 0.1), n((width,), 0.0, 0.05)


def _gamma(n, dim):
    return n((dim,), 0.1, 0.03)


def _block_weights(n, dim, dtype, qk_norm) -> dict:
    def lin(rows, cols):
        return n((rows, cols), 0.0, cols ** -0.5, dtype)

    return {"ln1": _norm(n, dim), "ln2": _norm(n, dim),
            "qn": _norm(n, 64) if qk_norm else None, "kn": _norm(n, 64) if qk_norm else None,
            "qkv_w": lin(3 * dim, dim), "qkv_b": n((3 * dim,), 0.0, 0.02),
            "proj_w": lin(dim, dim), "proj_b": n((dim,), 0.0, 0.02), "ls1": _gamma(n, dim),
            "fc1_w": lin(4 * dim, dim), "fc1_b": n((4 * dim,), 0.0, 0.02),
            "fc2_w": lin(dim, 4 * dim), "fc2_b": n((dim,), 0.0, 0.02), "ls2": _gamma(n, dim)}


def _wrap(w) -> BlockWeights:
    p = BlockParams(ln1=w["ln1"], ln2=w["ln2"], qn=w["qn"], kn=w["kn"], proj_b=w["proj_b"],
                    ls1=w["ls1"], fc1_b=w["fc1_b"], fc2_b=w["fc2_b"], ls2=w["ls2"])
    return BlockWeights(p, w["qkv_w"], w["qkv_b"], w["proj_w"], w["fc1_w"], w["fc2_w"])


def _rope_tables(gh, gw):
    """The axial tables a session builds once: (sin, cos), each (gh gw, 64)
    f32, channels [0, 16) from the row, [16, 32) from the column, repeated."""
    periods = 100.0 ** (torch.arange(16, dtype=torch.float64) / 16.0)
    side = max(gh, gw)

    def angles(count):
        coord = 2.0 * ((torch.arange(count, dtype=torch.float64) + 0.5) / side) - 1.0
        return 2.0 * math.pi * coord[:, None] / periods

    rows = angles(gh)[:, None, :].expand(gh, gw, 16)
    cols = angles(gw)[None, :, :].expand(gh, gw, 16)
    a = torch.cat([rows, cols, rows, cols], dim=-1).reshape(gh * gw, 64)
    return (a.sin().float().contiguous().to(DEVICE), a.cos().float().contiguous().to(DEVICE))


def _rope(case):
    if not case["gh"]:
        return None
    return (*_rope_tables(case["gh"], case["gw"]), case["prefix"])


def _inputs(case, seed) -> dict:
    """The case's input tensors, from the seed alone."""
    n, dt, kind = _Draws(seed), _dtype(case), case["kind"]
    if kind == "block":
        dim = case["dim"]
        return {"w": _block_weights(n, dim, dt, case["qk_norm"]), "rope": _rope(case),
                "x": n((case["seqs"] * case["tokens"], dim), dtype=dt)}
    if kind == "attention":
        shape = (case["seqs"], case["heads"], case["tokens"], 64)
        # queries of spread 1.5: scores of standard deviation 1.5, so that a
        # query prefers some keys and attends to the rest too
        return {"q": n(shape, 0.0, 1.5, dt), "k": n(shape, dtype=dt), "v": n(shape, dtype=dt)}
    if kind == "mlp":
        rows = case["rows"]
        return {"x": n((rows, 1024), dtype=dt), "res": n((rows, 1024), dtype=dt),
                "fc1_w": n((4096, 1024), 0.0, 1 / 32, dt), "fc1_b": n((4096,), 0.0, 0.02),
                "fc2_w": n((1024, 4096), 0.0, 1 / 64, dt), "fc2_b": n((1024,), 0.0, 0.02),
                "gamma": _gamma(n, 1024)}
    if kind == "qkv":
        return {"x": n((case["seqs"] * case["tokens"], 1024), dtype=dt),
                "w": n((3072, 1024), 0.0, 1 / 32, dt), "b": n((3072,), 0.0, 0.02),
                "qn": _norm(n, 64) if case["qk_norm"] else None,
                "kn": _norm(n, 64) if case["qk_norm"] else None, "rope": _rope(case)}
    p, frames = case["gh"] * case["gw"], case["frames"]
    if kind == "pass_ops":
        rows = frames * (p + case["prefix"])
        r = case["prefix"] - 1
        return {"patches": n((frames * p, 1024)), "cam": n((2, 1024), dtype=dt),
                "reg": n((2 * r, 1024), dtype=dt), "ln1": _norm(n, 1024), "ln2": _norm(n, 1024),
                "qn": _norm(n, 64), "kn": _norm(n, 64), "proj_b": n((1024,), 0.0, 0.02),
                "ls1": _gamma(n, 1024), "fc1_b": n((4096,), 0.0, 0.02),
                "fc2_b": n((1024,), 0.0, 0.02), "ls2": _gamma(n, 1024), "rope": _rope(case),
                "q_raw": n((rows, 1024), dtype=dt), "k_raw": n((rows, 1024), dtype=dt),
                "proj_raw": n((rows, 1024), dtype=dt), "fc1_raw": n((rows, 4096), dtype=dt),
                "fc2_raw": n((rows, 1024), dtype=dt)}
    assert kind == "trunk"
    return {"cam": n((2, 1024), dtype=dt), "reg": n((32, 1024), dtype=dt),
            "frame": [_block_weights(n, 1024, dt, True) for _ in range(24)],
            "inter": [_block_weights(n, 1024, dt, True) for _ in range(24)],
            "dino": n((frames * p, 1024))}


# ---------------------------------------------------------------------------
# one pass


def prepare(case, seed) -> dict:
    a = _inputs(case, seed)
    state = {"case": case, "ctx": HipContext(DEVICE), "a": a}
    kind = case["kind"]
    if kind == "block":
        state["w"] = _wrap(a["w"])
    elif kind == "trunk":
        periods = (100.0 ** (torch.arange(16, dtype=torch.float64) / 16.0)).float().numpy()
        state["trunk"] = Trunk(a["cam"], a["reg"], [_wrap(w) for w in a["frame"]],
                               [_wrap(w) for w in a["inter"]], periods, _dtype(case))
    elif kind == "pass_ops":
        rows = a["q_raw"].shape[0]
        x = torch.empty((rows, 1024), device=DEVICE, dtype=_dtype(case))
        state["io"] = BlockIO.empty_like_inputs(x, a["q_raw"], a["k_raw"], a["proj_raw"],
                                                a["fc1_raw"], a["fc2_raw"])
        state["cache"] = torch.empty((rows, 2048), device=DEVICE)
        state["p"] = BlockParams(ln1=a["ln1"], ln2=a["ln2"], qn=a["qn"], kn=a["kn"],
                                 proj_b=a["proj_b"], ls1=a["ls1"], fc1_b=a["fc1_b"],
                                 fc2_b=a["fc2_b"], ls2=a["ls2"])
    return state


def run(state):
    case, ctx, a = state["case"], state["ctx"], state["a"]
    kind = case["kind"]
    if kind == "block":
        return block_forward(ctx, state["w"], a["x"], case["seqs"], case["tokens"],
                             heads=case["heads"], rope=a["rope"], eps=EPS, fuse_ln=case["fuse_ln"])
    if kind == "attention":
        return ctx.attention_merged(a["q"], a["k"], a["v"])
    if kind == "mlp":
        act = ctx.linear_gelu(a["x"], a["fc1_w"], a["fc1_b"])
        return act, ctx.linear_ls_residual(act, a["fc2_w"], a["gamma"], a["res"], a["fc2_b"])
    if kind == "qkv":
        return ctx.linear_qkv_heads(a["x"], a["w"], a["b"], case["seqs"], case["tokens"], 16,
                                    qn=a["qn"], kn=a["kn"], rope=a["rope"], eps=EPS)
    if kind == "pass_ops":
        io, t = state["io"], case["gh"] * case["gw"] + case["prefix"]
        ctx.assemble_tokens(a["patches"], case["frames"], case["gh"] * case["gw"], a["cam"],
                            a["reg"], out_dtype=_dtype(case), out=io.x)
        run_block_ops(ctx, state["p"], io, case["frames"], t, 16, 64, rope=a["rope"], eps=EPS)
        ctx.cache_build(io.x, io.x_out, out=state["cache"])
        return {"x": io.x, "normed": io.normed, "q": io.q_head, "k": io.k_head, "x1": io.x1,
                "normed2": io.normed2, "act": io.act, "x_out": io.x_out, "cache": state["cache"]}
    return state["trunk"].forward(ctx, a["dino"], case["frames"], case["gh"], case["gw"])


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _block_work(rows, seqs, tokens, dim, esz):
    flops = 2 * rows * 12 * dim * dim + 4 * seqs * tokens * tokens * dim
    return 12 * dim * dim * esz + 2 * rows * dim * esz + 60 * dim, flops


def work(case) -> dict:
    kind = case["kind"]
    esz = 2 if case["dtype"] == "f16" else 4
    if kind == "block":
        rows = case["seqs"] * case["tokens"]
        b, f = _block_work(rows, case["seqs"], case["tokens"], case["dim"], esz)
    elif kind == "attention":
        s, t, h = case["seqs"], case["tokens"], case["heads"]
        b, f = 4 * s * t * h * 64 * esz, 4 * s * h * t * t * 64
    elif kind == "mlp":
        rows = case["rows"]
        b = rows * (1024 * 3 + 4096) * esz + 2 * 4096 * 1024 * esz
        f = 4 * rows * 4096 * 1024
    elif kind == "qkv":
        rows = case["seqs"] * case["tokens"]
        b = rows * 4096 * esz + 3072 * 1024 * esz + 2 * case["gh"] * case["gw"] * 64 * 4
        f = 2 * rows * 3072 * 1024
    elif kind == "pass_ops":
        p = case["gh"] * case["gw"]
        rows = case["frames"] * (p + case["prefix"])
        wide = rows * 1024
        # patches in; q, k, proj, fc2 and fc1 products in; the eight results out, the cache in f32
        b = case["frames"] * p * 4096 + 2 * wide * (4 + 4) + 2 * wide * (1 + 1 + 2 + 1 + 1 + 4 + 1) + 8 * wide
        f = rows * 1024 * 80
    else:
        n, p = case["frames"], case["gh"] * case["gw"]
        t = p + TRUNK_PREFIX
        b, f = n * p * 4096 + len(CACHED_LAYERS) * n * t * 2048 * 4, 0
        for k in range(24):
            reg = k in REGISTER_ATTENTION_LAYERS
            joint = n * (TRUNK_PREFIX if reg else t)
            for rows, s, tok in ((n * t, n, t), (joint, 1, joint)):
                f += _block_work(rows, s, tok, 1024, 2)[1]
                b += 12 * 1024 * 1024 * 2
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    """About four times the error against 64-bit sums that the kernels show
    over the ranges of ``draw``: half a unit in the last place of f16 for one
    layer or block, that error carried through 48 blocks for the trunk, and
    f32 sums of 1024 to 4096 products (a block's output is mostly its
    residual input, so its relative error is smaller than a layer's)."""
    if case["kind"] == "trunk":
        return {"rel": 8e-3, "max": 6e-2}
    if case["dtype"] == "f16":
        return {"rel": 1.4e-3, "max": 1.5e-2}
    if case["kind"] == "block":
        return {"rel": 6e-7, "max": 8e-6}
    return {"rel": 3.5e-6, "max": 4.5e-5}


# ---------------------------------------------------------------------------
# the same in 64 bits


def _d(t):
    return t.to(torch.float64)


def _ln(x, wb, eps=EPS):
    mean = x.mean(-1, keepdim=True)
    c = x - mean
    return c * torch.rsqrt((c * c).mean(-1, keepdim=True) + eps) * _d(wb[0]) + _d(wb[1])


def _lin(x, w, b):
    return x @ _d(w).t().contiguous() + _d(b)


def _rot(x, rope):
    """x (S, H, T, 64) rotated past the prefix."""
    if rope is None:
        return x
    sin, cos, prefix = _d(rope[0]), _d(rope[1]), rope[2]
    body = x[..., prefix:, :]
    half = torch.cat([-body[..., 32:], body[..., :32]], dim=-1)
    return torch.cat([x[..., :prefix, :], body * cos + half * sin], dim=-2)


def _heads(x, s, t, h):
    return x.reshape(s, t, h, -1).permute(0, 2, 1, 3).contiguous()


def _attend(q, k, v):
    """(S, H, T, D) in, (S*T, H*D) out, one sequence and head at a time."""
    s, h, t, d = q.shape
    out = torch.empty((s, t, h, d), dtype=torch.float64, device=q.device)
    step = max(64, min(t, (1 << 27) // max(1, t)))
    for i in range(s):
        for j in range(h):
            kt = k[i, j].t().contiguous() / math.sqrt(d)
            for r in range(0, t, step):
                out[i, r:r + step, j] = torch.softmax(q[i, j, r:r + step] @ kt, dim=-1) @ v[i, j]
    return out.reshape(s * t, h * d)


def _exact_block(w, x, s, t, h, rope):
    dim = x.shape[-1]
    qkv = _lin(_ln(x, w["ln1"]), w["qkv_w"], w["qkv_b"])
    q, k, v = (_heads(qkv[:, i * dim:(i + 1) * dim], s, t, h) for i in range(3))
    if w["qn"] is not None:
        q, k = _ln(q, w["qn"]), _ln(k, w["kn"])
    a = _attend(_rot(q, rope), _rot(k, rope), v)
    x1 = x + _d(w["ls1"]) * _lin(a, w["proj_w"], w["proj_b"])
    act = torch.nn.functional.gelu(_lin(_ln(x1, w["ln2"]), w["fc1_w"], w["fc1_b"]))
    return x1 + _d(w["ls2"]) * _lin(act, w["fc2_w"], w["fc2_b"])


def exact(case, seed):
    a, kind = _inputs(case, seed), case["kind"]
    if kind == "block":
        return _exact_block(a["w"], _d(a["x"]), case["seqs"], case["tokens"], case["heads"], a["rope"])
    if kind == "attention":
        return _attend(_d(a["q"]), _d(a["k"]), _d(a["v"]))
    if kind == "mlp":
        act = torch.nn.functional.gelu(_lin(_d(a["x"]), a["fc1_w"], a["fc1_b"]))
        return act, _d(a["res"]) + _d(a["gamma"]) * _lin(act, a["fc2_w"], a["fc2_b"])
    if kind == "qkv":
        qkv = _lin(_d(a["x"]), a["w"], a["b"])
        q, k, v = (_heads(qkv[:, i * 1024:(i + 1) * 1024], case["seqs"], case["tokens"], 16)
                   for i in range(3))
        if a["qn"] is not None:
            q, k = _ln(q, a["qn"]), _ln(k, a["kn"])
        return _rot(q, a["rope"]), _rot(k, a["rope"]), v
    frames, p = case["frames"], case["gh"] * case["gw"]
    if kind == "pass_ops":
        r, t = case["prefix"] - 1, p + case["prefix"]
        x = torch.stack([torch.cat([_d(a["cam"][v:v + 1]), _d(a["reg"][v * r:(v + 1) * r]),
                                    _d(a["patches"][i * p:(i + 1) * p])])
                         for i in range(frames) for v in [int(i != 0)]]).reshape(frames * t, 1024)
        q, k = (_rot(_ln(_heads(_d(a[raw]), frames, t, 16), a[nm]), a["rope"])
                for raw, nm in (("q_raw", "qn"), ("k_raw", "kn")))
        x1 = x + _d(a["ls1"]) * (_d(a["proj_raw"]) + _d(a["proj_b"]))
        out = x1 + _d(a["ls2"]) * (_d(a["fc2_raw"]) + _d(a["fc2_b"]))
        return {"x": x, "normed": _ln(x, a["ln1"]), "q": q, "k": k, "x1": x1,
                "normed2": _ln(x1, a["ln2"]),
                "act": torch.nn.functional.gelu(_d(a["fc1_raw"]) + _d(a["fc1_b"])), "x_out": out,
                "cache": torch.cat([x, out], dim=-1)}
    t = p + TRUNK_PREFIX
    x = torch.cat([torch.cat([_d(a["cam"][v:v + 1]), _d(a["reg"][v * 16:(v + 1) * 16]),
                              _d(a["dino"][i * p:(i + 1) * p])])
                   for i in range(frames) for v in [int(i != 0)]])
    rope = (*_rope_tables(case["gh"], case["gw"]), TRUNK_PREFIX)
    caches = []
    for k in range(24):
        f = _exact_block(a["frame"][k], x, frames, t, 16, rope)
        if k in REGISTER_ATTENTION_LAYERS:
            g = f.reshape(frames, t, 1024)
            reg = g[:, :TRUNK_PREFIX].reshape(frames * TRUNK_PREFIX, 1024)
            reg = _exact_block(a["inter"][k], reg, 1, frames * TRUNK_PREFIX, 16, None)
            x = torch.cat([reg.reshape(frames, TRUNK_PREFIX, 1024), g[:, TRUNK_PREFIX:]],
                          dim=1).reshape(frames * t, 1024)
        else:
            x = _exact_block(a["inter"][k], f, 1, frames * t, 16, None)
            if k in CACHED_LAYERS:
                caches.append(torch.cat([f, x], dim=-1))
    return caches
