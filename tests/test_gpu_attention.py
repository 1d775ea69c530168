"""Attention (hs_attention, hs_attention_merged) and the head merge
(hs_attn_merge) against the oracle on the reference's own test shapes, at
tile edges, and at full size against a float32 torch reference on the device.

Bars:
- f32: within 1e-5 (abs + rel) of the oracle, and 1e-4 absolute of the
  float64 naive softmax as tests/kernels.rs:232-235.
- f16: within 2e-3*max(1,|e|) of the oracle's f16 result (f32 math on the
  same f16 inputs, output rounded). The matrix-core path rounds the softmax
  weights to f16 for the P.V product; this bound covers that.
- f16 vs f32 on the same values: 5e-3 relative (tests/kernels.rs:377-401).
- attn_merge bit-exact; attention_merged bit-exact against
  attn_merge(attention(...)).
"""
import numpy as np
import pytest
import torch

from headshot_amd import _lib
from headshot_amd.parity import assert_bit_exact, assert_close, f16_close
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NP = {torch.float32: np.float32, torch.float16: np.float16}
DTYPES = [torch.float32, torch.float16]


def host(a: np.ndarray, dtype) -> np.ndarray:
    return O.to_f16(a) if dtype == torch.float16 else np.ascontiguousarray(a, np.float32)


def dev(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def back(t: torch.Tensor) -> np.ndarray:
    torch.cuda.synchronize()
    return t.cpu().numpy()


def check(got: np.ndarray, want: np.ndarray, what: str):
    assert got.dtype == want.dtype, f"{what}: dtype {got.dtype} vs {want.dtype}"
    if got.dtype == np.float32:
        assert_close(got, want, 1e-5, what)
    else:
        f16_close(got.astype(np.float32), want.astype(np.float32), what)


def naive64(q, k, v):
    """tests/kernels.rs:207-231 in float64."""
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    s = np.matmul(q, np.swapaxes(k, -1, -2)) / np.sqrt(q.shape[-1])
    p = np.exp(s - s.max(-1, keepdims=True))
    return np.matmul(p / p.sum(-1, keepdims=True), v)


def torch_attention32(q, k, v, q_rows=None):
    """float32 reference on the device; q_rows selects queries (dim 2)."""
    q32, k32, v32 = (x.float() for x in (q, k, v))
    if q_rows is not None:
        q32 = q32[:, :, q_rows].contiguous()
    scale = 1.0 / float(np.sqrt(q.shape[-1]))
    s = torch.matmul(q32, k32.transpose(-1, -2).contiguous()) * scale
    return torch.matmul(torch.softmax(s, dim=-1), v32)


def rand_qkv(seed, shape, dtype):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return [torch.randn(shape, generator=g).to(dtype).to("cuda:0") for _ in range(3)]


# ------------------------------------------------------ the reference's cases

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("t", [17, 64, 150])
def test_attention_reference_cases(ctx, dtype, t):
    """tests/kernels.rs:185-238: (s, h, d) = (2, 3, 64), q, k, v from Rng(5 + t)."""
    s, h, d = 2, 3, 64
    stream = O.rng_vec(5 + t, 3 * s * h * t * d).reshape(3, s, h, t, d)
    q, k, v = (host(stream[i], dtype) for i in range(3))
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    check(got, O.attention(q, k, v), f"attention t={t} {dtype}")
    if dtype == torch.float32:
        assert np.abs(got - naive64(q, k, v)).max() < 1e-4


def test_attention_f16_matches_f32(ctx):
    """tests/kernels.rs:377-401: (1, 2, 33, 64), Rng(9), 5e-3."""
    s, h, t, d = 1, 2, 33, 64
    stream = O.rng_vec(9, 3 * s * h * t * d).reshape(3, s, h, t, d)
    f32 = back(ctx.attention(*(dev(stream[i]) for i in range(3))))
    f16 = back(ctx.attention(*(dev(O.to_f16(stream[i])) for i in range(3))))
    assert_close(f16.astype(np.float32), f32, 5e-3, "attention f16 vs f32")


# ------------------------------------------------------------- tile edges

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("t", [1, 2, 31, 63, 65, 127, 128, 129, 257])
@pytest.mark.parametrize("s,h", [(1, 1), (3, 5), (2, 13)])
def test_attention_edges(ctx, dtype, t, s, h):
    rng = np.random.default_rng(1000 * t + 10 * s + h)
    q, k, v = (host(rng.standard_normal((s, h, t, 64)), dtype) for _ in range(3))
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    check(got, O.attention(q, k, v), f"attention t={t} s={s} h={h} {dtype}")


@pytest.mark.parametrize("scale", [0.25, 4.0])
def test_attention_f16_score_range(ctx, scale):
    """Flat (scale 0.25) and peaked (scale 4: scores of std 16) softmax."""
    rng = np.random.default_rng(77)
    s, h, t = 2, 4, 300
    q = O.to_f16(scale * rng.standard_normal((s, h, t, 64)))
    k = O.to_f16(rng.standard_normal((s, h, t, 64)))
    v = O.to_f16(rng.standard_normal((s, h, t, 64)))
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    check(got, O.attention(q, k, v), f"attention score scale {scale}")


@pytest.mark.parametrize("case", ["ramp", "spike", "mixed"])
def test_attention_f16_reference_moves(ctx, case):
    """Scores that rise from tile to tile, so that later 64-key tiles take the
    max path (a tile's weights against the kept reference would overflow
    f16): "ramp" raises every tile's scores by ~18 (log2 units), "spike" puts
    one dominant key in the last tile, "mixed" gives half the queries of each
    wave a rising and half a falling ramp (the max path then runs for the
    whole wave while half its queries keep their reference)."""
    rng = np.random.default_rng(5)
    s, h, t = 1, 2, 300
    q = np.zeros((s, h, t, 64))
    k = 0.5 * rng.standard_normal((s, h, t, 64))
    v = rng.standard_normal((s, h, t, 64))
    q[..., 0] = 8.0  # score = k[..., 0] (q.k / 8)
    if case == "spike":
        k[..., 0] += 2.0 * rng.standard_normal((s, h, t))
        k[:, :, t - 3, 0] = 120.0
    else:
        k[..., 0] += 12.5 * (np.arange(t) // 64)  # 12.5 * log2(e) = 18 per tile
        if case == "mixed":
            q[:, :, 1::2, 0] = -8.0  # odd queries: scores fall tile to tile
    q, k, v = O.to_f16(q), O.to_f16(k), O.to_f16(v)
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    check(got, O.attention(q, k, v), f"attention reference moves ({case})")


@pytest.mark.parametrize("v_scale", [1.0, 1000.0])
def test_attention_f16_row_sum_rounding_worst_case(ctx, v_scale):
    """The f16 matrix-core kernel sums each lane's weights in groups of four
    keys (the keys of one 32-key block that agree mod 8) by two levels of
    f16 additions, then in f32. Its worst case: one weight of 1 per group
    and three that f16 drops, one (just under half an f16 ulp of 1) at the
    first level beside the 1 and two (together just under it) at the
    second. Every group then loses ~1.97 * 2^-11 of its 1 + 1.97 * 2^-11,
    so l is low by ~9.6e-4 relative, and with V constant the output is high
    by as much (the numerator adds the same f16 weights in f32). Bound: at
    most 2^-10 from the two rounding levels plus 2^-11 from the output's
    f16 rounding, relative, which is also inside the f16 gate."""
    s_, h, t, d = 1, 2, 512, 64
    k = np.zeros((s_, h, t, d), np.float32)
    m32 = np.arange(t) % 32
    # scores q.k / 8 = a * 8 / 8 = a: weights exp(a) against the max 0
    a = np.where(m32 < 8, 0.0, np.where((m32 >= 16) & (m32 < 24), -7.6328125, -8.3359375))
    k[..., 0] = a
    q = np.zeros((s_, h, t, d), np.float32)
    q[..., 0] = 8.0
    v = np.full((s_, h, t, d), v_scale, np.float32)
    qh, kh, vh = (O.to_f16(x) for x in (q, k, v))
    w = np.exp2(np.float64(a) * np.log2(np.e))
    lost = w[(m32 >= 8)].reshape(-1)  # every non-dominant weight is dropped by the f16 sums
    assert np.all(w[(m32 >= 16) & (m32 < 24)] < 2.0 ** -11), "first-level weight below half an ulp"
    assert np.all(2 * w[(m32 >= 8) & (m32 < 16)] < 2.0 ** -11), "second-level pair below half an ulp"
    got = back(ctx.attention(dev(qh), dev(kh), dev(vh))).astype(np.float64)
    want = naive64(qh, kh, vh)
    rel = np.abs(got - want) / np.abs(want)
    # the construction reaches the bound's order: l low by ~lost / total
    assert rel.max() > 0.5 * lost.sum() / w.sum(), "the worst case did not show"
    assert rel.max() <= 2.0 ** -10 + 2.0 ** -11, f"row-sum rounding {rel.max():.3g} beyond its bound"
    f16_close(got.astype(np.float32), want.astype(np.float32), "row-sum worst case")


@pytest.mark.parametrize("case", range(24))
def test_attention_f16_random_sweep(ctx, case):
    """Seeded random shapes and score statistics against float32 torch: T
    from 1 to 3000 (partial tiles of every size), 1-4 sequences x 1-5
    heads, score scales from flat to peaked, and in half the cases a drift
    that raises or lowers the scores along the keys by a random amount per
    64-key tile, so that the max path runs at random tiles and not only at
    the first."""
    rng = np.random.default_rng(1000 + case)
    s, h = int(rng.integers(1, 5)), int(rng.integers(1, 6))
    t = int(rng.integers(1, 3001))
    scale = float(rng.choice([0.1, 0.5, 1.0, 2.0, 4.0]))
    q = scale * rng.standard_normal((s, h, t, 64))
    k = rng.standard_normal((s, h, t, 64))
    v = rng.standard_normal((s, h, t, 64))
    if case % 2:
        # every query leans on one direction u; key j moves along u by a
        # random walk over the tiles, so its scores move by ~2 * drift
        u = rng.standard_normal(64)
        u /= np.linalg.norm(u)
        q = q + 2.0 * u
        drift = rng.normal(0.0, 6.0, -(-t // 64)).cumsum()
        k = k + (4.0 * drift[np.arange(t) // 64])[None, None, :, None] * u
    q, k, v = (dev(O.to_f16(a)) for a in (q, k, v))
    got = back(ctx.attention(q, k, v)).astype(np.float32)
    ref = back(torch_attention32(q, k, v))
    f16_close(got, ref, f"attention sweep case {case}: s={s} h={h} t={t} scale={scale}")


@pytest.mark.parametrize("t", [257, 300, 511])
def test_attention_partial_tile_launch(ctx, t):
    """32 sequences x 16 heads with a partial last 256-query tile: the tile
    runs as its own launch with the waves past T idle (t = 257 leaves one
    live query in it), plain and merged outputs against float32 torch."""
    s, h = 32, 16
    q, k, v = rand_qkv(t, (s, h, t, 64), torch.float16)
    got = ctx.attention(q, k, v)
    f16_close(back(got).astype(np.float32), back(torch_attention32(q, k, v)),
              f"partial-tile launch t={t}")
    assert_bit_exact(back(ctx.attention_merged(q, k, v)), back(ctx.attn_merge(got)),
                     f"partial-tile launch merged t={t}")


# ------------------------------------------- f32 head_dim 64 (matrix cores)

@pytest.mark.parametrize("scale", [0.25, 4.0])
def test_attention_f32_score_range(ctx, scale):
    """Flat (scale 0.25) and peaked (scale 4: scores of std 16) softmax in
    f32, against the oracle and the float64 softmax."""
    rng = np.random.default_rng(78)
    s, h, t = 2, 4, 300
    q = (scale * rng.standard_normal((s, h, t, 64))).astype(np.float32)
    k, v = (rng.standard_normal((s, h, t, 64)).astype(np.float32) for _ in range(2))
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    check(got, O.attention(q, k, v), f"f32 attention score scale {scale}")
    assert np.abs(got - naive64(q, k, v)).max() < 1e-4


@pytest.mark.parametrize("case", ["ramp", "falling", "spike"])
def test_attention_f32_running_max(ctx, case):
    """Scores that rise from one 64-key tile to the next by ~18 (log2
    units), so every tile rescales what came before; that fall, so the first
    tile's max holds; and one dominant key in the last tile."""
    rng = np.random.default_rng(6)
    s, h, t = 1, 2, 300
    q = np.zeros((s, h, t, 64))
    k = 0.5 * rng.standard_normal((s, h, t, 64))
    v = rng.standard_normal((s, h, t, 64))
    q[..., 0] = 8.0  # score = k[..., 0] (q.k / 8)
    if case == "spike":
        k[:, :, t - 3, 0] = 120.0
    else:
        k[..., 0] += (12.5 if case == "ramp" else -12.5) * (np.arange(t) // 64)
    q, k, v = (a.astype(np.float32) for a in (q, k, v))
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    check(got, O.attention(q, k, v), f"f32 attention running max ({case})")
    assert np.abs(got - naive64(q, k, v)).max() < 1e-4


def test_attention_f32_unaligned_takes_generic(ctx):
    """Inputs 4 bytes off 16-byte alignment take the generic kernel: the
    same results within the f32 bar."""
    rng = np.random.default_rng(79)
    s, h, t = 1, 3, 100
    q, k, v = (rng.standard_normal((s, h, t, 64)).astype(np.float32) for _ in range(3))
    want = O.attention(q, k, v)
    bufs = [torch.zeros(a.size + 1, dtype=torch.float32, device="cuda:0") for a in (q, k, v)]
    views = []
    for b_, a in zip(bufs, (q, k, v)):
        b_[1:].copy_(torch.from_numpy(a.reshape(-1)))
        views.append(b_[1:].view(s, h, t, 64))
    assert views[0].data_ptr() % 16 != 0
    check(back(ctx.attention(*views)), want, "f32 attention, unaligned inputs")


@pytest.mark.parametrize("s,t", [(2, 1374), (1, 2748), (16, 782)])
def test_attention_f32_block_shapes(ctx, s, t):
    """The f32 block's frame and global attention at S=2 (2 x 1374 tokens)
    and the 21x37 frame (782 tokens), 16 heads: every query against a
    float64 softmax on the device, sampled queries against the oracle,
    and the merged output bit-exact against the merge of the plain one."""
    q, k, v = rand_qkv(s * 10000 + t, (s, 16, t, 64), torch.float32)
    got = ctx.attention(q, k, v)
    sc = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) / 8.0
    ref = torch.matmul(torch.softmax(sc, dim=-1), v.double())
    err = (got.double() - ref).abs().max().item()
    assert err < 1e-4, f"f32 attention ({s}, 16, {t}): max error {err} against float64"
    rows = np.array([0, 1, 31, 32, 127, 128, t - 1])
    qs, ks, vs = back(q), back(k), back(v)
    check(back(got)[:, :, rows], O.attention(qs, ks, vs, rows), f"f32 attention ({s}, 16, {t}) vs oracle")
    assert_bit_exact(back(ctx.attention_merged(q, k, v)), back(ctx.attn_merge(got)),
                     f"f32 attention merged ({s}, 16, {t})")
    del sc, ref


def test_attention_d128_f32(ctx):
    """The camera head's head_dim 128 (f32 only, engine/ops.rs:233-238)."""
    rng = np.random.default_rng(128)
    q, k, v = (rng.standard_normal((1, 2, 40, 128)).astype(np.float32) for _ in range(3))
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    check(got, O.attention(q, k, v), "attention d128")
    assert np.abs(got - naive64(q, k, v)).max() < 1e-4


@pytest.mark.parametrize("s,h,t", [(1, 16, 1), (2, 3, 15), (1, 16, 16), (3, 2, 17), (1, 4, 63),
                                   (1, 4, 64), (1, 2, 65), (2, 16, 200)])
@pytest.mark.parametrize("spread", [1.0, 6.0])
def test_attention_d128_f32_edges(ctx, s, h, t, spread):
    """attention_d128_kernel (16-query tiles, 16-key blocks over four waves,
    waves without keys below 49 tokens) against the float64 softmax: within
    the error of the one-thread-per-query kernel, which unaligned buffers
    take, and of 1e-5 (f32 scores of 128 products, |score| up to ~60 at the
    larger spread: 60 x 2^-23 relative on a weight)."""
    rng = np.random.default_rng(s * 100 + t)
    q, k, v = (rng.standard_normal((s, h, t, 128)).astype(np.float32) for _ in range(3))
    q *= np.float32(spread)
    want = naive64(q, k, v)
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    assert np.abs(got - want).max() < 1e-5 * spread
    merged = back(ctx.attention_merged(dev(q), dev(k), dev(v)))
    assert_bit_exact(merged.reshape(s, t, h, 128).transpose(0, 2, 1, 3).copy(), got, "merged d128")

    def odd(a):  # one float past a 16-byte boundary
        buf = torch.empty(a.size + 1, device="cuda:0")
        return buf[1:].view(a.shape).copy_(dev(a))

    ref = back(ctx.attention(odd(q), odd(k), odd(v)))
    assert np.linalg.norm(got - want) <= 1.25 * np.linalg.norm(ref - want) + 1e-7 * np.linalg.norm(want)


def test_attention_unsupported_shapes(ctx):
    x16 = torch.zeros((1, 1, 8, 128), dtype=torch.float16, device="cuda:0")
    with pytest.raises(_lib.HsError) as e:
        ctx.attention(x16, x16, x16)
    assert e.value.status == _lib.HS_EUNSUPPORTED
    x32 = torch.zeros((1, 1, 8, 32), dtype=torch.float32, device="cuda:0")
    with pytest.raises(_lib.HsError):
        ctx.attention(x32, x32, x32)
    with pytest.raises(AssertionError):
        ctx.attention(x32, x32, torch.zeros((1, 1, 9, 32), device="cuda:0"))


# ------------------------------------------------------------------ merge

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("s,h,t,d", [(2, 4, 5, 8), (2, 16, 37, 64), (1, 3, 11, 6), (3, 2, 7, 128),
                                     (1, 8, 13, 64), (3, 16, 131, 64)])
def test_attn_merge_exact(ctx, dtype, s, h, t, d):
    """Covers the token-per-wave kernel at 64, 128 and 256 vectors per token
    (odd token counts leave a half-filled wave) and the flat kernel."""
    rng = np.random.default_rng(s * 1000 + t)
    x = host(rng.standard_normal((s, h, t, d)), dtype)
    got = back(ctx.attn_merge(dev(x)))
    want = np.ascontiguousarray(x.transpose(0, 2, 1, 3).reshape(s * t, h * d))
    assert_bit_exact(got, want, f"attn_merge {dtype} {(s, h, t, d)}")
    assert_bit_exact(got, O.attn_merge(x), "attn_merge vs oracle")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("s,h,t", [(2, 3, 150), (3, 5, 65)])
def test_attention_merged_is_merge_of_attention(ctx, dtype, s, h, t):
    q, k, v = rand_qkv(s + h + t, (s, h, t, 64), dtype)
    a = ctx.attn_merge(ctx.attention(q, k, v))
    m = ctx.attention_merged(q, k, v)
    assert_bit_exact(back(m), back(a), f"attention_merged {dtype}")


# -------------------------------------------------------------- full size

def test_attention_frame_blocks_full_size(ctx):
    """Frame attention of the S=32 aggregator: (32, 16, 1374, 64) f16, every
    output against float32 torch on the same f16 inputs; two sequences
    against the oracle; the merged variant bit-exact."""
    s, h, t = 32, 16, 1374
    q, k, v = rand_qkv(32, (s, h, t, 64), torch.float16)
    got = ctx.attention(q, k, v)
    ref = torch_attention32(q, k, v)
    f16_close(back(got).astype(np.float32), back(ref), "frame attention vs torch f32")
    qs, ks, vs = (back(x)[[0, 31]][:, [0, 15]] for x in (q, k, v))
    sub = np.ascontiguousarray(back(got)[[0, 31]][:, [0, 15]])
    check(sub, O.attention(np.ascontiguousarray(qs), np.ascontiguousarray(ks),
                           np.ascontiguousarray(vs)), "frame attention vs oracle")
    merged = ctx.attention_merged(q, k, v)
    assert_bit_exact(back(merged), back(ctx.attn_merge(got)), "frame attention merged")


def test_attention_global_blocks_sampled(ctx):
    """Global attention of the S=32 aggregator: one sequence of 32*1374 =
    43968 tokens, 16 heads. Sampled queries against float32 torch and the
    oracle; constant V rows reproduce that row everywhere."""
    s, h, t = 1, 16, 32 * 1374
    q, k, v = rand_qkv(43968, (s, h, t, 64), torch.float16)
    got = back(ctx.attention(q, k, v))
    rows = torch.from_numpy(np.random.default_rng(5).choice(t, 256, replace=False)).to("cuda:0")
    ref = back(torch_attention32(q, k, v, rows))
    r = rows.cpu().numpy()
    f16_close(got[:, :, r].astype(np.float32), ref, "global attention vs torch f32")
    idx = np.sort(r[:6]).astype(np.int32)
    want = O.attention(back(q), back(k), back(v), q_idx=idx)
    check(np.ascontiguousarray(got[:, :, idx]), want, "global attention vs oracle")
    vc = v[:, :, :1].expand(s, h, t, 64).contiguous()
    out = back(ctx.attention(q, k, vc)).astype(np.float32)
    f16_close(out, np.broadcast_to(back(vc).astype(np.float32), out.shape), "constant V")


def _rel(got, want):
    return (np.linalg.norm(got - want) / np.linalg.norm(want)).item()


@pytest.mark.parametrize("s,h,t", [(1, 2, 1), (1, 3, 31), (1, 2, 64), (2, 2, 65), (1, 2, 127), (1, 1, 129),
                                   (3, 5, 200), (1, 260, 40), (1, 300, 257), (2, 130, 300)])
@pytest.mark.parametrize("spread", [1.0, 8.0])
def test_attention_f32_split_edges(ctx, s, h, t, spread):
    """flash_split_kernel at the edges of its key tiles (64; up to there with
    one buffer), query tiles (128
    and, past 256 of those, 256), and wave-dead tails: f32 precision (2^-24
    per rounding; the scores' spread of up to ~30 log2 units enters the
    weights' relative error)."""
    rng = np.random.default_rng(t)
    q, k, v = (rng.standard_normal((s, h, t, 64)).astype(np.float32) for _ in range(3))
    q *= np.float32(spread)
    want = naive64(q, k, v)
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    assert _rel(got, want) < 1.2e-6
    assert np.abs(got - want).max() < 1e-5 * max(1.0, spread)
    merged = back(ctx.attention_merged(dev(q), dev(k), dev(v)))
    assert_bit_exact(merged.reshape(s, t, h, 64).transpose(0, 2, 1, 3).copy(), got, "merged split")


@pytest.mark.parametrize("what", ["q", "k", "v", "vcol", "qrow", "krow"])
@pytest.mark.parametrize("scale", [1e-8, 1e6])
def test_attention_f32_split_ranges(ctx, what, scale):
    """Operands, V columns, query and key rows of any magnitude: the same
    relative error."""
    rng = np.random.default_rng(4)
    q, k, v = (rng.standard_normal((1, 3, 300, 64)).astype(np.float32) for _ in range(3))
    if what == "q":
        q *= np.float32(scale)
        k *= np.float32(1 / scale)
    elif what == "k":
        k *= np.float32(scale)
        q *= np.float32(1 / scale)
    elif what == "v":
        v *= np.float32(scale)
    elif what == "vcol":
        v[..., 17] *= np.float32(scale)
    elif what == "qrow":
        q[:, :, 150] *= np.float32(min(scale, 1e5))
    else:
        k[:, :, 299] *= np.float32(min(scale, 1e5))
    want = naive64(q, k, v)
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    ok = np.isfinite(want)
    assert ok.all() and np.isfinite(got).all()
    if what in ("qrow", "krow") and scale > 1:
        # scores of 1e5: their rounding alone moves weights by 1e5 x 2^-24
        assert np.abs(got - want).max() < 0.1
        rows = np.ones(300, bool)
        if what == "qrow":
            rows[150] = False
            assert _rel(got[:, :, rows], want[:, :, rows]) < 1.2e-6
    else:
        err = np.abs(got - want).max(axis=(0, 1, 2)) / np.abs(want).max(axis=(0, 1, 2))
        assert err.max() < 4e-6


def test_attention_f32_split_special_values(ctx):
    """Zero rows stay on the split path and exact; a NaN key or an infinite
    value reaches what the float64 softmax gives it to."""
    rng = np.random.default_rng(8)
    q, k, v = (rng.standard_normal((1, 2, 200, 64)).astype(np.float32) for _ in range(3))
    q[0, 0, 3] = 0
    k[0, 0] = 0  # equal scores: the mean of V
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    assert np.abs(got[0, 0] - v[0, 0].astype(np.float64).mean(0)).max() < 1e-6
    assert _rel(got, naive64(q, k, v)) < 1.2e-6
    v[0, 1, 7, 5] = np.inf
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    assert np.isposinf(got[0, 1, :, 5]).all()
    keep = np.arange(64) != 5
    assert np.isfinite(got[0, 1][:, keep]).all() and np.isfinite(got[0, 0]).all()
    k[0, 1, 9, 2] = np.nan
    got = back(ctx.attention(dev(q), dev(k), dev(v)))
    assert np.isnan(got[0, 1]).all() and np.isfinite(got[0, 0]).all()


@pytest.mark.parametrize("near,far,gap", [(1e-3, 6e4, 22.0), (1e-9, 1.0, 30.0), (1e-20, 1e-3, 60.0),
                                          (1e-28, 1e2, 65.0)])
@pytest.mark.parametrize("t", [200, 1374])
def test_attention_f32_split_wide_values(ctx, near, far, gap, t):
    """Large values under small weights beside small values under large ones:
    each weight and each value enters with f32's relative precision. A score is
    up to A = gap / ln 2 + 20 log2 units large; four accumulations of it and the
    exponent's argument round it by 2^-24 of that each, which is 5 ln 2 2^-24 A
    of the weight, below 2^-22 A (all weights are above 2^-126, where exp2
    ends)."""
    rng = np.random.default_rng(t)
    q, k, v = (rng.standard_normal((1, 8, t, 64)).astype(np.float32) for _ in range(3))
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, :, ::2, 0] = -gap  # scores lower by gap
    v *= np.float32(near)
    v[:, :, ::2] *= np.float32(far / near)
    want = naive64(q, k, v)
    mag = naive64(q, k, np.abs(v))
    err = np.abs(back(ctx.attention(dev(q), dev(k), dev(v))) - want) / mag
    assert err.max() < 2.0 ** -22 * (gap / np.log(2) + 20), err.max()


@pytest.mark.parametrize("s", [1e-2, 1e-4, 1e-6, 1e-9])
@pytest.mark.parametrize("swap", [False, True])
def test_attention_f32_split_wide_rows(ctx, s, swap):
    """Keys (or queries) with one large element that the other operand ignores
    and small ones that make the scores."""
    rng = np.random.default_rng(3)
    q, k, v = (rng.standard_normal((1, 3, 300, 64)).astype(np.float32) for _ in range(3))
    a, b = (k, q) if swap else (q, k)
    a *= np.float32(s)
    a[..., 5] = 100.0
    b *= np.float32(1 / s)
    b[..., 5] = 0.0
    assert _rel(back(ctx.attention(dev(q), dev(k), dev(v))), naive64(q, k, v)) < 1.2e-6


def test_attention_f32_split_one_key_is_its_value(ctx):
    """One token of score zero (weight one): every bit of its value, over
    magnitudes of 2^-98 to 2^49, and past both ends, where it is computed
    again."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    q, k, v = (torch.randn((40, 3, 1, 64), generator=g, device="cuda") for _ in range(3))
    q.zero_()
    v = torch.where(v.abs() < 0.5, torch.ones_like(v), v).clamp(-1.9, 1.9)
    v *= torch.exp2(torch.randint(-97, 49, v.shape, generator=g, device="cuda").float())
    v[3, 1, 0, 5], v[4, 2, 0, 6], v[5, 0, 0, 0] = 1e-35, 1e30, 0.0
    v[6, 0, 0, 1], v[7, 0, 0, 2] = 1e-39, 2.0 ** -149
    assert torch.equal(ctx.attention(q, k, v), v)


def test_attention_f32_split_queries_do_not_see_each_other(ctx):
    """A query's result follows its own row and its head's keys and values:
    beside queries that are computed again (huge, infinite, NaN) and in any
    batch (128 and 256 queries per workgroup) it keeps its bits."""
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    q, k, v = (torch.randn((34, 8, 333, 64), generator=g, device="cuda") for _ in range(3))
    whole = ctx.attention(q, k, v)
    for n in (1, 2, 17):
        assert torch.equal(ctx.attention(q[:n], k[:n], v[:n]), whole[:n]), n
    odd = q.clone()
    odd[0, :, 40] *= 1e20
    odd[0, :, 300, 7] = float("inf")
    odd[33, 3, 332, 1] = float("nan")
    keep = torch.ones((34, 8, 333), dtype=torch.bool)
    keep[0, :, 40] = keep[0, :, 300] = keep[33, 3, 332] = False
    again = ctx.attention(odd, k, v)
    assert torch.equal(again[keep], whole[keep])
    one = ctx.attention(odd[:1], k[:1], v[:1])
    assert torch.equal(one.nan_to_num(7.0), again[:1].nan_to_num(7.0))
    # scores that rise along the keys move the running max of some queries only
    rise = k * torch.linspace(0.5, 6, 333, device="cuda")[:, None]
    mixed = q * torch.logspace(-2, 0.7, 333, device="cuda")[torch.randperm(333, generator=g, device="cuda")][:, None]
    both = ctx.attention(mixed, rise, v)
    for part in (0, 1):
        some = mixed.clone()
        some[:, :, part::2] = 0
        assert torch.equal(ctx.attention(some, rise, v)[:, :, 1 - part::2], both[:, :, 1 - part::2])
    v2 = v.clone()
    v2[1, 2, 9, 3] = 1e-35  # head (1, 2) is computed again, the others not
    heads = torch.ones((34, 8), dtype=torch.bool)
    heads[1, 2] = False
    assert torch.equal(ctx.attention(q, k, v2)[heads], whole[heads])


@pytest.mark.parametrize("t", [1, 31, 33, 65, 97, 200])
@pytest.mark.parametrize("s", [1, 300])
def test_attention_f32_split_reads_its_own_rows(ctx, t, s):
    """Rows behind the last token (the next head's, and past the last head
    memory that is not the call's) reach no result: with NaN and infinities
    there every bit stays."""
    g = torch.Generator(device="cuda")
    g.manual_seed(t)
    size = s * t * 64

    def guarded(fill):
        bufs = [torch.full((size + 64 * 128,), fill, device="cuda") for _ in range(3)]
        return bufs, [b[:size].view(s, 1, t, 64) for b in bufs]

    src = [torch.randn((s, 1, t, 64), generator=g, device="cuda") for _ in range(3)]
    outs = []
    for fill in (0.0, float("nan"), float("inf")):
        _, views = guarded(fill)
        for a, b in zip(views, src):
            a.copy_(b)
        outs.append(ctx.attention(*views))
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    if s > 1:  # the next head's rows
        q, k, v = (a.clone() for a in src)
        k[1::2] = float("nan")
        v[1::2] = float("inf")
        assert torch.equal(ctx.attention(q, k, v)[::2], outs[0][::2])


@pytest.mark.parametrize("s,h,t", [(1, 2, 65), (1, 2, 129), (1, 3, 193), (2, 16, 300), (1, 16, 2100),
                                   (1, 40, 1600), (1, 260, 300)])
@pytest.mark.parametrize("spread", [1.0, 6.0])
def test_attention_f16_small_grids(ctx, s, h, t, spread):
    """f16 grids of at most one 128-query workgroup per CU take four waves, the
    others eight (the last shapes). Against the float64 softmax of the f16
    values: weights and the result round to f16."""
    rng = np.random.default_rng(h * 1000 + t)
    q, k, v = (rng.standard_normal((s, h, t, 64)).astype(np.float16) for _ in range(3))
    q *= np.float16(spread)
    # keys that rise along the sequence: the running max moves
    k[:, :, t // 2:] *= np.float16(1.5)
    got = back(ctx.attention(dev(q), dev(k), dev(v))).astype(np.float64)
    heads = [0, h - 1]
    want = naive64(q[:, heads].astype(np.float32), k[:, heads].astype(np.float32), v[:, heads].astype(np.float32))
    assert np.abs(got[:, heads] - want).max() < 4e-3
    assert _rel(got[:, heads], want) < 1e-3


@pytest.mark.parametrize("t", [1, 33, 64, 65, 127, 129, 257, 1386])
def test_attention_f16_alone_is_the_batch(ctx, t):
    """A sequence's result does not follow the grid: alone (four waves per
    workgroup), in a batch past one workgroup per CU (eight) and past two
    (a partial last tile in a launch of its own) bit for bit the same."""
    heads = 16
    g = torch.Generator(device="cuda")
    g.manual_seed(t)
    q, k, v = (torch.randn((33, heads, t, 64), generator=g, device="cuda").half() for _ in range(3))
    q *= 4.0
    whole = ctx.attention(q, k, v)
    for s in (1, 2, 17):
        part = ctx.attention(q[:s], k[:s], v[:s])
        assert torch.equal(part, whole[:s]), s
    one = ctx.attention(q[:1, :1].contiguous(), k[:1, :1].contiguous(), v[:1, :1].contiguous())
    assert torch.equal(one[0, 0], whole[0, 0])
