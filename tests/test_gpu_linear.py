"""Linear layers (hs_linear, hs_linear_gelu, hs_linear_ls_residual) against
the oracle (linear.wesl restated) and, at the trunk's full shapes, against a
float32 torch product on the device.

Bars: f32 within 1e-5 * (1 + |e|) * 4 of the oracle (the oracle sums in k
order; the kernel's order differs); f16 within 2e-3 * max(1, |e|);
small-integer inputs bit-exact (every product and partial sum is exact).
"""
import numpy as np
import pytest
import torch

from headshot_amd import _lib
from headshot_amd.parity import assert_bit_exact, assert_close, f16_close, ulp_diff_f16
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NP = {torch.float32: np.float32, torch.float16: np.float16}


def dev(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def back(t: torch.Tensor) -> np.ndarray:
    torch.cuda.synchronize()
    return t.cpu().numpy()


def check(got, want, what):
    if got.dtype == np.float32:
        assert_close(got, want, 4e-5, what)
    else:
        f16_close(got.astype(np.float32), want.astype(np.float32), what)


def operands(seed, m, n, k, dt, scale=1.0):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((m, k)) * scale).astype(dt)
    w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(dt)
    b = (rng.standard_normal(n) * 0.02).astype(np.float32)
    return x, w, b


@pytest.mark.parametrize("m,n,k", [(1, 128, 32), (37, 128, 64), (256, 256, 1024), (300, 384, 96),
                                   (513, 128, 32), (37, 48, 80), (5, 100, 40)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("with_bias", [True, False])
def test_linear_vs_oracle(ctx, m, n, k, dtype, with_bias):
    x, w, b = operands(m * 7 + n + k, m, n, k, NP[dtype])
    bias = b if with_bias else None
    got = back(ctx.linear(dev(x), dev(w), None if bias is None else dev(bias)))
    check(got, O.linear(x, w, bias), f"linear {(m, n, k)} {dtype}")


@pytest.mark.parametrize("m,n,k", [(300, 256, 128), (37, 128, 1024)])
def test_linear_f16_integers_exact(ctx, m, n, k):
    rng = np.random.default_rng(m + n + k)
    x = rng.integers(-3, 4, (m, k)).astype(np.float16)
    w = rng.integers(-3, 4, (n, k)).astype(np.float16)
    got = back(ctx.linear(dev(x), dev(w)))
    assert_bit_exact(got, O.linear(x, w), "integer linear f16")


@pytest.mark.parametrize("m,n,k", [(300, 256, 128), (37, 48, 80)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_linear_gelu_vs_reference_sequence(ctx, m, n, k, dtype):
    x, w, b = operands(m + 3 * n + k, m, n, k, NP[dtype], scale=2.0)
    got = back(ctx.linear_gelu(dev(x), dev(w), dev(b)))
    check(got, O.linear_gelu(x, w, b), f"linear_gelu {(m, n, k)} {dtype}")


@pytest.mark.parametrize("m,n,k", [(300, 256, 128), (37, 48, 80)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("in_place", [False, True])
def test_linear_ls_residual_vs_reference_sequence(ctx, m, n, k, dtype, in_place):
    x, w, b = operands(m + 5 * n + k, m, n, k, NP[dtype])
    rng = np.random.default_rng(9)
    res = rng.standard_normal((m, n)).astype(NP[dtype])
    g = rng.standard_normal(n).astype(np.float32)
    r = dev(res)
    got = ctx.linear_ls_residual(dev(x), dev(w), dev(g), r, dev(b), out=r if in_place else None)
    check(back(got), O.linear_ls_residual(x, w, g, res, b), f"linear_ls_residual {(m, n, k)}")


# the trunk's GEMMs at S=32 (43968 rows), f16
FULL = {"qkv": (3072, 1024), "proj": (1024, 1024), "fc1": (4096, 1024), "fc2": (1024, 4096)}


@pytest.mark.parametrize("name", list(FULL))
def test_linear_full_size(ctx, name):
    n, k = FULL[name]
    m = 32 * 1374
    g = torch.Generator(device="cpu").manual_seed(n + k)
    x = torch.randn((m, k), generator=g).half().to("cuda:0")
    w = (torch.randn((n, k), generator=g) / k ** 0.5).half().to("cuda:0")
    b = (torch.randn(n, generator=g) * 0.02).to("cuda:0")
    ref = (x.float() @ w.float().t().contiguous()) + b
    if name == "fc1":
        got = ctx.linear_gelu(x, w, b)
        ref = torch.nn.functional.gelu(ref.half().float())  # reference sequence: stored, then GELU
    elif name in ("proj", "fc2"):
        res = torch.randn((m, n), generator=g).half().to("cuda:0")
        # LayerScale magnitudes (the trunk's are ~1e-5 .. 0.1): with |gamma|
        # near 1, a one-ulp difference in the stored linear output (the sum
        # order differs from torch's) would already reach the f16 gate.
        gam = (torch.randn(n, generator=g) * 0.1).to("cuda:0")
        got = ctx.linear_ls_residual(x, w, gam, res, b)
        ref = res.float() + gam * ref.half().float()
    else:
        got = ctx.linear(x, w, b)
    f16_close(back(got).astype(np.float32), back(ref), f"full-size {name}")
    rows = np.array([0, 1, 255, 256, 20000, m - 1])
    xs, ws = back(x), back(w)
    if name == "qkv":
        check(back(got)[rows], O.linear(xs, ws, back(b), rows), f"full-size {name} vs oracle")


@pytest.mark.parametrize("case", range(16))
def test_linear_epilogues_random_sweep(ctx, case):
    """Seeded random shapes on the matrix-core path (n a multiple of 256, k
    of 64) and off it, each epilogue against float32 torch of the
    reference's sequence: bias; bias then GELU of the stored (f16) value;
    bias then LayerScale + residual of the stored value. m from 1 to 3000
    covers every remainder of the 256-row tile."""
    rng = np.random.default_rng(500 + case)
    m = int(rng.integers(1, 3001))
    fast = case % 4 != 3
    n = int(rng.choice([256, 512, 768, 1024])) if fast else int(rng.integers(1, 300))
    k = int(rng.choice([64, 128, 192, 512, 1024])) if fast else int(rng.integers(1, 200))
    g = torch.Generator(device="cpu").manual_seed(500 + case)
    x = torch.randn((m, k), generator=g).half().to("cuda:0")
    w = (torch.randn((n, k), generator=g) / k ** 0.5).half().to("cuda:0")
    b = (torch.randn(n, generator=g) * 0.02).to("cuda:0")
    stored = ((x.float() @ w.float().t().contiguous()) + b).half().float()
    what = f"sweep case {case}: m={m} n={n} k={k}"
    f16_close(back(ctx.linear(x, w, b)).astype(np.float32), back(stored), what + " bias")
    f16_close(back(ctx.linear_gelu(x, w, b)).astype(np.float32),
              back(torch.nn.functional.gelu(stored)), what + " gelu")
    res = torch.randn((m, n), generator=g).half().to("cuda:0")
    gam = (torch.randn(n, generator=g) * 0.1).to("cuda:0")
    f16_close(back(ctx.linear_ls_residual(x, w, gam, res, b)).astype(np.float32),
              back(res.float() + gam * stored), what + " layerscale")


# f32 shapes on the f32 matrix-core kernel (n % 128 == 0, k % 32 == 0): 64
# x 128 tiles below 512 tiles of 128 x 128, 128 x 128 tiles from there.
# Narrow: a last row tile of 56 rows; of 19 rows; one k stage (k = 32) with
# a last row tile of one row; an odd stage count; a single column tile (n =
# 128) with 2 stages (the smaller shapes of the tests above with n % 128 ==
# 0 and k % 32 == 0 run on it too). 128 x 128: a last row tile of 57 rows
# and 3 stages; one stage and a last row tile of one row; an odd stage
# count and n = 1024. Long k on few tiles: 16 x 8 tiles at k = 2048; 5 x 2
# tiles at k = 2080 (65 stages).
F32_MATRIX = [(3000, 2048, 64), (6163, 1024, 96), (6145, 1024, 32), (24577, 256, 160),
              (2815, 128, 64), (12345, 768, 96), (8193, 1024, 32), (8300, 1024, 160),
              (1000, 1024, 2048), (301, 256, 2080)]


@pytest.mark.parametrize("m,n,k", F32_MATRIX)
def test_linear_f32_matrix_core_epilogues(ctx, m, n, k):
    x, w, b = operands(m + 11 * n + k, m, n, k, np.float32, scale=2.0)
    rng = np.random.default_rng(m + k)
    res = rng.standard_normal((m, n)).astype(np.float32)
    g = (rng.standard_normal(n) * 0.5).astype(np.float32)
    y = O.linear(x, w, b)
    xd, wd, bd = dev(x), dev(w), dev(b)
    check(back(ctx.linear(xd, wd, bd)), y, f"f32 linear {(m, n, k)}")
    check(back(ctx.linear(xd, wd)), O.linear(x, w), f"f32 linear without bias {(m, n, k)}")
    check(back(ctx.linear_gelu(xd, wd, bd)), O.gelu(y), f"f32 linear_gelu {(m, n, k)}")
    want = O.residual_ls(res, y, g)
    check(back(ctx.linear_ls_residual(xd, wd, dev(g), dev(res), bd)), want,
          f"f32 linear_ls_residual {(m, n, k)}")
    r = dev(res)
    ctx.linear_ls_residual(xd, wd, dev(g), r, bd, out=r)
    check(back(r), want, f"f32 linear_ls_residual in place {(m, n, k)}")


@pytest.mark.parametrize("case", range(12))
def test_linear_f32_random_sweep(ctx, case):
    """Seeded random f32 shapes on the f32 matrix-core kernel, each epilogue
    against a float64 product on the device; m from 1 to 3000 covers every
    remainder of the 128-row tile."""
    rng = np.random.default_rng(900 + case)
    m = int(rng.integers(1, 3001))
    n = int(rng.choice([128, 256, 384, 640, 1024]))
    k = int(rng.choice([32, 64, 96, 160, 512, 1024]))
    g = torch.Generator(device="cpu").manual_seed(900 + case)
    x = torch.randn((m, k), generator=g).to("cuda:0")
    w = (torch.randn((n, k), generator=g) / k ** 0.5).to("cuda:0")
    b = (torch.randn(n, generator=g) * 0.02).to("cuda:0")
    res = torch.randn((m, n), generator=g).to("cuda:0")
    gam = torch.randn(n, generator=g).to("cuda:0")
    y = x.double() @ w.double().t().contiguous() + b.double()
    what = f"f32 sweep case {case}: m={m} n={n} k={k}"
    check(back(ctx.linear(x, w, b)), back(y), what + " bias")
    check(back(ctx.linear_gelu(x, w, b)), back(torch.nn.functional.gelu(y)), what + " gelu")
    check(back(ctx.linear_ls_residual(x, w, gam, res, b)), back(res.double() + gam.double() * y),
          what + " layerscale")


def test_linear_f32_integers_exact(ctx):
    """Small-integer f32 operands on the f32 matrix-core kernel: every
    product and partial sum is an integer below 2^24, so any summation order
    gives the oracle's value exactly."""
    m, n, k = 6000, 1024, 256
    rng = np.random.default_rng(77)
    x = rng.integers(-3, 4, (m, k)).astype(np.float32)
    w = rng.integers(-3, 4, (n, k)).astype(np.float32)
    assert_bit_exact(back(ctx.linear(dev(x), dev(w))), O.linear(x, w), "integer linear f32")


@pytest.mark.parametrize("name", ["qkv", "fc1", "fc2"])
def test_linear_f32_full_size(ctx, name):
    """The trunk's f32 products at S=32 (43968 rows) on the f32 matrix-core
    kernel against a float64 product on the device, and sampled rows
    against the oracle."""
    n, k = FULL[name]
    n = n // 3 if name == "qkv" else n  # the f32 q|k|v runs one product per third
    m = 32 * 1374
    g = torch.Generator(device="cpu").manual_seed(n + k + 1)
    x = torch.randn((m, k), generator=g).to("cuda:0")
    w = (torch.randn((n, k), generator=g) / k ** 0.5).to("cuda:0")
    b = (torch.randn(n, generator=g) * 0.02).to("cuda:0")
    ref = x.double() @ w.double().t().contiguous() + b.double()
    if name == "fc1":
        got = ctx.linear_gelu(x, w, b)
        ref = torch.nn.functional.gelu(ref)
    elif name == "fc2":
        res = torch.randn((m, n), generator=g).to("cuda:0")
        gam = (torch.randn(n, generator=g) * 0.1).to("cuda:0")
        got = ctx.linear_ls_residual(x, w, gam, res, b)
        ref = res.double() + gam.double() * ref
    else:
        got = ctx.linear(x, w, b)
    torch.cuda.synchronize()
    err = ((got.double() - ref).abs() / (ref.abs() + 1)).max().item()
    assert err < 4e-5, f"f32 full-size {name}: max relative error {err}"
    rows = np.array([0, 1, 255, 256, 20000, m - 1])
    xs, ws, bs = back(x), back(w), back(b)
    y = O.linear(xs, ws, bs, rows)
    if name == "fc1":
        want = O.gelu(y)
    elif name == "fc2":
        want = O.residual_ls(back(res)[rows], y, back(gam))
    else:
        want = y
    check(back(got)[rows], want, f"f32 full-size {name} vs oracle")
    del ref


def test_linear_contract(ctx):
    x = torch.zeros((4, 32), dtype=torch.float16, device="cuda:0")
    with pytest.raises(AssertionError):
        ctx.linear(x, torch.zeros((128, 16), dtype=torch.float16, device="cuda:0"))
    with pytest.raises(AssertionError):
        ctx.linear(x, torch.zeros((128, 32), dtype=torch.float32, device="cuda:0"))
    w = torch.zeros((128, 32), dtype=torch.float16, device="cuda:0")
    with pytest.raises(_lib.HsContractError):
        _lib.check(ctx.lib.hs_linear_ls_residual(torch.cuda.current_stream().cuda_stream, _lib.HS_F16,
                                                 x.data_ptr(), w.data_ptr(), None, None,
                                                 x.data_ptr(), x.data_ptr(), 4, 128, 32),
                   "linear_ls_residual")


# ---------------------------------------------------- fused q|k|v projection

def qkv_sequence(ctx, x, w, b, s, t, h, qn, kn, rope, eps):
    """The unfused sequence: linear per third, then qknorm_rope (q, k) or the
    plain head split (v)."""
    hd = h * 64
    outs = []
    for i, norm in enumerate((qn, kn, None)):
        proj = ctx.linear(x, w[i * hd:(i + 1) * hd], None if b is None else b[i * hd:(i + 1) * hd])
        outs.append(ctx.qknorm_rope(proj, s, t, h, 64, norm=norm, rope=rope if i < 2 else None,
                                    eps=eps))
    return outs


def qkv_case(seed, s, t, h, k, norm, prefix):
    from headshot_amd import rope as rp
    g = torch.Generator(device="cpu").manual_seed(seed)
    x = torch.randn((s * t, k), generator=g).half().to("cuda:0")
    w = (torch.randn((3 * h * 64, k), generator=g) / k ** 0.5).half().to("cuda:0")
    b = (torch.randn(3 * h * 64, generator=g) * 0.02).to("cuda:0")
    nrm = lambda: ((1 + 0.1 * torch.randn(64, generator=g)).to("cuda:0"),  # noqa: E731
                   (0.1 * torch.randn(64, generator=g)).to("cuda:0"))
    qn, kn = (nrm(), nrm()) if norm else (None, None)
    rope = None
    if prefix is not None:
        sin, cos = (torch.from_numpy(a).to("cuda:0") for a in rp.tables(rp.periods(), 1, t - prefix))
        rope = (sin, cos, prefix)
    return x, w, b, qn, kn, rope


# (s, t, h, k, QK-norm, RoPE prefix or None); t = 3 and 1 are shorter than
# the epilogue's 8-row step (its token counter wraps within a step)
QKV_CASES = [(2, 41, 16, 256, True, 5), (1, 300, 16, 1024, True, None), (3, 20, 8, 64, False, 17),
             (50, 3, 8, 128, True, 1), (1, 1, 8, 64, True, None), (5, 77, 32, 192, False, None),
             (7, 30, 4, 128, True, 3), (4, 9, 12, 64, True, None)]


@pytest.mark.parametrize("s,t,h,k,norm,prefix", QKV_CASES)
def test_linear_qkv_heads_is_the_sequence(ctx, s, t, h, k, norm, prefix):
    """hs_linear_qkv_heads against hs_linear + hs_qknorm_rope per third:
    bit-exact where hs_qknorm_rope runs its row kernel (8, 16 or 32 heads:
    the same head-vector code), within one f16 ulp where it runs its generic
    kernel (other head counts: another reduction order); q against the
    oracle's reference sequence (linear.wesl, split_heads, layernorm,
    rope_apply) within the f16 gate."""
    x, w, b, qn, kn, rope = qkv_case(s * 1000 + t, s, t, h, k, norm, prefix)
    got = ctx.linear_qkv_heads(x, w, b, s, t, h, qn=qn, kn=kn, rope=rope, eps=1e-5)
    want = qkv_sequence(ctx, x, w, b, s, t, h, qn, kn, rope, 1e-5)
    for name, a, e in zip("qkv", got, want):
        assert tuple(a.shape) == (s, h, t, 64)
        what = f"{name} {(s, t, h, k, norm, prefix)}"
        if h in (8, 16, 32) or name == "v":
            assert_bit_exact(back(a), back(e), what)
        else:
            assert ulp_diff_f16(back(a), back(e)).max() <= 1, what
    qproj = O.linear(back(x), back(w[:h * 64]), back(b[:h * 64]))
    tabs = (None, None, 0) if rope is None else (back(rope[0]), back(rope[1]), prefix)
    qo = O.qknorm_rope(qproj, *(tuple(back(a) for a in qn) if qn else (None, None)),
                       tabs[0], tabs[1], s, t, h, 64, tabs[2], 1e-5)
    f16_close(back(got[0]).astype(np.float32), qo.astype(np.float32), "q vs oracle")


def test_linear_qkv_heads_full_size_frame(ctx):
    """The S=32 frame block's projection (43,968 tokens, 37x37 grid, prefix
    5, 16 heads, dim 1024) bit-exact against the unfused sequence."""
    from headshot_amd import rope as rp
    s, t, h, k = 32, 1374, 16, 1024
    g = torch.Generator(device="cpu").manual_seed(77)
    x = torch.randn((s * t, k), generator=g).half().to("cuda:0")
    w = (torch.randn((3 * h * 64, k), generator=g) / k ** 0.5).half().to("cuda:0")
    b = (torch.randn(3 * h * 64, generator=g) * 0.02).to("cuda:0")
    qn = (torch.ones(64, device="cuda:0") * 1.1, torch.full((64,), 0.05, device="cuda:0"))
    kn = (torch.ones(64, device="cuda:0") * 0.9, torch.full((64,), -0.05, device="cuda:0"))
    sin, cos = (torch.from_numpy(a).to("cuda:0") for a in rp.tables(rp.periods(), 37, 37))
    got = ctx.linear_qkv_heads(x, w, b, s, t, h, qn=qn, kn=kn, rope=(sin, cos, 5), eps=1e-6)
    want = qkv_sequence(ctx, x, w, b, s, t, h, qn, kn, (sin, cos, 5), 1e-6)
    for name, a, e in zip("qkv", got, want):
        assert torch.equal(a, e), f"full-size {name}"


@pytest.mark.parametrize("s,t,h,k,norm,prefix", QKV_CASES)
def test_linear_qkv_heads_f32_is_the_sequence(ctx, s, t, h, k, norm, prefix):
    """The f32 q|k|v epilogue (f32 matrix-core kernel) against hs_linear +
    hs_qknorm_rope per third: bit-exact where hs_qknorm_rope runs its row
    kernel (8, 16 or 32 heads: the same head-vector code in the same lane
    layout), within 1e-6 relative where it runs its generic kernel (another
    reduction order); q against the oracle's reference sequence within the
    f32 bar."""
    x, w, b, qn, kn, rope = qkv_case(s * 1000 + t + 1, s, t, h, k, norm, prefix)
    x, w = x.float(), w.float()
    got = ctx.linear_qkv_heads(x, w, b, s, t, h, qn=qn, kn=kn, rope=rope, eps=1e-5)
    want = qkv_sequence(ctx, x, w, b, s, t, h, qn, kn, rope, 1e-5)
    for name, a, e in zip("qkv", got, want):
        assert tuple(a.shape) == (s, h, t, 64) and a.dtype == torch.float32
        what = f"f32 {name} {(s, t, h, k, norm, prefix)}"
        if h in (8, 16, 32) or name == "v":
            assert_bit_exact(back(a), back(e), what)
        else:
            assert_close(back(a), back(e), 1e-6, what)
    qproj = O.linear(back(x), back(w[:h * 64]), back(b[:h * 64]))
    tabs = (None, None, 0) if rope is None else (back(rope[0]), back(rope[1]), prefix)
    qo = O.qknorm_rope(qproj, *(tuple(back(a) for a in qn) if qn else (None, None)),
                       tabs[0], tabs[1], s, t, h, 64, tabs[2], 1e-5)
    check(back(got[0]), qo, "f32 q vs oracle")


def test_linear_qkv_heads_f32_block_shape(ctx):
    """The S=2 f32 frame block's projection (2 x 1374 tokens, 37x37 grid,
    prefix 5, 16 heads, dim 1024: 64 x 128 tiles) and the same at 8 frames
    (128 x 128 tiles), bit-exact against the unfused sequence."""
    from headshot_amd import rope as rp
    sin, cos = (torch.from_numpy(a).to("cuda:0") for a in rp.tables(rp.periods(), 37, 37))
    for s in (2, 8):
        x, w, b, qn, kn, _ = qkv_case(77 + s, s, 1374, 16, 1024, True, None)
        x, w = x.float(), w.float()
        got = ctx.linear_qkv_heads(x, w, b, s, 1374, 16, qn=qn, kn=kn, rope=(sin, cos, 5), eps=1e-6)
        want = qkv_sequence(ctx, x, w, b, s, 1374, 16, qn, kn, (sin, cos, 5), 1e-6)
        for name, a, e in zip("qkv", got, want):
            assert_bit_exact(back(a), back(e), f"f32 {name} at S={s}")


def test_linear_qkv_heads_fallback_f32(ctx):
    """f32 shapes the fused kernel does not cover (3 * H * 64 not a multiple
    of 128: H odd) run the unfused sequence; the C entry point refuses them."""
    x, w, b, qn, kn, rope = qkv_case(3, 2, 41, 3, 64, True, 5)
    x, w = x.float(), w.float()
    got = ctx.linear_qkv_heads(x, w, b, 2, 41, 3, qn=qn, kn=kn, rope=rope)
    want = qkv_sequence(ctx, x, w, b, 2, 41, 3, qn, kn, rope, 1e-5)
    for a, e in zip(got, want):
        assert torch.equal(a, e)
    with pytest.raises(_lib.HsError):
        _lib.check(ctx.lib.hs_linear_qkv_heads(
            torch.cuda.current_stream().cuda_stream, _lib.HS_F32, x.data_ptr(), w.data_ptr(),
            None, None, None, None, None, None, None, got[0].data_ptr(), got[1].data_ptr(),
            got[2].data_ptr(), 2, 41, 3, 64, 64, 0, 1e-5), "linear_qkv_heads")


@pytest.mark.parametrize("k", [64, 128, 192, 320, 1024])
@pytest.mark.parametrize("n", [256, 1024])
def test_linear_f16_tile_shapes_agree(ctx, n, k):
    """The tile shape follows the tile count (64 x 64, 128 x 128 with four
    and two stages, 192 x 256, 256 x 256 at 256 CUs and n = 1024) and sums k
    in one order: rows of a call of any size equal the same rows of a larger
    one, at the edges and remainders of every shape and with fewer k stages
    than a shape has buffers. The largest is checked against the float64
    product: f32 sums of k f16 products and one f16 rounding (2^-11)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    m_max = 12290 * 1024 // n if n < 1024 else 12290
    x = torch.randn((m_max, k), generator=g, device="cuda").half()
    w = (torch.randn((n, k), generator=g, device="cuda") / k ** 0.5).half()
    b = torch.randn(n, generator=g, device="cuda") * 0.02
    big = ctx.linear(x, w, b)
    want = x.double() @ w.double().t().contiguous() + b.double()
    err = (big.double() - want).abs()
    assert bool((err <= 2.0 ** -11 * want.abs() + k * 2.0 ** -24 * (1.0 + want.abs())).all())
    scale = 1024 // n
    for m in (1, 63, 65, 2048 * scale, 2049 * scale, 4097 * scale, 8191 * scale, 8193 * scale,
              8192 * scale + 193):
        assert torch.equal(ctx.linear(x[:m], w, b), big[:m]), m


@pytest.mark.parametrize("n,k", [(128, 32), (256, 96), (2048, 544), (6144, 2048), (2048, 8192)])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 33, 48, 49, 128, 129])
def test_linear_f32_few_rows(ctx, m, n, k):
    """Up to 128 rows the weights stream through gemm_skinny_kernel (tiles of
    1 to 2 x 1 to 3 blocks of 16, K over 16 waves, some without a piece at
    small k); more, and wide outputs, take the tiles. Every epilogue against float64: f32
    sums of k products (error below k 2^-24 of the sum of magnitudes, which
    is about sqrt(k) of the result's scale), and the parts of a product's
    columns equal to the whole."""
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    x, w, b, gamma, res = r(m, k), r(n, k) / k ** 0.5, r(n) * 0.02, r(n), r(m, n)
    lin = x.double() @ w.double().t().contiguous() + b.double()
    mag = x.double().abs() @ w.double().abs().t().contiguous() + 1.0
    tol = mag * (k ** 0.5 + 8) * 2.0 ** -23

    out = ctx.linear(x, w, b)
    assert bool(((out.double() - lin).abs() <= tol).all())
    half = n // 2
    if half % 128 == 0:
        assert torch.equal(ctx.linear(x, w[half:], b[half:]), out[:, half:])
    act = ctx.linear_gelu(x, w, b)
    # A&S 7.1.26: 1.5e-7 absolute on erf, times |v| / 2
    gel = torch.nn.functional.gelu(lin)
    assert bool(((act.double() - gel).abs() <= 1.2 * tol + 2e-7 * (1 + lin.abs())).all())
    want = res.double() + gamma.double() * lin
    got = ctx.linear_ls_residual(x, w, gamma, res, b, out=res)  # res may be out
    assert bool(((got.double() - want).abs() <= (1 + gamma.abs()) * tol).all())


@pytest.mark.parametrize("s,t", [(1, 1), (1, 16), (3, 17), (2, 64), (1, 129)])
@pytest.mark.parametrize("norm", [True, False])
def test_linear_f32_few_rows_heads_and_prologue(ctx, s, t, norm):
    """The same kernel's q|k|v epilogue and LayerNorm prologue, bit for bit the
    ops apart."""
    h, k = 4, 160
    g = torch.Generator(device="cuda")
    g.manual_seed(s * 1000 + t)
    r = lambda *sh: torch.randn(sh, generator=g, device="cuda")  # noqa: E731
    x, w, b = r(s * t, k), r(3 * h * 64, k) / k ** 0.5, r(3 * h * 64) * 0.02
    ln = (1 + 0.1 * r(k), 0.1 * r(k))
    nrm = lambda: (1 + 0.1 * r(64), 0.1 * r(64)) if norm else None  # noqa: E731
    qn, kn = nrm(), nrm()
    prefix = min(5, t)
    ang = r(max(t - prefix, 1), 64)
    rope = (ang.sin()[:t - prefix].contiguous(), ang.cos()[:t - prefix].contiguous(), prefix) if t > prefix else None
    got = ctx.linear_qkv_heads(x, w, b, s, t, h, qn=qn, kn=kn, rope=rope)
    lin = ctx.linear(x, w, b)
    for i, n in enumerate((qn, kn, None)):
        part = lin[:, i * h * 64:(i + 1) * h * 64].contiguous()
        want = ctx.qknorm_rope(part, s, t, h, 64, norm=n, rope=rope if i < 2 else None)
        tol = 0 if h in (8, 16, 32) else 2e-6
        assert bool(((got[i] - want).abs() <= tol * (1 + want.abs())).all())
    fused = ctx.linear_ln_qkv_heads(x, ln, w, b, s, t, h, qn=qn, kn=kn, rope=rope)
    apart = ctx.linear_qkv_heads(ctx.layernorm(x, *ln), w, b, s, t, h, qn=qn, kn=kn, rope=rope)
    for a, c in zip(fused, apart):
        assert torch.equal(a, c)
    assert torch.equal(ctx.linear_ln_gelu(x, ln, w, b), ctx.linear_gelu(ctx.layernorm(x, *ln), w, b))


@pytest.mark.parametrize("m,n", [(32, 24704), (33, 12288), (33, 12416), (64, 12288), (65, 8192), (65, 8320),
                                 (96, 8320), (97, 6144), (97, 6272), (128, 2048), (128, 6144), (128, 8192)])
def test_linear_f32_few_rows_or_wide(ctx, m, n):
    """Both sides of the line between the few-row kernel and the tiles, every
    epilogue against float64 (sums of 64 products)."""
    x, w, b = _split_operands(m, n, 64, m + n)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    gamma, res = (torch.randn(s, generator=g, device="cuda") for s in ((n,), (m, n)))
    lin = x.double() @ w.double().t().contiguous() + b.double()
    tol = (x.double().abs() @ w.double().abs().t().contiguous() + 1.0) * 16 * 2.0 ** -23
    assert bool(((ctx.linear(x, w, b).double() - lin).abs() <= tol).all())
    # A&S 7.1.26: 1.5e-7 absolute on erf, times |v| / 2
    gel = torch.nn.functional.gelu(lin)
    assert bool(((ctx.linear_gelu(x, w, b).double() - gel).abs() <= 1.2 * tol + 2e-7 * (1 + lin.abs())).all())
    want = res.double() + gamma.double() * lin
    assert bool(((ctx.linear_ls_residual(x, w, gamma, res, b).double() - want).abs() <= (1 + gamma.abs()) * tol).all())


@pytest.mark.parametrize("t", [17, 32, 64, 65, 128])
@pytest.mark.parametrize("h,d", [(16, 64), (32, 64), (44, 64), (40, 128)])
def test_linear_f32_few_rows_fused_is_apart(ctx, t, h, d):
    """q|k|v as one product and as three, over the line between the few-row
    kernel and the tiles: the same bits for 8, 16 and 32 heads of 64 and for
    heads of 128 without norms (one product and one split, or three)."""
    k, hd = 64, h * d
    x, w, b = _split_operands(t, 3 * hd, k, t + h)
    got = ctx.linear_qkv_heads(x, w, b, 1, t, h)
    for i in range(3):
        part = ctx.linear(x, w[i * hd:(i + 1) * hd], b[i * hd:(i + 1) * hd])
        want = ctx.split_heads(part, 1, t, h, d)
        if h == 44:  # 64-wide heads past 32: promised to f32's rounding only
            assert bool(((got[i] - want).abs() <= 2e-6 * (1 + want.abs())).all())
        else:
            assert torch.equal(got[i], want), i


def _split_operands(m, n, k, seed, w_scale=1.0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn((m, k), generator=g, device="cuda")
    w = torch.randn((n, k), generator=g, device="cuda") / k ** 0.5 * w_scale
    return x, w, torch.randn(n, generator=g, device="cuda") * 0.02


# (m, n): 64 x 128 tiles, 128 x 128 by 8 waves, 128 x 128 by 4 (256 CUs), with
# row remainders
@pytest.mark.parametrize("m,n", [(129, 128), (191, 1024), (2049, 1024), (2177, 2048), (4200, 1024),
                                 (5000, 3072)])
@pytest.mark.parametrize("k", [32, 64, 96, 1024])
def test_linear_f32_split(ctx, m, n, k):
    """f32 products as six bf16 ones: closer to the float64 product than a
    plain f32 chain of k / 2 terms is (relative 2-norm; 2^-24 per rounding, a
    chain's error grows with sqrt(k)), and rows and column parts of a call
    equal the same of a larger one."""
    x, w, b = _split_operands(m, n, k, m + n + k)
    out = ctx.linear(x, w, b)
    want = x.double() @ w.double().t().contiguous() + b.double()
    err = ((out.double() - want).norm() / want.norm()).item()
    assert err < 2.0 ** -24 * (1.5 + 0.12 * k ** 0.5), err
    for rows in (129, m - 1):
        if rows > 128:
            assert torch.equal(ctx.linear(x[:rows], w, b), out[:rows]), rows
    if n > 1024:
        assert torch.equal(ctx.linear(x, w[1024:], b[1024:]), out[:, 1024:])


@pytest.mark.parametrize("xs,ws", [(1e-3, 1.0), (200.0, 1e-2), (3000.0, 100.0), (1e-9, 1.0), (1.0, 1e-12),
                                   (1e6, 1.0), (1e20, 1e10)])
def test_linear_f32_split_ranges(ctx, xs, ws):
    """Operands of any magnitude: the same relative error everywhere."""
    x, w, _ = _split_operands(300, 256, 512, 5)
    x *= xs
    w *= ws
    want = x.double() @ w.double().t().contiguous()
    err = ((ctx.linear(x, w).double() - want).norm() / want.norm()).item()
    assert err < 6e-7, err


def test_linear_f32_split_mixed_rows(ctx):
    """Zero rows, tiny rows, huge rows, infinities and NaN beside ordinary
    rows, in x and in w: every row as precise as alone, non-finite values only
    where the float64 product has them."""
    x, w, b = _split_operands(400, 384, 640, 11)
    x[3] = 0
    x[140] *= 1e-20
    x[141, ::2] = 0
    x[270] *= 1e8
    x[271, 5] = float("inf")
    x[272, 7] = float("nan")
    x[399, 100] = 7e4
    w[5] *= 1e-15
    w[200] = 0
    w[383, 639] = float("-inf")
    out = ctx.linear(x, w, b).double()
    want = x.double() @ w.double().t().contiguous() + b.double()
    fin = torch.isfinite(want)
    assert torch.equal(fin, torch.isfinite(out))
    assert torch.equal(torch.isnan(want), torch.isnan(out))
    assert torch.equal(want[torch.isinf(want)], out[torch.isinf(want)])
    mag = torch.nan_to_num(x.double(), 0, 0, 0).abs() @ torch.nan_to_num(w.double(), 0, 0, 0).abs().t().contiguous()
    bound = (mag + b.abs()) * 640 ** 0.5 * 2.0 ** -23 + 1e-45
    assert bool(((out - want).abs()[fin] <= bound[fin]).all())


def test_linear_f32_split_keeps_every_bit(ctx):
    """x times the identity is x, bit for bit, over rows whose elements span 2^-100
    to 2^100, and with smaller elements, subnormals among them, which are
    computed again."""
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    x = torch.randn((300, 256), generator=g, device="cuda").clamp(-8, 8)
    x = torch.where(x.abs() < 2.0 ** -10, torch.ones_like(x), x)
    x *= torch.exp2(torch.randint(-90, 97, x.shape, generator=g, device="cuda").float())
    x[0, :4] = torch.tensor([1.0, 1e-8, 1e-10, 1e-11])
    x[1, ::3] = 0
    x[130, 7], x[131, 8], x[132] = 1e-33, -(2.0 ** -126), 2.0 ** -101
    x[133, 9], x[134, 10], x[135] = 1e-39, 2.0 ** -149, 3e-41
    x[140, 3], x[141, 4] = torch.finfo(torch.float32).max, -2.0 ** 127
    eye = torch.eye(256, device="cuda")
    assert torch.equal(ctx.linear(x, eye), x)
    xt = x[:256].contiguous()
    assert torch.equal(ctx.linear(eye, xt), xt.t())


@pytest.mark.parametrize("s", [1e-3, 1e-6, 1e-8, 1e-11, 1e-20, 1e-29, 1e-36])
def test_linear_f32_split_wide_rows(ctx, s):
    """An ordinary element that the other operand ignores beside small ones:
    the small ones' sum as precise as if they were alone (f32's precision is
    relative, 2^-24 per rounding, over chains of k / 2 terms at most)."""
    k = 512
    small, other, b = _split_operands(300, 256, k, 3, k ** 0.5)
    small, other = small * s, other.clone()
    small[:, 0], other[:, 0] = 1, 0
    for x, w in ((small, other), (other, small)):
        want = x.double() @ w.double().t().contiguous()
        err = (ctx.linear(x, w).double() - want).norm() / want.norm()
        assert err.item() < 2.0 ** -24 * (1.5 + (k / 2) ** 0.5), (s, err.item())


@pytest.mark.parametrize("c", [1 + 2.0 ** -11 - 3 * 2.0 ** -23, 1 + 2.0 ** -9 - 2.0 ** -23, 1 + 2.0 ** -8 + 2.0 ** -17 - 2.0 ** -23,
                               2 - 2.0 ** -23])
def test_linear_f32_split_equal_operands(ctx, c):
    """Every product the same, on values whose parts are largest beside the
    ones above them, so that nothing averages out: the three terms left out
    (2^-24) and a rounding each of two k slices, their small products and the
    final sum (2^-24 each)."""
    x, w = torch.full((129, 32), c, device="cuda"), torch.full((128, 32), c, device="cuda")
    want = 32 * (float(np.float32(c)) ** 2)
    err = ((ctx.linear(x, w).double() - want).abs() / want).max().item()
    assert err <= 5 * 2.0 ** -24, err


def test_linear_f32_split_rows_do_not_see_each_other(ctx):
    """An output follows its own x and w rows only, whatever shares its tile:
    beside rows that are computed again (tiny, infinite, NaN, overflowing)
    every other row keeps its bits, in tiles of 64 and of 128 rows, and the
    fused q|k|v stays the parts' products."""
    t, h, k = 1374, 16, 256  # 264 tiles of 128 rows fused, 64-row tiles for a third
    x, w, b = _split_operands(t, 3 * h * 64, k, 7)
    odd = x.clone()
    rows = [70, 71, 200, 1373]
    odd[70] *= 1e-36
    odd[71, 5] = float("inf")
    odd[200, 9] = float("nan")
    odd[1373] = 3e38
    ow = w.clone()
    cols = [65, 1500]
    ow[65, 3] = 1e-35
    ow[1500, 3] = float("inf")
    keep = torch.ones(t, dtype=torch.bool)
    keep[rows] = False
    wkeep = torch.ones(w.shape[0], dtype=torch.bool)
    wkeep[cols] = False
    part = slice(1024, 2048)
    for n in (slice(0, 3072), part):
        clean = ctx.linear(x, w[n], b[n])
        assert torch.equal(ctx.linear(odd, w[n], b[n])[keep], clean[keep])
        assert torch.equal(ctx.linear(x, ow[n], b[n])[:, wkeep[n]], clean[:, wkeep[n]])
    whole = ctx.linear(odd, ow, b)
    assert torch.equal(ctx.linear(odd, ow[part], b[part]).nan_to_num(7.0), whole[:, part].nan_to_num(7.0))
    got = ctx.linear_qkv_heads(odd, ow, b, 1, t, h)
    for i in range(3):
        want = ctx.split_heads(ctx.linear(odd, ow[i * 1024:(i + 1) * 1024], b[i * 1024:(i + 1) * 1024]), 1, t, h, 64)
        assert torch.equal(got[i].nan_to_num(7.0), want.nan_to_num(7.0))


def test_linear_f32_split_tiny_products(ctx):
    """Products near the bottom of f32's range (2^-120; their small parts are
    subnormal) keep f32's relative precision."""
    x, w, _ = _split_operands(300, 256, 64, 9, 8.0)
    x, w = x * 2.0 ** -58, w * 2.0 ** -58
    want = x.double() @ w.double().t().contiguous()
    err = ((ctx.linear(x, w).double() - want).norm() / want.norm()).item()
    assert err < 2.0 ** -24 * (1.5 + 32 ** 0.5), err


@pytest.mark.parametrize("s,t,h", [(1, 129, 4), (2, 700, 16), (3, 1400, 16)])
def test_linear_f32_split_heads_and_prologue(ctx, s, t, h):
    """The q|k|v epilogue and the LayerNorm prologue of the three tile
    shapes, bit for bit the ops apart (within 2e-6 for 4 heads)."""
    k = 256
    x, w, b = _split_operands(s * t, 3 * h * 64, k, t)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    r = lambda *sh: torch.randn(sh, generator=g, device="cuda")  # noqa: E731
    ln, qn, kn = ((1 + 0.1 * r(n), 0.1 * r(n)) for n in (k, 64, 64))
    ang = r(t - 5, 64)
    rope = (ang.sin(), ang.cos(), 5)
    got = ctx.linear_qkv_heads(x, w, b, s, t, h, qn=qn, kn=kn, rope=rope)
    hd = h * 64
    for i, n in enumerate((qn, kn, None)):
        part = ctx.linear(x, w[i * hd:(i + 1) * hd], b[i * hd:(i + 1) * hd])
        want = ctx.qknorm_rope(part, s, t, h, 64, norm=n, rope=rope if i < 2 else None)
        tol = 0 if h in (8, 16, 32) else 2e-6
        assert bool(((got[i] - want).abs() <= tol * (1 + want.abs())).all())
    xn = ctx.layernorm(x, *ln)
    for a, c in zip(ctx.linear_ln_qkv_heads(x, ln, w, b, s, t, h, qn=qn, kn=kn, rope=rope),
                    ctx.linear_qkv_heads(xn, w, b, s, t, h, qn=qn, kn=kn, rope=rope)):
        assert torch.equal(a, c)
    assert torch.equal(ctx.linear_ln_gelu(x, ln, w, b), ctx.linear_gelu(xn, w, b))


@pytest.mark.parametrize("t,h,d,k,dtype", [(8, 16, 128, 2048, torch.float32), (1, 2, 128, 64, torch.float32),
                                           (200, 4, 128, 96, torch.float32), (33, 3, 64, 100, torch.float32),
                                           (40, 8, 32, 128, torch.float16), (7, 5, 24, 40, torch.float16),
                                           (7, 1, 3, 40, torch.float16)])
@pytest.mark.parametrize("with_bias", [True, False])
def test_linear_qkv_heads_one_sequence(ctx, t, h, d, k, dtype, with_bias):
    """One sequence without norms or RoPE, shapes the fused kernel does not
    cover: one product and one split, equal to the three apart, contiguous."""
    g = torch.Generator(device="cuda")
    g.manual_seed(t + k)
    x = torch.randn((t, k), generator=g, device="cuda").to(dtype)
    w = (torch.randn((3 * h * d, k), generator=g, device="cuda") / k ** 0.5).to(dtype)
    b = torch.randn(3 * h * d, generator=g, device="cuda") * 0.02 if with_bias else None
    got = ctx.linear_qkv_heads(x, w, b, 1, t, h)
    outs = tuple(torch.empty((1, h, t, d), device="cuda", dtype=dtype) for _ in range(3))
    apart = ctx.linear_qkv_heads(x, w, b, 1, t, h, out=outs)  # given outputs: the three apart
    for a, c in zip(got, apart):
        assert a.shape == c.shape == (1, h, t, d) and a.is_contiguous() and a.data_ptr() % 16 == 0
        assert torch.equal(a, c)
