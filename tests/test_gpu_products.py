"""Products with few output tiles (gemm_rows.hip) and large fp32 products on the bf16 matrix
cores (gemm_split.hip), against float64 sums of the same inputs.

Bars: fp32 max_rel 2e-6 sqrt(K / 256) + 2e-6 (fp32 sums of K terms: K 2^-24 at worst, sqrt(K)
2^-24 in practice; activations and the output add a few ulps); bf16 outputs are rounded once,
so max_rel 2^-8 plus the fp32 part, doubled."""
import ctypes

import numpy as np
import pytest

from oracle import numpy_ref as ref

pytestmark = pytest.mark.gpu

F32 = np.float32


@pytest.fixture(scope="module")
def xp():
    import tl_hip
    tl_hip.ctx()
    return tl_hip


class _Rows(ctypes.Structure):
    _fields_ = [("tile", ctypes.c_int), ("splits", ctypes.c_int), ("us", ctypes.c_float)]


class _Split(ctypes.Structure):
    _fields_ = [("tile", ctypes.c_int), ("full", ctypes.c_int), ("splits", ctypes.c_int),
                ("us", ctypes.c_float)]


def plan(xp, dt, M, N, K, cus=256):
    """What tl_gemm makes of an unbatched [M, K] x [N, K] product with a plain tile hint: ("rows",
    tile, splits), ("split", tile, whole tiles, splits), or None for the other kernels."""
    def call(symbol, result, *more):
        f = getattr(xp.load_library(), symbol)
        f.restype, f.argtypes = result, [ctypes.c_int64] * 3 + [ctypes.c_int] + [ctypes.c_bool] * len(more)
        return f(M, N, K, cus, *more)
    if dt == "bf16":
        r = call("_ZN2tl14gemm_rows_planElllib", _Rows, True)
        return ("rows", r.tile, r.splits) if r.tile >= 0 else None
    r, s = call("_ZN2tl18gemm_rows_plan_f32Ellli", _Rows), call("_ZN2tl15gemm_split_planEllli", _Split)
    if r.tile >= 0 and (s.tile < 0 or r.us <= s.us):
        return ("rows", r.tile, r.splits)
    return ("split", s.tile, s.full, s.splits) if s.tile >= 0 else None


def bar(dt, K):
    return 2 * 2.0 ** -8 if dt == "bf16" else 2e-6 * (K / 256) ** 0.5 + 2e-6


def inputs(xp, dt, M, N, K, seed=0):
    rng = np.random.default_rng(seed + M * 7 + N * 3 + K)
    r = ref.round_bf16 if dt == "bf16" else (lambda a: a)
    a = r(rng.standard_normal((M, K), dtype=F32))
    w = r(rng.standard_normal((N, K), dtype=F32) / F32(K ** 0.5))
    bias = r(rng.standard_normal(N, dtype=F32))
    res = r(rng.standard_normal((M, N), dtype=F32))
    return a, w, bias, res


# (M, N, K): one row to several tiles, last tiles of one row and one column, one to many K
# slices, K parts (the second line: too few tiles for the chip), many columns (the third)
ROWS = [(1, 65, 128), (17, 33, 64), (24, 2304, 768), (33, 130, 192), (65, 516, 320), (129, 257, 448),
        (24, 768, 3072), (100, 72, 4096), (300, 128, 2048), (90, 40, 8192),
        (20, 40008, 128), (3, 32776, 192), (128, 50257, 64), (40, 33000, 128)]


@pytest.mark.parametrize("dt", ["fp32", "bf16"])
@pytest.mark.parametrize("mnk", ROWS)
def test_few_tiles(xp, dt, mnk):
    M, N, K = mnk
    a, w, bias, res = inputs(xp, dt, M, N, K)
    da, dw, db, dres = (xp.array(t, dtype=dt) for t in (a, w, bias, res))
    y = a.astype(np.float64) @ w.astype(np.float64).T
    for kind in ("plain", "gelu", "residual"):
        out = xp.empty((M, N), dt, pitch=(N + 7) // 8 * 8)
        kw, want = {}, y
        if kind != "plain":
            kw, want = dict(bias=db), y + bias
        if kind == "gelu":
            kw["act"], want = xp.TL_ACT_GELU, ref.gelu(want).astype(np.float64)
        if kind == "residual":
            kw.update(residual=dres, ldr=N)
            want = want + res
        xp.gemm(da, dw, M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK, C=out, ldc=out.pitch, **kw)
        err = ref.max_rel(out.get(), want)
        assert err <= bar(dt, K), (dt, mnk, kind, err)


# Every tile of gemm_rows_kernel (by its number in the tile table: ring depth and K slices per stage
# 4 x 4, 3 x 2, 5 x 1, 4 x 1, 3 x 1, 2 x 1) at one stage, one short of the ring, the ring and more than
# twice the ring, whole and in K parts (even, a short last part, an empty last part).
# dtype, tile, stages, parts, (M, N, K)
RINGS = [("bf16", 0, 1, 1, (17, 33, 64)), ("bf16", 0, 3, 1, (17, 33, 576)), ("bf16", 0, 4, 1, (17, 33, 832)),
         ("bf16", 0, 9, 1, (33, 1500, 2112)), ("bf16", 0, 16, 3, (17, 2052, 12288)),
         ("bf16", 0, 9, 3, (17, 2052, 6208)), ("bf16", 0, 1, 8, (17, 33, 1600)),
         ("bf16", 1, 1, 1, (17, 8200, 64)), ("bf16", 1, 2, 1, (17, 8200, 192)), ("bf16", 1, 3, 1, (17, 8200, 320)),
         ("bf16", 1, 7, 1, (17, 8200, 832)), ("bf16", 1, 7, 5, (17, 3000, 4160)), ("bf16", 1, 11, 3, (17, 4100, 4160)),
         ("bf16", 2, 1, 1, (33, 33, 64)), ("bf16", 2, 4, 1, (33, 8200, 256)), ("bf16", 2, 5, 1, (33, 4100, 320)),
         ("bf16", 2, 11, 1, (33, 4100, 704)), ("bf16", 2, 12, 16, (513, 33, 12288)),
         ("bf16", 2, 11, 6, (65, 1000, 4160)), ("bf16", 2, 9, 16, (700, 33, 8320)), ("bf16", 2, 32, 8, (48, 2048, 16384)),
         ("bf16", 3, 1, 1, (1, 32776, 64)), ("bf16", 3, 3, 1, (1, 32776, 192)), ("bf16", 3, 4, 1, (1, 32776, 256)),
         ("bf16", 3, 9, 1, (1, 32776, 576)), ("bf16", 3, 10, 5, (18, 8200, 3200)), ("bf16", 3, 9, 12, (17, 4100, 6208)),
         ("bf16", 4, 1, 1, (33, 32776, 64)), ("bf16", 4, 2, 1, (33, 32776, 128)), ("bf16", 4, 3, 1, (33, 32776, 192)),
         ("bf16", 4, 7, 1, (33, 32776, 448)), ("bf16", 4, 17, 3, (33, 16400, 3136)),
         ("bf16", 5, 1, 1, (65, 50257, 64)), ("bf16", 5, 2, 1, (65, 50257, 128)), ("bf16", 5, 3, 1, (65, 50257, 192)),
         ("bf16", 5, 5, 1, (65, 50257, 320)), ("bf16", 5, 17, 6, (65, 8200, 6208)),
         ("fp32", 0, 1, 1, (1, 33, 32)), ("fp32", 0, 3, 1, (1, 33, 288)), ("fp32", 0, 4, 1, (1, 2052, 416)),
         ("fp32", 0, 9, 1, (16, 6000, 1056)), ("fp32", 0, 16, 3, (129, 516, 6144)), ("fp32", 0, 11, 6, (1, 1025, 8192)),
         ("fp32", 0, 2, 16, (1, 33, 3104)), ("fp32", 1, 1, 1, (1, 8200, 32)), ("fp32", 1, 2, 1, (1, 8200, 96)),
         ("fp32", 1, 3, 1, (1, 8200, 160)), ("fp32", 1, 7, 1, (1, 12000, 416)), ("fp32", 1, 8, 16, (1, 1500, 8192)),
         ("fp32", 1, 7, 3, (1, 8200, 1280)), ("fp32", 1, 3, 12, (1, 2052, 2048)), ("fp32", 2, 1, 1, (33, 33, 32)),
         ("fp32", 2, 4, 1, (33, 8200, 128)), ("fp32", 2, 5, 1, (33, 8200, 160)), ("fp32", 2, 11, 1, (33, 8200, 352)),
         ("fp32", 2, 16, 16, (513, 33, 8192)), ("fp32", 2, 11, 12, (33, 1025, 4096)), ("fp32", 2, 6, 12, (33, 1025, 2048))]


@pytest.mark.parametrize("dt,tile,stages,parts,mnk", RINGS)
def test_few_tiles_rings(xp, dt, tile, stages, parts, mnk):
    M, N, K = mnk
    assert plan(xp, dt, M, N, K) == ("rows", tile, parts)
    per_part = -(-(K // (64 if dt == "bf16" else 32)) // parts)
    assert -(-per_part // (4, 2, 1, 1, 1, 1)[tile]) == stages
    a, w, bias, res = inputs(xp, dt, M, N, K)
    out = xp.empty((M, N), dt, pitch=(N + 7) // 8 * 8)
    xp.gemm(xp.array(a, dtype=dt), xp.array(w, dtype=dt), M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK,
            C=out, ldc=out.pitch, bias=xp.array(bias, dtype=dt), residual=xp.array(res, dtype=dt), ldr=N)
    want = a.astype(np.float64) @ w.astype(np.float64).T + bias + res
    assert ref.max_rel(out.get(), want) <= bar(dt, K)


@pytest.mark.parametrize("dt", ["fp32", "bf16"])
@pytest.mark.parametrize("cfg", [(24, 1, 4, 4, 64, 40, 37, 256), (3, 21, 8, 2, 32, 64, 5, 2048),
                                 (40, 7, 4, 1, 64, 16, 8, 128), (5, 300, 2, 2, 64, 304, 0, 128),
                                 (5, 401, 8, 2, 64, 416, 7, 2048), (6, 11, 24, 24, 128, 16, 1, 832),
                                 (66, 1, 64, 64, 256, 8, 0, 192), (4, 500, 8, 8, 64, 512, 3, 256),
                                 (4, 1000, 12, 12, 64, 1008, 0, 768)])
def test_few_tiles_head_scatter(xp, dt, cfg):
    """The QKV scatter into q and a cache at an odd position (one new position per sequence,
    short odd prompts), with and without parts of K, and over the larger tiles of both kernels;
    untouched cache rows stay."""
    B, T, Hq, Hkv, D, L, pos0, K = cfg
    M, N = B * T, (Hq + 2 * Hkv) * D
    a, w, bias, _ = inputs(xp, dt, M, N, K)
    q, k, vt = (xp.empty(s, dt).fill(7) for s in ((B, Hq, T, D), (B, Hkv, L, D), (B, Hkv, D, L)))
    xp.gemm(xp.array(a, dtype=dt), xp.array(w, dtype=dt), M=M, N=N, K=K, lda=K, ldb=K,
            b_layout=xp.TL_B_NK, bias=xp.array(bias, dtype=dt),
            qkv=(q, k, vt, T, Hq, Hkv, D, L, pos0))
    y = (a.astype(np.float64) @ w.astype(np.float64).T + bias).reshape(B, T, Hq + 2 * Hkv, D)
    y = y.transpose(0, 2, 1, 3)
    kw, vw = np.full((B, Hkv, L, D), 7.0), np.full((B, Hkv, D, L), 7.0)
    kw[:, :, pos0:pos0 + T] = y[:, Hq:Hq + Hkv]
    vw[..., pos0:pos0 + T] = y[:, Hq + Hkv:].transpose(0, 1, 3, 2)
    for got, want in ((q, y[:, :Hq]), (k, kw), (vt, vw)):
        assert ref.max_rel(got.get(), want) <= bar(dt, K), cfg


@pytest.mark.parametrize("dt", ["fp32", "bf16"])
@pytest.mark.parametrize("mnk", [(24, 512, 512), (48, 1000, 4096), (100, 200, 128), (17, 66000, 64), (17, 8200, 320),
                                 (33, 16400, 3136), (65, 1000, 4160), (1281, 1538, 1024)])
def test_few_tiles_gated(xp, mnk, dt):
    M, N, K = mnk
    a, w, _, _ = inputs(xp, dt, M, N, K)
    out = xp.empty((M, N // 2), dt)
    xp.gemm(xp.array(a, dtype=dt), xp.array(w, dtype=dt), M=M, N=N, K=K, lda=K, ldb=K,
            b_layout=xp.TL_B_NK, C=out, ldc=N // 2, act=xp.TL_ACT_SILU, geglu=True)
    y = a.astype(np.float64) @ w.astype(np.float64).T
    want = ref.silu(y[:, 0::2]).astype(np.float64) * y[:, 1::2]
    assert ref.max_rel(out.get(), want) <= bar(dt, K)


# whole tiles only, a last round split over K, everything split, tails of one row and column,
# one K step
SPLIT = [(2048, 2048, 256), (1281, 3073, 96), (4000, 2304, 768), (1281, 769, 3072), (4097, 1025, 32),
         (13050, 256, 256), (6145, 1025, 32), (12289, 513, 64)]


@pytest.mark.parametrize("mnk", SPLIT)
def test_fp32_pieces(xp, mnk):
    M, N, K = mnk
    assert plan(xp, "fp32", M, N, K)[0] == "split"
    a, w, bias, res = inputs(xp, "fp32", M, N, K)
    da, dw, db, dres = (xp.array(t, dtype="fp32") for t in (a, w, bias, res))
    y = a.astype(np.float64) @ w.astype(np.float64).T
    out = xp.empty((M, N), "fp32", pitch=(N + 7) // 8 * 8)
    args = dict(M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK, C=out, ldc=out.pitch)
    xp.gemm(da, dw, **args)
    assert ref.max_rel(out.get(), y) <= bar("fp32", K)
    rel = np.linalg.norm(out.get() - y) / np.linalg.norm(y)
    assert rel <= 2.0 ** -24 * 2 * max(1.0, (K / 32) ** 0.5), rel  # 6 roundings per 32 of K
    xp.gemm(da, dw, bias=db, residual=dres, ldr=N, **args)
    assert ref.max_rel(out.get(), y + bias + res) <= bar("fp32", K)


# one product per form of gemm_split_kernel: small tiles, large tiles with the last ones split over K
FORMS = [(2048, 2048, 256), (4000, 2304, 768)]


def fp32_product(xp, a, w, tile="auto"):
    (M, K), N = a.shape, w.shape[0]
    if tile == "auto":
        assert plan(xp, "fp32", M, N, K)[0] == "split"
    out = xp.empty((M, N), "fp32")
    xp.gemm(xp.array(a, dtype="fp32"), xp.array(w, dtype="fp32"), M=M, N=N, K=K, lda=K, ldb=K,
            b_layout=xp.TL_B_NK, C=out, ldc=N, tile=tile)
    return out.get()


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("ea,ew", [(-120, 100), (-124, 123), (-136, 115), (-136, 0)])
@pytest.mark.parametrize("mnk", FORMS)
def test_fp32_pieces_tiny_beside_huge(xp, mnk, ea, ew, swap):
    """Tiny elements, whose pieces are lost in part or whole, times huge ones (ordinary sums), and
    times ordinary ones (sums of no pieces at all): as close as the fp32 MFMA, whose sums of K
    products of normal operands are within the bar of float64."""
    M, N, K = mnk
    a, w, _, _ = inputs(xp, "fp32", M, N, K)
    w *= F32(K ** 0.5)
    a, w = np.ldexp(a, ew if swap else ea), np.ldexp(w, ea if swap else ew)
    got, old = fp32_product(xp, a, w), fp32_product(xp, a, w, tile="128x128")
    want = a.astype(np.float64) @ w.astype(np.float64).T
    floor = K * 2.0 ** -149 / np.abs(want).max()  # of sums that are fp32 denormals
    assert ref.max_rel(got, old) <= 2 * bar("fp32", K) + floor
    if ea > -126:
        assert ref.max_rel(got, want) <= bar("fp32", K) + floor


@pytest.mark.parametrize("mnk", FORMS)
def test_fp32_pieces_mixed_magnitudes(xp, mnk):
    """One tiny row against one huge column, the rest ordinary, with zero rows: every row and every
    column is as close to float64 as among its own kind."""
    M, N, K = mnk
    a, w, _, _ = inputs(xp, "fp32", M, N, K)
    a[7], w[11] = np.ldexp(a[7], -122), np.ldexp(w[11], 120)
    a[64:70], w[100] = 0, 0
    got = fp32_product(xp, a, w)
    want = a.astype(np.float64) @ w.astype(np.float64).T
    assert abs(got[7, 11] / want[7, 11] - 1) <= 1e-4  # one sum, which may cancel
    rows, cols = np.arange(M) != 7, np.arange(N) != 11
    for r, c in ((rows, cols), (rows, ~cols)):
        assert ref.max_rel(got[r][:, c], want[r][:, c]) <= bar("fp32", K)
    assert np.abs(got[7, cols] - want[7, cols]).max() <= K * 2.0 ** -149 + 1e-6 * np.abs(want[7, cols]).max()
    assert not got[64:70].any() and not got[:, 100].any()


@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1e12, 1e30])
@pytest.mark.parametrize("mnk", FORMS)
def test_fp32_pieces_scales(xp, mnk, scale):
    """Operands far from 1: sums as close as at scale 1 (the smallest are redone in fp32)."""
    M, N, K = mnk
    a, w, _, _ = inputs(xp, "fp32", M, N, K)
    a = (a * F32(scale)).astype(F32)
    assert ref.max_rel(fp32_product(xp, a, w), a.astype(np.float64) @ w.astype(np.float64).T) <= bar("fp32", K)


@pytest.mark.parametrize("mnk", [(2048, 2048, 128), (2305, 1025, 1024), (4000, 2304, 768)])
def test_fp32_pieces_not_finite(xp, mnk):
    """Infinities, NaN and values past bf16's largest give what fp32 sums give, in their rows
    and columns alone; a denormal row gives what the fp32 MFMA kernel gives."""
    M, N, K = mnk
    a, w, _, _ = inputs(xp, "fp32", M, N, K)
    a[3, 5], a[70, 0], a[700, K - 1], a[900, 7] = np.inf, -np.inf, np.nan, 3.4e38
    w[10, 9], w[600, 1] = np.inf, np.nan
    w[20] *= F32(1e-3)  # 3.4e38 stays finite there
    a[1000] = F32(1e-40)
    got, old = fp32_product(xp, a, w), fp32_product(xp, a, w, tile="128x128")  # the fp32 MFMA kernel
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ w.astype(np.float64).T
        want[np.abs(want) > 3.5e38] *= np.inf
    far = np.abs(np.abs(want) - 3.4e38) > 1e36  # not at fp32's very edge
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want) & far
    assert np.array_equal(got[inf], want[inf])
    ok = np.isfinite(want) & far & np.isfinite(got)
    assert ok.sum() >= np.isfinite(want).sum() - 4
    rows = np.ones(M, bool)
    rows[[900, 1000]] = False
    assert ref.max_rel(np.where(ok, got, 0)[rows], np.where(ok, want, 0)[rows]) <= bar("fp32", K)
    assert ref.max_rel(np.where(ok, got, 0)[900], np.where(ok, want, 0)[900]) <= bar("fp32", K)
    with np.errstate(all="ignore"):
        low = np.where(ok, got - old, 0)[1000]
    assert np.abs(low).max() <= K * 2.0 ** -149


@pytest.mark.parametrize("dt,mnk", [("bf16", (24, 768, 3072)), ("fp32", (24, 768, 3072)),
                                    ("fp32", (1281, 769, 3072)), ("bf16", (4, 32776, 4096))])
def test_parts_without_workspace(dt, mnk):
    """A fresh context whose first product is captured: the workspace cannot grow then, so the
    product takes one workgroup per tile; replays and a later eager call agree."""
    import tl_hip as xp
    M, N, K = mnk
    a, w, _, _ = inputs(xp, dt, M, N, K)
    old, xp._ctx = xp._ctx, None
    try:
        da, dw = xp.array(a, dtype=dt), xp.array(w, dtype=dt)
        out = xp.empty((M, N), dt, pitch=(N + 7) // 8 * 8)
        call = lambda: xp.gemm(da, dw, M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK, C=out,  # noqa: E731
                               ldc=out.pitch)
        assert xp.ctx().workspace_bytes() == 0
        with xp.capture() as g:
            call()
        want = a.astype(np.float64) @ w.astype(np.float64).T
        for _ in range(2):
            g.launch()
            assert ref.max_rel(out.get(), want) <= bar(dt, K)
        call()
        assert xp.ctx().workspace_bytes() > 0
        assert ref.max_rel(out.get(), want) <= bar(dt, K)
        g.destroy()
    finally:
        xp.synchronize()
        xp._ctx = old


# M, N, K, and the kernel that takes it in fp32 and in bf16 (None: the tiles of gemm.hip, or gemm_pp_kernel)
ODD_FORMS = [(21, 131, 576, "rows", "rows"), (65, 258, 4096, "rows", "rows"), (1029, 770, 1024, "rows", "rows"),
             (2051, 1030, 256, "split", "rows"), (1281, 769, 3072, "split", "rows"), (2050, 8197, 320, "split", None)]


@pytest.mark.parametrize("out_dt", ["fp32", "bf16"])
@pytest.mark.parametrize("dt", ["fp32", "bf16"])
@pytest.mark.parametrize("M,N,K,k32,k16", ODD_FORMS)
def test_odd_operand_forms(xp, M, N, K, k32, k16, dt, out_dt):
    """Rows apart by more than their length and operands that start inside a buffer (16 bytes in, the
    least that the matrix-core kernels take), outputs and residuals at odd offsets and pitches, a
    divisor, either type in and out, the residual overwritten by the result; nothing outside the
    output's rows is written."""
    got = plan(xp, dt, M, N, K)
    assert (got and got[0]) == (k32 if dt == "fp32" else k16)
    a, w, bias, res = inputs(xp, dt, M, N, K)
    if out_dt == "bf16":
        res = ref.round_bf16(res)
    y = a.astype(np.float64) @ w.astype(np.float64).T

    def strided(host, dtype, pitch, first):
        rows, cols = host.shape
        flat = np.full(first + rows * pitch, 7, F32)
        flat[first:].reshape(rows, pitch)[:, :cols] = host
        t = xp.array(flat, dtype=dtype)
        return t, xp.DeviceTensor((1,), dtype, buf=t.buf, offset=first * t.dtype.itemsize)

    step = 4 if dt == "fp32" else 8
    _, da = strided(a, dt, K + 2 * step, step)
    _, dw = strided(w, dt, K + 3 * step, step)
    db = xp.array(np.r_[F32(9), bias], dtype=dt)
    bias_at = xp.DeviceTensor((N,), dt, buf=db.buf, offset=db.dtype.itemsize)
    tol = 2 * bar(out_dt, K)  # the activation and the residual add their own roundings
    for pitch, first, in_place in ((N + 3, 1, False), (N + 1, 3, True), ((N + 11) // 8 * 8, 8, False)):
        whole, out = strided(res if in_place else np.zeros_like(res), out_dt, pitch, first)
        _, dres = strided(res, out_dt, N + 5, 3)
        xp.gemm(da, dw, M=M, N=N, K=K, lda=K + 2 * step, ldb=K + 3 * step, b_layout=xp.TL_B_NK, C=out, ldc=pitch,
                out_dtype=out_dt, bias=bias_at, act=xp.TL_ACT_SILU, divisor=2.0,
                residual=out if in_place else dres, ldr=pitch if in_place else N + 5)
        flat = whole.get()
        rows = flat[first:].reshape(M, pitch)
        want = ref.silu(y / 2 + bias).astype(np.float64) + res
        assert ref.max_rel(rows[:, :N], want) <= tol, (pitch, first)
        assert np.all(flat[:first] == 7) and np.all(rows[:, N:] == 7), (pitch, first)


def attention_exact(q, k, vt, causal, offset, Tk):
    """float64 attention of q [B, H, T, D] over the first Tk keys, heads merged [B, T, H D]."""
    q, k, v = (t.astype(np.float64) for t in (q, k[:, :, :Tk], np.swapaxes(vt[..., :Tk], 2, 3)))
    g = q.shape[1] // k.shape[1]
    k, v = np.repeat(k, g, 1), np.repeat(v, g, 1)
    s = q @ np.swapaxes(k, 2, 3) / q.shape[-1] ** 0.5
    if causal:
        T = q.shape[2]
        s = np.where(np.arange(Tk)[None] <= np.arange(T)[:, None] + offset, s, -np.inf)
    e = np.exp(s - s.max(-1, keepdims=True))
    y = (e / e.sum(-1, keepdims=True)) @ v
    return y.transpose(0, 2, 1, 3).reshape(q.shape[0], q.shape[2], -1)


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("case", [(1, 4, 2, 65, 97, 104, True, 32), (2, 2, 2, 130, 130, 136, False, 0),
                                  (1, 4, 1, 1, 300, 304, True, 299), (3, 2, 1, 33, 129, 136, True, 96),
                                  (1, 2, 2, 97, 193, 200, False, 0), (2, 3, 3, 321, 321, 328, True, 0),
                                  # head dim 32 without pairs of row blocks, below and beyond its lines
                                  (2, 2, 2, 225, 225, 232, False, 0), (3, 2, 1, 33, 257, 264, True, 224),
                                  (65, 4, 4, 64, 161, 168, True, 97), (64, 4, 4, 64, 161, 168, True, 97)])
def test_fp32_attention_pieces(xp, D, case):
    """Row blocks and key halves with remainders, grouped heads, a cache whose padding holds NaN,
    masked halves. Probabilities sum to 1, so errors are a few fp32 ulps of the values."""
    B, Hq, Hkv, T, Tk, L, causal, off = case
    rng = np.random.default_rng(T + Tk + D)
    q = rng.standard_normal((B, Hq, T, D), dtype=F32) * 2
    k, vt = (rng.standard_normal(s, dtype=F32) for s in ((B, Hkv, L, D), (B, Hkv, D, L)))
    k[:, :, Tk:], vt[..., Tk:] = np.nan, np.nan
    out = xp.empty((B, T, Hq * D), "fp32")
    xp.attention(*(xp.array(t, dtype="fp32") for t in (q, k, vt)), out, n_heads_q=Hq, n_heads_kv=Hkv,
                 divisor=float(F32(D ** 0.5)), causal=causal, offset=off, seq_k=Tk)
    assert ref.max_rel(out.get(), attention_exact(q, k, vt, causal, off, Tk)) <= 4e-6


@pytest.mark.parametrize("D", [32, 64])
def test_fp32_attention_pieces_not_finite(xp, D):
    """Rows that see an infinite score or value, a NaN, or only tiny values give what float64
    gives; a key with score -inf drops out."""
    B, H, T = 1, 2, 200
    rng = np.random.default_rng(D)
    q, k = (rng.standard_normal((B, H, T, D), dtype=F32) for _ in range(2))
    vt = rng.standard_normal((B, H, D, T), dtype=F32)
    q[..., 0] = np.abs(q[..., 0]) + F32(0.1)
    k[0, 0, 40, 0] = -np.inf         # head 0: key 40 drops out of every later row
    vt[0, 0, 3, 150] = np.inf        # and value 150 is infinite in one dimension
    vt[0, 0, 4, 180] = np.nan
    vt[0, 1] *= F32(1e-33)           # head 1: pieces of the values underflow
    out = xp.empty((B, T, H * D), "fp32")
    xp.attention(*(xp.array(t, dtype="fp32") for t in (q, k, vt)), out, n_heads_q=H, n_heads_kv=H,
                 divisor=float(F32(D ** 0.5)), causal=True, offset=0, seq_k=T)
    with np.errstate(all="ignore"):
        want = attention_exact(q, np.where(np.isinf(k), -1e300, k.astype(np.float64)), vt, True, 0, T)
    # probabilities of masked keys are 0, and 0 * inf is NaN in the oracle and within a 16-row
    # tile of the kernel: rows before the infinite and the NaN value's tiles never see them
    got = out.get()
    clean = vt.copy()
    clean[~np.isfinite(clean)] = 0
    low = attention_exact(q, np.where(np.isinf(k), -1e300, k.astype(np.float64)), clean, True, 0, T)
    want[:, :144, 3], want[:, :176, 4] = low[:, :144, 3], low[:, :176, 4]
    assert np.array_equal(np.isnan(got[0, 180:, 4]), np.isnan(want[0, 180:, 4]))
    assert np.all(np.isposinf(got[0, 150:, 3]))
    for cols in (slice(0, 3), slice(5, D), slice(D, 2 * D)):
        assert ref.max_rel(got[..., cols], want[..., cols]) <= 4e-6, cols
    assert ref.max_rel(got[0, :144, 3], want[0, :144, 3]) <= 4e-6
    assert ref.max_rel(got[0, :176, 4], want[0, :176, 4]) <= 4e-6


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("eq,ek", [(-122, 122), (-136, 124), (-104, 100)])
@pytest.mark.parametrize("D", [32, 64])
def test_fp32_attention_pieces_tiny_beside_huge(xp, D, eq, ek, swap):
    """Tiny queries against huge keys, or the other way round: ordinary scores (their products carry
    one rounding of each operand, which the inputs already hold), so ordinary outputs."""
    B, H, T = 2, 2, 150
    rng = np.random.default_rng(D + 200 + eq)
    q, k, vt = (rng.standard_normal(s, dtype=F32) for s in ((B, H, T, D), (B, H, T + 2, D), (B, H, D, T + 2)))
    q, k = np.ldexp(q, ek if swap else eq), np.ldexp(k, eq if swap else ek)
    out = xp.empty((B, T, H * D), "fp32")
    xp.attention(*(xp.array(t, dtype="fp32") for t in (q, k, vt)), out, n_heads_q=H, n_heads_kv=H,
                 divisor=float(F32(D ** 0.5)), causal=True, offset=0, seq_k=T)
    assert ref.max_rel(out.get(), attention_exact(q, k, vt, True, 0, T)) <= 4e-6


@pytest.mark.parametrize("D", [32, 64])
def test_fp32_attention_pieces_tiny_probabilities(xp, D):
    """Values that are huge where the probabilities are tiny and 0 at the key that takes them all;
    scores of up to 124 in log2 units carry 2^-17 of themselves into such a probability. And values
    that are all tiny: outputs within fp32's denormal steps."""
    B, H, T = 1, 2, 240
    rng = np.random.default_rng(D)
    q, k = (rng.standard_normal((B, H, T, D), dtype=F32) * F32(0.05) for _ in range(2))
    vt = np.ldexp(rng.standard_normal((B, H, D, T), dtype=F32), 122)
    q[..., 0], k[..., 0], k[:, :, 0, 0] = 1, 0, F32(119 * np.log(2) * D ** 0.5)
    vt[..., 0] = 0
    vt[0, 1] = np.ldexp(rng.standard_normal((D, T), dtype=F32), -136)
    out = xp.empty((B, T, H * D), "fp32")
    xp.attention(*(xp.array(t, dtype="fp32") for t in (q, k, vt)), out, n_heads_q=H, n_heads_kv=H,
                 divisor=float(F32(D ** 0.5)), causal=False, offset=0, seq_k=T)
    got, want = out.get(), attention_exact(q, k, vt, False, 0, T)
    assert ref.max_rel(got[..., :D], want[..., :D]) <= 2.0 ** -13
    assert np.abs(got[..., D:] - want[..., D:]).max() <= 4 * 2.0 ** -149


# 256x256 tiles that fill the chip: one to many K steps (odd and even counts), remainders of rows
# and columns, more than one round, a K beyond the late-load form's
@pytest.mark.parametrize("mnk", [(8192, 2048, 256), (8192, 2048, 320), (4096, 4096, 384),
                                 (7950, 2000, 2048), (2048, 8192, 8256), (16384, 4104, 256)])
def test_half_tiles_in_turn(xp, mnk):
    M, N, K = mnk
    a, w, bias, res = inputs(xp, "bf16", M, N, K)
    da, dw, db, dres = (xp.array(t, dtype="bf16") for t in (a, w, bias, res))
    rows = np.unique(np.r_[0:3, 120:132, 250:260, M - 140:M - 120, M - 3:M])
    y = a[rows].astype(np.float64) @ w.astype(np.float64).T
    for kind in ("plain", "silu", "residual"):
        out = xp.empty((M, N), "bf16")
        kw, want = {}, y
        if kind != "plain":
            kw, want = dict(bias=db), y + bias
        if kind == "silu":
            kw["act"], want = xp.TL_ACT_SILU, ref.silu(want).astype(np.float64)
        if kind == "residual":
            kw.update(residual=dres, ldr=N)
            want = want + res[rows]
        xp.gemm(da, dw, M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK, C=out, ldc=N, **kw)
        old = xp.empty((M, N), "bf16")  # a named tile: the same sums in the same order
        xp.gemm(da, dw, M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK, C=old, ldc=N,
                tile="dma128x128", **kw)
        assert np.array_equal(out.get_raw(), old.get_raw()), (mnk, kind)
        assert ref.max_rel(out.get()[rows], want) <= bar("bf16", K), (mnk, kind)


def test_half_tiles_in_turn_scatter_and_gated(xp):
    """The QKV scatter (slabs inside one part and across parts) and the gated epilogue on the
    same tiles, bit for bit against a named tile."""
    B, T, Hq, Hkv, D, K = 32, 256, 12, 2, 128, 256
    M, N = B * T, (Hq + 2 * Hkv) * D
    a, w, bias, _ = inputs(xp, "bf16", M, N, K)
    da, dw, db = (xp.array(t, dtype="bf16") for t in (a, w, bias))
    got = []
    for tile in ("auto", "dma128x128"):
        q, k, vt = (xp.empty(s, "bf16").fill(3) for s in ((B, Hq, T, D), (B, Hkv, T, D), (B, Hkv, D, T)))
        xp.gemm(da, dw, M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK, bias=db, tile=tile,
                qkv=(q, k, vt, T, Hq, Hkv, D, T, 0))
        out = xp.empty((M, N // 2), "bf16")
        xp.gemm(da, dw, M=M, N=N, K=K, lda=K, ldb=K, b_layout=xp.TL_B_NK, C=out, ldc=N // 2, tile=tile,
                act=xp.TL_ACT_GELU, geglu=True)
        got.append([t.get_raw() for t in (q, k, vt, out)])
    for x, y in zip(*got):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("D,Hkv", [(256, 1), (128, 2), (64, 4)])
@pytest.mark.parametrize("pos", [0, 63, 64, 500, 1023])
def test_decode_trims_dead_blocks(xp, D, Hkv, pos):
    """A grid of more than one round at a device position: only live key blocks are read (the
    others hold NaN), several per workgroup, also when the position reaches the capacity; the
    rotated new key is written back."""
    B, L, Hq = 160, 1024, 8
    rng = np.random.default_rng(pos + D)
    r = ref.round_bf16
    q = r(rng.standard_normal((B, Hq, 1, D), dtype=F32))
    k, vt = (r(rng.standard_normal(s, dtype=F32)) for s in ((B, Hkv, L, D), (B, Hkv, D, L)))
    k[:, :, pos + 1:], vt[..., pos + 1:] = np.nan, np.nan
    dk = xp.array(k, dtype="bf16")
    out = xp.empty((B, 1, Hq * D), "bf16")
    xp.attention_decode_dev(xp.array(q, dtype="bf16"), dk, xp.array(vt, dtype="bf16"), out,
                            xp.array(np.array([pos], np.int64)), n_heads_q=Hq, n_heads_kv=Hkv,
                            divisor=float(F32(D ** 0.5)), rope=xp.rope_table(1, D, 10000.0, pos))
    cos, sin = ref.rope_table(1, D, 10000.0, pos)
    qr = r(ref.rope(q, cos, sin))
    k[:, :, pos:pos + 1] = r(ref.rope(k[:, :, pos:pos + 1], cos, sin))
    want = attention_exact(qr, k, vt, True, pos, pos + 1)
    assert ref.max_rel(out.get(), want) <= 2e-2
    got = dk.get()
    assert np.array_equal(np.isnan(got), np.isnan(k))
    assert ref.max_rel(np.nan_to_num(got), np.nan_to_num(k)) <= 2.0 ** -7


@pytest.mark.parametrize("D,Hq,Hkv,Tq,L,pos", [(32, 8, 8, 1, 512, 0), (32, 8, 8, 2, 512, 300), (32, 4, 2, 3, 1024, 1021),
                                              (64, 8, 2, 2, 1024, 126), (128, 4, 2, 4, 1024, 700),
                                              (256, 8, 1, 2, 1024, 1022), (64, 8, 4, 1, 512, 512), (32, 8, 8, 2, 512, 511)])
def test_decode_trims_several_positions(xp, D, Hq, Hkv, Tq, L, pos):
    """The trimmed grid with one to four query positions, at head dim 32 too, up to the last key and
    at a position that the capacity cuts off (rows past it see the keys that there are)."""
    B = -(-2100 * 64 // (Hkv * L))
    rng = np.random.default_rng(pos + D)
    q = ref.round_bf16(rng.standard_normal((B, Hq, Tq, D), dtype=F32))
    k, vt = (ref.round_bf16(rng.standard_normal(s, dtype=F32)) for s in ((B, Hkv, L, D), (B, Hkv, D, L)))
    k[:, :, pos + Tq:], vt[..., pos + Tq:] = np.nan, np.nan
    out = xp.empty((B, Tq, Hq * D), "bf16")
    xp.attention_decode_dev(*(xp.array(t, dtype="bf16") for t in (q, k, vt)), out,
                            xp.array(np.array([pos], np.int64)), n_heads_q=Hq, n_heads_kv=Hkv,
                            divisor=float(F32(D ** 0.5)))
    want = attention_exact(q, k, vt, True, pos, min(pos + Tq, L))
    assert ref.max_rel(out.get(), want) <= 2e-2
