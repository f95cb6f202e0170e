"""The GEMM kernel for launches of few tiles against the closed form: the edges of its tiles, of the units its waves share K
in, of its short-K instances (one to four units per wave) and of the loop behind them."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import segq_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FORMATS = {"int8": (O.FMT_INT8, O.FMT_INT8), "e4m3": (O.FMT_E4M3, O.FMT_E4M3), "int4": (O.FMT_INT8, O.FMT_INT4)}


@pytest.fixture(scope="module")
def ops():
    from segquant_amd import ops as _ops
    _ops.L.lib()
    return _ops


def _codes(g, shape, fmt):
    if fmt == O.FMT_INT4:
        return g.integers(-8, 8, size=shape).astype(np.int8)
    if fmt == O.FMT_INT8:
        return g.integers(-128, 128, size=shape).astype(np.int8)
    c = g.integers(0, 256, size=shape).astype(np.uint8)
    c[(c & 0x7F) == 0x7F] = 0x3A  # no NaN codes
    return c


def _dev(c, fmt, pad=0):
    t = torch.from_numpy(np.stack([O.pack_int4(r) for r in c]) if fmt == O.FMT_INT4 else c).to(DEV)
    if not pad:
        return t
    wide = torch.full((t.shape[0], t.shape[1] + pad), 0x55, dtype=torch.uint8, device=DEV).view(t.dtype)  # what lies between the rows
    wide[:, :t.shape[1]] = t
    return wide[:, :t.shape[1]]


def _check(ops, kind, M, N, K, tile, dt, g, group=False, k0=0, row_sx=True, col_sw=True, has_bias=True, neg=False, add=False, pad=0):
    fa, fb = FORMATS[kind]
    a, b = _codes(g, (M, k0 + K), fa), _codes(g, (N, k0 + K), fb)
    sx = (g.random(M if row_sx else 1) * 30 + 10).astype(np.float32)
    sw = np.ones(1, np.float32) if group else (g.random(N if col_sw else 1) * 30 + 10).astype(np.float32)
    av, bv = O.code_values(a, fa)[:, k0:].astype(np.float64), O.code_values(b, fb)[:, k0:].astype(np.float64)
    gd = None
    if group:
        fac = np.zeros(((k0 + K) // 128, N), np.float32)
        fac[:] = g.random(fac.shape) * 0.09 + 0.01
        bv = bv * np.repeat(fac.astype(np.float64).T, 128, axis=1)[:, k0:]
        gd = torch.from_numpy(fac).to(DEV)
    den = sx.astype(np.float64)[:, None] * sw.astype(np.float64)[None, :]
    want, mag = av @ bv.T / den, np.abs(av) @ np.abs(bv).T / den
    bias = g.standard_normal(N).astype(np.float32) if has_bias else None
    bias_t = None
    if has_bias:
        bias_t = torch.from_numpy(bias).to(DEV).to(dt)
        bias = bias_t.float().cpu().numpy()
        want, mag = want + bias, mag + np.abs(bias)
    addend = None
    if add:
        addend = torch.randn(M, N, device=DEV).to(dt)
        want, mag = want + addend.double().cpu().numpy(), mag + addend.double().abs().cpu().numpy()
    ad, bd = _dev(a, fa, pad), _dev(b, fb, pad)
    esz = 2 if fb == O.FMT_INT4 else 1
    rg = [ops.Range(k0, K, torch.from_numpy(sx).to(DEV), torch.from_numpy(sw).to(DEV), 1 if neg else 0, int(row_sx), int(col_sw and not group))]
    gdesc = ops.gemm_desc(torch.zeros_like(ad) if neg else ad, bd, rg, m=M, n=N, a_fmt=fa, b_fmt=fb, out_dtype=dt, lda=k0 + K + pad,
                          ldb=(k0 + K) // esz + pad, bias=bias_t, a_neg=ad if neg else None, tile=tile, group_dequant=gd, addend=addend)
    ws = torch.empty(ops.gemm_workspace_bytes(gdesc), dtype=torch.uint8, device=DEV) if group else None
    assert tile == 0 or ops.gemm_plan(gdesc, ws)["tile"] == tile
    got = ops.gemm_launch(gdesc, ws).double().cpu().numpy()
    # fp32 arithmetic of the scaling (and of the group sums: one rounding per group and per share), the matrix cores' e4m3
    # sums, and the output's one rounding
    tol = (4e-6 + (2.0 ** -23 * ((k0 + K) // 128 + 8) if group else 0.0)) * mag + 1e-30
    if kind == "e4m3":  # 3e-4 as elsewhere; of 16 or 32 products none averages out, and each is cut at 2^-15 of the largest
        tol = tol + (3e-4 if K > 32 else 16 * 2.0 ** -15) * mag
    tol = tol + {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dt] * np.abs(want) + (2.0 ** -24 if dt == torch.float16 else 0.0)
    err = np.abs(got - want)
    assert np.isfinite(got).all() and (err <= tol).all(), (kind, M, N, K, tile, dt, float((err - tol).max()))


@pytest.mark.parametrize("kind,group", [("int8", False), ("e4m3", False), ("int4", False), ("int4", True)])
@pytest.mark.parametrize("tile", [22, 23, 24, 25])
def test_edges_of_tiles_and_of_k(ops, kind, group, tile):
    g = np.random.default_rng(100 * tile + len(kind) + group)
    step = 128 if group else 32 if kind == "int4" else 16
    for K in (step, 128, 1024 - step, 1024, 1024 + step, 2048 + step, 3072, 4096, 4096 + step, 6144 + step):
        K = max(step, K // step * step)
        M, N = int(g.choice([1, 2, 15, 16, 17, 31, 33, 50])), int(g.choice([4, 16, 36, 64, 100])) + (0 if group else int(g.integers(0, 3)))
        _check(ops, kind, M, N, K, tile, [torch.float32, torch.bfloat16, torch.float16][int(g.integers(0, 3))], g, group=group)


@pytest.mark.parametrize("kind,group", [("int8", False), ("e4m3", False), ("int4", False), ("int4", True)])
def test_forms_of_the_call(ops, kind, group):
    g = np.random.default_rng(7)
    for i, opt in enumerate([dict(), dict(row_sx=False, col_sw=False), dict(has_bias=False), dict(neg=True), dict(add=True), dict(pad=16),
                             dict(k0=128), dict(k0=256, pad=32, add=True)]):
        _check(ops, kind, 37, 104, 640, (22, 23, 24, 25, 0)[i % 5], (torch.bfloat16, torch.float32)[i & 1], g, group=group, **opt)


@pytest.mark.parametrize("kind", ["int8", "e4m3"])
@pytest.mark.parametrize("M,N,K", [(200, 1536, 6144), (333, 1152, 4608), (500, 2048, 2048), (129, 4092, 4096), (280, 2432, 2432)])
def test_several_hundred_rows(ops, kind, M, N, K):
    """More tiles than CUs, by the library's own choice: one unit of K in a wave's loop and several, ragged rows and columns."""
    g = np.random.default_rng(M)
    one = torch.ones(1, device=DEV)
    d = ops.gemm_desc(torch.empty(M, K, dtype=torch.uint8, device=DEV), torch.empty(N, K, dtype=torch.uint8, device=DEV), [ops.Range(0, K, one, one)],
                      m=M, n=N, a_fmt=FORMATS[kind][0], b_fmt=FORMATS[kind][1], out_dtype=torch.float32, lda=K, ldb=K)
    assert ops.gemm_plan(d)["tile"] in (22, 23, 24, 25)
    _check(ops, kind, M, N, K, 0, torch.float32, g)


@pytest.mark.parametrize("kind", ["int8", "e4m3", "int4"])
def test_raw_accumulators_and_batches(ops, kind):
    fa, fb = FORMATS[kind]
    g = np.random.default_rng(3)
    M, N, K = 21, 70, 1184
    a, b = _codes(g, (2 * M, K), fa), _codes(g, (2 * N, K), fb)
    av, bv = O.code_values(a, fa).astype(np.float64), O.code_values(b, fb).astype(np.float64)
    kb = K // 2 if kind == "int4" else K
    for tile in (22, 23, 24, 25):
        out = ops.gemm(_dev(a, fa), _dev(b, fb), [ops.Range(0, K, None, None)], m=M, n=N, a_fmt=fa, b_fmt=fb, out_dtype="acc", lda=K, ldb=kb,
                       tile=tile, batch=2, batch_stride_a=M * K, batch_stride_b=N * kb)
        got = out.double().cpu().numpy().reshape(2, M, N)
        for z in range(2):
            x, y = av[z * M:(z + 1) * M], bv[z * N:(z + 1) * N]
            if kind == "e4m3":
                assert (np.abs(got[z] - x @ y.T) <= 3e-4 * (np.abs(x) @ np.abs(y).T)).all()
            else:
                assert (got[z] == x @ y.T).all()


def test_what_the_tiles_do_not_serve_is_refused(ops):
    g = np.random.default_rng(1)
    a, b = _dev(_codes(g, (40, 256), O.FMT_INT8), O.FMT_INT8), _dev(_codes(g, (64, 256), O.FMT_INT8), O.FMT_INT8)
    one = torch.ones(1, device=DEV)
    kw = dict(m=40, n=64, a_fmt=O.FMT_INT8, b_fmt=O.FMT_INT8, out_dtype=torch.float32, lda=256, ldb=256, tile=24)
    for ranges in ([ops.Range(0, 256, one, one, 2)], [ops.Range(0, 128, one, one), ops.Range(128, 128, one, one)]):
        with pytest.raises(RuntimeError, match="tiles 22 to 25"):
            ops.gemm(a, b, ranges, **kw)
    with pytest.raises(RuntimeError, match="is not in 0.."):
        ops.gemm(a, b, [ops.Range(0, 256, one, one)], **{**kw, "tile": ops.L.lib().segq_gemm_tile_count() + 1})


# ---- one walk of K on the 8-wave tiles: a ragged end of K, DualScale's two ranges -----------------------------------------------
@pytest.mark.parametrize("kind", ["int8", "e4m3"])
@pytest.mark.parametrize("tile", [26, 27, 28])
def test_ragged_end_of_k(ops, kind, tile):
    g = np.random.default_rng(tile)
    for K in (16, 112, 128, 144, 256, 272, 1168, 1280):  # one, two and several steps, ragged and whole
        M, N = int(g.choice([1, 63, 130, 256, 300])), int(g.choice([16, 100, 129, 256, 390]))
        _check(ops, kind, M, N, K, tile, [torch.float32, torch.bfloat16, torch.float16][int(g.integers(0, 3))], g)
    for opt in (dict(row_sx=False, col_sw=False), dict(has_bias=False), dict(neg=True), dict(add=True), dict(pad=16), dict(k0=16), dict(k0=48, pad=32, add=True)):
        _check(ops, kind, 70, 208, 400, tile, torch.bfloat16, g, **opt)


@pytest.mark.parametrize("tile", [26, 27, 28])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_ragged_end_of_k_scales_as_the_general_kernel(ops, tile, dt):
    """int8 sums are exact and both kernels multiply them by quotients: the same bits, with aligned rows of the output and others."""
    g = np.random.default_rng(tile)
    for M, N, K in ((200, 300, 208), (65, 257, 1040), (256, 384, 144)):
        a, b = (_dev(_codes(g, (r, K), O.FMT_INT8), O.FMT_INT8) for r in (M, N))
        rg = [ops.Range(0, K, *(torch.from_numpy((g.random(r) * 30 + 10).astype(np.float32)).to(DEV) for r in (M, N)), 0, 1, 1)]
        out = [ops.gemm(a, b, rg, m=M, n=N, a_fmt=O.FMT_INT8, b_fmt=O.FMT_INT8, out_dtype=dt, lda=K, ldb=K, tile=t) for t in (tile, 4)]
        assert torch.equal(*out), (M, N, K, float((out[0] - out[1]).abs().max()))


@pytest.mark.parametrize("kind", ["int8", "e4m3"])
@pytest.mark.parametrize("M,N,K,tiles", [(1300, 1500, 784, (26, 27, 28)), (2000, 2300, 1040, (26, 27, 28)), (748, 384, 208, (26, 27, 28)),
                                         (748, 383, 208, (4,)), (869, 479, 160, (4,)), (2000, 2301, 1040, (26, 27, 28)), (722, 5554, 2320, (28,)), (2100, 5550, 2320, (26, 27))])
def test_ragged_launch_takes_a_walk(ops, kind, M, N, K, tiles):
    """... unless K is short and the rows of the output start off the boundaries of whole stores; on small tiles where they fill the CUs better."""
    g = np.random.default_rng(5)
    one = torch.ones(1, device=DEV)
    d = ops.gemm_desc(torch.empty(M, K, dtype=torch.uint8, device=DEV), torch.empty(N, K, dtype=torch.uint8, device=DEV), [ops.Range(0, K, one, one)],
                      m=M, n=N, a_fmt=FORMATS[kind][0], b_fmt=FORMATS[kind][1], out_dtype=torch.float32, lda=K, ldb=K)
    assert ops.gemm_plan(d)["tile"] in tiles
    _check(ops, kind, M, N, K, 0, torch.float32, g)


def _check_dual(ops, kind, S, M, N, K, tile, dt, g, k0=0, pad=0, empty=None, per_row=True, per_col=True, add=False, lend=None):
    fa = FORMATS[kind][0]
    a, b = _codes(g, (S * M, k0 + K), fa), _codes(g, (S * N, k0 + K), fa)
    pick = g.random(a.shape) < 0.5
    zero = np.zeros_like(a)
    sides = [np.where(pick, a, zero), np.where(pick, zero, a)]
    sx = [(g.random((S, M if per_row else 1)) * 30 + 10).astype(np.float32) for _ in range(2)]
    if empty is not None:  # a side that holds nothing has the scale limit / 0
        sides[empty][:M] = 0
        sx[empty][0] = np.inf
    sw = (g.random((S, N if per_col else 1)) * 30 + 10).astype(np.float32)
    bias = g.standard_normal(N).astype(np.float32)
    want, mag = np.zeros((S, M, N)), np.zeros((S, M, N))
    for z in range(S):
        bv = O.code_values(b[z * N:(z + 1) * N, k0:], fa).astype(np.float64)
        for side, s in zip(sides, sx):
            av = O.code_values(side[z * M:(z + 1) * M, k0:], fa).astype(np.float64)
            with np.errstate(divide="ignore"):
                den = s[z].astype(np.float64)[:, None] * sw[z].astype(np.float64)[None, :]
            want[z] += av @ bv.T / den
            mag[z] += np.abs(av) @ np.abs(bv).T / den
    want, mag = want + bias, mag + np.abs(bias)
    ad, nd, bd = _dev(sides[0], fa, pad), _dev(sides[1], fa, pad), _dev(b, fa, pad)
    p, n, w = (torch.from_numpy(t.reshape(-1)).to(DEV) for t in (sx[0], sx[1], sw))
    rg = [ops.Range(k0, K, p, w, 0, int(per_row), int(per_col)), ops.Range(k0, K, n, w, 1, int(per_row), int(per_col))]
    addend = None
    if add:
        addend = torch.randn(M, N, device=DEV).to(dt)
        want, mag = want + addend.double().cpu().numpy(), mag + addend.double().abs().cpu().numpy()
    kw = dict(batch=S, batch_stride_a=M * (k0 + K + pad), batch_stride_b=N * (k0 + K + pad), batch_stride_sx=sx[0].shape[1],
              batch_stride_sw=sw.shape[1]) if S > 1 else dict(addend=addend)
    gd = ops.gemm_desc(ad, bd, rg, m=M, n=N, a_fmt=fa, b_fmt=fa, out_dtype=dt, lda=k0 + K + pad, ldb=k0 + K + pad, a_neg=nd, own_sums=lend is None,
                       finite_scales=lend is not None, bias=torch.from_numpy(bias).to(DEV), tile=tile, **kw)
    ws = torch.empty(ops.gemm_workspace_bytes(gd), dtype=torch.uint8, device=DEV) if lend else None
    plan = ops.gemm_plan(gd, ws)
    took = plan["tile"]
    assert took == tile if tile else lend is not None or took in (29, 30)
    got = ops.gemm_launch(gd, ws).double().cpu().numpy().reshape(S, M, N)
    # per range an exact int32 sum, its conversion, two quotients and two products, then the addition of the two and of the bias
    # (finite scales: sums carried from range to range by a ratio of two scales, or added in shares of K)
    tol = (4e-6 if lend is not None and kind == "int8" else 1e-6 if kind == "int8" else 3e-4 if K > 32 else 16 * 2.0 ** -15) * mag + {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8}[dt] * np.abs(want)
    assert np.isfinite(got).all() and (np.abs(got - want) <= tol).all(), (kind, S, M, N, K, tile, dt, float((np.abs(got - want) - tol).max()))
    return plan


@pytest.mark.parametrize("kind", ["int8", "e4m3"])
@pytest.mark.parametrize("tile", [29, 30, 0])
def test_dual_ranges_in_one_walk(ops, kind, tile):
    g = np.random.default_rng(tile + 1)
    for S, M, N, K in ((1, 1, 16, 272), (1, 64, 128, 640), (1, 129, 193, 1024 if tile else 1168), (2, 127, 200, 1040), (3, 65, 130, 528), (1, 300, 500, 640)):
        _check_dual(ops, kind, S, M, N, K, tile, [torch.float32, torch.bfloat16][int(g.integers(0, 2))], g)
    if tile:
        for K in (16, 128, 144, 256):
            _check_dual(ops, kind, 1, 70, 100, K, tile, torch.float32, g)
    for opt in (dict(empty=0), dict(empty=1), dict(per_row=False, per_col=False), dict(pad=32), dict(k0=16, pad=16), dict(add=True)):
        _check_dual(ops, kind, 1, 140, 210, 656, tile, torch.float32, g, **opt)


@pytest.mark.parametrize("kind", ["int8", "e4m3"])
def test_dual_ranges_with_finite_scales(ops, kind):
    """Scales that are finite leave the way to the library: one walk, shares of K where room is lent for them, or in turn."""
    g = np.random.default_rng(17)
    took = {}
    for M, N, K in ((300, 500, 1024), (400, 1024, 12288), (130, 640, 6144)):
        for lend in (False, True):
            plan = _check_dual(ops, kind, 1, M, N, K, 0, torch.bfloat16, g, lend=lend)
            took[M, lend] = plan["tile"] in (29, 30), plan["splits"] > 1
    assert took[300, False] == took[300, True] == took[400, False] == (True, False) and took[400, True] == (False, True)


def _check_mix(ops, kind, M, N, K0, K1, tile, dt, g, shares=0, first=True, gap=0, empty=None, per_row=True, add=False, lend=True,
               merged=False):
    """DualScale's two ranges of K1 and a plain one of K0 (0: none; in front of or behind them in memory, `gap` apart), from two
    code tensors or from one of both signs."""
    fa = FORMATS[kind][0]
    k0, k1 = (0, K0 + gap if K0 else gap) if first else (K1 + gap, 0)
    K = max(k0 + K0, k1 + K1)
    a, b = _codes(g, (M, K), fa), _codes(g, (N, K), fa)
    neg = _codes(g, (M, K), fa)  # (outside the pair it holds what is never read)
    pick = a[:, k1:k1 + K1].view(np.uint8) >= 0x80 if merged else g.random((M, K1)) < 0.5
    if merged:
        neg[:, k1:k1 + K1] = a[:, k1:k1 + K1]
    a[:, k1:k1 + K1][pick] = 0
    neg[:, k1:k1 + K1][~pick] = 0
    scale = lambda n: (g.random(n) * 30 + 10).astype(np.float32)
    sx, sw = [scale(M if per_row else 1) for _ in range(3)], [scale(N), scale(N)]
    if empty is not None:
        (a if empty == 0 else neg)[:, k1:k1 + K1] = 0
        sx[empty][:] = np.inf
    parts = [(a, k1, K1, sx[0], sw[0]), (neg, k1, K1, sx[1], sw[0])] + ([(a, k0, K0, sx[2], sw[1])] if K0 else [])
    bias = g.standard_normal(N).astype(np.float32)
    want, mag = np.zeros((M, N)) + bias, np.zeros((M, N)) + np.abs(bias)
    for c, k, n, s, w in parts:
        av, bv = (O.code_values(t[:, k:k + n], fa).astype(np.float64) for t in (c, b))
        den = s.astype(np.float64)[:, None] * w.astype(np.float64)[None, :]
        want += av @ bv.T / den
        mag += np.abs(av) @ np.abs(bv).T / den
    up = lambda t: torch.from_numpy(t).to(DEV)
    rg = [ops.Range(k, n, up(s), up(w), int(c is neg) + (2 if merged and k == k1 else 0), int(per_row), 1) for c, k, n, s, w in parts]
    if merged:
        a = a.copy()
        a[:, k1:k1 + K1] |= neg[:, k1:k1 + K1]
    if first and K0:
        rg = rg[2:] + rg[:2]
    addend = None
    if add:
        addend = torch.randn(M, N, device=DEV).to(dt)
        want, mag = want + addend.double().cpu().numpy(), mag + addend.double().abs().cpu().numpy()
    gd = ops.gemm_desc(_dev(a, fa), _dev(b, fa), rg, m=M, n=N, a_fmt=fa, b_fmt=fa, out_dtype=dt, lda=K, ldb=K, a_neg=None if merged else _dev(neg, fa), finite_scales=True,
                       bias=up(bias), addend=addend, tile=tile, split_k=shares)
    # (a workspace that holds NaN: nothing of it is read before it is written)
    ws = torch.full((ops.gemm_workspace_bytes(gd) // 4 + 4,), float("nan"), device=DEV).view(torch.uint8) if lend else None
    plan = ops.gemm_plan(gd, ws)
    assert plan["tile"] == tile if tile else plan["tile"] in (31, 32, 33)
    assert not plan["parked"] and (not shares or plan["splits"] <= shares)
    got = [ops.gemm_launch(gd, ws).double().cpu().numpy() for _ in range(2)]
    # an exact int32 sum, its conversion, two quotients and two products per range and share (5 x 2^-24), the additions of up to
    # three ranges, 16 shares, bias and addend (their running sums stay below mag, 21 x 2^-24); e4m3: the matrix cores' limited-width adder
    tol = (1.6e-6 if kind == "int8" else 3e-4) * mag + {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dt] * np.abs(want)
    assert np.isfinite(got[0]).all() and (np.abs(got[0] - want) <= tol).all(), (kind, M, N, K0, K1, tile, dt, float((np.abs(got[0] - want) - tol).max()))
    assert (got[0] == got[1]).all()
    return plan


@pytest.mark.parametrize("kind", ["int8", "e4m3"])
@pytest.mark.parametrize("tile", [31, 32, 33, 0])
@pytest.mark.parametrize("merged", [False, True])
def test_dual_and_plain_ranges_in_one_walk(ops, kind, tile, merged):
    """Edges of the tiles; one, two and three steps of either kind (the loop loads two ahead); shares that begin or end in the
    plain range; three ranges in any order; sides that hold nothing; rules that a workspace or none is given to."""
    g = np.random.default_rng(tile + 2)
    dts = (torch.float32, torch.bfloat16, torch.float16)
    for i, (M, N, k0, k1) in enumerate(((1, 16, 1, 1), (64, 128, 2, 1), (193, 130, 1, 2), (129, 257, 3, 3), (192, 192, 2, 5), (300, 500, 7, 4), (257, 70, 5, 2))):
        for lend in (False, True):
            _check_mix(ops, kind, M, N, 128 * k0, 128 * k1, tile, dts[i % 3], g, first=bool(i % 2), lend=lend, merged=merged)
    for opt in (dict(empty=0), dict(empty=1), dict(empty=2), dict(per_row=False), dict(gap=128), dict(gap=128, first=False), dict(add=True)):
        _check_mix(ops, kind, 140, 210, 384, 640, tile, torch.float32, g, merged=merged, **opt)
    if tile:
        for i, shares in enumerate((2, 3, 5, 9)):  # of 18, 5 and 4 steps: whole ranges, one step, less
            for k0, k1 in ((1024, 1280), (384, 256), (0, 512)):
                _check_mix(ops, kind, 200, 300, k0, k1, tile, dts[i % 3], g, shares=shares, first=bool(i % 2), add=i == 1, empty=2 if i == 2 and k0 else None,
                           merged=merged)
    else:
        # the library's shares: two that meet, more that a second kernel sums; the pair alone; up to 128 rows its own choice is another
        for M, N, k0, k1, splits in ((1024, 3072, 512, 2048, (2, 3, 4)), (300, 640, 640, 4096, range(3, 17)), (600, 2048, 0, 8192, (3, 4, 5))):
            assert _check_mix(ops, kind, M, N, k0, k1, 0, torch.bfloat16, g, merged=merged)["splits"] in splits


@pytest.mark.parametrize("kind", ["int8", "e4m3"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_codes_of_both_signs_written_by_the_gemm(ops, kind, dt):
    """The epilogue that writes a DualScale layer's codes into one tensor against the quantise launch that does, bit for bit."""
    g = np.random.default_rng(23)
    fa = FORMATS[kind][0]
    for M, N, K, op in ((130, 208, 256, "gelu_tanh"), (1, 16, 128, None), (257, 272, 384, "silu")):
        a, b = _dev(_codes(g, (M, K), fa), fa), _dev(_codes(g, (N, K), fa), fa)
        s = [torch.full((1,), v, device=DEV) for v in (900.0, 3.0, 40.0, 900.0)]
        kw = dict(m=M, n=N, a_fmt=fa, b_fmt=fa, out_dtype=dt, lda=K, ldb=K, bias=torch.randn(N, device=DEV))
        rg = [ops.Range(0, K, s[0], s[1])]
        want = ops.quantize(ops.gemm(a, b, rg, tile=14, **kw), fa, s[2], s[3], dual=True, pre_op=op)
        got = ops.gemm(a, b, rg, out_codes=dict(fmt=fa, scale=s[2], scale_neg=s[3], pre_op=op, one_tensor=True), **kw)
        got = got[0] if isinstance(got, tuple) else got
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))


# ---- a linear of up to 16 rows in one launch ---------------------------------------------------------------------------------
@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,group", [("int8", False), ("e4m3", False), ("int4", False), ("int4", True)])
@pytest.mark.parametrize("dynamic", [False, True])
def test_linear_in_one_launch(ops, kind, group, dynamic, dt):
    """``segq_linear`` on 1 to 17 rows against its two launches apart: codes, scales and outputs bit for bit, rows that hold
    zeros, NaN, infinities and the largest value, inputs that are column slices, K of one to four units per wave and beyond."""
    fa, fb = FORMATS[kind]
    g = np.random.default_rng(11)
    for M, N, K in ((1, 64, 256), (16, 100, 1024), (5, 36, 1152), (9, 260, 2048), (16, 132, 3072), (3, 96, 4096), (2, 64, 4224), (17, 64, 512)):
        K = K if group or kind == "int4" else K - 16
        w = _dev(_codes(g, (N, K), fb), fb)
        wide = torch.randn(M, K + 32, device=DEV)
        wide[:, 7] *= 20
        if dynamic and M > 4:
            wide[0, 3] = float("nan")
            wide[1, 5] = float("inf")
            wide[2] = 0
            wide[3, K - 1] = torch.finfo(dt).max
        x = wide.to(dt)[:, 16:16 + K]
        sw = torch.rand(N, device=DEV) + 0.5
        gd = torch.rand(K // 128, N, device=DEV) if group else None
        bias = torch.randn(N, device=DEV).to(dt)

        def descs():
            scale = torch.full((M,), 7.0, device=DEV) if dynamic else torch.rand(M, device=DEV, generator=torch.Generator(device=DEV).manual_seed(M)) * 20 + 1
            q = ops.quantize_desc(x, fa, scale, row_stride=1, dynamic=dynamic)
            d = ops.gemm_desc(q[1], w, [ops.Range(0, K, scale, sw, 0, 1, 1)], m=M, n=N, a_fmt=fa, b_fmt=fb, out_dtype=dt, lda=K,
                              ldb=K // 2 if kind == "int4" else K, bias=bias, group_dequant=gd)
            nb = ops.gemm_workspace_bytes(d)
            return q, d, torch.empty(nb, dtype=torch.uint8, device=DEV) if nb else None, scale
        q, d, ws, scale = descs()
        out = ops.linear(q, d, ws)
        q2, d2, ws2, scale2 = descs()
        ops.quantize_launch(q2)
        want = ops.gemm_launch(d2, ws2)
        what = (kind, group, dynamic, dt, M, N, K)
        assert torch.equal(q[1].view(torch.uint8), q2[1].view(torch.uint8)), what
        assert torch.equal(scale.view(torch.int32), scale2.view(torch.int32)), what
        assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.nan_to_num(), want.nan_to_num()), what


def _captured(call):
    """The graph of one call and the number of launches in it."""
    hip = ctypes.CDLL("libamdhip64.so")
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph(keep_graph=True)
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=stream):
        call()
    count = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    graph.instantiate()
    return graph, count.value


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,group", [("int8", False), ("e4m3", False), ("int4", False), ("int4", True)])
@pytest.mark.parametrize("scales", ["tensor", "row", "dynamic"])
def test_wide_linear_in_one_launch(ops, kind, group, scales, dt):
    """Layers of many column tiles, on 16 x 64 too, and one scale for the tensor: codes, scales and outputs of the two launches apart
    bit for bit, from every replay of a graph as well, and in one launch wherever the estimate says so."""
    fa, fb = FORMATS[kind]
    g = np.random.default_rng(13)
    taken = set()  # tiles that did the quantise step
    for M, N, K in ((8, 12288, 1536), (8, 12300, 512), (5, 12288, 2944), (3, 12300, 1024), (8, 18432, 2048), (16, 12288, 3072), (2, 9216, 1536), (16, 36864, 3072), (17, 1024, 1024), (4, 512, 4224)):
        w = _dev(_codes(g, (N, K), fb), fb)
        dyn = scales == "dynamic"
        sw = torch.rand(1 if group else N, device=DEV) + 0.5
        gd = torch.rand(K // 128, N, device=DEV) if group else None
        x, scale = torch.randn(M, K, device=DEV).to(dt), torch.rand(1 if scales == "tensor" else M, device=DEV) * 20 + 1

        def descs(scale):
            q = ops.quantize_desc(x, fa, scale, row_stride=int(scales != "tensor"), dynamic=dyn)
            d = ops.gemm_desc(q[1], w, [ops.Range(0, K, scale, sw, 0, int(scales != "tensor"), int(not group))], m=M, n=N, a_fmt=fa, b_fmt=fb, out_dtype=dt,
                              lda=K, ldb=K // 2 if kind == "int4" else K, group_dequant=gd)
            nb = ops.gemm_workspace_bytes(d)
            return q, d, torch.empty(nb, dtype=torch.uint8, device=DEV) if nb else None
        what = (kind, group, scales, dt, M, N, K)
        q, d, ws = descs(scale.clone())
        tile = ops.gemm_plan(d, ws)["tile"]
        graph, launches = _captured(lambda: ops.linear(q, d, ws))
        tiles, most = -(-N // (32 if tile == 22 else 64)), 1024 * (4 if tile == 22 else 3)
        rounds = -(-tiles // torch.cuda.get_device_properties(0).multi_processor_count)
        f32, second = dt == torch.float32, M > 8
        extra = rounds * (0.9 if dyn else 0.1) + K / 1024 * (rounds * (0.83 + 0.36 * second + (0.44 if second else 0.12) * f32) - 0.55)
        if tile in (22, 23) or M > 16:  # (elsewhere the library has other launches for several rows)
            assert launches == (1 if M <= 16 and K <= most and extra <= 5.8 else 2), (what, tile, launches)
        if launches == 1:
            taken.add(tile)
        for _ in range(3):
            x.copy_(torch.randn(M, K, device=DEV))
            q2, d2, ws2 = descs(scale.clone())
            ops.quantize_launch(q2)
            want = ops.gemm_launch(d2, ws2)
            for out in (d[1], None):  # the replay's, then an eager call's
                if out is None:
                    out = ops.linear(q, d, ws)
                else:
                    out.zero_(); q[1].zero_()
                    graph.replay()
                assert torch.equal(q[1].view(torch.uint8), q2[1].view(torch.uint8)), what
                assert torch.equal(q[3][1].view(torch.int32), q2[3][1].view(torch.int32)) and torch.equal(out, want), what
    assert taken == {22, 23}, taken


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dynamic", [False, True])
def test_linear_over_its_own_input(ops, dynamic, dt):
    """A square linear whose output takes the place of its input, whole and shifted by some rows: the codes are those of the
    input, and the result is that of the call with an output of its own, however the workgroups follow each other."""
    g = np.random.default_rng(12)
    K = 2048
    w = _dev(_codes(g, (K, K), O.FMT_INT8), O.FMT_INT8)
    one = torch.ones(1, device=DEV)
    for M in (1, 16):
        for shift in (0, 1, M - 1, M):
            x = torch.randn(M, K, device=DEV).to(dt)

            def run(buf, out):
                buf[:M] = x
                scale = torch.full((M,), 20.0, device=DEV)
                q = ops.quantize_desc(buf[:M], O.FMT_INT8, scale, row_stride=1, dynamic=dynamic)
                d = ops.gemm_desc(q[1], w, [ops.Range(0, K, scale, one, 0, 1, 0)], m=M, n=K, a_fmt=O.FMT_INT8, b_fmt=O.FMT_INT8, out_dtype=dt,
                                  lda=K, ldb=K, out=out)
                return ops.linear(q, d), q[1], scale
            buf = torch.empty(2 * M, K, device=DEV, dtype=dt)
            want, codes, scale = run(buf, torch.empty(M, K, device=DEV, dtype=dt))
            for _ in range(10):
                got, c2, s2 = run(buf, buf[shift:shift + M])
                assert torch.equal(c2, codes) and torch.equal(s2, scale) and torch.equal(got, want), (dynamic, dt, M, shift)
