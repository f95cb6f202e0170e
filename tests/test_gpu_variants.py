"""Kernel variants at the sizes where they can go wrong: edges of tiles, remainders, unaligned views."""
import numpy as np
import pytest
import torch

from oracle import segq_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TDT = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


@pytest.mark.parametrize("dt", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("n", [1, 3, 4, 7, 8, 9, 2048, 4095, 4096, 4099, 20001])
@pytest.mark.parametrize("off", [0, 1, 8])
def test_fake_e4m3_sizes_and_offsets(dt, n, off):
    """16-byte accesses and their remainder, one value per thread for views off the 16-byte grid: the values of
    the CPU path bit for bit, signs of zeros among them; a NaN keeps its sign and payload and is quiet."""
    from segquant_amd import ops
    from segquant_amd.utils.extension import FakeQuantFp8Ext
    g = torch.Generator().manual_seed(n + off)
    x = (torch.randn(n + off, generator=g) * 200).to(TDT[dt])
    inf = float("inf")
    # odd in number, so that in every repetition they fall on the other half of a dword
    special = torch.tensor([0.0, -0.0, 1e4, -1e4, 2.0 ** -10, -(2.0 ** -11), 2.0 ** -7, inf, -inf]).to(TDT[dt])
    bits, quiet, exponent = {"fp32": (torch.int32, 1 << 22, 0x7F800000), "bf16": (torch.int16, 1 << 6, 0x7F80), "fp16": (torch.int16, 1 << 9, 0x7C00)}[dt]
    nans = [exponent | 1, exponent | quiet, exponent | quiet | 5, exponent | 3]  # signalling and quiet, payloads, either sign below
    sign = torch.iinfo(bits).min
    special = torch.cat([special, torch.tensor([nans[0], nans[1] + sign, nans[2], nans[3] + sign], dtype=bits).view(TDT[dt])])
    for at in range(off, n + off, 29):
        x[at:at + 13] = special[:n + off - at]
    x[max(off, n + off - 13):] = special[:min(n, 13)].flip(0)
    got = ops.fake_e4m3fy(x.to(DEV)[off:]).cpu()
    nan = x[off:].isnan()
    want = torch.where(nan, x[off:].view(bits) | quiet, FakeQuantFp8Ext.fake_e4m3fy(x[off:]).view(bits))
    assert got.dtype == x.dtype
    if dt == "fp32":  # (a 32-bit NaN is passed on as it is)
        want = torch.where(nan, x[off:].view(bits), want)
    np.testing.assert_array_equal(got.view(bits).numpy(), want.numpy())


@pytest.mark.parametrize("fmt", [O.FMT_INT8, O.FMT_E4M3])
@pytest.mark.parametrize("S,M,N,K", [(1, 5, 18, 128), (2, 300, 200, 384), (3, 130, 515, 256), (2, 77, 130, 208)])
def test_dual_operator_batches(fmt, S, M, N, K):
    """DualScale over several segments with per-segment scales that differ, K in whole steps and not, against the closed
    form in fp64, on the general kernel (test_dual_operator_sides has the sizes of the others)."""
    from segquant_amd import ops
    g = torch.Generator().manual_seed(S * M + K)
    x = torch.nn.functional.gelu(torch.randn(S, M, K, generator=g) * torch.tensor([1.0, 3.0, 0.5])[:S, None, None])
    lim = (127.0, 128.0) if fmt == O.FMT_INT8 else (448.0, 448.0)
    pos, neg = lim[0] / x.amax(dim=(1, 2)), lim[1] / (-x).amax(dim=(1, 2))
    rng = np.random.default_rng(7)
    w = rng.integers(-128, 128, size=(S, N, K)).astype(np.int8) if fmt == O.FMT_INT8 else \
        np.where((c := rng.integers(0, 256, size=(S, N, K)).astype(np.uint8)) & 0x7F == 0x7F, 0x3A, c).astype(np.uint8)
    sw = torch.rand(S, N, generator=g) * 30 + 10
    out = ops.real_quantized_gemm_dual_scaled(fmt, fmt, x.to(DEV), torch.from_numpy(w).to(DEV), pos.to(DEV), neg.to(DEV), sw.to(DEV)).cpu().numpy()
    for s in range(S):
        yp, yn = O.quantize_act_dual(x[s:s + 1].numpy(), [pos[s].numpy()], [neg[s].numpy()], fmt)
        wv = O.code_values(w[s], fmt)
        p, n = O.code_values(yp[0], fmt), O.code_values(yn[0], fmt)
        want = ((p @ wv.T) / np.float64(pos[s]) + (n @ wv.T) / np.float64(neg[s])) / sw[s].numpy().astype(np.float64)[None, :]
        mag = ((np.abs(p) @ np.abs(wv).T) / np.float64(pos[s]) + (np.abs(n) @ np.abs(wv).T) / np.float64(neg[s])) / sw[s].numpy()[None, :]
        # fp32 scaling of int32 sums; e4m3: the matrix cores' limited-width adder
        assert (np.abs(out[s] - want) <= (2e-6 if fmt == O.FMT_INT8 else 3e-4) * mag + 1e-30).all()


@pytest.mark.parametrize("off", [0, 8, 3])
@pytest.mark.parametrize("rows", [1, 5, 130])
def test_layers_read_column_slices_where_they_lie(rows, off):
    """Inputs and gates that are column slices of a wider tensor (16-byte aligned: read in place; off the grid, with
    rows that are no multiple of 16 bytes apart, repeated or reversed by a transposition: copied) give the bits of
    their contiguous copies, on the first call of a token count and on later ones, plain and with a fused activation."""
    from segquant_amd.layers.SegmentLinear import SegmentLinear
    K, N = 256, 144
    off = off & ~7 if rows == 1 else off  # (a single row is contiguous wherever it starts: unaligned, it is refused as ever)
    g = torch.Generator().manual_seed(rows + off)
    args = {"real_quant": True, "axis": -1, "dynamic": True}
    layer = SegmentLinear(K, N, bias=True, custom_weight_tensor=torch.randn(N, K, generator=g) * 0.02,
                          custom_bias_tensor=torch.randn(N, generator=g).to(torch.bfloat16), input_quant_type="int8", weight_quant_type="int8",
                          input_quant_args=args, weight_quant_args={"real_quant": True, "axis": 1}, device=DEV)
    layer.calibrate(torch.randn(64, K, generator=g).to(DEV))
    layer.finish_calibrate()
    for width in (2 * K + 16, 2 * K + 21):
        wide = torch.randn(rows, width, generator=g).to(torch.bfloat16).to(DEV)
        a, b = wide[:, off:off + K], wide[:, K + off:2 * K + off]
        t = torch.randn(K, rows, generator=g).to(torch.bfloat16).to(DEV).t()
        e = wide[:1, off:off + K].expand(rows, K)
        for v in (a, b, t, e, a):
            assert torch.equal(layer(v), layer(v.contiguous().clone()))
            assert torch.equal(layer(v), layer(v.contiguous().clone()))
        assert torch.equal(layer(a, pre_op="gelu", gate=b), layer(a.contiguous().clone(), pre_op="gelu", gate=b.contiguous().clone()))
        assert torch.equal(layer(t, pre_op="silu", gate=a), layer(t.contiguous().clone(), pre_op="silu", gate=a.contiguous().clone()))


@pytest.mark.parametrize("fa,fb", [(O.FMT_INT8, O.FMT_INT8), (O.FMT_E4M3, O.FMT_E4M3), (O.FMT_INT8, O.FMT_INT4)])
@pytest.mark.parametrize("lens", [(32,), (160,), (384,), (512,), (544,), (640,), (1184,), (96, 160, 544), (512, 32), (32, 32, 32, 1056)])
def test_general_gemm_steps_in_flight(fa, fb, lens):
    """One to ten K steps around the number the general kernel keeps in flight, ends inside a step, and ranges whose
    steps are loaded while the range before is multiplied; odd N, each bias type, on the tiles of each depth."""
    from segquant_amd import ops
    M, N, K = 67, 131, sum(lens)
    rng = np.random.default_rng(K + len(lens))
    lo = -8 if fb == O.FMT_INT4 else -128

    def codes(rows, fmt):
        if fmt == O.FMT_E4M3:
            c = rng.integers(0, 256, size=(rows, K)).astype(np.uint8)
            return np.where(c & 0x7F == 0x7F, 0x3A, c).astype(np.uint8)
        return rng.integers(lo if fmt == fb else -128, 8 if fmt == O.FMT_INT4 else 128, size=(rows, K)).astype(np.int8)

    a, b = codes(M, fa), codes(N, fb)
    ad = torch.from_numpy(a).to(DEV)
    bd = torch.from_numpy(np.stack([O.pack_int4(r) for r in b]) if fb == O.FMT_INT4 else b).to(DEV)
    sx = rng.uniform(0.5, 1.5, size=(len(lens), M)).astype(np.float32)
    sw = rng.uniform(0.5, 1.5, size=(len(lens), N)).astype(np.float32)
    sxd, swd = torch.from_numpy(sx).to(DEV), torch.from_numpy(sw).to(DEV)
    va, vb = O.code_values(a, fa), O.code_values(b, fb)
    want, mag, ranges, k = 0.0, 0.0, [], 0
    for i, n in enumerate(lens):
        f = 1.0 / (sx[i].astype(np.float64)[:, None] * sw[i].astype(np.float64)[None, :])
        want = want + (va[:, k:k + n] @ vb[:, k:k + n].T) * f
        mag = mag + (np.abs(va[:, k:k + n]) @ np.abs(vb[:, k:k + n]).T) * f
        ranges.append(ops.Range(k, n, sxd[i], swd[i], 0, 1, 1))
        k += n
    for bt in (None, torch.float32, torch.bfloat16, torch.float16):
        bias = None if bt is None else torch.from_numpy(rng.normal(size=N)).to(bt)
        exact = want if bt is None else want + bias.double().numpy()[None, :]
        for tile in (2, 3, 4):
            y = ops.gemm(ad, bd, ranges, m=M, n=N, a_fmt=fa, b_fmt=fb, out_dtype=torch.float32, lda=K, ldb=bd.shape[1],
                         bias=None if bias is None else bias.to(DEV), tile=tile)
            # int8: fp32 scaling of exact sums, a few roundings of 2^-24 per range; e4m3: the matrix cores' limited-width adder
            tol = 3e-4 if fa == O.FMT_E4M3 else 1e-6
            assert (np.abs(y.cpu().numpy().astype(np.float64) - exact) <= tol * mag + 2.0 ** -22 * np.abs(exact)).all(), (lens, bt, tile)


class _Plans:
    """What each GEMM launched through ``ops.gemm`` from here on runs as (``gemm_plan`` of its descriptor)."""

    def __init__(self, monkeypatch):
        from segquant_amd import ops
        self.seen = []
        desc = ops.gemm_desc

        def record(*args, **kw):
            g = desc(*args, **kw)
            self.seen.append(dict(ops.gemm_plan(g), two=g[0].a_neg is not None, workspace=g[0].workspace))
            return g
        monkeypatch.setattr(ops, "gemm_desc", record)


def _dual_case(fmt, S, M, N, K, per_token, sides, seed, int4=False, dtype=torch.float32):
    """Inputs, unclamped scales and the fp64 result of the DualScale operator; ``sides``: which signs each segment (or
    token, in turn) holds, an empty one having the scale limit / 0 = inf.  Column 1 of the weights is zero, its scale too."""
    g = torch.Generator().manual_seed(seed)
    x = torch.nn.functional.gelu(torch.randn(S, M, K, generator=g)) * 10.0 ** torch.randint(-2, 3, (S, 1, 1), generator=g)
    for i in range(S * (M if per_token else 1)):
        part = x.view(S * M, K)[i] if per_token else x[i]
        side = sides[i % len(sides)]
        if side == "+":
            part.clamp_(min=0.0)
        elif side == "-":
            part.copy_(-(part.abs() + 1e-3))
    lim = (127.0, 128.0) if fmt == O.FMT_INT8 else (448.0, 448.0)
    over = 2 if per_token else (1, 2)
    x = x.to(dtype).float()
    pos, neg = lim[0] / x.amax(dim=over).clamp(min=0.0), lim[1] / (-x).amax(dim=over).clamp(min=0.0)
    rng = np.random.default_rng(seed)
    lo = -8 if int4 else -128
    w = rng.integers(lo, -lo, size=(S, N, K)).astype(np.int8) if fmt == O.FMT_INT8 else \
        np.where((c := rng.integers(0, 256, size=(S, N, K)).astype(np.uint8)) & 0x7F == 0x7F, 0x3A, c).astype(np.uint8)
    sw = torch.rand(S, N, generator=g) * 30 + 10
    w[:, 1], sw[:, 1] = 0, float("inf")
    want, mag = np.empty((S, M, N)), np.empty((S, M, N))
    for s in range(S):
        rows = lambda t: t[s].numpy().astype(np.float64).reshape(-1, 1) + np.zeros((M, 1))
        with np.errstate(invalid="ignore"):
            yp, yn = O.quantize_act_dual(x[s:s + 1].numpy(), pos[s].numpy().reshape(-1), neg[s].numpy().reshape(-1), fmt)
        wv, p, n = O.code_values(w[s], fmt), O.code_values(yp[0], fmt), O.code_values(yn[0], fmt)
        col = sw[s].numpy().astype(np.float64)[None, :]
        want[s] = ((p @ wv.T) / rows(pos) + (n @ wv.T) / rows(neg)) / col
        mag[s] = ((np.abs(p) @ np.abs(wv).T) / rows(pos) + (np.abs(n) @ np.abs(wv).T) / rows(neg)) / col
    return x.to(dtype), w, pos, neg, sw, want, mag


@pytest.mark.parametrize("fmt", [O.FMT_INT8, O.FMT_E4M3])
@pytest.mark.parametrize("S,M,N,K,tile,two", [(2, 300, 200, 256, "64x128", False), (1, 1100, 1000, 208, "64x128", False),
                                              (2, 600, 700, 256, "128x128", True), (3, 400, 600, 384, "128x128", True), (3, 500, 900, 384, "128x128", False),
                                              (1, 3000, 1500, 384, "256x128", False), (2, 2000, 2000, 512, "256x128", True),
                                              (1, 300, 20000, 512, "128x256", True)])
@pytest.mark.parametrize("per_token,sides", [(False, ["+-"]), (False, ["+", "-", "+-"]), (False, ["-"]), (True, ["+-", "+", "-"])])
def test_dual_operator_sides(monkeypatch, fmt, S, M, N, K, tile, two, per_token, sides):
    """The DualScale operator on every kernel that serves it, from one merged code tensor and from two: batches, ragged
    edges, scales far apart from segment to segment or token to token, and sides that hold nothing, whose scale is
    infinite and whose contribution is zero.  It borrows no workspace and shares no tile's K steps."""
    from segquant_amd import ops
    x, w, pos, neg, sw, want, mag = _dual_case(fmt, S, M, N, K, per_token, sides, S + M + N + K)
    plans = _Plans(monkeypatch)
    out = ops.real_quantized_gemm_dual_scaled(fmt, fmt, x.to(DEV), torch.from_numpy(w).to(DEV), pos.reshape(-1).to(DEV),
                                              neg.reshape(-1).to(DEV), sw.to(DEV)).cpu().numpy()
    assert [(p["shape"], p["two"], p["parked"], p["splits"], p["workspace"]) for p in plans.seen] == [(tile, two, False, 1, None)]
    # int8: per range an exact sum, its conversion, two reciprocals (1 ulp each) and two products, then the addition:
    # 8 x 2^-24 = 4.8e-7; e4m3: the matrix cores' limited-width adder
    assert (np.abs(out - want) <= (5e-7 if fmt == O.FMT_INT8 else 3e-4) * mag).all()


@pytest.mark.parametrize("fmt", [O.FMT_INT8, O.FMT_E4M3])
@pytest.mark.parametrize("M,N,K", [(3, 300, 4096), (64, 520, 2048), (200, 1000, 4096), (520, 1032, 4096), (1500, 1500, 4096)])
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("per_token,sides", [(False, ["+-"]), (False, ["+"]), (True, ["+-", "+", "-"])])
def test_dual_operator_in_k_shares(monkeypatch, fmt, M, N, K, dt, per_token, sides):
    """One segment, few tiles, a long K: with 16-bit outputs the K steps are shared, in a workspace of the call's own
    that no other launch ever sees; fp32 outputs keep whole tiles.  Sides that hold nothing have an infinite scale."""
    from segquant_amd import ops
    x, w, pos, neg, sw, want, mag = _dual_case(fmt, 1, M, N, K, per_token, sides, M + N + K, dtype=TDT[dt])
    sw, want, mag = sw * 1024, want / 1024, mag / 1024  # (within fp16)
    plans = _Plans(monkeypatch)
    monkeypatch.setattr(ops, "int4_workspace", None)  # the buffer that layers share is not asked for
    args = (x.to(DEV), torch.from_numpy(w).to(DEV), pos.reshape(-1).to(DEV), neg.reshape(-1).to(DEV), sw.to(DEV))
    junk = torch.full((1 << 26,), 0x7FC00000, dtype=torch.int32, device=DEV)  # what the workspace finds in its memory: NaNs
    del junk
    outs = [ops.real_quantized_gemm_dual_scaled(fmt, fmt, *args) for _ in range(3)]
    for p in plans.seen:
        assert (p["splits"] > 2) == (p["workspace"] is not None)
        if dt == "fp32":
            assert p["splits"] == 1
        elif K == 4096 and M > 100 or (fmt == O.FMT_E4M3 and M == 64):
            assert p["splits"] > 2
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])  # the shares are added in their order
    # the sums as in whole tiles, one more fp32 rounding per share; the output's one rounding
    rounding = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 0.0}[dt]
    bound = (2e-6 if fmt == O.FMT_INT8 else 3e-4) * mag + rounding * np.abs(want) + (2.0 ** -24 if dt == "fp16" else 0.0)
    assert (np.abs(outs[0].cpu().float().numpy().astype(np.float64) - want) <= bound).all()


@pytest.mark.parametrize("S,M,N,K,two", [(1, 700, 500, 512, False), (2, 1000, 1000, 256, False), (1, 2100, 2100, 512, True)])
def test_dual_operator_sides_int4(monkeypatch, S, M, N, K, two):
    """The same with int4 weights, which are unpacked on their way into LDS."""
    from segquant_amd import ops
    x, w, pos, neg, sw, want, mag = _dual_case(O.FMT_INT8, S, M, N, K, True, ["+-", "+", "-"], S + M + N + K, int4=True)
    packed = np.stack([np.stack([O.pack_int4(r) for r in ws]).reshape(-1) for ws in w])
    plans = _Plans(monkeypatch)
    out = ops.real_quantized_gemm_dual_scaled(O.FMT_INT8, O.FMT_INT4, x.to(DEV), torch.from_numpy(packed).to(DEV), pos.reshape(-1).to(DEV),
                                              neg.reshape(-1).to(DEV), sw.to(DEV)).cpu().numpy()
    assert [(p["two"], p["workspace"]) for p in plans.seen] == [(two, None)]
    assert (np.abs(out - want) <= 5e-7 * mag).all()


@pytest.mark.parametrize("empty", [0, 1, 2])
@pytest.mark.parametrize("split_k", [1, 2, 3])
@pytest.mark.parametrize("tile", [11, 12, 13, 14, 15, 16, 17, 18])
def test_parked_ranges_with_an_infinite_scale(tile, split_k, empty):
    """int8 ranges whose sums are parked, whole tiles and K shares: a range of zero codes with an infinite scale (the
    first, the middle or the last one) adds nothing to the others, whose scales lie nine orders of magnitude apart."""
    from segquant_amd import ops
    M, N, lens = 300, 333, (256, 128, 384)
    K = sum(lens)
    rng = np.random.default_rng(tile * 10 + split_k)
    a, b = rng.integers(-128, 128, size=(M, K)).astype(np.int8), rng.integers(-128, 128, size=(N, K)).astype(np.int8)
    sx, sw = rng.uniform(1, 2, size=(3, M)).astype(np.float32), rng.uniform(1, 2, size=(3, N)).astype(np.float32)
    sx[1] *= 1e9
    sx[empty, ::2] = np.inf
    sw[empty, 5] = np.inf
    k0 = sum(lens[:empty])
    a[::2, k0:k0 + lens[empty]] = 0
    b[5, k0:k0 + lens[empty]] = 0
    ad, bd = torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV)
    sxd, swd = torch.from_numpy(sx).to(DEV), torch.from_numpy(sw).to(DEV)
    want, mag, ranges, k = 0.0, 0.0, [], 0
    for i, n in enumerate(lens):
        f = 1.0 / (sx[i].astype(np.float64)[:, None] * sw[i].astype(np.float64)[None, :])
        va, vb = a[:, k:k + n].astype(np.float64), b[:, k:k + n].astype(np.float64)
        want, mag = want + (va @ vb.T) * f, mag + (np.abs(va) @ np.abs(vb).T) * f
        ranges.append(ops.Range(k, n, sxd[i], swd[i], 0, 1, 1))
        k += n
    ws = torch.full((ops.split_bytes(M, N, split_k, park=True),), 0xFF, dtype=torch.uint8, device=DEV)
    kw = dict(m=M, n=N, a_fmt=O.FMT_INT8, b_fmt=O.FMT_INT8, out_dtype=torch.float32, lda=K, ldb=K, tile=tile, split_k=split_k)
    g = ops.gemm_desc(ad, bd, ranges, workspace=ws, **kw)
    if split_k == 1 or tile not in (13, 12, 14):  # (the smaller tiles' K shares keep a second register set)
        assert ops.gemm_plan(g)["parked"]
    out = ops.gemm_launch(g).cpu().numpy()
    # 8 roundings of 2^-24 per term as above, one more per K share
    assert (np.abs(out - want) <= 8e-7 * mag).all()


@pytest.mark.parametrize("M,N,K", [(500, 1100, 2048), (900, 2100, 512), (2100, 4000, 512), (130, 70, 512)])
def test_dual_operator_lies_as_close_as_single_precision_allows(M, N, K):
    """int8, fp32 out: no further from the exact result than the same sums scaled in single precision with correctly
    rounded reciprocals."""
    from segquant_amd import ops
    rng = np.random.default_rng(K + M)
    codes, b = rng.integers(-128, 128, size=(M, K)).astype(np.int8), rng.integers(-128, 128, size=(N, K)).astype(np.int8)
    sx, sw = rng.uniform(1, 2, size=(2, M)).astype(np.float32), rng.uniform(1, 2, size=N).astype(np.float32)
    x = codes / np.where(codes >= 0, sx[0][:, None], sx[1][:, None])  # (x times its scale lies within 1e-5 of the code)
    out = ops.real_quantized_gemm_dual_scaled(O.FMT_INT8, O.FMT_INT8, torch.from_numpy(x[None].astype(np.float32)).to(DEV), torch.from_numpy(b[None]).to(DEV),
                                              *(torch.from_numpy(t).to(DEV) for t in (sx[0], sx[1], sw)))[0].cpu().numpy()
    sums = [f(codes, 0).astype(np.float64) @ b.T.astype(np.float64) for f in (np.maximum, np.minimum)]
    exact = sum(s / (v[:, None].astype(np.float64) * sw[None, :].astype(np.float64)) for s, v in zip(sums, sx))
    one = np.float32(1)
    single = sum(s.astype(np.float32) * (one / v)[:, None] * (one / sw)[None, :] for s, v in zip(sums, sx))
    rms = lambda e: np.sqrt(np.mean(np.square(e)))
    assert rms(out - exact) <= 1.02 * rms(single - exact)


@pytest.mark.parametrize("fa,fb", [(O.FMT_INT8, O.FMT_INT8), (O.FMT_E4M3, O.FMT_E4M3), (O.FMT_INT8, O.FMT_INT4)])
@pytest.mark.parametrize("M,N,K", [(1100, 2001, 1184), (1100, 2001, 96), (1020, 2001, 1184)])
def test_general_gemm_on_more_tiles_than_compute_units(fa, fb, M, N, K):
    """64 x 128 tiles of one range on either side of one per compute unit, where the number of steps in flight changes."""
    from segquant_amd import ops
    rng = np.random.default_rng(M + K)

    def codes(rows, fmt):
        if fmt == O.FMT_E4M3:
            c = rng.integers(0, 256, size=(rows, K)).astype(np.uint8)
            return np.where(c & 0x7F == 0x7F, 0x3A, c).astype(np.uint8)
        return rng.integers(-8 if fmt == O.FMT_INT4 else -128, 8 if fmt == O.FMT_INT4 else 128, size=(rows, K)).astype(np.int8)

    a, b = codes(M, fa), codes(N, fb)
    bd = torch.from_numpy(np.stack([O.pack_int4(r) for r in b]) if fb == O.FMT_INT4 else b).to(DEV)
    sx, sw = rng.uniform(0.5, 1.5, size=M).astype(np.float32), rng.uniform(0.5, 1.5, size=N).astype(np.float32)
    y = ops.gemm(torch.from_numpy(a).to(DEV), bd, [ops.Range(0, K, torch.from_numpy(sx).to(DEV), torch.from_numpy(sw).to(DEV), 0, 1, 1)], m=M, n=N,
                 a_fmt=fa, b_fmt=fb, out_dtype=torch.float32, lda=K, ldb=bd.shape[1], tile=4).cpu().numpy()
    va, vb = O.code_values(a, fa), O.code_values(b, fb)
    f = 1.0 / (sx.astype(np.float64)[:, None] * sw.astype(np.float64)[None, :])
    # int8: fp32 scaling of exact sums, a few roundings of 2^-24; e4m3: the matrix cores' limited-width adder, which
    # aligns the products to the largest one: of these 2.2 million sums of 96 products one lies 3.3e-4 of sum |a||b| off,
    # on this tile as on 128 x 128 (1184 products: 4.8e-5)
    assert (np.abs(y - (va @ vb.T) * f) <= (5e-4 if fa == O.FMT_E4M3 else 5e-7) * (np.abs(va) @ np.abs(vb).T) * f).all()


def _smoothed(opt_type, K=256, N=144, M=40):
    from segquant_amd.layers.SegmentLinear import SegmentLinear
    g = torch.Generator().manual_seed(5)
    x = torch.randn(M, K, generator=g) * (torch.rand(K, generator=g) * 4 + 0.2)
    layer = SegmentLinear(K, N, bias=True, custom_weight_tensor=torch.randn(N, K, generator=g) * 0.02, custom_bias_tensor=torch.randn(N, generator=g),
                          input_quant_type="int8", weight_quant_type="int8", input_quant_args={"real_quant": True, "axis": -1, "dynamic": True},
                          weight_quant_args={"real_quant": True, "axis": 1}, opt_type=opt_type,
                          opt_kwargs={"low_rank": 32, "precision": "float32"} if opt_type == "svd" else None, device=DEV)
    x = x.to(DEV)
    layer.trace(x)
    layer.smooth()
    layer.calibrate(x)
    layer.finish_calibrate()
    return layer, x


def test_a_smoothed_layer_first_seen_in_a_dtype_under_capture():
    """The first call in fp16 of a layer in use in bf16 is one that is only recorded: eager calls before the graph's
    first replay, and the replays, give what a layer that was never captured gives."""
    layer, x = _smoothed("smooth")
    want = _smoothed("smooth")[0](x.half())
    layer(x.bfloat16())
    buf = torch.zeros_like(x.half())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(buf)
    assert torch.equal(layer(x.half()), want)
    for _ in range(3):
        buf.copy_(x.half())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(layer(x.half()), want)
        buf.zero_()
    assert set(layer.optimizer._plan["col_div_cast"]) == set(TDT.values())


def test_low_rank_factors_are_cast_before_the_first_call():
    """A layer with a low-rank branch makes nothing on the first call of a dtype that later calls read: that call may be
    recorded into a graph, or run on another stream."""
    layer, x = _smoothed("svd")
    out = layer(x.bfloat16())
    kept = {dt: [t.data_ptr() for t in l1] + [l2.data_ptr()] for dt, (l1, l2) in layer.optimizer._plan["l12_cast"].items()}
    assert set(kept) == set(TDT.values())
    for dt in (torch.float16, torch.float32, torch.bfloat16):
        again = layer(x.to(dt))
        assert (again.float() - out.float()).norm() <= 2e-2 * out.float().norm()
    assert kept == {dt: [t.data_ptr() for t in l1] + [l2.data_ptr()] for dt, (l1, l2) in layer.optimizer._plan["l12_cast"].items()}
