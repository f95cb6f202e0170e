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
    the CPU path bit for bit, a NaN staying one."""
    from segquant_amd import ops
    from segquant_amd.utils.extension import FakeQuantFp8Ext
    g = torch.Generator().manual_seed(n + off)
    x = (torch.randn(n + off, generator=g) * 200).to(TDT[dt])
    x[off:off + 6] = torch.tensor([float("nan"), -0.0, 1e4, -1e4, 2.0 ** -10, 2.0 ** -7])[:n].to(TDT[dt])
    got = ops.fake_e4m3fy(x.to(DEV)[off:]).cpu()
    want = FakeQuantFp8Ext.fake_e4m3fy(x[off:])
    assert torch.isnan(got[0]) and got.dtype == want.dtype
    np.testing.assert_array_equal(got[1:].float().numpy(), want[1:].float().numpy())


@pytest.mark.parametrize("fmt", [O.FMT_INT8, O.FMT_E4M3])
@pytest.mark.parametrize("S,M,N,K", [(1, 5, 18, 128), (2, 300, 200, 384), (3, 130, 515, 256), (2, 77, 130, 208)])
def test_dual_operator_batches(fmt, S, M, N, K):
    """DualScale over several segments: two code tensors and parked sums per segment (K in whole steps), the merged
    tensor otherwise; per-segment scales that differ, against the closed form in fp64."""
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
        assert (np.abs(out[s] - want) <= (4e-6 if fmt == O.FMT_INT8 else 3e-4) * mag + 1e-30).all()


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
