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
