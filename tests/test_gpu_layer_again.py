"""Repeated forwards of one layer."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(seed, dynamic, dt, m=40):
    from segquant_amd.layers.SegmentLinear import SegmentLinear
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randn(1000, 1168, generator=g, device=DEV) * 0.02
    x = torch.randn(m, 1168, generator=g, device=DEV)
    args = {"real_quant": True, "dual_scale": False, "axis": -1 if dynamic else None, "dynamic": dynamic}
    layer = SegmentLinear(1168, 1000, bias=True, custom_weight_tensor=w, custom_bias_tensor=torch.randn(1000, generator=g, device=DEV).to(dt),
                          input_quant_type="int8", weight_quant_type="int8", input_quant_args=args,
                          weight_quant_args={"real_quant": True, "axis": 1}, device=DEV)
    layer.calibrate(x)
    layer.finish_calibrate()
    return layer


def test_what_a_repeated_call_refuses():
    layer = _layer(5, False, torch.bfloat16)
    x = torch.randn(40, 1168, device=DEV).to(torch.bfloat16)
    for _ in range(3):
        layer(x)
    with pytest.raises(RuntimeError):
        layer(x[:, :1167])
    with pytest.raises(RuntimeError):
        layer(x.cpu())
    wide = torch.randn(40 * 1168 + 1, device=DEV).to(torch.bfloat16)
    with pytest.raises(RuntimeError, match="aligned"):
        layer(wide[1:].view(40, 1168))
