"""The workgroup-per-row quantise kernel where it takes over: one run of 16 per thread, up to eight waves a row."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt", ["int8", "fpe4m3"])
@pytest.mark.parametrize("cols", [16, 1008, 1024, 1040, 2064, 4096, 4112, 7184, 8192])
def test_workgroup_per_row_equals_wave_per_row(dt, fmt, cols):
    """Dividing by ones changes nothing but the kernel: codes and scales equal the plain launch's (one wave per row) bit for bit,
    on both sides of the row count (three per compute unit) where longer rows change kernels."""
    from segquant_amd import ops
    edge = 3 * torch.cuda.get_device_properties(0).multi_processor_count
    for rows in (1, 5, edge, edge + 1):
        x = torch.randn(rows, cols, device=DEV)
        x[:, cols // 2] *= 30
        if rows > 4:
            x[0] = 0
            x[1, 3] = float("nan")
            x[2, cols - 1] = float("inf")
        x = x.to(dt)
        out = []
        for div in (None, torch.ones(cols, device=DEV)):
            scale = torch.empty(rows, device=DEV)
            out.append((ops.quantize(x, fmt, scale, row_stride=1, dynamic=True, col_div=div).view(torch.uint8), scale.view(torch.int32)))
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1]), (dt, fmt, rows, cols)


@pytest.mark.parametrize("cols", [1280, 5120])
def test_gated_rows_do_not_depend_on_the_row_count(cols):
    from segquant_amd import ops
    edge = 3 * torch.cuda.get_device_properties(0).multi_processor_count
    x, gate = (torch.randn(edge + 8, cols, device=DEV).to(torch.bfloat16) for _ in range(2))
    out = []
    for rows in (edge + 8, edge):
        pos, neg = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
        kw = dict(row_stride=1, dynamic=True, pre_op="gelu", gate=gate[:rows], dual=True, two_tensors=True)
        a, b = ops.quantize(x[:rows], "int8", pos, neg, **kw)
        out.append([t[:edge] for t in (a, b, pos, neg)])
    assert all(torch.equal(p, q) for p, q in zip(*out))
