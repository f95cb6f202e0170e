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


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cols", [1040, 2064, 3072, 3088])
def test_many_rows_with_divisors_equal_plain_rows(dt, cols, dual):
    """A wave per row or a workgroup: both sides of the row counts (6 and 14 per compute unit) between which they change."""
    from segquant_amd import ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for rows in (6 * cus, 6 * cus + 1, 10 * cus + 1, 14 * cus, 14 * cus + 1):
        x = torch.randn(rows, cols, device=DEV)
        x[0], x[1, 3], x[2, cols - 1] = 0, float("nan"), float("inf")
        x = x.to(dt)
        out = []
        for div in (None, torch.ones(cols, device=DEV)):
            pos, neg = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
            codes = ops.quantize(x, "int8", pos, neg if dual else None, row_stride=1, dynamic=True, col_div=div, dual=dual, two_tensors=dual)
            out.append([t.view(torch.uint8) for t in (codes if dual else (codes,))] + [t.view(torch.int32) for t in ((pos, neg) if dual else (pos,))])
        assert all(torch.equal(p, q) for p, q in zip(*out)), (dt, cols, dual, rows)


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("widths", [(16, 1024), (16, 48, 1040), (512, 1008, 16, 528), (1024, 4096)])
def test_segments_equal_their_own_launches(dt, widths, dual):
    """Column segments of a wave at most, and of more, against launches of one segment each: codes and scales bit for bit."""
    from segquant_amd import ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    bounds = [sum(widths[:i]) for i in range(len(widths) + 1)]
    for rows in (1, 7, 14 * cus, 14 * cus + 1):
        x = torch.randn(rows, bounds[-1], device=DEV)
        x[0, bounds[1]] = float("nan")
        x[rows - 1, :16] = 0
        x = x.to(dt)
        pos, neg = torch.empty(len(widths), rows, device=DEV), torch.empty(len(widths), rows, device=DEV)
        kw = dict(row_stride=1, dynamic=True, dual=dual, two_tensors=dual)
        got = ops.quantize(x, "int8", pos, neg if dual else None, kseg_bounds=bounds, kseg_stride=rows, **kw)
        for s, (c0, c1) in enumerate(zip(bounds, bounds[1:])):
            p, n = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
            want = ops.quantize(x[:, c0:c1].contiguous(), "int8", p, n if dual else None, **kw)
            assert torch.equal(p.view(torch.int32), pos[s].view(torch.int32)) and (not dual or torch.equal(n.view(torch.int32), neg[s].view(torch.int32))), (dt, widths, rows, s)
            for g, w in zip(got if dual else (got,), want if dual else (want,)):
                assert torch.equal(g[:, c0:c1], w), (dt, widths, rows, s)


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cols", [16, 5136, 7184, 8192, 12304, 16400])
def test_divisors_alone_equal_a_division_in_front(cols, dt, dual):
    """A wave, a workgroup with four runs a thread, and a row that is longer than those; scales of the row and given ones.  The
    division is one of fp32 rounded to the type, as torch's, so codes and scales are equal bit for bit."""
    from segquant_amd import ops
    rows = 3 * torch.cuda.get_device_properties(0).multi_processor_count + 1
    x, div = torch.randn(rows, cols, device=DEV).to(dt), (torch.rand(cols, device=DEV) * 4 + 0.05).to(dt)
    x[0], x[1, 3], x[2, cols - 1] = 0, float("nan"), float("inf")
    for dynamic in (True, False):
        out = []
        for t, kw in ((x, dict(col_div=div)), (x / div, {})):
            pos, neg = torch.full((rows,), 30.0, device=DEV), torch.full((rows,), 50.0, device=DEV)
            codes = ops.quantize(t, "int8", pos, neg if dual else None, row_stride=1, dynamic=dynamic, dual=dual, two_tensors=dual, **kw)
            out.append(list(codes if dual else (codes,)) + [s.view(torch.int32) for s in (pos, neg)])
        assert all(torch.equal(p, q) for p, q in zip(*out)), (dt, cols, dual, dynamic)
