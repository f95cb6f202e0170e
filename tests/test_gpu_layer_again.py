"""Repeated forwards of one layer take the short way; each must be bit-equal to a fresh layer's first forward."""
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


@pytest.mark.parametrize("dynamic", [False, True])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_repeated_forwards(dynamic, dt):
    layer = _layer(5, dynamic, dt)
    kept, want = [], []
    side = torch.cuda.Stream()
    for i in range(12):
        x = torch.randn(40, 1168, device=DEV).to(dt)
        form = i % 6
        if form == 1:
            x = x.view(2, 20, 1168)
        elif form == 2:  # rows of a wider tensor
            x = torch.cat([x, x], dim=1)[:, :1168]
        elif form == 3:  # another token count
            x = x[:24]
        if form == 4:
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                y = layer(x)
            torch.cuda.current_stream().wait_stream(side)
            x.record_stream(side)
            y.record_stream(torch.cuda.current_stream())
        else:
            y = layer(x)
        assert y.shape == (*x.shape[:-1], 1000) and y.dtype == dt
        kept.append(y)
        want.append(_layer(5, dynamic, dt)(x))
    for y, w in zip(kept, want):  # earlier outputs are not overwritten by later calls
        assert torch.equal(y, w)


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


@pytest.mark.parametrize("m", [8, 40])
@pytest.mark.parametrize("dynamic", [False, True])
def test_a_captured_forward_outlives_the_layers_buffers(dynamic, m):
    """Recorded on the stream that the layer was warmed up on, and replayed after that stream's buffers were given back (other
    token counts have taken the layer's few places): one launch for 8 rows, two for 40, each replay as a fresh layer's forward."""
    dt = torch.bfloat16
    layer, fresh = _layer(5, dynamic, dt), _layer(5, dynamic, dt)
    xs = [torch.randn(m, 1168, device=DEV).to(dt) for _ in range(3)]
    want = [fresh(x).clone() for x in xs]
    held = xs[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            layer(held)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = layer(held)
    with torch.cuda.stream(side):
        for other in range(50, 62):
            for _ in range(2):
                layer(torch.randn(other, 1168, device=DEV).to(dt))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    for i in (0, 1, 2, 1):
        junk = [torch.full((1 << 12,), 0x7FC0, dtype=torch.int16, device=DEV) for _ in range(200)]
        held.copy_(xs[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[i]) and all(int((t != 0x7FC0).sum()) == 0 for t in junk), (dynamic, m, i)


@pytest.mark.parametrize("dynamic", [False, True])
def test_two_threads_on_one_stream(dynamic):
    """The code buffer and the descriptors of a layer are one set per stream, whichever thread calls."""
    import threading
    layer, fresh = _layer(5, dynamic, torch.bfloat16), _layer(5, dynamic, torch.bfloat16)
    xs = [torch.randn(40, 1168, device=DEV).to(torch.bfloat16) for _ in range(3)]
    want = [fresh(x).clone() for x in xs]
    for _ in range(2):
        layer(xs[0])
    torch.cuda.synchronize()
    got = [[] for _ in xs]
    threads = [threading.Thread(target=lambda i=i: got[i].extend(layer(xs[i]) for _ in range(100))) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i, outs in enumerate(got):
        assert len(outs) == 100 and all(torch.equal(o, want[i]) for o in outs), (dynamic, i)
