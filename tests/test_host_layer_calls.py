"""What a layer keeps between calls, on the host: descriptors filled for CPU buffers, nothing launched."""
import pytest
import torch

from segquant_amd import ops
from segquant_amd.optimum import optimizer as opt_mod

M, N, K = 4, 8, 16


def _hit(need=0, workspace=None):
    """What the first call of a token count leaves behind (``fused_launches``)."""
    q, g = ops.L.QuantDesc(), ops.L.GemmDesc()
    g.workspace, g.workspace_bytes = workspace, need
    return dict(q=(q, {}), g=(g, {}), need=need, dyn=False, dual=False, S=1, M=M, N=N, sx_src=[(0, 0)], code_shape=(M, K),
                code_dtype=torch.int8, out_dtype=torch.float32, static=None)


@pytest.fixture
def layer(monkeypatch):
    """An optimiser without weights, and the current stream under the test's control."""
    opt = object.__new__(opt_mod.DefaultOptimizer)
    opt.stream, opt.capture = "A", False
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: opt.capture)
    monkeypatch.setattr(ops, "_stream", lambda device=None: opt.stream)
    monkeypatch.setattr(ops, "_int4_ws", {})
    return opt


def test_descriptors_of_another_stream_get_that_streams_workspace(layer):
    """The first call ran on stream A with A's workspace; the descriptors that a later call on B leaves for the ones after it
    name B's, whether or not that call's own launch has been enqueued yet."""
    hit = _hit(64, ops.int4_workspace("cpu", 64).data_ptr())
    x = torch.empty(M, K)
    for stream in ("B", "A"):
        layer.stream = stream
        layer._relaunch(hit, x)
        kept = hit["buffers"][stream][1]
        assert kept.workspace == ops.int4_workspace("cpu", 64).data_ptr() and kept.workspace_bytes == 64


def test_a_capture_takes_buffers_of_its_own(layer):
    """What a graph replays must not lie where eager calls, or another graph captured on the same stream, put theirs, nor where
    a layer fed with many token counts gives its buffers back."""
    room = ops.int4_workspace("cpu", 64)
    hit, x = _hit(64, room.data_ptr()), torch.empty(M, K)
    eager = layer._relaunch(hit, x)
    layer.capture = True
    first, second = layer._relaunch(hit, x), layer._relaunch(hit, x)
    layer.capture = False
    after = layer._relaunch(hit, x)
    assert after[0][0].codes == eager[0][0].codes and after[1][0].workspace == room.data_ptr()  # eager calls reuse theirs
    for at in (lambda r: r[0][0].codes, lambda r: r[1][0].workspace, lambda r: r[2].data_ptr()):
        assert len({at(r) for r in (eager, first, second)}) == 3
    assert list(hit["buffers"]) == ["A"] and ops.int4_workspace("cpu", 64) is room
