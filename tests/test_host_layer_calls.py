"""What a layer keeps between calls, on the host: descriptors filled for CPU buffers, nothing launched."""
import copy
import pickle
import threading
import time
import types

import pytest
import torch

from segquant_amd import ops
from segquant_amd.optimum import optimizer as opt_mod, smooth  # noqa: F401 (registers the smoothing optimisers)
from segquant_amd.optimum.optimizer import OptimizerRegistry

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


class _OnTheGpu:
    """Enough of a tensor for a repeated call, wherever its memory is."""
    is_cuda = True
    device = torch.device("cpu")

    def __init__(self):
        self.t = torch.empty(M, K)
        self.shape, self.dtype = self.t.shape, self.t.dtype
        self.is_contiguous, self.numel, self.data_ptr = self.t.is_contiguous, self.t.numel, self.t.data_ptr


def test_repeated_calls_of_two_threads_keep_their_tensors_together(layer, monkeypatch):
    """Two threads on one stream share the descriptors and buffers of a layer: between one call's addresses and the end of its
    launches no other call may write its own (the library is entered without the interpreter's lock)."""
    inside, seen = [0], []

    class Library:
        def segq_linear(self, qd, gd, stream):
            q, g = qd._obj, gd._obj
            inside[0] += 1
            first = (q.x, g.out, inside[0])
            time.sleep(1e-3)
            seen.append((first, (q.x, g.out, inside[0])))
            inside[0] -= 1
            return 0

    monkeypatch.setattr(ops.L, "lib", lambda: Library())
    hit = _hit()
    layer._relaunch(hit, torch.empty(M, K))
    layer._plan = {"K": K, "launches": {(M, torch.float32, None): hit}}
    outs = {}

    def calls(x):
        outs[x] = [layer._again(x, None) for _ in range(25)]

    xs = [_OnTheGpu() for _ in range(3)]
    threads = [threading.Thread(target=calls, args=(x,)) for x in xs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(a == b and a[2] == 1 for a, b in seen) and len(seen) == 75
    owner = {o.data_ptr(): x.data_ptr() for x in xs for o in outs[x]}
    assert all(owner[out] == x for (x, out, _), _ in seen)


def test_the_default_stream_is_not_asked_for_a_capture(monkeypatch):
    """It records no graph, and the question costs a repeated call of a small layer some of its time."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: pytest.fail("asked"))
    assert ops.capturing(0) is False


def test_calls_that_share_no_buffers_take_no_lock(layer, monkeypatch):
    """A layer that keeps nothing between its calls, and any call with more than an input, go straight to their launches; the
    others hold the lock of their stream."""
    held = []

    class Lock:
        def __enter__(self):
            held.append(True)

        def __exit__(self, *exc):
            held.pop()

    monkeypatch.setattr(ops, "stream_lock", {"A": Lock()})
    monkeypatch.setattr(layer, "_again", lambda x, bias: None, raising=False)
    monkeypatch.setattr(layer, "_enqueue", lambda *a: bool(held), raising=False)
    x = torch.empty(M, K)
    for plan, kw, locked in ((None, {}, False), ({"K": K}, {}, False), ({"K": K, "launches": {}}, {}, True),
                             ({"K": K, "launches": {}}, {"pre_op": "gelu"}, False), ({"K": K, "launches": {}}, {"addend": x}, False)):
        layer._plan = plan
        assert layer.forward_fused(x, **kw) is locked


def _fused_layer(layer, monkeypatch, rows, k, n, l2t=None):
    """The layer's fused route on CPU tensors (never read: nothing is launched), with a plan for int8 codes; what it lends."""
    lent = []
    monkeypatch.setattr(ops, "_need_cuda", lambda *ts: None)
    monkeypatch.setattr(ops, "int4_workspace", lambda device, need: lent.append(need) or torch.empty(1, dtype=torch.uint8))
    one = torch.ones(1)
    layer.chunks, layer.seg_mode, layer.dual_scale, layer.dual_segments = 1, "weight", False, [False]
    layer.input_calibrators = [types.SimpleNamespace(dynamic=False)]
    layer._plan = dict(fa="int8", fw="int8", w=torch.empty(n, k, dtype=torch.int8), sw=one, sw_cs=0, bounds=[0, k], N=n, K=k, sx=(one[None], None))
    if l2t is not None:
        layer._plan["l2t"] = l2t
        layer._lowrank_operands = lambda plan, x2: (torch.empty(rows, l2t.shape[1], dtype=x2.dtype), l2t.to(x2.dtype))
    return lent


def test_a_launch_without_shares_leaves_those_of_other_launches_their_workspace(layer, monkeypatch):
    """256 x 3072 x 12288 is shared along K, but not with codes out or with a low-rank branch in the epilogue: whichever comes
    first, every launch is lent what it can use itself."""
    rows, k, n = 256, 12288, 3072
    x = torch.empty(rows, k, dtype=torch.bfloat16)
    spec = dict(fmt="int8", scale=torch.ones(1))
    for calls in (("codes", "plain"), ("plain", "codes")):
        lent = _fused_layer(layer, monkeypatch, rows, k, n)
        for call in calls:
            ws = layer.fused_launches(x, out_codes=spec if call == "codes" else None)[2]
            assert (ws is None) == (call == "codes")
        assert len(lent) == 1 and lent[0] > 0
    lent = _fused_layer(layer, monkeypatch, rows, k, n, l2t=torch.empty(n, 32))
    assert layer.fused_launches(x)[2] is None  # the branch is in the epilogue
    assert layer.fused_launches(x.float())[2] is not None and lent[0] > 0  # 32-bit outputs have it as an addend


def test_answers_kept_per_token_count_are_bounded(layer, monkeypatch):
    """A layer fed with ever-changing token counts keeps no more of the library's answers than a fixed number."""
    k, n, most = 128, 256, opt_mod._MAX_ANSWERS
    counts = range(1, 2 * most + 3)
    monkeypatch.setattr(ops, "lowrank_tile", lambda g: 0)
    _fused_layer(layer, monkeypatch, 0, k, n)
    layer._lowrank_operands = lambda plan, x2: (torch.empty(x2.shape[0], 32, dtype=x2.dtype), torch.empty(n, 32, dtype=x2.dtype))
    layer._plan["l2t"] = torch.empty(n, 32)
    for m in counts:
        layer.fused_launches(torch.empty(m, k, dtype=torch.bfloat16))
    layer.dual_segments = [True]
    plan = {k_: v for k_, v in layer._plan.items() if k_ != "l2t"}
    monkeypatch.setattr(ops, "dual_in_one_tensor", lambda *a: True)
    for m in counts:
        assert layer._one_code_tensor(plan, m, torch.bfloat16) is True
    for table in (layer._plan["lr_ok"], layer._plan["lr_tile"], layer._plan["ws_need"], plan["one_tensor"]):
        assert 0 < len(table) <= most
    assert layer._plan["lr_ok"][counts[-1], torch.bfloat16] is True  # (a full table starts anew: the newest is there)


@pytest.mark.parametrize("again", [lambda o: pickle.loads(pickle.dumps(o)), copy.deepcopy])
def test_a_loaded_layer_makes_a_plan_of_its_own(again):
    """A layer saved after its first call has a plan in the file, of the version that saved it: one from before the transposed
    low-rank factors has none of them, and the layer must not look for them there."""
    opt = object.__new__(OptimizerRegistry.get("svd"))
    opt.__dict__.update(low_rank=32, chunks=1, _plan=dict(K=K, N=N, l2t=torch.empty(N, 32), l12_cast={}))
    loaded = again(opt)
    assert loaded._plan is None and (loaded.low_rank, loaded.chunks) == (32, 1) and opt._plan is not None


@pytest.mark.parametrize("again", [lambda o: pickle.loads(pickle.dumps(o)), copy.deepcopy])
def test_a_copy_of_a_planned_layer_is_ready_for_a_capture(again):
    """A plan that is made while a graph is recorded holds tensors without contents until the graph runs: the copy of a layer that
    has one keeps it."""
    opt = object.__new__(OptimizerRegistry.get("smooth"))
    one = torch.ones(N)
    opt.__dict__.update(chunks=1, seg_mode="weight", chunksizes=[N], kernel_type="Wint8Aint8", s=[torch.ones(K)], _plan=None,
                        weight_manager=types.SimpleNamespace(out_features=N, in_features=K, weight_tensor=torch.zeros(N, K, dtype=torch.int8)),
                        weight_calibrators=[types.SimpleNamespace(scale=one)])
    opt._build_plan(torch.device("cpu"))
    loaded = again(opt)
    assert loaded._plan is not None and loaded._plan is not opt._plan and torch.equal(loaded._plan["w"], opt._plan["w"])
