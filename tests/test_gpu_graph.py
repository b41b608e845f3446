"""The decode layer under HIP graph capture, the way a serving stack replays a decode step:
`ts_decode_layer` only launches kernels (its side jobs, clearing counters and tickets, are
kernels too), so a captured call replays with new queries, new lengths and new table
contents in the same buffers.  Every replay is checked against an eager call of a second
layer object on the same inputs, with eager work and synchronisations in between."""

import ctypes
import dataclasses

import pytest
import torch

from helpers import say
from tokenselect_amd import _lib, ops, workloads

pytestmark = pytest.mark.gpu

SHAPE = dict(num_heads=32, num_kv_heads=8, rope_theta=5e5)


@pytest.fixture
def fused_select(request):
    previous = ops.set_fused_select(request.param)
    yield request.param
    ops.set_fused_select(previous)


def _capture(layer, q, k_pool, v_pool, bt):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the first calls load code objects and size the grids
        for _ in range(2):
            layer(q, k_pool, v_pool, dataclasses.replace(bt, workspace_clean=False))
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = layer(q, k_pool, v_pool, bt)
    return graph, outputs


@pytest.mark.parametrize("fused_select", [True, False], indirect=True, ids=["fused", "separate"])
@pytest.mark.parametrize("pool_kernel", [-1, 5], ids=["plain", "max-pool"])
def test_decode_layer_replays_in_a_graph(dev, fused_select, pool_kernel):
    lens, ks = [5000, 100, 2048, 901], [256, 256, 200, 256]
    say(f"decode_layer in a graph: fused={fused_select} pool_kernel={pool_kernel}")
    wl = workloads.build("small", SHAPE, lens, ks, 16, dev, 61, n_init=16, n_local=32, top_k=256,
                         pool_kernel=pool_kernel)
    c, bt = wl.cfg, wl.batch
    q = wl.q.clone()
    layer = ops.DecodeLayer(c, len(lens), max(lens), dev)
    eager = ops.DecodeLayer(c, len(lens), max(lens), dev)
    graph, (out, sel, sel_pos, sel_len) = _capture(layer, q, wl.k_pool, wl.v_pool, bt)
    gen = torch.Generator(device=dev).manual_seed(62)
    for replay in range(5):
        # new inputs in the captured buffers: another query, shorter contexts from the
        # third replay on (a request of 100 tokens stays dense), new keys in the pool
        q.copy_(torch.randn(q.shape, device=dev, generator=gen).to(q.dtype))
        if replay >= 2:
            bt.seq_lens.sub_(torch.tensor([37, 0, 5, 1], dtype=torch.int32, device=dev))
        if replay == 3:
            wl.k_pool[::7].mul_(-1)
        graph.replay()
        torch.cuda.synchronize()
        layer.check()
        got = [t.clone() for t in (out, sel, sel_pos, sel_len)]
        want = eager(q, wl.k_pool, wl.v_pool, bt)
        torch.cuda.synchronize()
        assert torch.equal(got[3], want[3]), f"replay {replay}: lengths"
        for b in range(len(lens)):
            S = int(want[3][b])
            assert torch.equal(got[2][b, :S], want[2][b, :S]), f"replay {replay} b={b}: positions"
            assert torch.equal(got[1][b, :S], want[1][b, :S]), f"replay {replay} b={b}: slots"
        assert torch.equal(got[0].view(torch.int16), want[0].view(torch.int16)), f"replay {replay}: out"
    # and the replays moved with their inputs: the last lengths are the shortened ones
    assert sel_len.tolist() == [16 + 256 + 32, 100, 16 + 200 + 32, 16 + 256 + 32]


@pytest.fixture
def stated(monkeypatch):
    """The layer calls reach a function that notes what they state of the workspace and launches
    nothing."""
    lib, flags = _lib.load(), []

    def note(cfg, bt, *rest):
        flags.append(bt.contents.workspace_clean)
        return _lib.TS_OK

    restype, argtypes = _lib.SIGNATURES["ts_decode_layer"]
    layer = ctypes.CFUNCTYPE(restype, *argtypes)(note)
    names = ("ts_decode_layer", "ts_decode_step_strided", "ts_prefill_chunk", "ts_prefill_step_strided",
             "ts_decode_layer_layout")
    real = [ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in names]
    bind = _lib.binding()
    bind.connect(ctypes.cast(layer, ctypes.c_void_p).value, *real[1:])
    yield flags
    bind.connect(*real)


def test_no_call_vouches_for_a_workspace_that_a_graph_uses(dev, stated):
    """What the object says of its workspace: nothing in a captured call, whatever ran before it,
    and nothing after one, since the object does not see the replays.  The caller may."""
    wl = workloads.build("small", SHAPE, [2048, 901], [256, 256], 16, dev, 63, n_init=16, n_local=32, top_k=256)
    bt = wl.batch
    longer = dataclasses.replace(bt, max_seq_len=bt.max_seq_len - 1)   # (of the same layout)
    some = torch.zeros(8, device=dev)

    def capture(layer, b, call=True):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            some.add_(1)
            if call:
                layer(wl.q, wl.k_pool, wl.v_pool, b)
            else:
                layer._clean_for = None   # (what votes() and attend() do)

    for call in (True, False):
        layer = ops.DecodeLayer(wl.cfg, 2, 2048, dev)
        del stated[:]
        for b in (longer, longer, bt):
            layer(wl.q, wl.k_pool, wl.v_pool, b)
        assert stated == [0, 1, 1] and layer._clean_for == (2, 2048)
        del stated[:]
        capture(layer, bt, call)
        for _ in range(3):
            layer(wl.q, wl.k_pool, wl.v_pool, bt)
        assert stated == ([0] if call else []) + [0, 0, 0] and layer._clean_for is None
        layer(wl.q, wl.k_pool, wl.v_pool, dataclasses.replace(bt, workspace_clean=True))
        assert stated[-1] == 1


def test_what_ends_the_memory_of_a_clean_workspace(dev, stated):
    """A call of the same layout states that the workspace is clean; the one after a call of another
    layout, with a selection cache, with the separate kernels or split at the vote does not."""
    wl = workloads.build("small", SHAPE, [2048, 901], [256, 256], 16, dev, 63, n_init=16, n_local=32, top_k=256)
    bt, args = wl.batch, (wl.q, wl.k_pool, wl.v_pool)
    layer = ops.DecodeLayer(wl.cfg, 2, 2048, dev)
    one = ops.Batch(bt.seq_lens[:1], bt.table[:1], 2048)
    short = dataclasses.replace(bt, max_seq_len=1000)
    cache = ops.SelectionCache.allocate(wl.cfg, 2, dev)

    def split():
        layer.attend(wl.q, layer.votes(wl.q, wl.k_pool, bt), wl.k_pool, wl.v_pool, bt)

    def refused():
        with pytest.raises(ValueError):
            layer(wl.q[:, 1:], wl.k_pool, wl.v_pool, bt)

    between = {"nothing": (lambda: None, 1),
               "same layout": (lambda: layer(*args, dataclasses.replace(bt, max_seq_len=2047)), 1),
               "batch": (lambda: layer(wl.q[:1], *args[1:], one), 0), "length": (lambda: layer(*args, short), 0),
               "cache": (lambda: layer(*args, bt, cache=cache), 0), "split": (split, 0),
               "separate": (lambda: layer(*args, dataclasses.replace(bt, separate_kernels=True)), 0),
               "refused before anything ran": (refused, 1)}
    for name, (call, after) in between.items():
        layer(*args, bt)
        layer(*args, bt)
        assert stated[-1] == 1, name
        call()
        layer(*args, bt)
        assert stated[-1] == after, name


@pytest.mark.parametrize("said", [False, True], ids=["full", "caller says clean"])
def test_replays_and_eager_steps_share_a_workspace(dev, said):
    """A captured step and eager steps of two other shapes on one object, in turn; where the
    caller says that the captured call finds its counters clean, only calls of its layout run
    between the replays."""
    say(f"replays and eager steps in turn: said={said}")
    wl = workloads.build("small", SHAPE, [5000, 100, 2048, 901], [256] * 4, 16, dev, 64, n_init=16, n_local=32,
                         top_k=256)
    bt, q = wl.batch, wl.q.clone()
    steps = [bt, dataclasses.replace(bt, max_seq_len=5001)]
    if not said:
        pair = ops.Batch(bt.seq_lens[2:], bt.table[2:].contiguous(), 2048)
        steps += [pair, pair, bt]
    layer = ops.DecodeLayer(wl.cfg, 4, 5001, dev)
    layout = {_lib.load().ts_decode_layer_layout(ctypes.byref(layer._c), 4, n) for n in (5000, 5001)}
    assert len(layout) == 1

    def check(got, b):
        fresh = ops.DecodeLayer(wl.cfg, 4, 5001, dev)
        want = fresh(q if b.batch == 4 else q[2:].contiguous(), wl.k_pool, wl.v_pool, b)
        torch.cuda.synchronize()
        layer.check()
        assert torch.equal(got[3], want[3])
        for r in range(b.batch):
            S = int(want[3][r])
            assert torch.equal(got[1][r, :S], want[1][r, :S]) and torch.equal(got[2][r, :S], want[2][r, :S])
        assert torch.equal(got[0].view(torch.int16), want[0].view(torch.int16))

    graph, outputs = _capture(layer, q, wl.k_pool, wl.v_pool, dataclasses.replace(bt, workspace_clean=said))
    gen = torch.Generator(device=dev).manual_seed(65)
    for replay in range(4):
        q.copy_(torch.randn(q.shape, device=dev, generator=gen).to(q.dtype))
        graph.replay()
        check([t.clone() for t in outputs], bt)
        for b in steps:
            mine = q if b.batch == 4 else q[2:].contiguous()
            check([t.clone() for t in layer(mine, wl.k_pool, wl.v_pool, b)], b)
