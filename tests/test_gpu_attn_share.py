"""The decode attention whose splits everybody merges (AttnShare, ts_attn.hip), as a layer without a selection cache
runs it, against the attention that merges in one workgroup (ts_sparse_decode_attn, tested against the oracle) over
the selection that the layer left: both sum in fp32, so that an output differs by the last bit of its rounding to bf16 (eight
significant bits: neighbours are up to 2^-7 of their value apart), or where its terms cancel by 2^-17 of their size (values of 4
at most, summed with weights that add up to one)."""

import ctypes
import dataclasses

import pytest
import torch

from tokenselect_amd import _lib, ops, workloads
from helpers import say

pytestmark = pytest.mark.gpu


def _workload(dev, heads, kv_heads, lens, n_init, n_local, top_k, seed=41):
    return workloads.build("share", dict(num_heads=heads, num_kv_heads=kv_heads, rope_theta=5e5), lens, [top_k] * len(lens), 1,
                           dev, seed=seed, n_init=n_init, n_local=n_local, top_k=top_k)


def _close(wl, got, q):
    out, sel, _, sel_len = got
    want = ops.sparse_decode_attention(wl.cfg, q, wl.k_pool, wl.v_pool, sel, sel_len, max_sel_len=wl.cfg.max_sel).float()
    torch.cuda.synchronize()
    assert (sel_len > 0).all()
    excess = ((out.float() - want).abs() - (2.0 ** -7 * want.abs() + 2.0 ** -15)).max().item()
    assert excess <= 0.0, excess


# (heads, KV heads, lengths, sink, window, top-k): 64 entries a workgroup and more, one to five sixteens of splits, heads'
# columns between one and 32 workgroups, splits that end within the list, short requests beside long ones
CASES = [(7, 1, [9000], 128, 512, 2048), (28, 4, [7000], 128, 512, 2048), (32, 8, [7000, 700], 128, 512, 2048),
         (1, 1, [7000], 16, 64, 600), (8, 1, [9000], 128, 512, 4096), (6, 2, [7000, 1, 3000], 64, 128, 513),
         (48, 8, [6000], 100, 300, 1700), (40, 8, [6000, 6500], 128, 512, 2048), (16, 8, [6000, 2000, 5000], 128, 512, 1024),
         (8, 8, [6000] * 4, 128, 512, 1024), (2, 1, [8000], 0, 1, 639), (2, 1, [8000], 0, 1, 640), (2, 1, [8000], 0, 1, 5119)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "H%dkv%d-%s-%d" % (c[0], c[1], "-".join(map(str, c[2])), sum(c[3:])))
def test_splits_merged_by_everybody(dev, case):
    """Steps one after the other on one workspace, the first of which clears it, between calls that use it otherwise."""
    say("attention merged by everybody H=%d kv=%d lens=%s %s" % (case[0], case[1], case[2], case[3:]))
    wl = _workload(dev, *case)
    B, longest = len(wl.seq_lens), max(wl.seq_lens)
    layer = ops.DecodeLayer(wl.cfg, B, longest, dev)
    g = torch.Generator(device=dev).manual_seed(42)
    first = None
    for step in range(5):
        q = wl.q if step % 2 == 0 else torch.randn(wl.q.shape, generator=g, device=dev).bfloat16()
        got = [t.clone() for t in layer(q, wl.k_pool, wl.v_pool, wl.batch)]
        torch.cuda.synchronize()
        assert not layer.gave_up() and layer._clean_for is not None
        _close(wl, got, q)
        if step == 0:
            first = got[0]
        elif step % 2 == 0:
            assert torch.equal(got[0].view(torch.int16), first.view(torch.int16)), step


def test_a_call_on_separate_kernels_leaves_the_words_zero(dev):
    """A workspace that a call on the separate kernels used last may be called clean: their scores are where the words lie."""
    say("separate kernels, then a clean workspace")
    wl = _workload(dev, 28, 4, [7000], 128, 512, 2048)
    c, n = wl.cfg, max(wl.seq_lens)
    lib, cc = _lib.load(), c.to_c()
    layer = ops.DecodeLayer(c, 1, n, dev)
    outs = []
    for options in (dict(), dict(separate_kernels=True), dict(workspace_clean=True), dict(workspace_clean=True)):
        bt = ops._c_batch(c, dataclasses.replace(wl.batch, **options))
        assert lib.ts_decode_layer(ctypes.byref(cc), ctypes.byref(bt), wl.q.data_ptr(), layer.q_cos.data_ptr(),
                                   layer.q_sin.data_ptr(), wl.k_pool.data_ptr(), wl.v_pool.data_ptr(), wl.k_pool.shape[0], None,
                                   layer.out.data_ptr(), layer.sel.data_ptr(), layer.sel_pos.data_ptr(), layer.sel.shape[1],
                                   layer.sel_len.data_ptr(), layer.workspace.data_ptr(), layer.workspace.numel(),
                                   torch.cuda.current_stream().cuda_stream) == _lib.TS_OK, lib.ts_last_error()
        torch.cuda.synchronize()
        outs.append(layer.out[0].view(torch.int16).clone())
    assert torch.equal(outs[0], outs[2]) and torch.equal(outs[0], outs[3])


@pytest.mark.parametrize("absent", [1, 3])
def test_an_attention_that_gives_up(dev, absent):
    """Splits that send nothing (forced from the host) and a 20 us bound: every kernel ends, the step is reported as one whose
    selection gave up, recover() repeats it on the separate kernels, and an object that nobody recovers raises."""
    say(f"attention gives up, {absent} splits absent")
    wl = _workload(dev, 32, 8, [7000, 700], 128, 512, 2048)
    forced = dataclasses.replace(wl.batch, wait_us=20, absent_workgroups=-absent)
    layer = ops.DecodeLayer(wl.cfg, 2, 7000, dev)
    for _ in range(2):
        want = [t.clone() for t in layer(wl.q, wl.k_pool, wl.v_pool, wl.batch)]
    out, _, _, sel_len = layer(wl.q, wl.k_pool, wl.v_pool, forced)
    torch.cuda.synchronize()
    assert layer.gave_up() and sel_len.tolist() == [-1, -1] and torch.isfinite(out.float()).all()
    got = layer.recover(wl.q, wl.k_pool, wl.v_pool, forced)
    torch.cuda.synchronize()
    assert got is not None and layer.separate and not layer.gave_up()
    assert torch.equal(got[3], want[3]) and torch.equal(got[1][0], want[1][0])
    _close(wl, got, wl.q)
    other = ops.DecodeLayer(wl.cfg, 2, 7000, dev)
    other(wl.q, wl.k_pool, wl.v_pool, forced)
    torch.cuda.synchronize()
    with pytest.raises(ops.SelectionGaveUp):
        other(wl.q, wl.k_pool, wl.v_pool, wl.batch)
    _close(wl, other(wl.q, wl.k_pool, wl.v_pool, wl.batch), wl.q)


def _nodes(graph):
    """Launches in a captured graph, of the runtime that captured it."""
    with open("/proc/self/maps") as maps:
        path = next(line.split()[-1] for line in maps if "libamdhip64.so" in line)
    count = ctypes.c_size_t(0)
    assert ctypes.CDLL(path).hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    return count.value


@pytest.mark.parametrize("stated", [False, True], ids=["unstated", "stated clean"])
@pytest.mark.parametrize("case", [(28, 4, [20000]), (32, 8, [9000, 3000])], ids=lambda c: "H%dkv%d" % c[:2])
def test_a_captured_layer(dev, case, stated):
    """At a model's sizes: the rotation (which clears the words where the caller states nothing), the selection and the attention,
    and no launch besides; replays with other queries, eager work and synchronisations in between, give the eager call's bits."""
    say(f"captured attention merged by everybody {case} stated={stated}")
    wl = _workload(dev, *case, 128, 512, 2048)
    B, longest = len(wl.seq_lens), max(wl.seq_lens)
    bt = dataclasses.replace(wl.batch, workspace_clean=stated)
    layer, eager = (ops.DecodeLayer(wl.cfg, B, longest, dev) for _ in range(2))
    q = wl.q.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the first calls load code objects and size the grids
        for _ in range(2):
            layer(q, wl.k_pool, wl.v_pool, wl.batch)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        out, sel, _, sel_len = layer(q, wl.k_pool, wl.v_pool, bt)
    assert _nodes(graph) == (2 if stated else 3)
    g = torch.Generator(device=dev).manual_seed(43)
    for replay in range(5):
        q.copy_(torch.randn(q.shape, generator=g, device=dev))
        if not stated and replay == 3:
            layer.workspace.fill_(0xa5)  # whatever used it in between
        graph.replay()
        torch.cuda.synchronize()
        layer.check()
        want = eager(q, wl.k_pool, wl.v_pool, wl.batch)
        torch.cuda.synchronize()
        assert torch.equal(sel_len, want[3]), replay
        for b, n in enumerate(sel_len.tolist()):
            assert torch.equal(sel[b, :n], want[1][b, :n]), replay
        assert torch.equal(out.view(torch.int16), want[0].view(torch.int16)), replay


# the contexts from which the words fit where separate kernels have their scores (k = 2048), and one below
LINE = [((28, 4, [4608]), False), ((28, 4, [4609]), True), ((12, 2, [4480]), False), ((12, 2, [4481]), True),
        ((4, 1, [4096]), False), ((4, 1, [4097]), True), ((32, 8, [2689]), True), ((28, 4, [2700, 2689]), True), ((64, 8, [2689]), True), ((56, 8, [5000, 900]), True)]


@pytest.mark.parametrize("case,shares", LINE, ids=lambda c: "H%dkv%d-%d" % (c[0], c[1], c[2][0]) if isinstance(c, tuple) else str(c))
def test_where_the_words_fit(dev, case, shares):
    """Both sides of the line give the other attention's output; splits forced to be absent tell who waits."""
    say(f"attention where the words fit: {case} {shares}")
    wl = _workload(dev, *case, 128, 512, 2048)
    B, longest = len(wl.seq_lens), max(wl.seq_lens)
    layer = ops.DecodeLayer(wl.cfg, B, longest, dev)
    for _ in range(3):
        got = layer(wl.q, wl.k_pool, wl.v_pool, wl.batch)
        _close(wl, got, wl.q)
    layer(wl.q, wl.k_pool, wl.v_pool, dataclasses.replace(wl.batch, wait_us=20, absent_workgroups=-1))
    torch.cuda.synchronize()
    assert layer.gave_up() == shares


@pytest.mark.parametrize("before", [0, 2], ids=["stored ahead", "stored by the selection"])
def test_a_step_whose_attention_gives_up(dev, before):
    """The store of a step that gives up has happened, whichever launch it rode in: recover() repeats selection and attention
    alone, lengths advance once, and pools, table and output are those of an object that nothing disturbed."""
    say(f"step whose attention gives up, {before} steps before it")
    wl = _workload(dev, 28, 4, [7000, 6000], 128, 512, 2048)
    g = torch.Generator(device=dev).manual_seed(44)
    width, steps = 7000 + 8, before + 2
    spare = torch.arange(wl.k_pool.shape[0], wl.k_pool.shape[0] + 2 * steps, dtype=torch.int32, device=dev).view(steps, 2)
    qs = torch.randn((steps, *wl.q.shape), generator=g, device=dev).bfloat16()
    kv = torch.randn((steps, 2, 2, 4, 128), generator=g, device=dev).bfloat16()

    def serve(forced_at):
        pools = [torch.cat((p, torch.zeros((2 * steps, 4, 128), dtype=p.dtype, device=dev))) for p in (wl.k_pool, wl.v_pool)]
        table = torch.zeros((2, width), dtype=torch.int32, device=dev)
        table[:, :wl.table.shape[1]] = wl.table
        lens = wl.seq_lens_dev.clone()
        layer = ops.DecodeLayer(wl.cfg, 2, 7000 + steps, dev)
        for t in range(steps):
            bt = ops.Batch(lens, table, 7000 + steps)
            if t == forced_at:
                bt = dataclasses.replace(bt, wait_us=20, absent_workgroups=-1)
            assert (layer._clean_for is not None) == (t > 0 and not layer.separate)
            got = layer.step(qs[t], kv[t, 0], kv[t, 1], spare[t], *pools, bt)
            torch.cuda.synchronize()
            assert lens.tolist() == [7000 + t + 1, 6000 + t + 1]
            if t == forced_at:
                assert layer.gave_up() and got[3].tolist() == [-1, -1]
                got = layer.recover(qs[t], *pools, bt)
                torch.cuda.synchronize()
            assert not layer.gave_up() and lens.tolist() == [7000 + t + 1, 6000 + t + 1]
        return [x.clone() for x in got], pools, table, lens

    (got, pools, table, lens), (want, pools_w, table_w, lens_w) = serve(before), serve(None)
    for a, b in ((pools[0], pools_w[0]), (pools[1], pools_w[1])):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert torch.equal(table, table_w) and torch.equal(lens, lens_w) and torch.equal(got[3], want[3])
    for b, n in enumerate(got[3].tolist()):  # (the separate kernels' votes are added up in another order: ties only)
        assert len(set(got[1][b, :n].tolist()) ^ set(want[1][b, :n].tolist())) <= 2
    full = dataclasses.replace(wl, k_pool=pools[0], v_pool=pools[1])
    _close(full, got, qs[-1])
