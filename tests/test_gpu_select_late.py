"""What a layer's selection does in place of meetings (ts_score.hip): the wide band around a hint and the candidates that
are sent late.  The selection of a layer against that of ts_select without a hint, which meets: the same slots,
positions and lengths, for hints right, off by any number of bins up to beyond the wide band, and nonsense; few
workgroups with many candidates each, more of them than fit, ties, batches, and calls without a hint."""

import dataclasses

import pytest
import torch

from tokenselect_amd import ops, workloads
from helpers import say

pytestmark = pytest.mark.gpu


def _workload(dev, heads, kv_heads, lens, top_k, page=1, seed=51, pool=-1, same=0):
    wl = workloads.build("late", dict(num_heads=heads, num_kv_heads=kv_heads, rope_theta=5e5), lens, [top_k] * len(lens), page,
                         dev, seed=seed, n_init=64, n_local=128, top_k=top_k)
    wl.cfg.pool_kernel = pool
    if same:  # runs of `same` tokens with one key: equal votes
        table = wl.table.long()
        for b, n in enumerate(lens):
            at = torch.arange(n, device=dev)
            rows = table[b, at // page] * page + at % page
            wl.k_pool[rows] = wl.k_pool[rows[at // same * same]]
    return wl


def _met(wl, q):
    """Un-hinted, with meetings: from the rotated query that the layer makes for itself."""
    c, B = wl.cfg, len(wl.seq_lens)
    cos, sin = ops.scoring_cos_sin(c.head_dim, c.rope_theta, c.rope_scale, c.n_local, q.device)
    qf = ops.rope_apply(q.view(B, c.num_heads, c.head_dim), cos, sin, None)
    sel, pos, n = ops.select(c, dataclasses.replace(wl.batch, hint=None), qf, wl.k_pool)[:3]
    torch.cuda.synchronize()
    return sel.clone(), pos.clone(), n.clone()


def _same(got, want, what):
    assert torch.equal(got[3], want[2]), what
    for b, n in enumerate(want[2].tolist()):
        assert torch.equal(got[1][b, :n], want[0][b, :n]) and torch.equal(got[2][b, :n], want[1][b, :n]), (what, b)


# one request over all workgroups, a few of some tokens, many of few workgroups each, runs of equal votes that fit a
# workgroup's words and that do not, a pooled one
CASES = [dict(heads=32, kv_heads=8, lens=[40000], top_k=512), dict(heads=28, kv_heads=4, lens=[9000, 40, 5000], top_k=1024),
         dict(heads=32, kv_heads=8, lens=[6000, 3000, 4500, 2000, 7000, 2500, 3300, 5000], top_k=700, page=16),
         dict(heads=8, kv_heads=2, lens=[20000, 1500], top_k=2000), dict(heads=4, kv_heads=1, lens=[12000], top_k=300, same=7),
         dict(heads=16, kv_heads=8, lens=[8000, 8000], top_k=500, same=40), dict(heads=8, kv_heads=1, lens=[15000], top_k=400, pool=5),
         dict(heads=12, kv_heads=2, lens=[30000], top_k=2048, pool=31)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "H%dkv%d-%d-same%d-pool%d" % (c["heads"], c["kv_heads"], sum(c["lens"]),
                                                                                 c.get("same", 0), c.get("pool", -1)))
def test_a_layers_selection_without_meetings(dev, case):
    say(f"late candidates {case}")
    wl = _workload(dev, **case)
    B, longest = len(wl.seq_lens), max(wl.seq_lens)
    layer = ops.DecodeLayer(wl.cfg, B, longest, dev)
    want = _met(wl, wl.q)
    _same(layer(wl.q, wl.k_pool, wl.v_pool, dataclasses.replace(wl.batch, hint=None)), want, "no hint")
    hint = torch.zeros(B, dtype=torch.int32, device=dev)
    bt = dataclasses.replace(wl.batch, hint=hint)
    _same(layer(wl.q, wl.k_pool, wl.v_pool, bt), want, "no hint yet")
    code = hint.clone()
    selects = code > 0
    for off in (0, -20, -17, -16, -15, -12, -9, -8, -5, -4, -3, -1, 1, 3, 4, 5, 6, 9, 11, 12, 13, 16, 17, 18, 300, 5000):
        hint.copy_(torch.where(selects, (code + off).clamp(min=0), code))
        got = layer(wl.q, wl.k_pool, wl.v_pool, bt)
        torch.cuda.synchronize()
        assert not layer.gave_up(), off
        _same(got, want, off)
        assert torch.equal(hint, code), off
    g = torch.Generator(device=dev).manual_seed(52)
    q = wl.q
    for step in range(6):  # hints left by another query, each request's off by a number of its own
        q = (0.8 * q.float() + 0.6 * torch.randn(q.shape, generator=g, device=dev)).bfloat16()
        _same(layer(q, wl.k_pool, wl.v_pool, bt), _met(wl, q), f"step {step}")
        assert not layer.gave_up()


@pytest.mark.parametrize("off", [0, 9, -9])
def test_a_wait_for_late_words_that_gives_up(dev, off):
    """Forced from the host (a member that all but a request's first workgroup wait for in vain, a 20 us bound): the layer
    reports it and recovers, whatever the hint."""
    say(f"late candidates, forced give-up, hint off by {off}")
    wl = _workload(dev, 32, 8, [9000, 3000], 300)
    layer = ops.DecodeLayer(wl.cfg, 2, 9000, dev)
    hint = torch.zeros(2, dtype=torch.int32, device=dev)
    bt = dataclasses.replace(wl.batch, hint=hint)
    want = _met(wl, wl.q)
    for _ in range(2):
        _same(layer(wl.q, wl.k_pool, wl.v_pool, bt), want, "before")
    hint += off
    forced = dataclasses.replace(bt, wait_us=20, absent_workgroups=1)
    _, _, _, sel_len = layer(wl.q, wl.k_pool, wl.v_pool, forced)
    torch.cuda.synchronize()
    assert layer.gave_up() and sel_len.tolist() == [-1, -1]
    got = layer.recover(wl.q, wl.k_pool, wl.v_pool, forced)
    torch.cuda.synchronize()
    assert got is not None and not layer.gave_up()
    _same(got, want, "recovered")


def test_each_request_with_a_k_of_its_own(dev):
    """The wide band finds each request's own k-th vote: hints off by bins on either side of it, a request among them that
    attends to everything."""
    say("late candidates, k per request")
    lens, ks = [9000, 3000, 7000, 900], [700, 31, 512, 700]
    wl = workloads.build("late", dict(num_heads=32, num_kv_heads=8, rope_theta=5e5), lens, ks, 1, dev, seed=53, n_init=64,
                         n_local=128, top_k=700)
    assert wl.batch.k_per_req is not None
    layer = ops.DecodeLayer(wl.cfg, 4, 9000, dev)
    hint = torch.zeros(4, dtype=torch.int32, device=dev)
    bt = dataclasses.replace(wl.batch, hint=hint)
    want = _met(wl, wl.q)
    assert want[2].tolist() == [64 + 700 + 128, 64 + 31 + 128, 64 + 512 + 128, 64 + 700 + 128]
    _same(layer(wl.q, wl.k_pool, wl.v_pool, bt), want, "no hint yet")
    code = hint.clone()
    for off in (0, -17, -16, -12, -9, -5, -4, 4, 5, 9, 12, 16, 17):
        hint.copy_(torch.where(code > 0, code + off, code))
        got = layer(wl.q, wl.k_pool, wl.v_pool, bt)
        torch.cuda.synchronize()
        assert not layer.gave_up(), off
        _same(got, want, off)
        assert torch.equal(hint, code), off


def test_every_head_shape_selects_in_one_launch(dev):
    """A single request, and a few, of any head shape the library serves."""
    for kv_heads in (1, 2, 4, 8):
        for group in range(1, 9):
            c = ops.LayerConfig(num_heads=group * kv_heads, num_kv_heads=kv_heads, page_size=1, n_init=64, n_local=128, top_k=512)
            for batch, longest in ((1, 1000), (1, 60000), (4, 9000)):
                say(f"selection form of {group * kv_heads} heads on {kv_heads}, {batch} of {longest}")
                assert ops.layer_selection_form(c, batch, longest) == 2 and ops.select_supported(c, batch, longest)


@pytest.mark.parametrize("case", [dict(heads=64, kv_heads=8, lens=[40000], top_k=512),
                                  dict(heads=40, kv_heads=8, lens=[9000, 3000, 700], top_k=700),
                                  dict(heads=48, kv_heads=8, lens=[7000, 6000], top_k=400, same=9)],
                         ids=lambda c: "H%dkv%d-%d" % (c["heads"], c["kv_heads"], sum(c["lens"])))
def test_five_to_eight_heads_on_each_of_eight(dev, case):
    """The shapes whose kernels take the most of a CU."""
    test_a_layers_selection_without_meetings(dev, case)
