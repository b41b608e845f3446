"""Steps whose every request is known to attend to all its tokens: the store writes the selection
and nothing is scored.  Compared with the general path, which a call takes when its requests have
a k of their own (the same k here).  And steps of a growing context, which start with the selection
as long as the workspace's layout stays what the step before left clean."""

import os

import numpy as np
import pytest
import torch

from tokenselect_amd import ops
from helpers import say

pytestmark = pytest.mark.gpu

MAX_TOKENS = 5000


def _state(cfg, lengths, extra, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    total = sum(lengths) + extra + 8
    order = torch.randperm(total, generator=g, device=dev).to(torch.int32)
    table = torch.zeros((len(lengths), MAX_TOKENS), dtype=torch.int32, device=dev)
    at = 0
    for b, n in enumerate(lengths):
        table[b, :n] = order[at:at + n]
        at += n
    pools = [torch.randn((total, cfg.num_kv_heads, 128), generator=g, device=dev).bfloat16() for _ in range(2)]
    return g, pools, table, torch.tensor(lengths, dtype=torch.int32, device=dev), order[at:].contiguous()


def _same(got, ref):
    """Lists, tables, lengths and stored rows are copies: equal.  The outputs are the same fp32 sums
    over another number of splits, rounded to bf16: one ulp of the larger."""
    assert torch.equal(got["lens"], ref["lens"]) and torch.equal(got["table"], ref["table"])
    assert torch.equal(got["k"], ref["k"]) and torch.equal(got["v"], ref["v"])
    assert torch.equal(got["sel_len"], ref["sel_len"])
    for b, n in enumerate(ref["sel_len"].tolist()):
        assert torch.equal(got["sel"][b, :n], ref["sel"][b, :n])
        assert torch.equal(got["sel_pos"][b, :n], ref["sel_pos"][b, :n])
    a, b = got["out"].float(), ref["out"].float()
    assert bool(((a - b).abs() <= b.abs() * 2.0 ** -7 + 1e-6).all())


@pytest.mark.parametrize("lengths,top_k", [([0], 2048), ([1], 2048), ([127], 2048), ([128, 1023, 1024], 2048),
                                           ([2687], 2048), ([2687, 640, 5, 4095 - 1408] , 2048),
                                           ([4095, 4096], 4096), ([4735], 4096)])
def test_dense_step_matches_the_general_path(dev, lengths, top_k):
    say(f"dense step lengths={lengths} k={top_k}")
    cfg = ops.LayerConfig(num_heads=8, num_kv_heads=2, n_init=128, n_local=512, top_k=top_k, rope_theta=5e5)
    B, got = len(lengths), []
    for own_k in (False, True):
        g, (k_pool, v_pool), table, lens, slots = _state(cfg, lengths, B, dev, 5)
        loc = slots[:B].clone()
        if B == 3:
            loc[1] = k_pool.shape[0]  # a slot outside the pool: the request is left untouched
        q, k, v = (torch.randn((B, n * 128), generator=g, device=dev).bfloat16() for n in (8, 2, 2))
        layer = ops.DecodeLayer(cfg, B, max(lengths) + 1, dev)
        for _ in range(2):  # the second call finds the counters that the first one left
            kpr = torch.full((B,), top_k, dtype=torch.int32, device=dev) if own_k else None
            lens.copy_(torch.tensor(lengths))
            bt = ops.Batch(lens, table, max(lengths) + 1, k_per_req=kpr)
            out, sel, sel_pos, sel_len = layer.step(q, k, v, loc, k_pool, v_pool, bt)
        got.append(dict(out=out.clone(), sel=sel.clone(), sel_pos=sel_pos.clone(), sel_len=sel_len.clone(), lens=lens,
                        table=table, k=k_pool, v=v_pool))
    torch.cuda.synchronize()
    _same(*got)


@pytest.mark.parametrize("length,rows", [(0, 1), (0, 300), (255, 1), (256, 8), (700, 9), (2176, 512), (2687, 1)])
def test_dense_chunk_matches_the_general_path(dev, length, rows):
    say(f"dense chunk length={length} rows={rows}")
    cfg = ops.LayerConfig(num_heads=8, num_kv_heads=2, n_init=128, n_local=512, top_k=2048, rope_theta=5e5)
    got = []
    for own_k in (False, True):
        g, (k_pool, v_pool), table, lens, slots = _state(cfg, [length], rows, dev, 6)
        loc = slots[:rows].clone()
        q, k, v = (torch.randn((rows, n * 128), generator=g, device=dev).bfloat16() for n in (8, 2, 2))
        chunk = ops.PrefillChunk(cfg, length + rows, dev, max_rows=512)
        kpr = torch.full((1,), 2048, dtype=torch.int32, device=dev) if own_k else None
        bt = ops.Batch(lens, table, length + rows, k_per_req=kpr)
        out, sel, sel_pos, sel_len = chunk.step(q, k, v, loc, k_pool, v_pool, bt)
        got.append(dict(out=out.clone(), sel=sel.view(1, -1).clone(), sel_pos=sel_pos.view(1, -1).clone(),
                        sel_len=sel_len.view(-1).clone(), lens=lens, table=table, k=k_pool, v=v_pool))
    torch.cuda.synchronize()
    _same(*got)


@pytest.mark.parametrize("first,steps,B,pool", [(2640, 80, 1, -1), (3180, 40, 3, -1), (3000, 70, 1, 9)])
def test_growing_context_on_one_workspace(dev, first, steps, B, pool):
    """Lengths that grow past dense, past 64-token and past workgroup boundaries, one object for
    all steps against a fresh one (whose first call clears everything) at each: the same
    selections and outputs, bit for bit."""
    say(f"growing context from {first}, {steps} steps, B={B} pool={pool}")
    cfg = ops.LayerConfig(num_heads=8, num_kv_heads=2, n_init=128, n_local=512, top_k=2048, rope_theta=5e5,
                          pool_kernel=pool)
    last = first + steps
    g, (k_pool, v_pool), table, lens, _ = _state(cfg, [last] * B, 0, dev, 8)
    layer = ops.DecodeLayer(cfg, B, last, dev)
    layer.workspace.fill_(0xa5)
    for n in range(first, last):
        q = torch.randn((B, 8 * 128), generator=g, device=dev).bfloat16()
        lens.copy_(torch.tensor([n - 300 * b for b in range(B)]))
        bt = ops.Batch(lens, table, n)
        got = [t.clone() for t in layer(q, k_pool, v_pool, bt)]
        fresh = ops.DecodeLayer(cfg, B, last, dev)
        want = fresh(q, k_pool, v_pool, bt)
        torch.cuda.synchronize()
        assert not layer.gave_up() and torch.equal(got[3], want[3]), n
        for b, s in enumerate(want[3].tolist()):
            assert torch.equal(got[1][b, :s], want[1][b, :s]) and torch.equal(got[2][b, :s], want[2][b, :s]), (n, b)
        assert torch.equal(got[0], want[0]), n


@pytest.mark.parametrize("page", [1, 16], ids=["tokens", "pages"])
@pytest.mark.parametrize("first,steps", [(0, 3), (126, 4), (637, 8), (2684, 8)])
def test_steps_on_one_workspace(dev, first, steps, page):
    """Steps that store their own tokens, over the ends of the sinks, of sinks and window (where a
    selection's counters begin) and of dense, one object for all against a fresh one at each, whose
    first call clears everything and stores in a launch of its own: the same bit for bit, outputs
    included (the same splits, the same roundings).  Request 1 is shorter, and its table is full for
    the last steps."""
    say(f"steps from {first}, pages of {page}")
    cfg = ops.LayerConfig(num_heads=14, num_kv_heads=2, n_init=128, n_local=512, top_k=2048, rope_theta=5e5,
                          page_size=page)
    last, B = first + steps, 2
    room = -(-last // page) * page
    lengths = [first, max(room - 2 - steps // 2, 0)]
    g = torch.Generator(device=dev).manual_seed(9)
    pages = 2 * (room // page) + 2 * steps
    order = torch.randperm(pages, generator=g, device=dev).to(torch.int32)
    table = torch.zeros((B, room // page), dtype=torch.int32, device=dev)
    at = 0
    for b, n in enumerate(lengths):
        held = -(-n // page)
        table[b, :held] = order[at:at + held]
        at += held
    free = order[at:].contiguous()
    start = [torch.randn((pages * page, 2, 128), generator=g, device=dev).bfloat16() for _ in range(2)]
    sides = []
    for _ in range(2):
        count = torch.tensor([free.shape[0]], dtype=torch.int32, device=dev)
        sides.append(dict(k=start[0].clone(), v=start[1].clone(), table=table.clone(),
                          lens=torch.tensor(lengths, dtype=torch.int32, device=dev),
                          pages=ops.PagePool(free.clone(), count, torch.zeros(1, dtype=torch.int32, device=dev))))
    one = ops.DecodeLayer(cfg, B, max(room, lengths[1]) + 1, dev)
    one.workspace.fill_(0xa5)
    for t in range(steps):
        q, kv = (torch.randn((B, n * 128), generator=g, device=dev).bfloat16() for n in (14, 4))
        loc = free[2 * t:2 * t + 2].clone()
        got = []
        for s, layer in zip(sides, (one, ops.DecodeLayer(cfg, B, max(room, lengths[1]) + 1, dev))):
            bt = ops.Batch(s["lens"], s["table"], min(max(first, lengths[1]) + t + 1, room))
            out, sel, sel_pos, sel_len = layer.step(q, kv[:, :256].contiguous(), kv[:, 256:].contiguous(),
                                                    loc if page == 1 else None, s["k"], s["v"], bt,
                                                    pages=None if page == 1 else s["pages"])
            got.append(dict(out=out.clone(), sel=sel, sel_pos=sel_pos, sel_len=sel_len, lens=s["lens"],
                            table=s["table"], k=s["k"], v=s["v"]))
        torch.cuda.synchronize()
        assert not one.gave_up()
        _same(*got)
        assert torch.equal(got[0]["out"], got[1]["out"]), t
        assert torch.equal(sides[0]["pages"].free_count, sides[1]["pages"].free_count)
    assert sides[0]["lens"].tolist() == [last, min(lengths[1] + steps, room)]


@pytest.mark.parametrize("case", ["one", "page begins", "page goes on", "batch", "batch of pages", "70 requests",
                                  "no window", "foreign slot", "bad page", "no page left", "table full",
                                  "own k", "separate kernels", "votes form", "pooled"])
def test_a_step_stores_as_the_store_does(dev, case):
    """A step whose launches score or rotate and store on the side, against ts_kv_store and the
    layer on a fresh object: lengths, tables, pools, free pages, selections and outputs bit for bit,
    over the first call (which rotates) and those that start with the selection."""
    say(f"step that stores on the side: {case}")
    page = 16 if "page" in case else 1
    B = {"batch": 4, "batch of pages": 5, "70 requests": 70, "no page left": 3, "own k": 2}.get(case, 1)
    if case in ("foreign slot", "bad page", "table full"):
        B = 2
    lengths = [3200 - 7 * b for b in range(B)]
    if case == "page begins":
        lengths = [3200]
    if case == "page goes on":
        lengths = [3205]
    if case in ("batch", "own k"):
        lengths[1] = 300  # dense among others
    if case in ("batch of pages", "bad page", "no page left"):
        lengths = [3200 + 16 * b for b in range(B)]
        lengths[-1] += 3
    top_k = 256 if case == "70 requests" else 1024
    if case == "votes form":
        lengths, B = [40000] * 9, 9
    cfg = ops.LayerConfig(num_heads=32 if case == "votes form" else 8, num_kv_heads=8 if case == "votes form" else 2,
                          n_init=16, n_local=0 if case == "no window" else 64, top_k=top_k, rope_theta=5e5,
                          page_size=page, pool_kernel=5 if case == "pooled" else -1)
    steps, H, row = 3, cfg.num_heads, cfg.num_kv_heads * 128
    g = torch.Generator(device=dev).manual_seed(12)
    width = (max(lengths) + steps) // page + 1
    if case == "table full":
        width = max(lengths) + 1  # (one more token of request 0; request 1 goes on)
    held = [-(-n // page) for n in lengths]
    pages = sum(held) + B * steps
    order = torch.randperm(pages, generator=g, device=dev).to(torch.int32)
    table, at = torch.zeros((B, width), dtype=torch.int32, device=dev), 0
    for b, n in enumerate(held):
        table[b, :n] = order[at:at + n]
        at += n
    free = order[at:].contiguous()
    if case == "bad page":
        free[-1] = pages + 5
    count = 1 if case == "no page left" else free.shape[0]
    start = [torch.randn((pages * page, cfg.num_kv_heads, 128), generator=g, device=dev).bfloat16() for _ in range(2)]
    sides = [dict(k=start[0].clone(), v=start[1].clone(), table=table.clone(),
                  lens=torch.tensor(lengths, dtype=torch.int32, device=dev),
                  hint=torch.zeros(B, dtype=torch.int32, device=dev),
                  pages=ops.PagePool(free.clone(), torch.tensor([count], dtype=torch.int32, device=dev),
                                     torch.zeros(1, dtype=torch.int32, device=dev))) for _ in range(2)]
    longest = min(max(lengths) + steps, width * page)
    one = ops.DecodeLayer(cfg, B, longest, dev)
    one.workspace.fill_(0xa5)
    kpr = torch.tensor([700, 256][:B], dtype=torch.int32, device=dev) if case == "own k" else None
    for t in range(steps):
        q = torch.randn((B, H * 128), generator=g, device=dev).bfloat16()
        kv = torch.randn((2, B, row), generator=g, device=dev).bfloat16()
        loc = None
        if page == 1:
            loc = free[t * B:t * B + B].clone()
            if case == "foreign slot":
                loc[1 - t % 2] = start[0].shape[0] if t else -1
        got = []
        for s, whole in zip(sides, (True, False)):
            most = min(max(lengths) + t + 1, width * page)
            bt = ops.Batch(s["lens"], s["table"], most, k_per_req=kpr, hint=s["hint"],
                           separate_kernels=case == "separate kernels")
            if whole:
                out, sel, sel_pos, sel_len = one.step(q, kv[0], kv[1], loc, s["k"], s["v"], bt,
                                                      pages=None if page == 1 else s["pages"])
            else:
                ops.kv_store(cfg, kv[0], kv[1], loc, s["k"], s["v"], s["table"], s["lens"],
                             pages=None if page == 1 else s["pages"])
                layer = ops.DecodeLayer(cfg, B, longest, dev)
                out, sel, sel_pos, sel_len = layer(q, s["k"], s["v"], bt)
            got.append(dict(out=out.clone(), sel=sel, sel_pos=sel_pos, sel_len=sel_len, lens=s["lens"],
                            table=s["table"], k=s["k"], v=s["v"]))
        torch.cuda.synchronize()
        assert not one.gave_up()
        _same(*got)
        assert torch.equal(got[0]["out"], got[1]["out"])
        assert torch.equal(sides[0]["pages"].free_count, sides[1]["pages"].free_count)
        assert int(sides[0]["pages"].ticket) == 0
    if case in ("one", "page begins", "70 requests", "votes form"):
        assert sides[0]["lens"].tolist() == [n + steps for n in lengths]


@pytest.mark.parametrize("padded", [[1], [0], [5, 1], [300, 40]])
def test_padded_requests_on_one_slot(dev, padded):
    """Requests that pad a batch list one slot over and over and store to it.  One of them: the step's
    output is that of the store and the layer, whose context holds the new row wherever the slot is
    listed.  Several: each attends to its own new row.  The request beside them as if alone."""
    say(f"padded requests of {padded} tokens")
    cfg = ops.LayerConfig(num_heads=14, num_kv_heads=2, n_init=128, n_local=512, top_k=2048, rope_theta=5e5)
    B, steps = 1 + len(padded), 3
    g, (k_pool, v_pool), table, lens, free = _state(cfg, [900], 8, dev, 17)
    slot = int(free[-1])
    table = torch.cat([table, torch.full((len(padded), MAX_TOKENS), slot, dtype=torch.int32, device=dev)])
    layer = ops.DecodeLayer(cfg, B, 1000, dev)
    now = torch.tensor([900] + padded, dtype=torch.int32, device=dev)
    for t in range(steps):
        q, k, v = (torch.randn((B, n * 128), generator=g, device=dev).bfloat16() for n in (14, 2, 2))
        loc = torch.cat([free[t:t + 1], torch.full((len(padded),), slot, dtype=torch.int32, device=dev)])
        want = []
        for b in range(B):   # each by itself
            pools, one, row = (k_pool.clone(), v_pool.clone()), now[b:b + 1].clone(), table[b:b + 1].clone()
            ops.kv_store(cfg, k[b:b + 1], v[b:b + 1], loc[b:b + 1], *pools, row, one)
            alone = ops.DecodeLayer(cfg, 1, 1000, dev)
            want.append(alone(q[b:b + 1], *pools, ops.Batch(one, row, 900 + t + 1))[0].clone())
        lens = now.clone()
        out = layer.step(q, k, v, loc, k_pool, v_pool, ops.Batch(lens, table, 900 + t + 1))[0]
        torch.cuda.synchronize()
        if t > 0 or len(padded) == 1:   # (a first call stores in a launch of its own: one row for all)
            ref = torch.cat(want).float()
            assert bool(((out.float() - ref).abs() <= ref.abs() * 2.0 ** -7 + 1e-6).all()), t   # (other splits: an ulp)
        now[0] += 1


@pytest.mark.parametrize("bound", [300, 511, 512, 700])
def test_a_dense_step_beyond_the_bound_is_stored(dev, bound):
    """max_seq_len below the length: attended to are the positions below it, as before, but the new
    token's row is stored and listed in the table by a first call and by those after it."""
    say(f"dense step beyond a bound of {bound}")
    cfg = ops.LayerConfig(num_heads=14, num_kv_heads=2, n_init=128, n_local=512, top_k=2048, rope_theta=5e5)
    length = 700
    g, (k_pool, v_pool), table, lens, free = _state(cfg, [length, 40], 8, dev, 16)
    layer = ops.DecodeLayer(cfg, 2, 800, dev)
    for t in range(3):
        q, k, v = (torch.randn((2, n * 128), generator=g, device=dev).bfloat16() for n in (14, 2, 2))
        want_k, want_v, loc = k_pool.clone(), v_pool.clone(), free[2 * t:2 * t + 2].clone()
        want_k[loc.long()], want_v[loc.long()] = k.view(2, 2, 128), v.view(2, 2, 128)
        _, sel, _, sel_len = layer.step(q, k, v, loc, k_pool, v_pool, ops.Batch(lens, table, bound))
        torch.cuda.synchronize()
        assert lens.tolist() == [length + t + 1, 41 + t] and table[0, length + t] == loc[0]
        assert torch.equal(k_pool, want_k) and torch.equal(v_pool, want_v), t
        assert sel_len.tolist() == [min(bound, length + t + 1), 41 + t]
        assert torch.equal(sel[0, :sel_len[0]], table[0, :sel_len[0]])


@pytest.mark.parametrize("page", [1, 16], ids=["tokens", "pages"])
@pytest.mark.parametrize("longest,cached", [(700, False), (3000, False), (3000, True)],
                         ids=["dense", "selected", "selection cache"])
def test_a_request_without_a_length_is_left_alone(dev, longest, cached, page):
    """A negative length is refused as a full table is, by whatever launch places the new token: the
    store alone, the first launch of a first call and that of the calls after it.  (Request 1's: an
    entry of its table written all the same would be one of request 0's last.)"""
    say(f"request without a length: longest={longest} cached={cached} pages of {page}")
    cfg = ops.LayerConfig(num_heads=8, num_kv_heads=2, n_init=128, n_local=512, top_k=1024, rope_theta=5e5,
                          page_size=page)
    g = torch.Generator(device=dev).manual_seed(15)
    pages = longest // page + 8
    order = torch.randperm(pages, generator=g, device=dev).to(torch.int32)
    held = -(-longest // page)
    table = torch.full((2, pages), -1, dtype=torch.int32, device=dev)
    table[0, :held] = order[:held]
    k_pool, v_pool = (torch.randn((pages * page, 2, 128), generator=g, device=dev).bfloat16() for _ in range(2))
    lens = torch.tensor([longest, -5 * page], dtype=torch.int32, device=dev)
    pool = None if page == 1 else ops.PagePool(order[held:].contiguous(),
                                               torch.tensor([pages - held], dtype=torch.int32, device=dev),
                                               torch.zeros(1, dtype=torch.int32, device=dev))
    cache = ops.SelectionCache.allocate(cfg, 2, dev) if cached else None
    layer = ops.DecodeLayer(cfg, 2, longest + 8, dev)
    now = longest
    for t in range(4):
        q, k, v = (torch.randn((2, n * 128), generator=g, device=dev).bfloat16() for n in (8, 2, 2))
        loc = None if pool else torch.stack([order[held + t], order[held + 4]])
        want_k = k_pool.clone()
        if t == 0:
            ops.kv_store(cfg, k, v, loc, k_pool, v_pool, table, lens, pages=pool)
        else:
            layer.step(q, k, v, loc, k_pool, v_pool, ops.Batch(lens, table, now + 1), cache, pages=pool)
        torch.cuda.synchronize()
        want_k[int(table[0, now // page]) * page + now % page] = k[0].view(2, 128)
        now += 1
        assert not layer.gave_up()
        assert lens.tolist() == [now, -5 * page] and torch.equal(k_pool, want_k), t
        assert bool((table[1] == -1).all()) and bool((table[0, -(-now // page):] == -1).all()), t


@pytest.mark.parametrize("length,rows,room,page", [(0, 40, 64, 1), (600, 512, 1200, 1), (1000, 100, 1050, 1), (31, 33, 64, 16),
                                                   (640, 512, 1200, 16), (1000, 100, 1040, 16), (2400, 288, 2688, 1)])
def test_a_dense_chunk_stores_as_the_store_does(dev, length, rows, room, page):
    """A dense chunk, whose gather stores its rows, against ts_kv_store_chunk and the chunk on a fresh
    object: length, table, pools, free pages, list and output bit for bit; tables that end within the
    chunk, slots that are none of the pool's (clamped, each to a row of its own)."""
    say(f"dense chunk that stores on the side: {length}+{rows} room {room} pages of {page}")
    cfg = ops.LayerConfig(num_heads=14, num_kv_heads=2, n_init=128, n_local=512, top_k=2048, rope_theta=5e5, page_size=page)
    g = torch.Generator(device=dev).manual_seed(14)
    pages = room // page + 4
    order = torch.randperm(pages - 2, generator=g, device=dev).to(torch.int32) + 1  # (the first and the last row stay free)
    held = -(-length // page)
    table = torch.zeros((1, room // page), dtype=torch.int32, device=dev)
    table[0, :held] = order[:held]
    start = [torch.randn((pages * page, 2, 128), generator=g, device=dev).bfloat16() for _ in range(2)]
    q, k, v = (torch.randn((rows, n * 128), generator=g, device=dev).bfloat16() for n in (14, 2, 2))
    loc = None
    if page == 1:
        loc = torch.cat([order[held:], order[:0]])[:rows].clone()
        loc = torch.nn.functional.pad(loc, (0, rows - loc.shape[0]), value=int(order[-1]))  # (past the table: not stored)
        loc[3], loc[5] = -7, pages + 11
    got = []
    for whole in (True, False):
        s = dict(k=start[0].clone(), v=start[1].clone(), table=table.clone(),
                 lens=torch.tensor([length], dtype=torch.int32, device=dev))
        pool = None if page == 1 else ops.PagePool(order[held:].contiguous(), torch.tensor([pages - 2 - held], dtype=torch.int32, device=dev),
                                                   torch.zeros(1, dtype=torch.int32, device=dev))
        chunk = ops.PrefillChunk(cfg, min(length + rows, room), dev, max_rows=512)
        chunk.workspace.fill_(0xff)
        bt = ops.Batch(s["lens"], s["table"], min(length + rows, room))
        if whole:
            out, sel, sel_pos, sel_len = chunk.step(q, k, v, loc, s["k"], s["v"], bt, pages=pool)
        else:
            ops.kv_store_chunk(cfg, k, v, loc, s["k"], s["v"], s["table"][0], s["lens"], pages=pool)
            out, sel, sel_pos, sel_len = chunk(q, s["k"], s["v"], bt)
        got.append(dict(out=out.clone(), sel=sel.view(1, -1).clone(), sel_pos=sel_pos.view(1, -1).clone(),
                        sel_len=sel_len.view(-1).clone(), lens=s["lens"], table=s["table"], k=s["k"], v=s["v"]))
    torch.cuda.synchronize()
    _same(*got)
    assert torch.equal(got[0]["out"], got[1]["out"])
    assert int(got[0]["lens"]) == min(length + rows, room)


ROUNDING = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "attn_rounding.npz")


def rounding_outputs(dev, heads, kv_heads):
    """Attention outputs (int16 bit patterns) of seeded inputs: the first step of an object, whose
    attention reads a list, and five more, whose attention reads the table."""
    cfg = ops.LayerConfig(num_heads=heads, num_kv_heads=kv_heads, n_init=128, n_local=512, top_k=2048, rope_theta=5e5)
    g = torch.Generator().manual_seed(heads)
    lengths = [2003, 1500, 517, 2600, 64, 1999, 1024, 300]
    B, total = len(lengths), 12000
    randn = lambda *shape: torch.randn(shape, generator=g).bfloat16().to(dev)
    order = torch.randperm(total, generator=g).to(torch.int32).to(dev)
    table, at = torch.zeros((B, 2700), dtype=torch.int32, device=dev), 0
    for b, n in enumerate(lengths):
        table[b, :n] = order[at:at + n]
        at += n
    k_pool, v_pool = randn(total, kv_heads, 128), randn(total, kv_heads, 128)
    lens = torch.tensor(lengths, dtype=torch.int32, device=dev)
    layer, outs = ops.DecodeLayer(cfg, B, 2688, dev), []
    for t in range(6):
        q, k, v = randn(B, heads * 128), randn(B, kv_heads * 128), randn(B, kv_heads * 128)
        loc = order[at + B * t:at + B * (t + 1)].clone()
        bt = ops.Batch(lens, table, max(lengths) + t + 1)
        outs.append(layer.step(q, k, v, loc, k_pool, v_pool, bt)[0].clone())
    torch.cuda.synchronize()
    return torch.stack(outs).cpu().contiguous().view(torch.int16).numpy()


@pytest.mark.parametrize("heads,kv_heads", [(8, 2), (7, 1), (4, 4)])
def test_attention_rounds_as_it_did(dev, heads, kv_heads):
    """The rotations of queries and keys say which of their products is rounded: the outputs keep their
    bits whatever else changes in the kernel.  The fixture holds rounding_outputs() of the kernel
    before its attention read tables (a compiler that contracts on its own gave others since)."""
    say(f"rounding of the attention: {heads} heads on {kv_heads}")
    want = np.load(ROUNDING)[f"{heads}_{kv_heads}"]
    got = rounding_outputs(dev, heads, kv_heads)
    assert got.shape == want.shape
    differ = np.argwhere(got != want)
    assert differ.shape[0] == 0, f"{differ.shape[0]} of {want.size} outputs: {differ[:8].tolist()}"
