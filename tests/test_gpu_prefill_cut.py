"""The prefill attention's jobs that are cut between workgroups (PrefillCuts, ts_prefill_shared.hip): a prompt's dense
rows and the chunks behind them, where their jobs are just enough, fill a wave and a little, almost fill one, and at rows
that fill neither a tile nor a job, against the oracle.  Bounds as in test_gpu_prefill_shared."""

import ctypes
import re

import pytest
import torch

import oracle
from tokenselect_amd import _lib, ops, workloads
from helpers import say

pytestmark = pytest.mark.gpu

N_INIT, N_LOCAL, TOP_K, CHUNK = 128, 512, 1024, 256


class _Prompt:
    def __init__(self, dev, heads, kv_heads, before, rows, cap=0.0):
        wl = workloads.build("cut", dict(num_heads=heads, num_kv_heads=kv_heads, rope_theta=5e5), [max(before, 1)], [TOP_K], 1,
                             dev, seed=31, n_init=N_INIT, n_local=N_LOCAL, top_k=TOP_K, extra_pages=rows)
        self.wl, self.c, self.dev, self.before, self.rows = wl, wl.cfg, dev, before, rows
        self.c.logit_cap = cap
        g = torch.Generator(device=dev).manual_seed(32)
        self.q = torch.randn((rows, heads * 128), generator=g, device=dev).bfloat16()
        self.k, self.v = (torch.randn((rows, kv_heads, 128), generator=g, device=dev).bfloat16() for _ in range(2))
        self.slots = wl.free_pages[:rows].contiguous()

    def fresh(self):
        self.k_pool, self.v_pool = self.wl.k_pool.clone(), self.wl.v_pool.clone()
        self.table = torch.zeros((1, self.before + self.rows + 64), dtype=torch.int32, device=self.dev)
        self.table[0, :self.before] = self.wl.table[0, :self.before]
        self.seq = torch.full((1,), self.before, dtype=torch.int32, device=self.dev)
        return torch.empty_like(self.q)

    def together(self, room=None):
        """The call with its own workspace's bytes, or with `room` of them; the bytes it cannot do without."""
        lib, cc, out = _lib.load(), self.c.to_c(), self.fresh()
        total = self.before + self.rows
        cos, sin = ops.rope_tables(128, self.c.rope_theta, self.c.rope_scale, N_LOCAL + CHUNK, self.dev)
        bt = _lib.TsBatch(1, total, self.seq.data_ptr(), self.table.data_ptr(), self.table.shape[1], None)
        kv = _lib.TsNewKv(self.k.data_ptr(), self.v.data_ptr(), self.slots.data_ptr(), None, self.table.shape[1])

        def call(space, nbytes):
            return lib.ts_prefill_prompt(ctypes.byref(cc), ctypes.byref(bt), ctypes.byref(kv), self.q.data_ptr(), 0, 0,
                                         self.rows, CHUNK, cos.data_ptr(), sin.data_ptr(), cos.shape[0],
                                         self.k_pool.data_ptr(), self.v_pool.data_ptr(), self.k_pool.shape[0],
                                         out.data_ptr(), space.data_ptr(), nbytes,
                                         torch.cuda.current_stream().cuda_stream)

        asked = lib.ts_prefill_prompt_workspace_bytes(ctypes.byref(cc), self.rows, CHUNK, total)
        space = torch.full((asked,), 0xa5, dtype=torch.uint8, device=self.dev)
        assert call(space, 0) == _lib.TS_EWORKSPACE
        need = int(re.search(r"required (\d+)", lib.ts_last_error().decode()).group(1))
        assert call(space, asked if room is None else need) == _lib.TS_OK, lib.ts_last_error()
        torch.cuda.synchronize()
        return out.cpu().float(), asked, need

    def one_by_one(self):
        """What each chunk attends to, from the chunks one by one."""
        out, lists = self.fresh(), []
        layer = ops.PrefillChunk(self.c, self.before + self.rows, self.dev, max_rows=CHUNK)
        for at in range(0, self.rows, CHUNK):
            here = min(CHUNK, self.rows - at)
            layer._serve(self.q, self.k, self.v, self.slots, self.k_pool, self.v_pool,
                         ops.Batch(self.seq, self.table, self.before + at + here), None, out, at, here)
            lists.append(layer.sel[0, :int(layer.sel_len)].clone())
        torch.cuda.synchronize()
        return lists

    def check(self, out, lists):
        c, kc, vc = self.c, self.k_pool.cpu(), self.v_pool.cpu()
        sm = c.sm_scale if c.sm_scale is not None else c.head_dim ** -0.5
        for i, sel in enumerate(lists):
            at = slice(i * CHUNK, min((i + 1) * CHUNK, self.rows))
            q = self.q[at].cpu().view(-1, c.num_heads, 128)
            ref = oracle.prefill.sparse_prefill_attention(q, kc, vc, sel.cpu(), sm, c.rope_theta, c.rope_scale, c.logit_cap,
                                                          c.rope_mode).reshape(q.shape[0], -1).float()
            excess = ((out[at] - ref).abs() - (2e-2 + 2.0 ** -6 * ref.abs())).max().item()
            assert excess <= 0.0, (i, excess)


# (heads, KV heads, tokens before, rows, cap): dense alone, chunks alone, both
CASES = [(28, 4, 0, 1664, 0.0), (48, 8, 0, 1205, 30.0), (32, 8, 3000, 5 * CHUNK - 37, 0.0), (28, 4, 3000, 9 * CHUNK + 1, 0.0),
         (24, 8, 3000, 12 * CHUNK - 200, 30.0), (32, 4, 0, 1664 + 5 * CHUNK + 90, 0.0), (8, 1, 5000, 19 * CHUNK - 3, 0.0),
         (16, 2, 3000, 14 * CHUNK, 0.0)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "H%dkv%d+%d-%d" % c[:4])
def test_jobs_that_are_cut(dev, case):
    """Twice the same bits, whoever comes last; with no room for the pieces as well, uncut."""
    say("cut prefill attention H=%d kv=%d before=%d rows=%d cap=%g" % case)
    p = _Prompt(dev, *case)
    lists = p.one_by_one()
    out, asked, need = p.together()
    assert asked > need
    p.check(out, lists)
    assert torch.equal(out, p.together()[0])
    p.check(p.together(room=0)[0], lists)


@pytest.mark.parametrize("heads,kv_heads,rows,top_k,cap,cut",
                         [(40, 8, 1584, 1024, 0.0, True), (32, 8, 1664, 1024, 0.0, False), (64, 8, 1024, 1024, 0.0, False),
                          (56, 8, 1664, 1024, 0.0, False), (24, 8, 2560, 2048, 0.0, True), (32, 8, 2688, 2048, 0.0, True),
                          (56, 8, 2560, 2048, 30.0, True), (40, 8, 2560, 2048, 0.0, False)])
def test_dense_rows_that_are_cut(dev, monkeypatch, heads, kv_heads, rows, top_k, cap, cut):
    """Dense rows alone, where sharing their jobs out pays (less than a wave, more, more than two) and where it does not (too few, jobs too
    short, so many that the longest is the launch either way): cut, some sums are added up in pieces; otherwise the bits are those
    without room."""
    say(f"dense rows, cut or not: {heads} on {kv_heads}, {rows}, top-k {top_k}")
    monkeypatch.setitem(globals(), "TOP_K", top_k)
    p = _Prompt(dev, heads, kv_heads, 0, rows, cap)
    lists = p.one_by_one()
    out, _, _ = p.together()
    p.check(out, lists)
    without = p.together(room=0)[0]
    p.check(without, lists)
    assert torch.equal(out, without) != cut
