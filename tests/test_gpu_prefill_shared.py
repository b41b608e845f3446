"""The prefill attention's workgroups of 256 columns (ts_prefill_shared.hip) against the oracle, at the
smallest numbers of rows that take them: every number of heads per KV head, rows that fill neither a
tile of 16 nor a workgroup, selections that are shorter than the chunk, exactly as long, and longer, the soft cap.

Within 2e-2 plus two bf16 units of the reference value: the rotated keys and the softmax weights
enter the matrix products as bf16, 2^-9 of a logit's terms each (the bound of the kernel for few rows and
queries of up to twice the unit; with three times the unit a logit of 15 is off by up to 2^-8 x 15 = 6 %, and
so is its weight)."""

import pytest
import torch

import oracle
from tokenselect_amd import ops, workloads
from helpers import say

pytestmark = pytest.mark.gpu

SHAPES = [dict(num_heads=h, num_kv_heads=kv, rope_theta=5e5)
          for h, kv in ((8, 8), (16, 8), (24, 8), (32, 8), (40, 8), (48, 8), (28, 4), (8, 1), (12, 2))]


def _fewest_rows(shape):
    """Rows that are the first to fill 0.8 of the device with workgroups of 16 column blocks."""
    per_head, group = -(-205 // shape["num_kv_heads"]), shape["num_heads"] // shape["num_kv_heads"]
    return 16 * (((per_head - 1) * 16) // group) + 1


def _check(dev, shape, m, S, rope_mode="ROPE_LLAMA", cap=0.0, scale=1.0):
    say(f"shared prefill attention H={shape['num_heads']} kv={shape['num_kv_heads']} m={m} S={S} {rope_mode} cap={cap}")
    wl = workloads.build("ps", shape, [S + 50], [64], 1, dev, seed=3, n_init=8, n_local=m)
    c = wl.cfg
    c.rope_mode, c.logit_cap = rope_mode, cap
    g = torch.Generator(device=dev).manual_seed(4)
    q = (scale * torch.randn((m, c.num_heads * 128), generator=g, device=dev)).bfloat16()
    sel = wl.table[0, torch.randperm(S + 50, generator=g, device=dev)[:S].long()].contiguous()
    out = ops.sparse_prefill_attention(c, q, wl.k_pool, wl.v_pool, sel, torch.tensor([S], dtype=torch.int32, device=dev))
    torch.cuda.synchronize()
    sm = c.sm_scale if c.sm_scale is not None else c.head_dim ** -0.5
    ref = oracle.prefill.sparse_prefill_attention(q.cpu().view(m, c.num_heads, 128), wl.k_pool.cpu(), wl.v_pool.cpu(),
                                                  sel.cpu(), sm, c.rope_theta, c.rope_scale, cap, rope_mode)
    ref = ref.reshape(m, -1).float()
    excess = ((out.cpu().float() - ref).abs() - (2e-2 + 2.0 ** -6 * ref.abs())).max().item()
    assert excess <= 0.0, excess


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"H{s['num_heads']}kv{s['num_kv_heads']}")
@pytest.mark.parametrize("more_rows,keys", [(0, 0), (14, 31), (16, 333), (7, -45)])
def test_shared_prefill_attention(dev, shape, more_rows, keys):
    m = _fewest_rows(shape) + more_rows
    _check(dev, shape, m, m + keys)


@pytest.mark.parametrize("rope_mode,cap,scale", [("NONE", 0.0, 2.0), ("ROPE_LLAMA", 30.0, 2.0), ("ROPE_LLAMA", 0.0, 2.0)])
def test_shared_prefill_attention_options(dev, rope_mode, cap, scale):
    _check(dev, SHAPES[3], 1777, 2555, rope_mode, cap, scale)


def test_shared_prefill_attention_without_keys(dev):
    """A selection that gave up reports -1, an empty one 0: the rows are zero."""
    m = 1777
    say("shared prefill attention without keys")
    wl = workloads.build("ps", SHAPES[3], [100], [8], 1, dev, seed=25, n_init=1, n_local=m)
    q = torch.ones((m, 4096), dtype=torch.bfloat16, device=dev)
    for reported in (-1, 0):
        out = ops.sparse_prefill_attention(wl.cfg, q, wl.k_pool, wl.v_pool, wl.table[0, :100].contiguous(),
                                           torch.tensor([reported], dtype=torch.int32, device=dev))
        torch.cuda.synchronize()
        assert torch.count_nonzero(out).item() == 0, reported


@pytest.mark.parametrize("shape", [SHAPES[3], SHAPES[6]], ids=["H32kv8", "H28kv4"])
@pytest.mark.parametrize("rows", [13 * 128 - 5, 17 * 128 - 60], ids=["all", "all but one chunk"])
def test_chunks_of_a_prompt_share(dev, shape, rows):
    """Chunks of 128 rows, 16 workgroups each, with selections of their own: thirteen take these workgroups,
    of seventeen all but the last.  Against the oracle on what the chunks one by one select, and so are those."""
    say(f"prompt of chunks that share H={shape['num_heads']} rows={rows}")
    before, chunk, top_k = 1000, 128, 200
    wl = workloads.build("pr", shape, [before], [top_k], 1, dev, seed=21, n_init=8, n_local=64, top_k=top_k,
                         extra_pages=rows)
    c = wl.cfg
    g = torch.Generator(device=dev).manual_seed(22)
    q = torch.randn((rows, c.num_heads * 128), generator=g, device=dev).bfloat16()
    k, v = (torch.randn((rows, c.num_kv_heads, 128), generator=g, device=dev).bfloat16() for _ in range(2))
    slots = wl.free_pages[:rows].contiguous()
    outs, lists = [], []
    for together in (True, False):
        k_pool, v_pool = wl.k_pool.clone(), wl.v_pool.clone()
        table = torch.zeros((1, before + rows), dtype=torch.int32, device=dev)
        table[0, :before] = wl.table[0, :before]
        seq = torch.full((1,), before, dtype=torch.int32, device=dev)
        out = torch.empty_like(q)
        layer = ops.PrefillChunk(c, before + rows, dev, max_rows=chunk)
        if together:
            layer._prompt(q, k, v, slots, k_pool, v_pool, ops.Batch(seq, table, before + rows), out, 0, rows, chunk)
        else:
            for at in range(0, rows, chunk):
                here = min(chunk, rows - at)
                layer._serve(q, k, v, slots, k_pool, v_pool, ops.Batch(seq, table, before + at + here), None, out, at, here)
                lists.append((layer.sel[0].clone(), layer.sel_len.clone()))
        torch.cuda.synchronize()
        outs.append(out.cpu().float())
    sm = c.sm_scale if c.sm_scale is not None else c.head_dim ** -0.5
    qc, kc, vc = q.cpu().view(rows, c.num_heads, 128), k_pool.cpu(), v_pool.cpu()
    for i, (sel, sel_len) in enumerate(lists):
        at = slice(i * chunk, min((i + 1) * chunk, rows))
        assert int(sel_len) == c.max_sel
        ref = oracle.prefill.sparse_prefill_attention(qc[at], kc, vc, sel[:int(sel_len)].cpu(), sm, c.rope_theta,
                                                      c.rope_scale, 0.0, c.rope_mode)
        ref = ref.reshape(qc[at].shape[0], -1).float()
        for name, out in zip(("together", "one by one"), outs):
            excess = ((out[at] - ref).abs() - (2e-2 + 2.0 ** -6 * ref.abs())).max().item()
            assert excess <= 0.0, (name, i, excess)
