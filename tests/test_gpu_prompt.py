"""A prompt's chunks taken together (``ts_prefill_prompt``) where the sizes are at their limits: tables that
get full, more rows than one launch takes, too little memory for the workspace, values that are not finite.
What is compared with is the chunks one by one (``ts_prefill_step_strided``)."""

import ctypes
import dataclasses

import pytest
import torch

from tokenselect_amd import _lib, ops, workloads
from tokenselect_amd.patcher import sglang_standins as sg
from tokenselect_amd.patcher import token_retrieval as tr
from helpers import say

pytestmark = pytest.mark.gpu


def _prompt(dev, heads, kv_heads, L0, T, top_k, seed=51, n_init=8, n_local=64, **config):
    """A layer's configuration, its pools and table, and T rows more."""
    shape = dict(num_heads=heads, num_kv_heads=kv_heads, rope_theta=5e5)
    wl = workloads.build("pp", shape, [max(L0, 1)], [top_k], 1, dev, seed=seed, n_init=n_init, n_local=n_local,
                         top_k=top_k, extra_pages=T)
    g = torch.Generator(device=dev).manual_seed(seed + 1)
    common = torch.randn((1, heads * 128), generator=g, device=dev)
    q = (common + torch.randn((T, heads * 128), generator=g, device=dev)).bfloat16()
    k, v = (torch.randn((T, kv_heads, 128), generator=g, device=dev).bfloat16() for _ in range(2))
    return wl, dataclasses.replace(wl.cfg, **config), q, k, v, wl.free_pages[:T].contiguous()


def _served(dev, wl, c, q, k, v, slots, L0, width, chunk, together, bound=None):
    """(K pool, V pool, table, length, output) after the rows, with a table of `width` tokens."""
    T = q.shape[0]
    k_pool, v_pool = wl.k_pool.clone(), wl.v_pool.clone()
    table = torch.zeros((1, width), dtype=torch.int32, device=dev)
    table[0, :L0] = wl.table[0, :L0]
    seq = torch.full((1,), L0, dtype=torch.int32, device=dev)
    out = torch.full_like(q, 7.0)
    layer = ops.PrefillChunk(c, width, dev, max_rows=chunk)
    if together:
        layer._prompt(q, k, v, slots, k_pool, v_pool, ops.Batch(seq, table, bound or min(L0 + T, width)), out, 0, T, chunk)
    else:
        for start in range(0, T, chunk):
            end = min(start + chunk, T)
            layer._serve(q, k, v, slots, k_pool, v_pool, ops.Batch(seq, table, min(L0 + end, width)), None, out, start,
                         end - start)
    torch.cuda.synchronize()
    assert not layer.gave_up()
    return k_pool, v_pool, table, seq, out


def _same(x, y, names=("k", "v", "table", "length", "out")):
    for name, a, b in zip(names, x, y):
        a, b = (t.view(torch.int16) if t.dtype == torch.bfloat16 else t for t in (a, b))
        assert torch.equal(a, b), f"{name}: {int((a != b).sum())} of {a.numel()} differ"


@pytest.mark.parametrize("top_k", [2048, 96], ids=["dense", "selecting"])
@pytest.mark.parametrize("L0,T,width", [(0, 1500, 1000), (0, 1500, 1500), (0, 1500, 1501), (700, 900, 1100),
                                        (700, 300, 700), (3, 500, 130)])
def test_a_table_that_gets_full(dev, top_k, L0, T, width):
    """Rows beyond the table are not stored, and every chunk's rows lie where they lie if it is taken alone:
    tables that end within a chunk, with the last chunk, and that are full from the start."""
    say(f"prompt of {T} on {L0} in a table of {width}, top_k {top_k}")
    case = _prompt(dev, 8, 2, L0, T, top_k)
    _same(*(_served(dev, *case, L0, width, 128, together) for together in (True, False)))


def test_more_rows_than_one_attention_takes(dev):
    """Ten chunks of 104900 rows: a launch of the attention takes 65535 x 16 = 1048560 rows.  Pools, table and
    length the same; outputs as the two kernels' (2^-8 of a mean of normal values, and the result's rounding)."""
    T, chunk = 1049000, 104900
    say(f"prompt of {T} rows in chunks of {chunk}")
    case = _prompt(dev, 1, 1, 0, T, 64, n_local=600)
    x, y = (_served(dev, *case, 0, T, chunk, together) for together in (True, False))
    _same(x[:4], y[:4])
    assert (x[4].float() - y[4].float()).abs().max().item() <= 2 ** -7 * y[4].float().abs().max().item()


def test_fewer_rows_than_a_chunk_need_no_longer_tables(dev):
    """The rotation tables cover the rows that are there, whatever a chunk may have."""
    L0, T = 1000, 20
    say("prompt of fewer rows than a chunk, tables of as many")
    wl, c, q, k, v, slots = _prompt(dev, 8, 2, L0, T, 96)
    want = _served(dev, wl, c, q, k, v, slots, L0, L0 + T, T, False)
    lib, cc = _lib.load(), c.to_c()
    k_pool, v_pool = wl.k_pool.clone(), wl.v_pool.clone()
    table = torch.zeros((1, L0 + T), dtype=torch.int32, device=dev)
    table[0, :L0] = wl.table[0, :L0]
    seq = torch.full((1,), L0, dtype=torch.int32, device=dev)
    out = torch.empty_like(q)
    cos, sin = ops.rope_tables(c.head_dim, c.rope_theta, c.rope_scale, c.n_local + T, dev)
    nbytes = lib.ts_prefill_prompt_workspace_bytes(ctypes.byref(cc), T, 512, L0 + T)
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    bt = _lib.TsBatch(1, L0 + T, seq.data_ptr(), table.data_ptr(), L0 + T, None)
    kv = _lib.TsNewKv(k.data_ptr(), v.data_ptr(), slots.data_ptr(), None, L0 + T)
    code = lib.ts_prefill_prompt(ctypes.byref(cc), ctypes.byref(bt), ctypes.byref(kv), q.data_ptr(), 0, 0, T, 512,
                                 cos.data_ptr(), sin.data_ptr(), cos.shape[0], k_pool.data_ptr(), v_pool.data_ptr(),
                                 k_pool.shape[0], out.data_ptr(), workspace.data_ptr(), nbytes,
                                 torch.cuda.current_stream().cuda_stream)
    assert code == _lib.TS_OK, lib.ts_last_error()
    torch.cuda.synchronize()
    _same((k_pool, v_pool, table, seq, out), want)


@pytest.mark.parametrize("where", ["key", "query"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("pool", [-1, 5], ids=["votes", "pooled"])
def test_values_that_are_not_finite(dev, where, value, pool):
    """A key of the context or a query row that is not finite: its head's scores, and with them the votes of the
    chunks that see it, are what they are for the chunks one by one, and so is what is selected and attended to."""
    L0, T, chunk = 900, 300, 64
    say(f"prompt with {value} in a {where}, pool {pool}")
    wl, c, q, k, v, slots = _prompt(dev, 8, 2, L0, T, 96, pool_kernel=pool)
    if where == "key":
        wl.k_pool[wl.table[0, 500].long(), 1, 7] = value
    else:
        q[chunk + 3, 2 * 128 + 9] = value
    x, y = (_served(dev, wl, c, q, k, v, slots, L0, L0 + T, chunk, together) for together in (True, False))
    _same([t.nan_to_num(nan=77.0) if t.dtype == torch.bfloat16 else t for t in x],
          [t.nan_to_num(nan=77.0) if t.dtype == torch.bfloat16 else t for t in y])


def test_a_prompt_without_memory_for_its_workspace(dev, monkeypatch):
    """Where a round's workspace (some 230 MB here) cannot be had, the chunks go one by one, in the memory that
    the request holds anyway: the results are those of the chunks together (kernels of either width: 2e-2)."""
    monkeypatch.setattr(tr, "PREFILL_CHUNK_SIZE", 512)
    H, Hkv, D, prompt = 8, 8, 128, 13000
    say("prompt without memory for its workspace")
    tr.patch(rope_base=5e5, rope_scale=1, rope_model="ROPE_LLAMA", max_n_tokens=16384, top_k=2048, n_init=128, n_local=512)
    g = torch.Generator(device=dev).manual_seed(61)
    common = torch.randn(1, H * D, generator=g, device=dev)
    q = (common + torch.randn(prompt, H * D, generator=g, device=dev)).bfloat16()
    k, v = (torch.randn(prompt, Hkv * D, generator=g, device=dev).bfloat16() for _ in range(2))
    slots = torch.randperm(prompt, generator=g, device=dev).to(torch.int32)
    pool = sg.TokenToKVPool(prompt, torch.bfloat16, Hkv, D, 1, dev)
    runner = sg.ModelRunner(model_config=sg.ModelConfig(1, D, H, Hkv), token_to_kv_pool=pool, dtype=torch.bfloat16)
    attn = sg.RadixAttention(H, D, D ** -0.5, Hkv, layer_id=0)

    def serve(name):
        retriever = runner.req_to_token_retriever.get_token_retriever(name)
        out = attn.forward(q, k, v, sg.InputMetadata(sg.ForwardMode.EXTEND, retriever, pool, slots))
        torch.cuda.synchronize()
        return out.float(), retriever.num_tokens[0], int(retriever._num_tokens_dev[0])

    want = serve("with")
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (192 << 20)) / total)
    try:
        held = []
        with pytest.raises(torch.OutOfMemoryError):
            while len(held) < 4096:
                held.append(torch.empty(64 << 20, dtype=torch.uint8, device=dev))
        del held[-2:]
        refused = torch.cuda.memory_stats(dev)["num_ooms"]
        got = serve("without")
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.cuda.memory_stats(dev)["num_ooms"] > refused
    assert got[1:] == want[1:] == (prompt, prompt)
    assert (got[0] - want[0]).abs().max().item() <= 2e-2
