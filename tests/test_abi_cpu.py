"""CPU-side checks of the C ABI: the built library loads without a GPU, exports
every symbol ``include/tokenselect.h`` declares, and rejects bad arguments on the
host (before any HIP call) with the documented error codes."""

import ctypes
import os
import re

import pytest
import torch

from tokenselect_amd import _lib, ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(_lib.LIB_PATH):
        from tokenselect_amd import build
        build.build(verbose=False)
    return _lib.load()


def cfg(**kw):
    base = dict(num_heads=32, num_kv_heads=8, head_dim=128, page_size=1, n_init=128, n_local=512,
                top_k=2048, pool_kernel=-1, head_map=0, rope_mode=1, rope_theta=5e5, rope_scale=1.0,
                sm_scale=0.088, logit_cap=0.0)
    base.update(kw)
    return _lib.TsConfig(*[base[name] for name, _ in _lib.TsConfig._fields_])


def err(lib):
    return lib.ts_last_error().decode()


def test_header_symbols_are_exported_and_bound(lib):
    header = open(os.path.join(ROOT, "include", "tokenselect.h")).read()
    declared = set(re.findall(r"\b(ts_[a-z_]+)\s*\(", header))
    assert declared, "no declarations found in the header"
    for name in declared:
        assert hasattr(lib, name), f"{name} is declared in the header but not exported"
    assert declared == set(_lib.SIGNATURES), "ctypes signatures and header disagree"
    assert lib.ts_version() == int(re.search(r"#define TS_VERSION (\d+)", header).group(1))


def test_struct_layouts_match_the_header():
    assert ctypes.sizeof(_lib.TsConfig) == 14 * 4
    assert ctypes.sizeof(_lib.TsBatch) == 8 + 8 + 8 + 8 + 8 + 8 + 8 + 8 + 4 * 4 + 8  # 5 ints, padded
    assert _lib.TsBatch.workspace_clean.offset == 80
    assert _lib.TsBatch.threshold_hint.offset == 56
    assert _lib.TsBatch.separate_kernels.offset == 64 and _lib.TsBatch.rerun.offset == 68
    assert _lib.TsBatch.wait_us.offset == 72 and _lib.TsBatch.absent_workgroups.offset == 76
    assert _lib.TsBatch.fault.offset == 40 and _lib.TsBatch.host_seq_lens.offset == 48
    assert _lib.TsBatch.seq_lens.offset == 8 and _lib.TsBatch.table_stride.offset == 24
    assert ctypes.sizeof(_lib.TsSelCache) == 4 * 8 + 8
    assert ctypes.sizeof(_lib.TsNewKv) == 4 * 8 + 8 and _lib.TsNewKv.max_tokens.offset == 32


def test_padding_of_the_structs_is_not_read(lib):
    """ts_batch and ts_new_kv end in four bytes of padding, in which a caller may leave anything:
    what is reported is what is wrong with the call (here its workspace)."""
    c, one = cfg(), ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first

    def padded(struct):
        raw = bytearray(struct)
        assert len(raw) == ctypes.sizeof(struct) and not any(raw[-4:])
        raw[-4:] = (12345).to_bytes(4, "little")
        return type(struct).from_buffer(raw)

    bt = padded(_lib.TsBatch(1, 4096, one, one, 4096, None))
    kv = padded(_lib.TsNewKv(one, one, one, None, 4096))
    cache = _lib.TsSelCache(one, one, one, one, 0.9)
    tail = (one, one, one, 4096, one, one, 64, None)
    assert lib.ts_decode_layer(ctypes.byref(c), ctypes.byref(bt), one, one, one, one, one, 10, None,
                               *tail) == _lib.TS_EWORKSPACE, err(lib)
    assert lib.ts_decode_step(ctypes.byref(c), ctypes.byref(bt), ctypes.byref(kv), one, one, one, one, one, 10,
                              ctypes.byref(cache), *tail) == _lib.TS_EWORKSPACE, err(lib)
    assert lib.ts_prefill_step(ctypes.byref(c), ctypes.byref(bt), ctypes.byref(kv), one, 8, one, one, 4096, one, one,
                               10, *tail) == _lib.TS_EWORKSPACE, err(lib)


def test_row_strides_are_checked_before_anything_is_launched(lib):
    """The strided steps: rows at least as far apart as they are long, in whole 16-byte pieces."""
    c, one = cfg(), ctypes.c_void_p(0x1000)
    bt = _lib.TsBatch(1, 4096, one, one, 4096, None)
    kv = _lib.TsNewKv(one, one, one, None, 4096)
    cache = _lib.TsSelCache(one, one, one, one, 0.9)
    tail = (one, one, one, 4096, one, one, 64, None)
    for q, rows, code in ((0, 0, _lib.TS_EWORKSPACE), (6144, 6144, _lib.TS_EWORKSPACE), (4096, 1024, _lib.TS_EWORKSPACE),
                          (4088, 1024, _lib.TS_EINVAL), (4100, 1024, _lib.TS_EINVAL), (-4096, 1024, _lib.TS_EINVAL),
                          (4096, 1016, _lib.TS_EINVAL), (4096, 1028, _lib.TS_EINVAL)):
        assert lib.ts_decode_step_strided(ctypes.byref(c), ctypes.byref(bt), ctypes.byref(kv), one, q, rows, one, one,
                                          one, one, 10, ctypes.byref(cache), *tail) == code, (q, rows, err(lib))
        assert lib.ts_prefill_step_strided(ctypes.byref(c), ctypes.byref(bt), ctypes.byref(kv), one, q, rows, 8, one,
                                           one, 4096, one, one, 10, *tail) == code, (q, rows, err(lib))


def test_config_validation(lib):
    assert lib.ts_check_config(ctypes.byref(cfg())) == _lib.TS_OK
    assert lib.ts_check_config(None) == _lib.TS_EINVAL
    assert lib.ts_check_config(ctypes.byref(cfg(head_dim=64))) == _lib.TS_ESHAPE
    assert "head_dim 64" in err(lib)
    assert lib.ts_check_config(ctypes.byref(cfg(num_heads=30))) == _lib.TS_ESHAPE
    assert lib.ts_check_config(ctypes.byref(cfg(num_heads=72, num_kv_heads=8))) == _lib.TS_ESHAPE
    assert lib.ts_check_config(ctypes.byref(cfg(num_heads=24, num_kv_heads=3))) == _lib.TS_ESHAPE
    assert lib.ts_check_config(ctypes.byref(cfg(page_size=12))) == _lib.TS_EINVAL
    assert lib.ts_check_config(ctypes.byref(cfg(top_k=0))) == _lib.TS_EINVAL
    assert lib.ts_check_config(ctypes.byref(cfg(rope_mode=7))) == _lib.TS_EINVAL
    assert lib.ts_check_config(ctypes.byref(cfg(rope_theta=0.0))) == _lib.TS_EINVAL
    for hkv, g in [(1, 8), (2, 2), (4, 7), (8, 4), (8, 8), (4, 1), (8, 3), (2, 6), (4, 5)]:
        assert lib.ts_check_config(ctypes.byref(cfg(num_heads=hkv * g, num_kv_heads=hkv))) == 0


def test_workspace_queries(lib):
    c = cfg()
    assert lib.ts_decode_layer_workspace_bytes(ctypes.byref(c), 1, 131072) > 32 * 131072 * 4
    assert lib.ts_decode_layer_workspace_bytes(ctypes.byref(cfg(head_dim=64)), 1, 1024) == 0
    assert lib.ts_score_partials_bytes(ctypes.byref(c), 1, 131072) % 256 == 0
    assert lib.ts_attn_workspace_bytes(ctypes.byref(c), 4, 2688) > 0


def test_null_and_range_errors_need_no_gpu(lib):
    c = cfg()
    one = ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first
    bt = _lib.TsBatch(1, 4096, one, one, 4096, None)
    assert lib.ts_score(ctypes.byref(c), None, one, one, 10, None, one, 4096, one, 1 << 20,
                        None) == _lib.TS_EINVAL
    assert lib.ts_score(ctypes.byref(c), ctypes.byref(bt), None, one, 10, None, one, 4096, one,
                        1 << 20, None) == _lib.TS_EINVAL
    assert "NULL" in err(lib)
    # score stride smaller than the candidate count
    assert lib.ts_score(ctypes.byref(c), ctypes.byref(bt), one, one, 10, None, one, 100, one,
                        1 << 20, None) == _lib.TS_EWORKSPACE
    # partials buffer too small
    assert lib.ts_score(ctypes.byref(c), ctypes.byref(bt), one, one, 10, None, one, 4096, one, 16,
                        None) == _lib.TS_EWORKSPACE
    bad = _lib.TsBatch(0, 4096, one, one, 4096, None)
    assert lib.ts_vote(ctypes.byref(c), ctypes.byref(bad), one, 4096, one, None, one, one, None,
                       4096, None) == _lib.TS_EINVAL
    # a host-side length beyond max_seq_len
    lens = (ctypes.c_int32 * 1)(5000)
    beyond = _lib.TsBatch(1, 4096, one, one, 4096, None, None, ctypes.cast(lens, ctypes.c_void_p))
    assert lib.ts_vote(ctypes.byref(c), ctypes.byref(beyond), one, 4096, one, None, one, one, None,
                       4096, None) == _lib.TS_EINVAL
    # table rows too short for a batch of 2
    short = _lib.TsBatch(2, 4096, one, one, 100, None)
    assert lib.ts_topk_ragged(ctypes.byref(c), ctypes.byref(short), one, 4096, None, None, one, one,
                              4096, one, one, 256, None) == _lib.TS_EINVAL
    # sel_stride below n_init + top_k + n_local
    assert lib.ts_topk_ragged(ctypes.byref(c), ctypes.byref(bt), one, 4096, None, None, one, one,
                              100, one, one, 256, None) == _lib.TS_EWORKSPACE
    # hit flags without a cache
    assert lib.ts_topk_ragged(ctypes.byref(c), ctypes.byref(bt), one, 4096, one, None, one, one,
                              4096, one, one, 256, None) == _lib.TS_EINVAL
    assert lib.ts_sparse_decode_attn(ctypes.byref(c), one, one, one, 10, one, 4096, one, 1, 2688,
                                     one, one, 16, None) == _lib.TS_EWORKSPACE
    assert lib.ts_paged_matmul(one, one, 10, one, one, 5, 10, 32, 8, 128, None) == _lib.TS_EINVAL
    assert lib.ts_paged_matmul(one, one, 10, one, one, 0, 10, 32, 8, 64, None) == _lib.TS_ESHAPE
    assert lib.ts_rope_apply(one, one, one, one, None, 1, 1, 4, 127, None) == _lib.TS_ESHAPE
    # pages of 16 tokens without a page pool
    assert lib.ts_kv_store(ctypes.byref(cfg(page_size=16)), one, one, one, None, one, one, 10, one, 100,
                           one, 1, 100, None) == _lib.TS_EINVAL
    assert "page pool" in err(lib)
    # more than 2^20 candidates per request
    huge = _lib.TsBatch(1, (1 << 20) + 641, one, one, 1 << 21, None)
    assert lib.ts_topk_ragged(ctypes.byref(c), ctypes.byref(huge), one, 1 << 21, None, None, one, one,
                              4096, one, one, 1 << 30, None) == _lib.TS_ESHAPE
    assert lib.ts_decode_layer(ctypes.byref(c), ctypes.byref(bt), one, one, one, one, one, 10, None,
                               one, one, one, 4096, one, one, 64, None) == _lib.TS_EWORKSPACE
    assert "workspace" in err(lib)


def test_misaligned_buffers_are_refused_on_the_host(lib):
    """Tensors are read with 16-byte vector loads and workspaces hold 8-byte atomics: a view at
    an odd offset fails the call instead of faulting the device."""
    c = cfg()
    one, odd = ctypes.c_void_p(0x1000), ctypes.c_void_p(0x1004)
    bt = _lib.TsBatch(1, 4096, one, one, 4096, None)
    big = 1 << 30
    assert lib.ts_score_vote(ctypes.byref(c), ctypes.byref(bt), one, odd, 10, None, one, 4096, one, big,
                             None) == _lib.TS_EINVAL
    assert "k_pool must be aligned" in err(lib)
    assert lib.ts_score_vote(ctypes.byref(c), ctypes.byref(bt), one, one, 10, None, one, 4096,
                             ctypes.c_void_p(0x1010), big, None) == _lib.TS_EINVAL
    assert "workspace must be aligned to 256" in err(lib)
    assert lib.ts_topk_ragged(ctypes.byref(c), ctypes.byref(bt), one, 4096, None, None, one, one, 4096,
                              one, ctypes.c_void_p(0x1008), big, None) == _lib.TS_EINVAL
    assert lib.ts_sparse_decode_attn(ctypes.byref(c), odd, one, one, 10, one, 4096, one, 1, 2688,
                                     one, one, big, None) == _lib.TS_EINVAL
    assert "q must be aligned" in err(lib)
    # the stores and the projection: rows are copied as 16-byte vectors
    assert lib.ts_kv_store(ctypes.byref(c), one, odd, one, None, one, one, 10, one, 4096, one, 1, 4096,
                           None) == _lib.TS_EINVAL
    assert "v must be aligned" in err(lib)
    assert lib.ts_kv_store_chunk(ctypes.byref(c), one, one, one, None, 4, one, odd, 10, one, one, 4096,
                                 None) == _lib.TS_EINVAL
    assert "v_pool must be aligned" in err(lib)
    assert lib.ts_qkv_store(ctypes.byref(c), one, odd, None, 4096, one, None, one, one, one, 10, one,
                            4096, one, 1, 4096, None) == _lib.TS_EINVAL
    assert "w must be aligned" in err(lib)
    assert lib.ts_fingerprint(ctypes.byref(c), odd, 4, one, one, 4096, one, one) == _lib.TS_EINVAL
    assert "q must be aligned" in err(lib)


def test_static_scratch_entry_point_rejects_what_does_not_fit(lib):
    assert lib.ts_attn_static_scratch_bytes() == 4 << 20
    one = ctypes.c_void_p(0x1000)  # never dereferenced: the size check fails first
    wide = cfg(num_heads=64, num_kv_heads=8, top_k=4096)
    # 130 requests x 64 heads x 512 bytes of partials per head and split: above 4 MiB
    assert lib.ts_sparse_decode_attn_static(ctypes.byref(wide), one, one, one, 10, one, 4736, one,
                                            130, 4736, one, None) == _lib.TS_EWORKSPACE
    assert "scratch" in err(lib)
    assert lib.ts_sparse_decode_attn_static(ctypes.byref(cfg()), one, one, one, 10, None, 2688, one,
                                            1, 2688, one, None) == _lib.TS_EINVAL


def test_python_layer_refuses_cpu_tensors(lib):
    c = ops.LayerConfig(num_heads=4, num_kv_heads=2, n_init=1, n_local=2, top_k=4)
    x = torch.zeros(1, 4, 128, dtype=torch.bfloat16)
    t = torch.zeros(4, 128)
    with pytest.raises(ValueError, match="no CPU path"):
        ops.rope_apply(x, t, t, None)
    bt = ops.Batch(torch.zeros(1, dtype=torch.int32), torch.zeros(1, 64, dtype=torch.int32), 64)
    with pytest.raises(ValueError, match="no CPU path"):
        ops.score(c, bt, x, torch.zeros(64, 2, 128, dtype=torch.bfloat16))
    with pytest.raises(TypeError):
        ops.rope_apply(x.float(), t, t, None)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libtokenselect_hip.so"))
    with pytest.raises(ImportError, match="no CPU fallback"):
        _lib.load()


def test_workspace_sizes_never_shrink_with_the_context_or_the_batch(lib):
    """A workspace sized for (batch, max_seq_len) must serve every smaller batch and every
    shorter context: the candidates per workgroup move in steps, so the sizes are taken
    from bounds that do not."""
    for heads, kv in ((32, 8), (28, 4), (8, 1)):
        c = cfg(num_heads=heads, num_kv_heads=kv)
        lens = list(range(700, 70000, 997)) + [32768, 32769, 131072, 131073, 262144, 262145, 1048576]
        for fn in (lib.ts_decode_layer_workspace_bytes, lib.ts_score_partials_bytes,
                   lib.ts_select_workspace_bytes, lib.ts_topk_workspace_bytes):
            sizes = [fn(ctypes.byref(c), 4, L) for L in sorted(lens)]
            assert all(x > 0 for x in sizes)
            assert sizes == sorted(sizes), fn.__name__
        by_batch = [lib.ts_decode_layer_workspace_bytes(ctypes.byref(c), B, 65536) for B in range(1, 33)]
        assert by_batch == sorted(by_batch)


def test_header_is_plain_c_and_agrees_with_the_ctypes_mirror(tmp_path):
    """The boundary is a C ABI: the header compiles as C99 (no C++ in it), and a C program
    sees the struct sizes and field offsets that the ctypes mirror and the library use."""
    import shutil
    import subprocess
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no C compiler")
    include = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include")
    # The mirror has the header's fields, all of them and in their order.
    header = re.sub(r"/\*.*?\*/", "", open(os.path.join(include, "tokenselect.h")).read(), flags=re.S)
    mirrors = {"ts_config": _lib.TsConfig, "ts_batch": _lib.TsBatch, "ts_selcache": _lib.TsSelCache,
               "ts_page_pool": _lib.TsPagePool, "ts_new_kv": _lib.TsNewKv}
    structs = dict(re.findall(r"typedef struct (\w+) \{(.*?)\}", header, flags=re.S))
    assert set(structs) == set(mirrors)
    for name, mirror in mirrors.items():
        assert re.findall(r"(\w+)\s*;", structs[name]) == [f[0] for f in mirror._fields_], name
    src = tmp_path / "layout.c"
    src.write_text(
        '#include <stddef.h>\n#include <stdio.h>\n#include "tokenselect.h"\n'
        'int main(void) {\n'
        + "".join(f'  printf("%zu\\n", sizeof({name}));\n' + "".join(
            f'  printf("%zu\\n", offsetof({name}, {field[0]}));\n' for field in mirror._fields_)
            for name, mirror in mirrors.items()) +
        '  return 0;\n}\n')
    exe = tmp_path / "layout"
    subprocess.run([gcc, "-std=c99", "-Wall", "-Wextra", "-Werror", "-pedantic", "-I", include, str(src),
                    "-o", str(exe)], check=True)
    got = [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    want = [n for mirror in mirrors.values() for n in
            (ctypes.sizeof(mirror), *(getattr(mirror, field[0]).offset for field in mirror._fields_))]
    assert got == want


def test_a_prompts_arguments_are_checked_before_anything_is_launched(lib):
    """ts_prefill_prompt: what it does not take is refused on the host."""
    c, one = cfg(), ctypes.c_void_p(0x1000)
    pool = ctypes.pointer(_lib.TsPagePool(one, one, one))

    def call(rows=4096, chunk=512, batch=1, config=c, q=one, pages=None, stride=0, nbytes=64, k_per_req=None, **options):
        bt = _lib.TsBatch(batch, 4096, one, one, 4096, k_per_req)
        for name, value in options.items():
            setattr(bt, name, value)
        kv = _lib.TsNewKv(one, one, one, pages, 4096)
        return lib.ts_prefill_prompt(ctypes.byref(config), ctypes.byref(bt), ctypes.byref(kv), q, stride, 0, rows, chunk,
                                     one, one, 4096, one, one, 10, one, one, nbytes, None)

    assert call() == _lib.TS_EWORKSPACE, err(lib)
    for bad in (dict(rows=0), dict(chunk=0), dict(batch=2), dict(q=None), dict(pages=pool), dict(stride=4088),
                dict(config=cfg(page_size=16)), dict(k_per_req=one), dict(chunk=4000), dict(rerun=1)):
        assert call(**bad) == _lib.TS_EINVAL, (bad, err(lib))
    assert lib.ts_prefill_prompt_workspace_bytes(ctypes.byref(c), 0, 512, 4096) == 0


def test_a_prompts_workspace_is_bounded(lib):
    """512 MiB, or what one chunk needs where that is more, however long the prompt."""
    for c in (cfg(), cfg(top_k=4096, pool_kernel=15), cfg(num_heads=28, num_kv_heads=4), cfg(n_local=65536),
              cfg(num_heads=4, num_kv_heads=1, top_k=64)):
        for length in (700, 31615, 131072, 1 << 20):
            one = lib.ts_prefill_prompt_workspace_bytes(ctypes.byref(c), 512, 512, length)
            few, many = (lib.ts_prefill_prompt_workspace_bytes(ctypes.byref(c), n * 512, 512, length) for n in (2, 2000))
            assert 0 < one <= few <= many <= max(512 << 20, one), (length, one, few, many)
