"""CPU-side checks of the product's host logic: the C ABI loads and exports everything
include/ksa_hip.h declares, rejects bad arguments before any launch, the closed-form
visibility rule used by the kernels equals the oracle predicate, and the cache class keeps
the reference's bookkeeping (checked against the oracle's integer model with a host row
mover injected by the test — the product itself has none)."""
import ctypes
import os
import re
import types

import numpy as np
import pytest
import torch

from oracle import ksa_oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    from ksa_amd import _lib
    L = _lib.lib()
    header = open(os.path.join(ROOT, "include", "ksa_hip.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(ksa_[a-z0-9_]+)\s*\(", header))
    assert declared, "no declarations found"
    assert declared == set(_lib.EXPORTS), declared ^ set(_lib.EXPORTS)
    for name in declared:
        assert getattr(L, name) is not None
    assert L.ksa_version() >= 100
    assert b"ok" == L.ksa_error_string(0)


def test_error_codes_before_launch():
    from ksa_amd import _lib
    L = _lib.lib()
    # bad sizes / null pointers are rejected without touching a device
    assert L.ksa_block_index(0, 10, 128, 8, 3, 10, 0, 128, 64, None, None, None, None, None) == -1
    assert L.ksa_block_index(100, 110, 128, 8, 3, 9, 0, 128, 64, None, None, None, None, None) == -1
    assert L.ksa_block_index(100, 110, 128, 8, 3, 10, 0, 128, 64, None, None, None, None, None) == -2
    null3 = ctypes.cast(None, ctypes.POINTER(ctypes.c_int64))
    assert L.ksa_prefill_fwd(None, None, None, None, None, 1, 128, 4, 2, 128, 0, null3, null3, null3,
                             128, 8, 3, 0, 0, 0, None, None, None, None, 2, 1.0, 0, None, None) == -2
    assert L.ksa_prefill_chunks_fwd(None, None, None, None, None, 1, 128, 4, 2, 128, 0, null3, null3, null3,
                                    128, 8, 3, 0, 1.0, 0, None, None) == -2
    assert L.ksa_decode_fwd(None, None, None, None, None, None, 0, 10, 1, 4, 2, 1, 128, 0, null3, null3,
                            null3, null3, 1.0, 1, None, 0, None) == -2
    assert L.ksa_decode_workspace_bytes(64, 32, 8, 1, 128, 1) == 0
    assert L.ksa_decode_workspace_bytes(64, 32, 8, 1, 128, 2) == 64 * 8 * 2 * 32 * 130 * 4
    assert L.ksa_decode_auto_splits(64, 8, 17288) == 1
    assert L.ksa_decode_auto_splits(8, 8, 17288) == 8
    assert L.ksa_decode_auto_splits(1, 8, 100) == 1
    assert 1 <= L.ksa_decode_auto_splits(1, 8, 100000) <= 64


@pytest.mark.parametrize("P_mode", ["prefix", "inline"])
def test_closed_form_counts_equal_predicate(P_mode):
    """ksa_count_visible (csrc/ksa_mask.h, the rule both the index kernel and the prefill
    mask are built on) against brute force over the oracle predicate."""
    from ksa_amd import _lib
    L = _lib.lib()
    rng = np.random.default_rng(1)
    for _ in range(60):
        C, S = int(rng.integers(1, 24)), int(rng.integers(1, 6))
        W = int(rng.integers(0, 6))
        n = int(rng.integers(1, 9))
        Sq = n * (C + S) + int(rng.integers(0, C + 1))
        P = (Sq // (C + S)) * S if P_mode == "prefix" else 0
        Sk = Sq + P
        skip = int(rng.integers(0, 2))
        vis = O.dense_mask_predicate(Sq, C, S, W, P, bool(skip))
        cum = np.concatenate([np.zeros((Sq, 1), np.int64), np.cumsum(vis, axis=1)], axis=1)
        for _ in range(40):
            q = int(rng.integers(0, Sq))
            a = int(rng.integers(0, Sk))
            b = int(rng.integers(a, Sk + 1))
            got = L.ksa_debug_count_visible(q, a, b, C, S, W, P, skip, Sq, Sk)
            assert got == cum[q, b] - cum[q, a], (C, S, W, P, skip, q, a, b)


def _host_mover(src, dst, nrows, src_start=0, dst_start=0, src_index=None):
    if nrows <= 0:
        return
    rows = src_index.long() if src_index is not None else torch.arange(src_start, src_start + nrows)
    dst[:, :, dst_start:dst_start + nrows, :] = src[:, :, rows[:nrows], :].clone()


def _make_cache(C, S, scns):
    from ksa_amd.cache import Qwen3RingBufferCache
    cfg = types.SimpleNamespace(summary_chunk_size=C, summary_token_num=S, num_hidden_layers=len(scns))

    class HostCache(Qwen3RingBufferCache):
        _move_rows = staticmethod(_host_mover)
    return HostCache(cfg, scns)


@pytest.mark.parametrize("C,S", [(4, 2), (8, 1)])
@pytest.mark.parametrize("n_prefill", [1, 7, 16, 37])
def test_cache_bookkeeping_matches_model(C, S, n_prefill):
    """Drives the product cache class and the oracle's integer model with the same tagged
    rows through prefill, reorganisation, decode steps and chunk boundaries."""
    scns = [2, 3, 1000]                # last layer is a large-window layer
    cache = _make_cache(C, S, scns)
    assert cache.is_large_window == [False, True, True]
    B = C + S
    n_full = n_prefill // C
    Sq = n_full * B + n_prefill % C
    sp = O.summary_positions(Sq, C, S)
    D, H = 8, 2
    tags = torch.arange(Sq, dtype=torch.float32)
    kv = tags[None, None, :, None].expand(1, H, Sq, D).to(torch.bfloat16).contiguous()
    models = [O.RingBufferModel(C, S, scn, large) for scn, large in zip(scns, cache.is_large_window)]
    spt = torch.from_numpy(sp)[None]
    for layer in range(3):
        k_all, v_all = cache.update(kv, kv, layer, {"summary_mask": spt})
        assert k_all.shape[2] == Sq
    # as in the reference, a small-window layer reports 0 until the cache is reorganised
    assert cache.get_true_token_num() == n_prefill and cache.get_seq_length(0) == 0 and cache.get_seq_length(1) == Sq
    cache.reorganize_after_prefill(spt)
    for m in models:
        m.reorganize_after_prefill(np.arange(Sq), sp)
    pos = Sq
    n_text = n_prefill

    def check():
        for layer, m in enumerate(models):
            a, b = m.attention_range()
            assert cache.attention_range(layer) == (a, b)
            k, v = cache.get_attention_kv(layer)
            assert k.shape[2] == b - a
            assert sorted(k[0, 0, :, 0].float().tolist()) == sorted(m.buf[a:b].tolist())
            assert cache._capacity[layer] == m.cap == cache.key_cache[layer].shape[2]
        assert cache.get_true_token_num() == n_text

    check()
    for _ in range(3 * C + 1):
        row = torch.full((1, H, 1, D), float(pos), dtype=torch.bfloat16)
        for layer, m in enumerate(models):
            cache.update_text(row, row, layer)
            m.update_text(pos)
        n_text += 1
        pos += 1
        check()
        if n_text % C == 0:
            stags = np.arange(pos, pos + S)
            srow = torch.from_numpy(stags.astype(np.float32))[None, None, :, None].expand(1, H, S, D).to(torch.bfloat16)
            for layer, m in enumerate(models):
                ks, vs = cache.get_summary_attention_kv(layer, srow, srow)
                assert sorted(ks[0, 0, :, 0].float().tolist()) == list(range(pos - C, pos + S))
                cache.update_summary(srow, srow, layer)
                m.update_summary(stags)
            pos += S
            assert cache.get_cur_chunk_size() == B
            cache.reset_chunk_counter()
            assert cache.get_cur_chunk_size() == 0
            check()


@pytest.mark.parametrize("C,S,n_prefill", [(4, 2, 7), (8, 1, 16), (4, 2, 1), (2, 1, 3)])
def test_cache_boundary_slots_equal_update_calls(C, S, n_prefill):
    """`boundary_slots` + the caller's own row moves (what the recorded boundary step does)
    against `update_text` + `get_summary_attention_kv` + `update_summary` on a second cache
    driven with the same rows: same counters, same ranges, same buffer contents wherever
    rows are attended, over many boundaries (ring wrap-around, growth of the summary region)."""
    scns = [2, 3, 1000]
    a_cache, b_cache = _make_cache(C, S, scns), _make_cache(C, S, scns)
    for c in (a_cache, b_cache):
        c._SUMMARY_INIT_CAP = 4
        c._APPEND_HEADROOM = 5
    B = C + S
    Sq = (n_prefill // C) * B + n_prefill % C
    sp = torch.from_numpy(O.summary_positions(Sq, C, S))[None]
    D, H = 8, 2
    kv = torch.arange(Sq, dtype=torch.float32)[None, None, :, None].expand(1, H, Sq, D).to(torch.bfloat16).contiguous()
    for c in (a_cache, b_cache):
        for layer in range(3):
            c.update(kv, kv, layer, {"summary_mask": sp})
        c.reorganize_after_prefill(sp)
    pos, n_text, n_boundaries = Sq, n_prefill, 0
    counters = ("_text_len", "_capacity", "_window_write_ptr", "_n_valid_window", "_chunk_buf_len",
                "_n_summaries", "cur_chunk_sizes", "true_tokens", "_total_chunks")
    for _ in range(40 * C):
        row = torch.full((1, H, 1, D), float(pos % 251), dtype=torch.bfloat16)
        boundary = n_text % C == C - 1
        if not boundary:
            for layer in range(3):
                a_cache.update_text(row, row, layer)
                b_cache.update_text(row, row, layer)
            pos += 1
        else:
            srow = (torch.arange(pos + 1, pos + 1 + S) % 251).float()[None, None, :, None].expand(1, H, S, D).to(torch.bfloat16)
            for layer in range(3):
                a_cache.update_text(row, row, layer)
                want_range = a_cache.attention_range(layer)
                ks, _ = a_cache.get_summary_attention_kv(layer, srow, srow)
                want_sum = ks[0, 0, :, 0].float().tolist()
                a_cache.update_summary(srow, srow, layer)
                # the same step from the rows `boundary_slots` names
                assert b_cache.boundary_fits_one_piece(layer)
                sl = b_cache.boundary_slots(layer, S)
                for buf in (b_cache.key_cache[layer], b_cache.value_cache[layer]):
                    _host_mover(row, buf, 1, 0, sl["text"])
                    assert sl["attend"] == want_range
                    if b_cache.is_large_window[layer]:
                        _host_mover(srow, buf, S, 0, sl["spare"])
                        got_sum = buf[0, 0, sl["spare"] - C:sl["spare"] + S, 0].float().tolist()
                    else:
                        _host_mover(srow, buf, S, 0, 0)
                        got_sum = buf[0, 0, :S + C, 0].float().tolist()
                        _host_mover(buf, buf, sl["flush_rows"], sl["flush_src"], sl["flush_dst"])
                        _host_mover(srow, buf, S, 0, sl["append"])
                    assert sorted(got_sum) == sorted(want_sum)
            pos += 1 + S
            n_boundaries += 1
            a_cache.reset_chunk_counter()
            b_cache.reset_chunk_counter()
        n_text += 1
        for name in counters:
            va, vb = getattr(a_cache, name), getattr(b_cache, name)
            if name == "_capacity":   # an append-only buffer also holds the step's spare rows
                assert va[0] == vb[0] and all(x <= y for x, y in zip(va[1:], vb[1:]))
            else:
                assert va == vb, name
        for layer in range(3):
            a, e = a_cache.attention_range(layer)
            assert b_cache.attention_range(layer) == (a, e)
            assert torch.equal(a_cache.key_cache[layer][:, :, a:e], b_cache.key_cache[layer][:, :, a:e])
            assert torch.equal(a_cache.value_cache[layer][:, :, a:e], b_cache.value_cache[layer][:, :, a:e])
    assert n_boundaries >= 30


def test_cache_summary_growth():
    """Summary region overflows its headroom -> buffer grows to the right, rows keep their place."""
    C, S = 2, 1
    cache = _make_cache(C, S, [1])
    cache._SUMMARY_INIT_CAP = 4
    model = O.RingBufferModel(C, S, 1)
    model.SUMMARY_INIT_CAP = 4
    Sq = 3
    sp = O.summary_positions(Sq, C, S)
    kv = torch.arange(Sq, dtype=torch.float32)[None, None, :, None].expand(1, 1, Sq, 8).to(torch.bfloat16).contiguous()
    cache.update(kv, kv, 0, {"summary_mask": torch.from_numpy(sp)[None]})
    cache.reorganize_after_prefill(torch.from_numpy(sp)[None])
    model.reorganize_after_prefill(np.arange(Sq), sp)
    pos = Sq
    for step in range(1200):
        row = torch.full((1, 1, 1, 8), float(pos % 251), dtype=torch.bfloat16)
        cache.update_text(row, row, 0)
        model.update_text(pos % 251)
        pos += 1
        if cache._chunk_buf_len[0] == C:
            srow = torch.full((1, 1, S, 8), float(pos % 251), dtype=torch.bfloat16)
            cache.update_summary(srow, srow, 0)
            model.update_summary([pos % 251])
            pos += 1
    assert cache._capacity[0] == model.cap > 300
    a, b = model.attention_range()
    assert cache.attention_range(0) == (a, b)
    assert cache.key_cache[0][0, 0, a:b, 0].float().tolist() == [float(x) for x in model.buf[a:b]]


def test_split_heuristics_are_host_only_and_bounded():
    """`ksa_gemm_rows_auto_splits` / `ksa_decode_auto_splits` run on the host: the decoder's
    shapes get the split counts the kernels were tuned with, and any shape gets a count the
    kernels accept (at least 1, at most 16, never a slice shorter than one 512-element chunk)."""
    from ksa_amd import _lib
    L = _lib.lib()
    known = {(6144, 2560): 5, (2560, 4096): 8, (19456, 2560): 5, (2560, 9728): 13, (151936, 2560): 1}
    for (N, K), want in known.items():
        assert L.ksa_gemm_rows_auto_splits(N, K) == want, (N, K)
    rng = np.random.default_rng(0)
    for _ in range(200):
        N, K = int(rng.integers(1, 200000)), 32 * int(rng.integers(1, 600))
        sp = L.ksa_gemm_rows_auto_splits(N, K)
        assert 1 <= sp <= 16 and sp <= max(1, K // 512), (N, K, sp)
        assert L.ksa_gemm_rows_workspace_bytes(N, sp) == (0 if sp == 1 else sp * 16 * N * 4)
    for b, h, rows in [(64, 8, 17288), (8, 8, 40000), (1, 1, 100), (1, 8, 1 << 20)]:
        assert 1 <= L.ksa_decode_auto_splits(b, h, rows) <= 64
    assert L.ksa_decode_auto_splits(64, 8, 17288) == 1


def test_summary_pos_analysis_runs_once_for_fresh_views():
    """The HF call site passes `summary_mask.squeeze(0)`, a new tensor object per layer
    (modeling_qwen3sa.py:807-815): the analysis (one host synchronisation) must run once per
    buffer, not once per view, also for masks made under torch.inference_mode(), whose tensors
    have no modification counter."""
    from ksa_amd import prefill
    C, S = 16, 2
    Sq = 5 * (C + S) + 7
    for inference in (False, True):
        prefill.clear_summary_pos_cache()
        ctx = torch.inference_mode() if inference else torch.no_grad()
        with ctx:
            mask = (torch.arange(Sq) % (C + S) >= C)[None].clone()
            mask[0, 5 * (C + S):] = False
            before = prefill._POS_ANALYSES
            res = [prefill._analyse_summary_pos(mask.squeeze(0), Sq, C, S) for _ in range(3)]
        assert prefill._POS_ANALYSES - before == 1, inference
        assert all(r is res[0] for r in res)
        assert res[0][0] == 5 * S and res[0][1] is True and res[0][2] is None
    # an in-place edit of a tracked tensor is seen
    prefill.clear_summary_pos_cache()
    mask = (torch.arange(Sq) % (C + S) >= C).clone()
    mask[5 * (C + S):] = False
    a = prefill._analyse_summary_pos(mask, Sq, C, S)
    mask[3] = True
    b = prefill._analyse_summary_pos(mask, Sq, C, S)
    assert a[1] is True and b[1] is False and b[0] == a[0] + 1
    assert b[2].tolist() == sorted([3] + [i for i in range(5 * (C + S)) if i % (C + S) >= C])
    # a new mask of the same shape that reuses nothing of the old one is analysed on its own
    other = torch.zeros(Sq, dtype=torch.bool)
    assert prefill._analyse_summary_pos(other, Sq, C, S)[0] == 0
    prefill.clear_summary_pos_cache()


@pytest.mark.parametrize("b,hq,hkv,q", [(1, 32, 8, 1), (1, 32, 8, 9), (8, 32, 4, 8), (16, 8, 8, 1), (64, 32, 8, 1), (3, 8, 1, 40)])
def test_decode_splits_rule(b, hq, hkv, q):
    """The split count of the decode calls: never more than two workgroups per CU need, never splits of less
    than a round of the workgroup (128 rows), one split for up to three rounds, defined for every input."""
    from ksa_amd import _lib
    L = _lib.lib()
    units = b * hkv * -(-q * (hq // hkv) // 32)
    last = 0
    for rows in (1, 128, 192, 193, 256, 300, 513, 1000, 4096, 16384, 131072, 2**31 - 1):
        n = L.ksa_decode_splits(b, hq, hkv, q, 128, rows)
        assert last <= n <= 64 and (n == 1 or (n - 1) * units < 2 * 256 and (n - 1) * 128 < rows)
        if rows <= 300:
            assert n == 1
        last = max(n, 1)
        wide = L.ksa_decode_splits(b, hq, hkv, q, 256, rows)   # one workgroup per CU: no split without rows
        assert 1 <= wide <= 64 and (wide == 1 or (wide - 1) * -(-rows // 128 // wide) * 128 < rows)
    assert L.ksa_decode_splits(1, 32, 7, 1, 128, 1000) == 1 and L.ksa_decode_splits(0, 32, 8, 1, 128, 1000) == 1


def test_rules_of_the_native_front_are_those_of_the_general_way():
    """Which prompts take chunk tiles and which launches get work queues, over chunks, summaries, head dimensions and lengths on
    both sides of every line: the same in the native front and in Python."""
    from ksa_amd import _lib, prefill
    if _lib.fast is _lib._GeneralWay:
        pytest.skip("no native front")
    for C in (0, 1, 64, 100, 127, 128, 129, 256, 384, 500, 512, 513, 640, 1024):
        for S in (0, 1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 32, 64):
            for D in (64, 128, 256):
                B = C + S
                for Sq in {1, 63, 64, 65, 127, 128, B - 1, B, B + 1, C, C + 1, 3 * B, 3 * B + C - 1, 3 * B + C, 3 * B + C + 1, 4 * B - 1,
                           9001, 139264, (1 << 29) - 1, 1 << 29, (1 << 31) - 1}:
                    if Sq <= 0:
                        continue
                    got, queue = _lib.fast.layout_rules(Sq, D, C, S)
                    want = C > 0 and S > 0 and prefill._chunk_tiles(Sq, D, C, S, Sq // B * S, False)
                    assert got == want and queue == prefill._QUEUE_ROWS, (C, S, D, Sq)


@pytest.mark.parametrize("broken", ["missing", "other"])
def test_package_without_its_native_front(broken):
    """A native front that does not load (it is built against one PyTorch) or that is another build's leaves the Python way,
    with a warning; the library itself stays indispensable."""
    import subprocess
    import sys
    module = "None" if broken == "missing" else "types.SimpleNamespace(bind=lambda *a: (_ for _ in ()).throw(TypeError('entry points')))"
    code = f"""
import sys, types, warnings, importlib
front = {module}
sys.modules['ksa_amd._fast'] = front
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter('always')
    import ksa_amd
from ksa_amd import _lib
assert any('_fast.so' in str(w.message) for w in seen), seen
assert _lib.lib().ksa_version() > 0
assert _lib.fast.decode(1, 2, 3, None, None, None, None) is None and _lib.fast.block_index(*range(8)) is None
assert _lib.fast.prefill(*range(11)) is None and _lib.fast.pre_attention(*range(12)) is None
"""
    res = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr


def test_decode_qkv_argument_checks():
    """Shapes the fused decode call does not take are refused on the host."""
    from ksa_amd import _lib, decode
    L = _lib.lib()
    assert decode.decode_qkv_supported(32, 8, 128) and not decode.decode_qkv_supported(32, 8, 256)
    assert not decode.decode_qkv_supported(33, 1, 64)
    st = (ctypes.c_int64 * 3)(8, 8, 8)
    base = dict(qkv=16, ks=2, qw=16, kw=16, cos=16, sin=16, cbs=0, eps=1e-6, kc=16, vc=16, out=16, row=None, row0=3,
                start=None, end=None, s0=0, e0=10, b=1, hq=4, hkv=2, d=64, dt=0, kst=st, vst=st, ost=st, scale=0.1, ns=1,
                ws=None, wb=0, stream=None)
    call = lambda **kw: L.ksa_decode_qkv_fwd(*{**base, **kw}.values())
    assert call(qkv=None) != 0 and call(d=256) != 0 and call(row0=10) != 0 and call(row0=-1) != 0 and call(e0=0) != 0
    assert call(hq=5) != 0 and call(ns=2) != 0 and call(out=None) != 0 and call(kc=8) != 0 and call(b=129) != 0


def _kernel_metadata(path):
    """name -> metadata of every kernel in the code objects that a library carries."""
    import msgpack
    import struct
    blob, magic, kernels = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", {}
    at = blob.find(magic)
    while at >= 0:
        pos = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", blob, at + len(magic))[0]):
            off, size, n = struct.unpack_from("<QQQ", blob, pos)
            target, pos = blob[pos + 24: pos + 24 + n], pos + 24 + n
            elf = blob[at + off: at + off + size]
            note = elf.find(b"AMDGPU\0\0")        # name of the note: name size, description size, type, name, description
            if b"amdgcn" in target and note >= 12:
                desc = elf[note + 8: note + 8 + struct.unpack_from("<I", elf, note - 8)[0]]
                kernels.update({k[".name"]: k for k in msgpack.unpackb(desc)["amdhsa.kernels"]})
        at = blob.find(magic, at + 1)
    return kernels


def test_no_kernel_keeps_arrays_in_scratch_memory():
    """Arrays and what lambdas share stay in registers: a function that the compiler does not inline takes them to
    scratch memory (six times the time of a prefill at head_dim 256)."""
    from ksa_amd import _lib
    pytest.importorskip("msgpack")
    kernels = _kernel_metadata(_lib.LIB_PATH)
    assert any("ksa_prefill_kernel" in n and "Li256ELi0E" in n for n in kernels)   # (head_dim 256, general addressing)
    # (a few spilled registers are no array)
    assert {n: k[".private_segment_fixed_size"] for n, k in kernels.items() if k[".private_segment_fixed_size"] > 32} == {}


@pytest.mark.parametrize("b,hq,hkv,q", [(64, 8, 1, 9), (20, 32, 4, 9), (64, 8, 2, 9), (8, 32, 4, 9), (3, 32, 8, 9), (40, 64, 8, 9), (4, 32, 2, 9)])
@pytest.mark.parametrize("D", [64, 128])
def test_decode_splits_of_column_blocks(b, hq, hkv, q, D):
    """Several blocks of columns per slice: never past two workgroups per CU by more than the alignment of the blocks asks
    for, splits of at least a round, and the blocks of a slice on one XCD wherever the count is large enough."""
    import math
    from ksa_amd import _lib
    blocks = -(-q * (hq // hkv) // 32)
    a, slices = 8 // math.gcd(8, hkv), b * hkv
    assert blocks > 1
    for rows in (1, 300, 513, 900, 1500, 4096, 20000, 131072, 2**31 - 1):
        n = _lib.lib().ksa_decode_splits(b, hq, hkv, q, D, rows)
        assert 1 <= n <= 64 and (n == 1 or (n - 1) * 128 < rows) and (n == 1 or (n - 1) * slices < 512)
        if rows >= 4096 and a * slices <= 512:
            assert n % a == 0 or n < a


def _cus_of_the_rules(L):
    if L.ksa_device_cu_count() not in (0, 256):
        pytest.skip("the figures are those of 256 CUs")


@pytest.mark.parametrize("b,Hq,Hkv,Q,D,rows,n", [
    (1, 32, 8, 1, 128, 150, 1), (1, 32, 8, 1, 128, 737, 12), (1, 32, 8, 1, 128, 1500, 24),          # slices of one tile
    (1, 32, 8, 1, 128, 2000, 0), (8, 32, 8, 1, 128, 500, 0), (3, 32, 8, 1, 128, 737, 0),            # of two: four waves of 32 rows
    (1, 32, 8, 1, 64, 2000, 16), (3, 32, 8, 1, 64, 1100, 6), (1, 32, 8, 1, 128, 4100, 22),          # (not at head_dim 64)
    (8, 32, 8, 1, 128, 737, 4), (8, 32, 8, 1, 128, 1500, 4), (8, 32, 8, 1, 128, 4352, 4),
    (1, 32, 8, 1, 128, 9000, 29), (1, 32, 8, 1, 128, 131072, 32), (32, 32, 8, 1, 128, 500, 1),
    (12, 32, 8, 1, 128, 4100, 2),                                                                   # one round, not two
    (33, 32, 8, 1, 128, 600, 0), (33, 32, 8, 1, 128, 601, 1), (33, 32, 8, 1, 128, 1200, 1), (33, 32, 8, 1, 128, 1201, 0),
    (33, 32, 8, 1, 128, 2500, 0), (33, 32, 8, 1, 128, 2501, 2), (48, 32, 8, 1, 128, 1100, 1), (49, 32, 8, 1, 128, 1100, 0),
    (64, 32, 8, 1, 128, 2500, 0), (64, 32, 8, 1, 128, 2501, 1), (64, 32, 8, 1, 128, 8704, 1),       # more slices than CUs
    (4, 32, 8, 1, 64, 24000, 8), (31, 8, 1, 1, 64, 131072, 8),
    (1, 32, 8, 4, 128, 737, 12), (1, 32, 8, 5, 128, 737, 0), (1, 32, 2, 1, 128, 737, 12), (1, 34, 2, 1, 128, 737, 0),   # columns
    (1, 32, 8, 1, 256, 737, 0), (1, 32, 8, 1, 96, 737, 0), (1, 33, 8, 1, 128, 737, 0), (1, 32, 8, 1, 128, 0, 0),
])
def test_decode_wide_splits_on_both_sides_of_each_line(b, Hq, Hkv, Q, D, rows, n):
    """Which decode calls take workgroups of eight waves, and with how many splits (0: the four-wave kernel is faster)."""
    from ksa_amd import _lib
    _cus_of_the_rules(_lib.lib())
    assert _lib.lib().ksa_decode_wide_splits(b, Hq, Hkv, Q, D, rows) == n


@pytest.mark.parametrize("b,Hq,Hkv,D,rows,n", [
    (1, 32, 8, 128, 737, 12), (1, 32, 8, 128, 2000, 0), (1, 32, 8, 64, 2000, 16), (8, 32, 8, 128, 4352, 4), (32, 32, 8, 128, 131072, 1),
    (33, 32, 8, 128, 737, 0), (1, 34, 2, 128, 737, 0), (1, 32, 8, 256, 737, 0), (1, 33, 8, 128, 737, 0), (1, 32, 8, 128, 0, 0),
    (12, 32, 8, 128, 5000, 2), (12, 32, 8, 128, 5001, 0), (13, 32, 8, 128, 5001, 2), (25, 32, 8, 128, 5001, 0), (26, 32, 8, 128, 5001, 1),
    (21, 32, 8, 64, 10000, 1), (21, 32, 8, 64, 10001, 0), (22, 32, 8, 64, 10001, 1), (12, 32, 8, 64, 10001, 2),
])
def test_decode_qkv_wide_splits_on_both_sides_of_each_line(b, Hq, Hkv, D, rows, n):
    """The same for a step with the pre-attention in it: one round of workgroups, and none that leaves CUs idle over long ranges."""
    from ksa_amd import _lib
    _cus_of_the_rules(_lib.lib())
    assert _lib.lib().ksa_decode_qkv_wide_splits(b, Hq, Hkv, D, rows) == n


@pytest.mark.parametrize("b,Hq,Hkv,D,N,rows,n,pays", [
    (1, 32, 8, 128, 2560, 737, 12, 1), (1, 32, 8, 128, 2560, 4097, 22, 1), (8, 32, 8, 128, 2560, 737, 2, 1),
    (8, 32, 8, 128, 2560, 4352, 4, 1), (16, 32, 8, 128, 2560, 4097, 2, 1),
    (17, 32, 8, 128, 2560, 737, 0, 0), (1, 136, 8, 64, 2560, 737, 0, 0), (1, 128, 8, 64, 2560, 737, 12, 1),             # batch, columns
    (1, 32, 8, 256, 2560, 737, 0, 0), (1, 32, 8, 128, 2568, 737, 0, 0), (1, 32, 8, 128, 2560, 0, 0, 0),
    (1, 64, 8, 128, 4096, 737, 12, 1), (1, 64, 8, 128, 4112, 737, 12, 0), (1, 64, 8, 128, 5120, 400, 7, 0),             # product > CUs
    (1, 16, 2, 128, 2048, 1100, 18, 1), (1, 16, 2, 128, 2048, 1101, 18, 0), (1, 32, 2, 128, 2048, 2048, 32, 1),         # few kv heads
    (1, 32, 2, 128, 2048, 2049, 33, 0), (1, 32, 4, 128, 2048, 2049, 33, 1),
    (12, 32, 8, 128, 2560, 5000, 2, 1), (12, 32, 8, 128, 2560, 5001, 0, 0), (13, 32, 8, 128, 2560, 5001, 2, 1),         # idle CUs
    (12, 32, 8, 64, 2048, 5001, 2, 1), (5, 32, 8, 128, 2560, 131072, 6, 1),
    (16, 16, 8, 128, 2048, 300, 1, 0), (15, 16, 8, 128, 2048, 300, 1, 1), (16, 32, 8, 128, 2048, 300, 1, 1),            # half the CUs
    (8, 32, 32, 128, 4096, 300, 1, 0), (4, 32, 32, 128, 4096, 300, 1, 1),
    (1, 32, 8, 64, 2048, 599, 10, 0), (1, 32, 8, 64, 2048, 600, 10, 1), (1, 32, 8, 64, 2048, 8192, 26, 1),              # head_dim 64
    (1, 32, 8, 64, 2048, 8193, 26, 0), (12, 32, 8, 64, 2048, 1000, 2, 1), (13, 32, 8, 64, 2048, 1000, 2, 0),
])
def test_wide_attention_and_o_projection_on_both_sides_of_each_line(b, Hq, Hkv, D, N, rows, n, pays):
    """The split count of the one launch in workgroups of eight waves (0: not taken), and whether it is faster than the two."""
    from ksa_amd import _lib
    L = _lib.lib()
    _cus_of_the_rules(L)
    assert L.ksa_decode_qkv_o_wide_splits(b, Hq, Hkv, D, N, rows) == n
    assert L.ksa_decode_qkv_o_wide_pays(b, Hq, Hkv, D, N, rows) == pays


def test_attention_and_o_projection_in_one_launch_where_it_is_faster():
    """The rule for the one launch at 256 CUs, both sides of each of its lines, and the split counts that it rests on (the
    counts of the attention alone beside them): what measured slower goes to the separate launches."""
    import ksa_amd._lib as _lib
    L = _lib.lib()
    if L.ksa_device_cu_count() not in (0, 256):
        pytest.skip("the figures are those of 256 CUs")
    for (b, Hq, Hkv, D, N, rows), alone, n, pays in [
        ((1, 32, 8, 128, 2560, 400), 4, 4, 1),
        ((1, 32, 8, 128, 2560, 4096), 32, 32, 1),
        ((1, 32, 8, 128, 2560, 16384), 64, 20, 1),
        ((1, 32, 8, 128, 2560, 131072), 64, 64, 1),
        ((8, 32, 8, 128, 2560, 131072), 8, 3, 1),
        ((16, 32, 8, 128, 4096, 4096), 4, 2, 1),
        ((1, 32, 1, 128, 2560, 16384), 64, 64, 0),    # too many sums
        ((1, 32, 1, 128, 2560, 32768), 64, 64, 1),    # ... for a range below this
        ((8, 32, 2, 128, 2560, 32768), 32, 8, 0),     # few kv heads: too few splits
        ((16, 32, 1, 128, 2560, 131072), 32, 4, 0),
        ((2, 16, 4, 128, 2048, 1400), 11, 11, 0),     # 22 sums at 16 heads
        ((1, 16, 4, 128, 2048, 2500), 20, 20, 1),
        ((1, 16, 8, 128, 2048, 16384), 64, 20, 0),
        ((1, 32, 8, 64, 2048, 2500), 20, 20, 1),
        ((1, 32, 8, 64, 2048, 4096), 32, 32, 0),
        ((1, 64, 8, 128, 5120, 400), 4, 4, 0),        # 640 workgroups of the product
        ((1, 32, 32, 128, 4096, 400), 4, 4, 0),
        ((8, 24, 8, 128, 3072, 1300), 8, 3, 0),
        ((8, 24, 8, 128, 3072, 1400), 8, 3, 1),       # 64 workgroups to a split
        ((4, 24, 8, 128, 3072, 4096), 16, 5, 0),
        ((8, 48, 8, 128, 4096, 4096), 8, 3, 1),
        ((8, 16, 8, 128, 2048, 4096), 8, 3, 0),
        ((12, 16, 8, 128, 2048, 4096), 5, 2, 1),
        ((8, 64, 8, 128, 5120, 4096), 8, 3, 0),
        ((16, 32, 4, 128, 2560, 4096), 8, 3, 0),      # 48 sums
        ((17, 32, 8, 128, 2560, 400), 1, 1, 0),
        ((1, 32, 8, 128, 2560, 0), 1, 1, 0),
    ]:
        got = (L.ksa_decode_splits(b, Hq, Hkv, 1, D, rows), L.ksa_decode_qkv_o_splits(b, Hq, Hkv, D, rows),
               L.ksa_decode_qkv_o_pays(b, Hq, Hkv, D, N, rows))
        assert got == (alone, n, pays), (b, Hq, Hkv, D, N, rows, got)


def test_norm_and_product_in_one_launch_where_it_is_faster():
    """The rule for the residual add + norm in front of a product at 256 CUs, both sides of each of its lines."""
    import ksa_amd._lib as _lib
    L = _lib.lib()
    if L.ksa_device_cu_count() not in (0, 256):
        pytest.skip("the figures are those of 256 CUs")
    for (M, N, H, ksplit), pays in [
        ((1, 6144, 2560, 19), 1), ((8, 6144, 2560, 19), 1), ((9, 6144, 2560, 19), 0),
        ((6, 6144, 2560, 28), 1), ((4, 6144, 2560, 29), 0), ((7, 6144, 2560, 20), 1), ((7, 6144, 2560, 21), 0),
        ((8, 6144, 4096, 28), 1), ((8, 6144, 4096, 29), 0),
        ((4, 2560, 2048, 4), 1), ((5, 2560, 2048, 8), 0), ((5, 2560, 2048, 9), 1),
        ((1, 4096, 1024, 16), 0), ((1, 4096, 1024, 17), 1), ((8, 4096, 1024, 17), 1),
        ((1, 16384, 2560, 19), 0), ((1, 12288, 4096, 19), 1), ((1, 16384, 4096, 19), 0), ((1, 16384, 1024, 20), 0), ((1, 12288, 2048, 19), 1), ((1, 12416, 2048, 19), 0),
        ((4, 4352, 3840, 9), 1), ((5, 4352, 3840, 16), 0), ((5, 4352, 3840, 17), 1),
        ((1, 6144, 2561, 19), 0), ((1, 6144, 4128, 19), 0),
    ]:
        assert L.ksa_add_rmsnorm_gemm_rows_pays(M, N, H, ksplit) == pays, (M, N, H, ksplit)
