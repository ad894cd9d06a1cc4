"""End-to-end module (`ksa_amd.model`): the caller of both hot paths.

What pins what
* `expand_with_summary_tokens` / `boundary_position_ids`: closed forms of the reference's
  position-id rules (examples/pretrain/hf_template/modeling_qwen3sa.py:1134-1175, :1497-1531)
  evaluated by brute-force loops here, and hand-computed values for C=8, S=2.
* prefill-vs-decode consistency (CPU, fp32 operators from oracle/): the logits for token n
  obtained by prefill(n tokens) must equal those of prefill(m tokens) followed by n - m decode
  steps.  The prefill mask rule is pinned to the reference in tests/test_oracle.py; this test
  carries that pin over to the decode side of the module (cache rows, ring order, hidden
  summaries, boundary step, position ids).  With S = 1 it holds across chunk boundaries; with
  S > 1 the reference's boundary step lets every summary query see all S summary keys while
  its prefill mask is causal among them, so the check then stays inside one chunk.
* GPU: the module on the HIP kernels (bf16) against the same module on the CPU operators
  (fp32, same bf16-rounded weights), teacher-forced with the CPU run's tokens: logits within a
  stated tolerance at every step, over prefill, in-chunk steps and boundary steps.
The reference's cache knows two kinds of layers only: those with the smallest window, and
"large window" layers (any larger window) that keep every text row and no summaries
(:114-115); configurations here therefore use one window size plus unbounded layers.
The reference's model itself is not importable here (it needs the transformers version it was
written for and the CUDA summary_attn wheel), so the module as a whole is pinned by the above
only: "parity unpinned" against a run of the reference's own model.
"""
import numpy as np
import pytest
import torch

from ksa_amd.model import (KsaQwen3Config, KsaQwen3ForCausalLM, boundary_position_ids, convert_weights,
                           expand_with_summary_tokens, init_weights)


def tiny_config(**kw):
    base = dict(hidden_size=64, num_hidden_layers=4, num_attention_heads=4, num_key_value_heads=2,
                head_dim=64, intermediate_size=96, vocab_size=200, summary_token_begin=200,
                summary_chunk_size=8, summary_token_num=1, rope_theta=10000.0,
                summary_sliding_chunk_num=[2, 2, 1 << 20, 2])
    base.update(kw)
    return KsaQwen3Config(**base)


def cpu_model(cfg, seed=0):
    from oracle.model_ops import OracleOps
    w = init_weights(cfg, "cpu", torch.bfloat16, seed)
    return KsaQwen3ForCausalLM(cfg, convert_weights(w, "cpu", torch.float32), OracleOps()), w


@pytest.mark.parametrize("kind", ["last_chunk_slice_right", "last_chunk_slice_left", "zeros"])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 29])
def test_expand_positions_brute_force(kind, n):
    C, S, begin = 8, 2, 500
    cfg = tiny_config(summary_token_num=S, summary_token_begin=begin, summary_token_position_ids_type=kind)
    ids_in = torch.arange(100, 100 + n)[None].repeat(2, 1)
    ids, pos, is_sum = expand_with_summary_tokens(ids_in, cfg)
    exp_ids, exp_pos, exp_sum = [], [], []
    for t in range(n):
        exp_ids.append(100 + t); exp_pos.append(t); exp_sum.append(False)
        if (t + 1) % C == 0:
            i = t // C
            for j in range(S):
                exp_ids.append(begin + j); exp_sum.append(True)
                if kind == "zeros":
                    exp_pos.append(0)
                else:
                    k = j + 1 if kind.endswith("right") else j
                    exp_pos.append(max(i * C + (k * C) // S - 1, i * C))
    assert ids.tolist() == [exp_ids, exp_ids]
    assert pos[0].tolist() == exp_pos
    assert is_sum.tolist() == exp_sum


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["last_chunk_slice_right", "last_chunk_slice_left", "zeros"])
@pytest.mark.parametrize("text,C,S,D", [("origin", 128, 8, 128), ("inner_chunk", 100, 7, 64), ("origin", 5, 3, 16)])
def test_gpu_expand_prompt_equals_host_form(text, C, S, D, kind, dtype):
    from ksa_amd.model import HipOps
    cfg = tiny_config(head_dim=D, summary_chunk_size=C, summary_token_num=S, summary_token_position_ids_type=kind,
                      summary_chunk_position_ids_type=text)
    inv = (1.0 / (1e6 ** (torch.arange(0, D, 2).float() / D))).cuda()
    for b, n in ((1, 1), (9, C - 1), (2, C), (2, 7 * C + 3), (1, 60 * C)):
        ids = torch.randint(0, 200, (b, 2 * n), device="cuda")[:, ::2]   # (a view with a stride)
        got_ids, cos, sin, mask = HipOps().expand_prompt(ids, cfg, inv, dtype)
        want_ids, pos, want_mask = expand_with_summary_tokens(ids, cfg)
        assert torch.equal(got_ids, want_ids) and torch.equal(mask, want_mask)
        angle = pos[0].float()[:, None] * torch.cat((inv, inv))[None]
        for got, want in ((cos, angle.cos()), (sin, angle.sin())):   # one rounding of the same fp32 function
            assert got.shape == (1, want.shape[0], D)
            torch.testing.assert_close(got[0], want.to(dtype), rtol=2.0 ** (-7 if dtype == torch.bfloat16 else -10), atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["last_chunk_slice_right", "last_chunk_slice_left", "zeros"])
@pytest.mark.parametrize("text,C,S,D", [("origin", 128, 8, 128), ("inner_chunk", 100, 7, 64), ("origin", 5, 3, 16)])
def test_gpu_step_rows_equal_host_form(text, C, S, D, kind, dtype):
    """Ids and rotary rows of a decode step at every kind of place, and stretches of the rotary table, bit for bit."""
    from ksa_amd.model import HipOps
    cfg = tiny_config(head_dim=D, summary_chunk_size=C, summary_token_num=S, summary_token_position_ids_type=kind,
                      summary_chunk_position_ids_type=text, num_hidden_layers=1, summary_sliding_chunk_num=[2])
    ops, model = HipOps(), KsaQwen3ForCausalLM(cfg, init_weights(cfg, "cuda", dtype, 0))
    inv = model.inv_freq_dev
    for b, index in ((1, 0), (3, C - 2), (2, C - 1), (1, C), (9, 7 * C - 1), (1, 20001 * C - 1), (1, 100003)):
        tok = torch.randint(0, 200, (b, 2), device="cuda")[:, 1:]
        boundary = index % C == C - 1
        ids, cos, sin = ops.expand_step(tok, index, boundary, cfg, inv, dtype)
        p = index if text == "origin" else index % C
        pos = boundary_position_ids(index, cfg, "cpu") if boundary else torch.tensor([[p]])
        want = model._rope_tables(pos)
        assert torch.equal(cos, want[0]) and torch.equal(sin, want[1]), index
        new = torch.arange(S)[None].expand(b, -1) + cfg.summary_token_begin
        assert torch.equal(ids.cpu(), torch.cat([tok.cpu(), new], 1) if boundary else tok.cpu()), index
    assert ops.expand_step(tok, C - 2, True, cfg, inv, dtype) is None and ops.expand_step(tok.int(), 3, False, cfg, inv, dtype) is None
    for first in (0, 1000, 130000):
        tab = ops.rope_rows(first, 33, cfg, inv, dtype)
        want = model._rope_tables(torch.arange(first, first + 33)[None])
        assert torch.equal(tab[:, 0], want[0][0]) and torch.equal(tab[:, 1], want[1][0])
    buf = torch.full((35, 2, D), 7.0, dtype=dtype, device="cuda")
    assert ops.rope_rows(5, 33, cfg, inv, dtype, out=buf[1:34]).data_ptr() == buf[1].data_ptr()
    assert torch.equal(buf[1:34], ops.rope_rows(5, 33, cfg, inv, dtype)) and (buf[0] == 7).all() and (buf[34] == 7).all()
    L = ops._lib.lib()
    call = lambda **kw: L.ksa_expand_slots(*{**dict(ids=tok.data_ptr(), rs=1, b=1, slot0=0, n=1, C=C, S=S, beg=0, inner=0, kind=0,
                                                    inv=inv.data_ptr(), D=D, out=None, cos=buf.data_ptr(), sin=buf.data_ptr(), rr=D,
                                                    dt=0, st=None), **kw}.values())
    for bad in (dict(b=0), dict(slot0=-1), dict(n=0), dict(slot0=2 ** 31 - 1), dict(C=0), dict(S=0), dict(C=2 ** 31 - 1), dict(D=24),
                dict(inv=None), dict(cos=None), dict(sin=buf.data_ptr() + 2), dict(rr=D + 4), dict(ids=None, out=tok.data_ptr()), dict(kind=3), dict(dt=2)):
        assert call(**bad) != 0, bad


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [False, True])
def test_gpu_steps_make_their_rows_without_torch(graph, monkeypatch):
    """No step of a generation - the first one, the first at a chunk's end, the first recorded one - leaves its positions or rotary rows to
    torch, whose kernels would have to be loaded in the middle of it; its logits are those of the torch form bit for bit."""
    import ksa_amd.model as M
    cfg = tiny_config(hidden_size=128, num_hidden_layers=2, summary_token_num=2, summary_sliding_chunk_num=[2, 1 << 20])
    w = init_weights(cfg, "cuda", torch.bfloat16, 1)

    class Plain(M.HipOps):
        expand_step = rope_rows = lambda self, *a, **k: None
    ids = torch.randint(0, 200, (2, 13), generator=torch.Generator().manual_seed(0)).cuda()
    runs = []
    for ops in (Plain(), M.HipOps()):
        model = KsaQwen3ForCausalLM(cfg, w, ops)
        model.BOUNDARY_GRAPH_AFTER = 2
        if runs:
            def refuse(*a, **k):
                raise AssertionError("left to torch")
            monkeypatch.setattr(model, "_rope_tables", refuse)
            monkeypatch.setattr(M, "boundary_position_ids", refuse)
        runs.append(model.generate(ids, 40, return_logits=True, use_graph=graph))
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][1], runs[1][1])


@pytest.mark.gpu
def test_gpu_prefill_of_short_prompts_keeps_its_results():
    """The head of a prefill in one launch, closed-form cache rows and the attention without a mask change no bit of a prompt up to
    `GRID_ROWS`: logits and cache rows are those of the torch head, the mask and the grid of the block index."""
    from ksa_amd import prefill
    from ksa_amd.model import HipOps

    class Plain(HipOps):
        expand_prompt = lambda self, *a: None

        def summary_attn_func(self, *args, **kwargs):
            return prefill.summary_attn_func(*args, chunk_tiles=False, **kwargs)
    cfg = tiny_config(hidden_size=256, num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=2, head_dim=128,
                      intermediate_size=512, vocab_size=4000, summary_token_begin=4000, summary_chunk_size=128, summary_token_num=8,
                      summary_sliding_chunk_num=[4, 1 << 20])
    w = init_weights(cfg, "cuda", torch.bfloat16, 3)
    model, plain = KsaQwen3ForCausalLM(cfg, w), KsaQwen3ForCausalLM(cfg, w, Plain())
    last = 4608 // 136 * 128 + 4608 % 136     # as many rows as the grid keeps
    for b, n in ((1, 1), (2, 127), (1, 128), (3, 300), (1, 1000), (8, 2049), (1, 4096), (1, last)):
        ids = torch.randint(0, cfg.vocab_size, (b, n), generator=torch.Generator().manual_seed(n)).cuda()
        (got, cache), (want, ref) = model.prefill(ids), plain.prefill(ids)
        assert torch.equal(got, want), (b, n)
        for layer in range(2):
            for x, y in zip(cache.get_attention_kv(layer), ref.get_attention_kv(layer)):
                assert torch.equal(x, y), (b, n, layer)


def test_expand_known_values():
    cfg = tiny_config(summary_token_num=2)
    ids, pos, is_sum = expand_with_summary_tokens(torch.arange(17)[None], cfg)
    # chunk 0: text 0..7, summaries at 3 and 7; chunk 1: text 8..15, summaries at 11 and 15; tail 16
    assert pos[0].tolist() == list(range(8)) + [3, 7] + list(range(8, 16)) + [11, 15] + [16]
    assert ids[0, 8:10].tolist() == [200, 201] and ids[0, -1].item() == 16
    # the boundary step that completes chunk 1 (token index 15) places its summaries like prefill does
    assert boundary_position_ids(15, cfg, "cpu")[0].tolist() == [15, 11, 15]


def _decode_logits(model, ids, m):
    """prefill the first m tokens, then feed the rest one by one; logits after every token >= m."""
    logits, cache = model.prefill(ids[:, :m])
    got = [logits]
    for t in range(m, ids.shape[1]):
        got.append(model.decode_step(ids[:, t:t + 1], cache))
    return torch.cat(got, dim=1)


@pytest.mark.parametrize("m,n", [(8, 30), (13, 27), (3, 20), (1, 18)])
@pytest.mark.parametrize("indep,mix", [(False, 1.0), (True, 1.0), (True, 0.0), (True, 0.35)])
def test_decode_matches_prefill_across_boundaries_S1(m, n, indep, mix):
    cfg = tiny_config(summary_independent_parameters=indep, mix_coeff=mix)
    model, _ = cpu_model(cfg, seed=1)
    ids = torch.randint(0, cfg.vocab_size, (2, n), generator=torch.Generator().manual_seed(m * 100 + n))
    dec = _decode_logits(model, ids, m)
    for j, t in enumerate(range(m, n + 1)):
        ref, _ = model.prefill(ids[:, :t])
        assert torch.allclose(dec[:, j], ref[:, 0], atol=2e-5, rtol=1e-4), (t, (dec[:, j] - ref[:, 0]).abs().max())


@pytest.mark.parametrize("m", [16, 19])
def test_decode_matches_prefill_inside_a_chunk_S2(m):
    cfg = tiny_config(summary_token_num=2, summary_token_begin=200)
    model, _ = cpu_model(cfg, seed=2)
    n = 23   # chunk 2 completes at token 24: stays inside the chunk
    ids = torch.randint(0, cfg.vocab_size, (1, n), generator=torch.Generator().manual_seed(m))
    dec = _decode_logits(model, ids, m)
    for j, t in enumerate(range(m, n + 1)):
        ref, _ = model.prefill(ids[:, :t])
        assert torch.allclose(dec[:, j], ref[:, 0], atol=2e-5, rtol=1e-4), t


def test_prefill_mlp_sliced_over_the_batch():
    """A prefill whose MLP activation exceeds `MLP_SLICE_BYTES` runs the MLP over slices of the batch: same
    logits as in one piece, and the same logits from the decode steps that follow (host operators; rows are
    independent, so only the library's blocking of the products may differ)."""
    cfg = tiny_config()
    model, _ = cpu_model(cfg, 2)
    ids = torch.randint(0, cfg.vocab_size, (5, 21), generator=torch.Generator().manual_seed(2))
    log0, c0 = model.prefill(ids)
    model.MLP_SLICE_BYTES = 2 * 21 * 2 * cfg.intermediate_size * 4   # two sequences per slice (fp32 host weights)
    seen = []
    inner = model.ops.silu_mul
    model.ops.silu_mul = lambda g, u=None: (seen.append(g.shape[0]), inner(g, u))[1]
    log1, c1 = model.prefill(ids)
    assert torch.allclose(log0, log1, atol=1e-5, rtol=1e-5)
    assert seen and max(seen) <= 2 and sum(seen) == 5 * cfg.num_hidden_layers
    model.ops.silu_mul = inner
    tok = log0.argmax(-1)
    for _ in range(4):   # the caches hold the same rows: a few decode steps across a chunk boundary agree as well
        d0, d1 = model.decode_step(tok, c0), model.decode_step(tok, c1)
        assert torch.allclose(d0, d1, atol=1e-5, rtol=1e-5)
        tok = d0.argmax(-1)


def test_generate_shapes_and_forcing():
    cfg = tiny_config()
    model, _ = cpu_model(cfg)
    ids = torch.randint(0, cfg.vocab_size, (2, 11), generator=torch.Generator().manual_seed(5))
    out, logits = model.generate(ids, 12, return_logits=True)
    assert out.shape == (2, 23) and logits.shape == (2, 12, cfg.vocab_size)
    assert (out[:, :11] == ids).all() and (out[:, 11:] == logits.argmax(-1)).all()
    out2, logits2 = model.generate(ids, 12, forced=out[:, 11:], return_logits=True)
    assert torch.equal(out, out2) and torch.allclose(logits, logits2)


def test_bad_config():
    with pytest.raises(ValueError):
        KsaQwen3Config(num_hidden_layers=3, summary_sliding_chunk_num=[1, 2]).sliding_chunk_nums()
    with pytest.raises(ValueError):
        cfg = tiny_config(summary_independent_parameters=True, mix_coeff=1.5)
        cpu_model(cfg)


@pytest.mark.parametrize("mix", [0.0, 0.35, 1.0])
def test_mix_coeff_blend_equals_reference_order(mix):
    """The reference blends the summary rows' normalised q and k (and v) from the two projections
    BEFORE the rotary embedding (modeling_qwen3sa.py:776-788, then :792-793); the module blends
    after its fused norm + rotary step.  Restated here in the reference's order with plain torch
    ops and compared with what the module hands to the attention call."""
    cfg = tiny_config(summary_independent_parameters=True, mix_coeff=mix, summary_token_num=2,
                      num_hidden_layers=1, summary_sliding_chunk_num=[2])
    model, _ = cpu_model(cfg, seed=3)
    lw = model.w["layers"][0]
    ids_in = torch.randint(0, cfg.vocab_size, (2, 21), generator=torch.Generator().manual_seed(1))
    ids, pos, is_sum = expand_with_summary_tokens(ids_in, cfg)
    seen = {}

    class SpyOps(type(model.ops)):
        @staticmethod
        def summary_attn_func(q, k, v, *a, **kw):
            seen["qkv"] = (q.clone(), k.clone(), v.clone())
            return type(model.ops).__mro__[1].summary_attn_func(q, k, v, *a, **kw)
    model.ops = SpyOps()
    model.prefill(ids_in)
    q, k, v = seen["qkv"]

    D, Hq, Hkv, eps = cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.rms_norm_eps
    x = model.w["embed_tokens"][ids]
    h = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * lw["input_layernorm"]

    def proj(w):
        y = h @ w.T
        b, L, _ = y.shape
        qq = y[..., :Hq * D].view(b, L, Hq, D)
        kk = y[..., Hq * D:(Hq + Hkv) * D].view(b, L, Hkv, D)
        vv = y[..., (Hq + Hkv) * D:].view(b, L, Hkv, D)
        norm = lambda t, wn: t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + eps) * wn
        return norm(qq, lw["q_norm"]), norm(kk, lw["k_norm"]), vv
    base, summ = proj(lw["qkv_proj"]), proj(lw["qkv_proj_summary"])
    sel = is_sum[None, :, None, None]
    mixed = [torch.where(sel, mix * s_ + (1 - mix) * b_, b_) if mix != 0 else b_ for b_, s_ in zip(base, summ)]
    cos, sin = model._rope_tables(pos)

    def rope(t):
        c, s_ = cos[:, :, None, :], sin[:, :, None, :]
        rot = torch.cat((-t[..., D // 2:], t[..., :D // 2]), dim=-1)
        return t * c + rot * s_
    want = (rope(mixed[0]), rope(mixed[1]), mixed[2])
    for got, exp, name in zip((q, k, v), want, "qkv"):
        assert torch.allclose(got, exp, atol=2e-5, rtol=1e-4), (name, (got - exp).abs().max())


# ------------------------------------------------------------------------------------ GPU
def _check_logits_and_tokens(log_g, log_c, tol_rel, what, rms_rel=None):
    """GPU logits against the CPU run's, teacher-forced with the CPU run's tokens: every logit
    within tol_rel of the logit scale (and their root-mean-square difference within rms_rel of
    it), and the greedy token identical wherever the CPU run's margin between its best and
    second-best logit exceeds twice that tolerance (where the margin is smaller the two runs
    may legitimately pick different tokens)."""
    scale = log_c.abs().max().item()
    tol = tol_rel * scale
    err = (log_g - log_c).abs().amax(dim=(0, 2))        # per step
    assert err.max().item() <= tol, (what, err.tolist(), scale)
    if rms_rel is not None:
        rms = (log_g - log_c).pow(2).mean().sqrt().item()
        print(f"{what}: rms logit error {rms / scale:.3e} of the logit scale")
        assert rms <= rms_rel * scale, (what, rms, scale)
    top2 = log_c.topk(2, dim=-1).values
    decided = (top2[..., 0] - top2[..., 1]) > 2 * tol
    same = log_g.argmax(-1) == log_c.argmax(-1)
    assert decided.any(), f"{what}: no step has a decided margin, the token check would be empty"
    assert bool(same[decided].all()), (what, "greedy ids differ at decided steps",
                                       torch.nonzero(decided & ~same).tolist())
    return err.max().item() / scale, same.float().mean().item(), decided.float().mean().item()


def _gpu_vs_cpu(cfg, batch, n_prompt, n_new, seed, tol_rel):
    from ksa_amd.model import HipOps
    cpu, w = cpu_model(cfg, seed)
    gpu = KsaQwen3ForCausalLM(cfg, convert_weights(w, "cuda", torch.bfloat16), HipOps())
    ids = torch.randint(0, cfg.vocab_size, (batch, n_prompt), generator=torch.Generator().manual_seed(seed))
    out_c, log_c = cpu.generate(ids, n_new, return_logits=True)
    out_g, log_g = gpu.generate(ids, n_new, forced=out_c[:, n_prompt:], return_logits=True)
    rel, agree, _ = _check_logits_and_tokens(log_g.cpu(), log_c, tol_rel, "eager")
    return rel, agree


@pytest.mark.gpu
@pytest.mark.parametrize("S,D,indep,mix", [(1, 64, False, 1.0), (2, 128, False, 1.0), (2, 64, True, 1.0),
                                          (2, 128, True, 0.35)])
def test_gpu_module_matches_cpu_module(S, D, indep, mix):
    """Prefill of 21 tokens (two complete chunks + a partial one), then 20 decode steps that
    cross two chunk boundaries; bf16 kernels vs fp32 host operators, teacher-forced.
    Tolerance: 1.5 % of the largest logit magnitude (measured 0.4-0.6 %) (bf16 activations through 4 layers)."""
    cfg = tiny_config(summary_token_num=S, head_dim=D, summary_independent_parameters=indep, mix_coeff=mix,
                      hidden_size=128, intermediate_size=256)
    rel, agree = _gpu_vs_cpu(cfg, batch=2, n_prompt=21, n_new=20, seed=3, tol_rel=1.5e-2)
    print(f"max logit error {rel:.3e} of the logit scale, arg-max agreement {agree:.2f}")


@pytest.mark.gpu
@pytest.mark.parametrize("batch,S", [(20, 2), (40, 1), (64, 1)])
def test_gpu_module_more_than_16_rows(batch, S):
    """A batch above 16: the steps inside a chunk (`batch` rows) and the chunk-boundary steps (batch x (1 + S)
    rows, up to 128) run their projections on the wide form of the few-rows GEMMs, with the K-split partial
    sums handed to the norms and the pre-attention step, and the MLP as two launches.  Same check and
    tolerance as `test_gpu_module_matches_cpu_module`; then the same steps replayed from HIP graphs against
    the eager ones."""
    from ksa_amd.model import HipOps
    cfg = tiny_config(summary_token_num=S, head_dim=64, hidden_size=128, intermediate_size=256)
    rel, agree = _gpu_vs_cpu(cfg, batch=batch, n_prompt=21, n_new=20, seed=5, tol_rel=1.5e-2)
    print(f"max logit error {rel:.3e} of the logit scale, arg-max agreement {agree:.2f}")
    _, w = cpu_model(cfg, 5)
    gpu = KsaQwen3ForCausalLM(cfg, convert_weights(w, "cuda", torch.bfloat16), HipOps())
    gpu.BOUNDARY_GRAPH_AFTER = 0
    ids = torch.randint(0, cfg.vocab_size, (batch, 21), generator=torch.Generator().manual_seed(6))
    out_e, log_e = gpu.generate(ids, 40, return_logits=True)
    out_g, log_g = gpu.generate(ids, 40, forced=out_e[:, 21:], return_logits=True, use_graph=True)
    scale = log_e.abs().max().item()
    assert (log_g - log_e).abs().max().item() <= 1e-2 * scale


@pytest.mark.gpu
def test_gpu_module_kernel_shape():
    """The real attention shape (C=128, S=8, 8/2 heads, D=128, windows 1 | unbounded | 1):
    prefill of 300 tokens, 120 decode steps (one boundary), batch 2."""
    cfg = tiny_config(summary_chunk_size=128, summary_token_num=8, head_dim=128, num_attention_heads=8,
                      num_key_value_heads=2, hidden_size=256, intermediate_size=512, num_hidden_layers=3,
                      summary_sliding_chunk_num=[1, 1 << 20, 1], vocab_size=1000, summary_token_begin=1000)
    rel, agree = _gpu_vs_cpu(cfg, batch=2, n_prompt=300, n_new=120, seed=4, tol_rel=1.5e-2)
    print(f"max logit error {rel:.3e} of the logit scale, arg-max agreement {agree:.2f}")


@pytest.mark.gpu
def test_gpu_module_config4_layer_shape():
    """Config 4's own layer shape - hidden 2560, 32 / 8 heads of 128, MLP 9728, vocabulary 151936,
    batch 8 - on one 3 : 1 group of layers (three Summary layers with a window of 4 chunks and one
    unbounded layer): a 300-token prompt (two complete chunks and a partial one), then 132 greedy
    steps that cross a chunk boundary, eagerly launched and replayed from the HIP graph, both
    against the same module on the fp32 host operators, teacher-forced with the host run's tokens.
    Asserts the logit tolerance and token-exact greedy ids at every step whose host-side margin
    decides the token; the share of decided steps is printed.  Tolerance: the largest of the
    160 million logit differences within 2.5 % of the logit scale (the extreme of that many
    bf16 rounding errors: measured 1.7 %, the same at the first step as at the last), their
    root mean square within 0.5 %."""
    from ksa_amd.model import HipOps
    from oracle.model_ops import OracleOps
    cfg = KsaQwen3Config(num_hidden_layers=4, summary_sliding_chunk_num=[4, 4, 4, 1 << 20])
    w = init_weights(cfg, "cuda", torch.bfloat16, 11)
    gpu = KsaQwen3ForCausalLM(cfg, w, HipOps())
    cpu = KsaQwen3ForCausalLM(cfg, convert_weights(w, "cpu", torch.float32), OracleOps())
    gpu.BOUNDARY_GRAPH_AFTER = 0     # the graph run replays its boundary step too
    batch, n_prompt, n_new = 8, 300, 132
    ids = torch.randint(0, cfg.vocab_size, (batch, n_prompt), generator=torch.Generator().manual_seed(12))
    out_c, log_c = cpu.generate(ids, n_new, return_logits=True)
    del cpu
    forced = out_c[:, n_prompt:]
    for what, graph in (("eager", False), ("graph", True)):
        _, log_g = gpu.generate(ids, n_new, forced=forced, return_logits=True, use_graph=graph)
        rel, agree, decided = _check_logits_and_tokens(log_g.cpu(), log_c, 2.5e-2, what, rms_rel=5e-3)
        print(f"{what}: max logit error {rel:.3e} of the logit scale, arg-max agreement {agree:.3f} over all "
              f"steps, {decided:.2f} of the steps decided by their margin")
        assert agree >= 0.9, (what, agree)
        del log_g


@pytest.mark.gpu
def test_gpu_graph_decode_equals_eager_decode():
    """The HIP-graph decode path against the eager one on the same inputs: 150 steps that cross a
    chunk boundary and one reallocation of the append-only buffers (forcing a second recording),
    every replay compared.  The two paths choose the decode kernel's split count differently
    (the graph path cannot look at the row range on the host), so the logits agree to rounding,
    not bit for bit: tolerance 1 % of the logit scale at every step."""
    from ksa_amd.model import HipOps
    cfg = tiny_config(summary_chunk_size=128, summary_token_num=8, head_dim=128, num_attention_heads=8,
                      num_key_value_heads=2, hidden_size=256, intermediate_size=512, num_hidden_layers=4,
                      summary_sliding_chunk_num=[1, 1 << 20, 1, 1 << 20], vocab_size=1000,
                      summary_token_begin=1000)
    w = init_weights(cfg, "cuda", torch.bfloat16, 7)
    model = KsaQwen3ForCausalLM(cfg, w, HipOps())
    model.BOUNDARY_GRAPH_AFTER = 0     # the boundary step is replayed from its own recording
    ids = torch.randint(0, cfg.vocab_size, (2, 200), generator=torch.Generator().manual_seed(9))
    n_new = 150
    out_e, log_e = model.generate(ids, n_new, return_logits=True)
    out_g, log_g = model.generate(ids, n_new, forced=out_e[:, 200:], return_logits=True, use_graph=True)
    torch.cuda.synchronize()
    err = (log_e - log_g).abs().amax(dim=(0, 2))
    scale = log_e.abs().max().item()
    print(f"graph vs eager: max logit difference {err.max().item() / scale:.3e} of the logit scale")
    assert err.max().item() <= 1e-2 * scale, (err / scale).tolist()


@pytest.mark.gpu
def test_gpu_graph_decode_survives_buffer_growth():
    """A small head-room makes the append-only text buffers grow during decoding, which moves
    them; the graph path must notice and record again."""
    from ksa_amd.model import HipOps
    cfg = tiny_config(summary_chunk_size=128, summary_token_num=8, head_dim=128, num_attention_heads=8,
                      num_key_value_heads=2, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                      summary_sliding_chunk_num=[1, 1 << 20], vocab_size=1000, summary_token_begin=1000)
    w = init_weights(cfg, "cuda", torch.bfloat16, 8)
    ops = HipOps()

    class SmallHeadroom(ops.cache_cls):
        _APPEND_HEADROOM = 16
    ops.cache_cls = SmallHeadroom
    model = KsaQwen3ForCausalLM(cfg, w, ops)
    ids = torch.randint(0, cfg.vocab_size, (1, 140), generator=torch.Generator().manual_seed(10))
    out_e, log_e = model.generate(ids, 60, return_logits=True)
    out_g, log_g = model.generate(ids, 60, forced=out_e[:, 140:], return_logits=True, use_graph=True)
    err = (log_e - log_g).abs().amax(dim=(0, 2))
    assert err.max().item() <= 1e-2 * log_e.abs().max().item(), err.tolist()


@pytest.mark.gpu
@pytest.mark.parametrize("S,indep,mix,after", [(1, False, 1.0, 0), (2, True, 0.35, 0), (2, False, 1.0, 6)])
def test_gpu_graph_boundary_steps_equal_eager(S, indep, mix, after):
    """Chunk-boundary steps replayed from their own recording against the eager path: chunks of 8
    tokens, 70 steps = 9 boundaries, a ring of two chunks (its write position wraps at every
    second boundary) next to a ring of one and an unbounded layer, and head-rooms so small that
    the summary region and the append-only buffers outgrow their buffers several times (each
    growth moves the buffers, so both recordings are made again).  `after` = how many boundary
    steps of a cache run eagerly before they are recorded (6: the switch happens in the middle of
    the run).  Tolerance as for the steps
    inside a chunk: 1 % of the logit scale at every step (the two paths choose the decode
    kernel's split count differently)."""
    from ksa_amd.model import HipOps
    cfg = tiny_config(summary_token_num=S, head_dim=128, summary_independent_parameters=indep, mix_coeff=mix,
                      hidden_size=128, intermediate_size=256, summary_sliding_chunk_num=[2, 1, 1 << 20, 2])
    w = init_weights(cfg, "cuda", torch.bfloat16, 5)
    ops = HipOps()

    class SmallHeadroom(ops.cache_cls):
        _APPEND_HEADROOM = 6
        _SUMMARY_INIT_CAP = 3
    ops.cache_cls = SmallHeadroom
    model = KsaQwen3ForCausalLM(cfg, w, ops)
    model.BOUNDARY_GRAPH_AFTER = after
    replays = []
    inner = model._replay
    model._replay = lambda st, which, body, cache: (replays.append(which), inner(st, which, body, cache))[1]
    ids = torch.randint(0, cfg.vocab_size, (2, 21), generator=torch.Generator().manual_seed(6))
    n_new = 71
    out_e, log_e = model.generate(ids, n_new, return_logits=True)
    assert not replays
    out_g, log_g = model.generate(ids, n_new, forced=out_e[:, 21:], return_logits=True, use_graph=True)
    torch.cuda.synchronize()
    n_b = sum(1 for t in range(21 + 1, 21 + n_new) if t % cfg.summary_chunk_size == 0)
    assert n_b == 9 and replays.count("boundary") == n_b - model.BOUNDARY_GRAPH_AFTER, replays
    assert replays.count("text") == n_new - 1 - n_b, replays
    err = (log_e - log_g).abs().amax(dim=(0, 2))
    scale = log_e.abs().max().item()
    print(f"graph vs eager over {n_b} boundaries: max logit difference {err.max().item() / scale:.3e} of the logit scale")
    assert err.max().item() <= 1e-2 * scale, (err / scale).tolist()


@pytest.mark.gpu
def test_gpu_module_fp16():
    """The module with fp16 weights and activations (every kernel of the step has an fp16 form):
    the real attention shape, a 300-token prompt, 120 steps across a chunk boundary, launched
    eagerly and replayed from the HIP graphs, against the fp32 host operators on the same
    weights, teacher-forced.  Tolerance 0.3 % of the logit scale (measured 0.07-0.08 %; fp16
    rounds eight times finer than bf16, whose bar is 1.5 %)."""
    from ksa_amd.model import HipOps
    from oracle.model_ops import OracleOps
    cfg = tiny_config(summary_chunk_size=128, summary_token_num=8, head_dim=128, num_attention_heads=8,
                      num_key_value_heads=2, hidden_size=256, intermediate_size=512, num_hidden_layers=3,
                      summary_sliding_chunk_num=[1, 1 << 20, 1], vocab_size=1000, summary_token_begin=1000)
    w = init_weights(cfg, "cuda", torch.float16, 21)
    gpu = KsaQwen3ForCausalLM(cfg, w, HipOps())
    gpu.BOUNDARY_GRAPH_AFTER = 0
    cpu = KsaQwen3ForCausalLM(cfg, convert_weights(w, "cpu", torch.float32), OracleOps())
    ids = torch.randint(0, cfg.vocab_size, (2, 300), generator=torch.Generator().manual_seed(22))
    out_c, log_c = cpu.generate(ids, 120, return_logits=True)
    for what, graph in (("eager", False), ("graph", True)):
        _, log_g = gpu.generate(ids, 120, forced=out_c[:, 300:], return_logits=True, use_graph=graph)
        assert log_g.dtype == torch.float32 and gpu.dtype == torch.float16
        rel, agree, _ = _check_logits_and_tokens(log_g.cpu(), log_c, 3e-3, what)
        print(f"fp16 {what}: max logit error {rel:.3e} of the logit scale, arg-max agreement {agree:.2f}")


def _mlp_rows_config():
    """A small decoder whose MLP shape the one-launch MLP kernel takes (hidden size a multiple of 128)."""
    return tiny_config(summary_chunk_size=128, summary_token_num=8, head_dim=128, num_attention_heads=8,
                       num_key_value_heads=2, hidden_size=256, intermediate_size=512, num_hidden_layers=3,
                       summary_sliding_chunk_num=[1, 1 << 20, 1], vocab_size=1000, summary_token_begin=1000)


def test_one_launch_forms_count_on_the_words_of_their_own_decoder(monkeypatch):
    """Two decoders of one hidden size and different MLP sizes on one operator set: each gets the workspace that its own
    one-launch MLP uses, whichever was made first, so that their steps may overlap; none where that MLP takes other launches
    (16 rows of 5120).  Host logic: the launches themselves are replaced by what they were given."""
    from ksa_amd import decode, gemm
    from ksa_amd.model import HipOps
    given = []
    monkeypatch.setattr(gemm, "MlpRowsWorkspace", lambda H, I, device: (H, I))
    monkeypatch.setattr(gemm, "add_rmsnorm_linear_rows", lambda *a: (given.append(a[-1]), (None, None))[1])
    monkeypatch.setattr(decode, "ksa_decode_qkv_o", lambda *a, **k: (given.append(a[-1]), "o")[1])
    monkeypatch.setattr(HipOps, "_streaming", lambda self, w, multiple=16: object.__new__(gemm.TiledWeight))
    monkeypatch.setattr(decode, "decode_qkv_o_pays", lambda *a: True)
    ops = HipOps()
    for H, b, sizes in ((2048, 2, (512, 1024)), (5120, 16, (512,))):
        models = []
        for I in sizes:
            cfg = tiny_config(hidden_size=H, intermediate_size=I, num_attention_heads=8, num_hidden_layers=1,
                              summary_sliding_chunk_num=1)
            models.append(KsaQwen3ForCausalLM(cfg, init_weights(cfg, "cpu", torch.bfloat16), ops))
            ops.prepare_mlp_rows(H, I, torch.device("cpu"))
        for model, I in list(zip(models, sizes))[::-1]:
            lw = model.w["layers"][0]
            part = lambda n: gemm.SplitKPartials(torch.zeros(17 * 16 * n * 4, dtype=torch.uint8), 17, b, (b, 1, n), torch.bfloat16)
            kc = torch.zeros(b, 2, 32, 64, dtype=torch.bfloat16)
            given.clear()
            if H == 2048:
                model._norm_qkv(lw, part(H), torch.zeros(b, 1, H, dtype=torch.bfloat16))
                assert model._text_attention(lw, part(12 * 64), None, None, kc, kc, 3, 0, 9, {}) == "o"
                assert given == [(H, I)] * 2
            else:
                assert ops.decode_qkv_o(part(12 * 64), *[None] * 5, kc, kc, 8, 3, 0, 9, 1.0, lw["o_proj"], I) is None


@pytest.mark.gpu
def test_gpu_one_model_serves_changing_batch_sizes():
    """Batch 8, then 2, then 8, then 1 on ONE model (one operator set, hence one workspace of the
    one-launch MLP, whose counting words go on from call to call): every call's logits equal, bit
    for bit, those of a model made fresh for that call."""
    from ksa_amd.model import HipOps
    cfg = _mlp_rows_config()
    w = init_weights(cfg, "cuda", torch.bfloat16, 31)
    shared = KsaQwen3ForCausalLM(cfg, w, HipOps())
    for i, (batch, graph) in enumerate([(8, True), (2, True), (8, False), (1, True), (2, False), (8, True)]):
        ids = torch.randint(0, cfg.vocab_size, (batch, 140), generator=torch.Generator().manual_seed(40 + i))
        out_a, log_a = shared.generate(ids, 12, return_logits=True, use_graph=graph)
        fresh = KsaQwen3ForCausalLM(cfg, w, HipOps())
        out_b, log_b = fresh.generate(ids, 12, return_logits=True, use_graph=graph)
        assert shared.ops.mlp_one_launch and fresh.ops.mlp_one_launch
        assert torch.equal(out_a, out_b), (i, batch)
        assert torch.equal(log_a, log_b), (i, batch, (log_a - log_b).abs().max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [False, True])
def test_gpu_generate_repeats_on_separate_launches_after_a_timeout(graph):
    """The one-launch MLP's give-up path through the model, forced from the host (the workspace word
    with the number of past launches is set far ahead, so its waits cannot be satisfied; every
    workgroup leaves through its bounded wait).  `generate` must notice at its check, switch the
    operator set to the separate launches, repeat the call, and return what a model that never used
    the one-launch MLP returns, bit for bit; the steps in between must not have raised or hung.
    A direct caller of the step functions gets the exception at the next chunk boundary."""
    from ksa_amd.gemm import MlpRowsTimeout
    from ksa_amd.model import HipOps
    cfg = _mlp_rows_config()
    w = init_weights(cfg, "cuda", torch.bfloat16, 33)
    ids = torch.randint(0, cfg.vocab_size, (2, 250), generator=torch.Generator().manual_seed(34))
    plain_ops = HipOps()
    plain_ops.mlp_one_launch = False
    want_ids, want_log = KsaQwen3ForCausalLM(cfg, w, plain_ops).generate(ids, 10, return_logits=True, use_graph=graph)

    model = KsaQwen3ForCausalLM(cfg, w, HipOps())
    ws = model.ops.prepare_mlp_rows(cfg.hidden_size, cfg.intermediate_size, model.device)
    ws.buf[:8].view(torch.int64).fill_(1 << 40)
    got_ids, got_log = model.generate(ids, 10, return_logits=True, use_graph=graph)
    assert not model.ops.mlp_one_launch
    assert torch.equal(got_ids, want_ids) and torch.equal(got_log, want_log)
    assert not model.ops.mlp_rows_failed()          # the workspace was cleared

    # the step functions themselves: 250 = 128 + 122, so the sixth step is a chunk boundary
    model2 = KsaQwen3ForCausalLM(cfg, w, HipOps())
    logits, cache = model2.prefill(ids)
    model2.ops.prepare_mlp_rows(cfg.hidden_size, cfg.intermediate_size, model2.device).buf[:8].view(
        torch.int64).fill_(1 << 40)
    step = model2.decode_step_graph if graph else model2.decode_step
    with pytest.raises(MlpRowsTimeout):
        for _ in range(6):
            logits = step(logits[:, 0].argmax(-1)[:, None], cache)
    assert cache.get_cur_chunk_size() == cfg.summary_chunk_size - 1   # raised in front of the boundary step
    assert not model2.ops.mlp_one_launch


@pytest.mark.gpu
def test_gpu_config4_full_depth_decode_equals_prefill():
    """Config 4 at its own size - 36 layers (three Summary layers with a window of 4 chunks to one
    unbounded layer, nine times), hidden 2560, 32 / 8 heads, MLP 9728, vocabulary 151936, batch 8,
    a prompt of 32k tokens: the logits for token n from `prefill(n tokens)` against those from
    `prefill(n - 9 tokens)` followed by 9 decode steps replayed from the HIP graphs, across the chunk
    boundary at 32768 tokens (the boundary step runs from its own recording).  The summaries that the
    boundary step stores are not visible to the text tokens of the next four chunks, so the two ways
    agree to rounding although the reference's boundary step treats the summary tokens differently
    from its prefill mask.  This is the decode == prefill invariant through prefill, cache
    reorganisation (256 chunks, nine text-only gathers of 32k rows), ring, boundary flush and the
    one-launch MLP at the depth and the size the benchmark's end-to-end run has.
    Tolerance: both sides are bf16 runs whose rounding errors differ (library GEMMs over 34k rows on one
    side, the few-rows kernels on the other; different summation orders in attention) and add up over
    nine times the depth of `test_gpu_module_config4_layer_shape`, i.e. about three times its noise:
    root mean square within 1 % of the logit scale (measured 0.56 %), largest of the 1.2 million
    differences within 5 % (measured 2.8 %).  A stale or misplaced cache row in one layer moves the
    logits by less than that; those are pinned row by row in tests/test_cache_gpu.py.  What this test
    catches is a step that went wrong as a whole at full depth: garbage or non-finite rows, a layer
    kind taking the wrong range, a timed-out launch."""
    from ksa_amd.model import HipOps
    cfg = KsaQwen3Config()
    assert cfg.num_hidden_layers == 36 and cfg.sliding_chunk_nums()[:4] == [4, 4, 4, 1 << 20]
    dev = torch.device("cuda")
    w = init_weights(cfg, dev, torch.bfloat16, 17)
    model = KsaQwen3ForCausalLM(cfg, w, HipOps())
    model.BOUNDARY_GRAPH_AFTER = 0
    batch, n, k = 8, 32768 + 5, 9
    ids = torch.randint(0, cfg.vocab_size, (batch, n), generator=torch.Generator().manual_seed(18)).to(dev)
    want, cache_full = model.prefill(ids)
    want = want[:, 0].float()
    assert cache_full.get_true_token_num() == n and cache_full.get_cur_chunk_size() == 5
    del cache_full
    torch.cuda.empty_cache()
    logits, cache = model.prefill(ids[:, :n - k])
    boundaries = 0
    for t in range(n - k, n):
        boundaries += cache.get_cur_chunk_size() == cfg.summary_chunk_size - 1
        logits = model.decode_step_graph(ids[:, t:t + 1], cache)
    got = logits[:, 0].float()
    model.check_steps(cache)                 # raises if a launch gave up waiting
    assert boundaries == 1 and cache.get_true_token_num() == n
    assert model.ops.mlp_one_launch
    assert torch.isfinite(got).all() and torch.isfinite(want).all()
    scale = want.abs().max().item()
    err = (got - want).abs().max().item()
    rms = (got - want).pow(2).mean().sqrt().item()
    agree = (got.argmax(-1) == want.argmax(-1)).float().mean().item()
    print(f"full depth: max logit difference {err / scale:.3e} of the logit scale, rms {rms / scale:.3e}, "
          f"arg-max agreement {agree:.2f}")
    assert err <= 5e-2 * scale and rms <= 1e-2 * scale, (err / scale, rms / scale)


@pytest.mark.gpu
def test_gpu_graph_decode_forms_of_token_ids():
    """A recorded step reads int64 ids where they are and takes every other form through a copy: the same
    logits bit for bit, and those of the separate launches that other operators' recordings hold."""
    from ksa_amd.model import HipOps
    cfg = tiny_config(summary_chunk_size=128, summary_token_num=8, head_dim=128, num_attention_heads=8,
                      num_key_value_heads=2, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                      summary_sliding_chunk_num=[1, 1 << 20], vocab_size=1000, summary_token_begin=1000)
    w = init_weights(cfg, "cuda", torch.bfloat16, 8)
    ids = torch.randint(0, cfg.vocab_size, (3, 140), generator=torch.Generator().manual_seed(10))
    tok = torch.tensor([[5], [999], [0]], device="cuda")

    class SeparateHead(HipOps):
        def __init__(self):
            super().__init__()
            self.embed_rmsnorm_supported = lambda table, weight: False

    forms = (tok, tok.int(), tok.cpu(), torch.cat((tok, tok), 1)[:, :1], tok - cfg.embedding_rows())
    got = []
    for ops, form in [(HipOps(), f) for f in forms] + [(SeparateHead(), tok)]:
        model = KsaQwen3ForCausalLM(cfg, w, ops)
        _, cache = model.prefill(ids)
        steps = [model.decode_step_graph(form, cache).clone() for _ in range(3)]
        got.append(torch.stack(steps))
    for g in got[1:]:
        assert torch.equal(g, got[0])
