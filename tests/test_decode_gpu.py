"""GPU parity of decode attention and the cache row mover against the CPU oracle."""
import numpy as np
import pytest
import torch

from conftest import to_np
from oracle import c_oracle

pytestmark = pytest.mark.gpu

ATOL = 2e-2   # bf16 GPU vs fp32 oracle, stated bar
RTOL_INF = 2e-2


def _mk(Bz, Hq, Hkv, Q, D, rows, seed, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(Bz, Hq, Q, D, generator=g).to(dtype)
    k = torch.randn(Bz, Hkv, rows, D, generator=g).to(dtype)
    v = torch.randn(Bz, Hkv, rows, D, generator=g).to(dtype)
    return q, k, v


def _check(q, k, v, start, end, nsplit, scale=None):
    import ksa_amd
    dev = torch.device("cuda")
    Bz = q.shape[0]
    st = torch.as_tensor(start, dtype=torch.int32, device=dev) if np.ndim(start) else int(start)
    en = torch.as_tensor(end, dtype=torch.int32, device=dev) if np.ndim(end) else int(end)
    out = ksa_amd.ksa_decode(q.to(dev), k.to(dev), v.to(dev), st, en, scale=scale, nsplit=nsplit)
    torch.cuda.synchronize()
    want = c_oracle.decode(to_np(q), to_np(k), to_np(v), np.broadcast_to(start, (Bz,)),
                           np.broadcast_to(end, (Bz,)), scale=scale)
    got = to_np(out)
    err = np.abs(got - want).max()
    assert np.isfinite(got).all()
    assert err <= ATOL and err <= RTOL_INF * np.abs(want).max(), (err, np.abs(want).max())


@pytest.mark.parametrize("nsplit", [1, 2, 5, None])
def test_decode_small(nsplit):
    q, k, v = _mk(3, 8, 2, 1, 128, 700, seed=0)
    _check(q, k, v, 0, 700, nsplit)


@pytest.mark.parametrize("nsplit", [1, 3])
def test_decode_per_sequence_ranges(nsplit):
    """ragged [start, end) per sequence, including one-row and sub-tile slices"""
    q, k, v = _mk(6, 8, 4, 1, 128, 1000, seed=1)
    start = np.array([0, 5, 136, 999, 100, 17], np.int32)
    end = np.array([1000, 6, 900, 1000, 131, 530], np.int32)
    _check(q, k, v, start, end, nsplit)


def test_decode_strided_view_like_hf():
    """HF hands in cache[:, :, start:end, :] views (non-contiguous batch/head strides)."""
    import ksa_amd
    dev = torch.device("cuda")
    q, k, v = _mk(2, 32, 8, 1, 128, 2000, seed=2)
    kd, vd = k.to(dev), v.to(dev)
    kview, vview = kd[:, :, 37:1500, :], vd[:, :, 37:1500, :]

    class M:
        num_key_value_groups = 4
    out, w = ksa_amd.decode_attention_forward(M(), q.to(dev), kview, vview, None, scaling=128 ** -0.5)
    assert w is None and out.shape == (2, 1, 32, 128)
    want = c_oracle.decode(to_np(q), to_np(k), to_np(v), 37, 1500)
    assert np.abs(to_np(out) - want).max() <= ATOL


def test_decode_boundary_queries():
    """chunk-boundary step: S = 8 summary queries x g = 4 heads fill one 32-column tile;
    Q = 9 needs two column blocks."""
    for Q in (8, 9):
        q, k, v = _mk(2, 8, 2, Q, 128, 136, seed=3)
        _check(q, k, v, 0, 136, 1)
        _check(q, k, v, 0, 136, 2)


def test_decode_head_dim_64_and_fp16():
    q, k, v = _mk(2, 4, 2, 1, 64, 555, seed=4)
    _check(q, k, v, 3, 555, 2)
    q, k, v = _mk(2, 4, 2, 1, 128, 555, seed=5, dtype=torch.float16)
    _check(q, k, v, 3, 555, 1)


@pytest.mark.parametrize("D", [256, 96, 192, 40])
def test_decode_other_head_dims(D):
    """Head dimension 256 (kernels of its own) and multiples of 8 without one (zero-padded copies of the
    attended rows at the next kernel size): scalar and per-sequence ranges, splits, the boundary step's
    9 query tokens, fp16."""
    q, k, v = _mk(3, 8, 2, 1, D, 900, seed=30 + D)
    _check(q, k, v, 5, 900, 1)
    _check(q, k, v, np.array([0, 100, 640], np.int32), np.array([900, 777, 641], np.int32), 3)
    q, k, v = _mk(2, 4, 2, 9, D, 300, seed=31 + D, dtype=torch.float16)
    _check(q, k, v, 0, 136, 2)


def test_decode_peaked_softmax():
    """large scale -> near one-hot attention: exercises the running-max rescale"""
    q, k, v = _mk(2, 8, 2, 1, 128, 3000, seed=6)
    _check(q, k, v, 0, 3000, 1, scale=1.0)
    _check(q, k, v, 0, 3000, 4, scale=1.0)


def test_decode_cfg3_shape_subset():
    """cfg 3 geometry (cap 17288, S=8, C=128, ring 512, 8192 summaries) on 4 of the 64
    sequences: slice [136 - cbl, 8808)."""
    Bz, cap = 4, 17288
    q, k, v = _mk(Bz, 32, 8, 1, 128, cap, seed=7)
    cbl = np.array([1, 128, 57, 100], np.int32)
    _check(q, k, v, 136 - cbl, np.full(Bz, 8808, np.int32), None)


def test_decode_cfg3_full_batch():
    """cfg 3 itself: batch 64, 32/8 heads, cap 17288, per-sequence slice [136 - cbl, 8808) with
    cbl uniform in [1, 128]: all 64 x 32 output rows against the oracle (one sequence at a
    time on the host), and the split-K identity (1 split == 4 splits up to rounding)."""
    import ksa_amd
    dev = torch.device("cuda")
    Bz, Hq, Hkv, D, cap = 64, 32, 8, 128, 17288
    g = torch.Generator(device=dev).manual_seed(11)
    k = torch.randn(Bz, Hkv, cap, D, generator=g, device=dev).to(torch.bfloat16)
    v = torch.randn(Bz, Hkv, cap, D, generator=g, device=dev).to(torch.bfloat16)
    q = torch.randn(Bz, Hq, 1, D, generator=g, device=dev).to(torch.bfloat16)
    cbl = torch.randint(1, 129, (Bz,), generator=g, device=dev, dtype=torch.int32)
    start = (136 - cbl).to(torch.int32)
    end = torch.full((Bz,), 8808, dtype=torch.int32, device=dev)
    out1 = ksa_amd.ksa_decode(q, k, v, start, end, nsplit=1)
    out4 = ksa_amd.ksa_decode(q, k, v, start, end, nsplit=4)
    outa = ksa_amd.ksa_decode(q, k, v, start, end)
    torch.cuda.synchronize()
    assert (out1.float() - out4.float()).abs().max().item() <= 2e-3
    assert (out1.float() - outa.float()).abs().max().item() <= 2e-3
    got = to_np(out1)
    st, en = start.cpu().numpy(), end.cpu().numpy()
    worst = 0.0
    for b in range(Bz):
        want = c_oracle.decode(to_np(q[b:b + 1]), to_np(k[b:b + 1]), to_np(v[b:b + 1]), st[b:b + 1], en[b:b + 1])
        err = np.abs(got[b:b + 1] - want).max()
        worst = max(worst, err)
        assert err <= ATOL and err <= RTOL_INF * np.abs(want).max(), (b, err)
    assert np.isfinite(got).all()


def test_copy_rows():
    import ksa_amd
    from ksa_amd.cache import _move_rows
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(0)
    src = torch.randn(2, 3, 50, 128, generator=g).bfloat16().to(dev)
    dst = torch.zeros(2, 3, 80, 128, dtype=torch.bfloat16, device=dev)
    _move_rows(src, dst, 20, 5, 33)
    assert torch.equal(dst[:, :, 33:53], src[:, :, 5:25]) and float(dst[:, :, :33].abs().sum()) == 0
    idx = torch.tensor([7, 3, 49, 0], dtype=torch.int32, device=dev)
    _move_rows(src, dst, 4, dst_start=60, src_index=idx)
    assert torch.equal(dst[:, :, 60:64], src[:, :, idx.long()])


def test_decode_empty_and_single_row_ranges():
    """Ragged extremes: a sequence whose row range is empty (the reference never produces one; this
    build defines its output as zeros, not NaN), one with a single row (output = that row of V) and
    ordinary ones in the same launch, with one and with several splits."""
    import ksa_amd
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(31)
    b, Hq, Hkv, D, rows = 4, 8, 2, 128, 900
    q = torch.randn(b, Hq, 1, D, generator=g).bfloat16()
    kc = torch.randn(b, Hkv, rows, D, generator=g).bfloat16()
    vc = torch.randn(b, Hkv, rows, D, generator=g).bfloat16()
    start = np.array([100, 500, 0, 37], np.int32)
    end = np.array([100, 501, 900, 300], np.int32)
    for nsplit in (1, 4):
        got = ksa_amd.ksa_decode(q.to(dev), kc.to(dev), vc.to(dev), torch.as_tensor(start, device=dev),
                                 torch.as_tensor(end, device=dev), nsplit=nsplit).float().cpu().numpy()
        assert np.isfinite(got).all()
        assert np.abs(got[0]).max() == 0.0
        want1 = vc[1, :, 500].float().numpy()                     # [Hkv, D]; head h reads kv head h // g
        assert np.array_equal(got[1, 0], np.repeat(want1, Hq // Hkv, axis=0))
        ref = c_oracle.decode(q[2:].float().numpy(), kc[2:].float().numpy(), vc[2:].float().numpy(), start[2:], end[2:])
        assert np.abs(got[2:] - ref).max() <= 2e-2


def _weights_oracle(q, k, start, end, scale, mask=None):
    """softmax(q K^T * scale + mask) in float64 per (sequence, head, query token) over rows [start, end)."""
    Bz, Hq, Q, D = q.shape
    g = Hq // k.shape[1]
    L = int(np.max(end - start))
    out = np.zeros((Bz, Hq, Q, L))
    for b in range(Bz):
        n = int(end[b] - start[b])
        for h in range(Hq):
            s = q[b, h].astype(np.float64) @ k[b, h // g, start[b]:end[b]].astype(np.float64).T * scale
            if mask is not None:
                s = s + np.broadcast_to(mask, (Bz, Hq, Q, L))[b, h, :, :n]
            s -= s.max(axis=-1, keepdims=True)
            e = np.exp(s)
            out[b, h, :, :n] = e / e.sum(axis=-1, keepdims=True)
    return out


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16), (256, torch.bfloat16), (96, torch.bfloat16)])
def test_decode_weights_match_softmax(D, dtype):
    """The probabilities of the eager decode variant (modeling_qwen3sa.py:569-588) against a float64
    soft-max of the same scores: per-sequence ranges of different lengths (zeros behind the shorter
    ones), one query token and the boundary step's nine, GQA, an additive mask; each row sums to 1.
    Tolerance: the rounding of a probability to the 16-bit type (relative 2^-8 for bf16, 2^-11 for
    fp16) plus an absolute 1e-6."""
    import ksa_amd
    dev = torch.device("cuda")
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for Q, rows, start, end in ((1, 900, np.array([0, 100, 640]), np.array([900, 777, 641])),
                                (9, 300, np.array([3, 3, 3]), np.array([139, 139, 139]))):
        q, k, v = _mk(3, 8, 2, Q, D, rows, seed=90 + Q + D, dtype=dtype)
        scale = D ** -0.5
        st, en = (torch.as_tensor(x, dtype=torch.int32, device=dev) for x in (start, end))
        w = ksa_amd.ksa_decode_weights(q.to(dev), k.to(dev), st, en)
        L = int((end - start).max())
        assert w.shape == (3, 8, Q, L) and w.dtype == dtype
        want = _weights_oracle(to_np(q), to_np(k), start, end, scale)
        got = to_np(w).astype(np.float64)
        assert (np.abs(got - want) <= rel * want + 1e-6).all(), np.abs(got - want).max()
        assert np.abs(got.sum(-1) - 1).max() <= 2e-2
        for b in range(3):
            assert (got[b, :, :, end[b] - start[b]:] == 0).all()
    # scalar range + additive mask that removes every third position and biases the rest
    q, k, v = _mk(2, 4, 4, 2, D, 200, seed=99, dtype=dtype)
    mask = torch.zeros(2, 1, 2, 150, dtype=dtype)
    mask[..., ::3] = float("-inf")
    mask[..., 1::3] = 0.5
    w = ksa_amd.ksa_decode_weights(q.to(dev), k.to(dev), 20, 170, mask=mask.to(dev))
    want = _weights_oracle(to_np(q), to_np(k), np.full(2, 20), np.full(2, 170), D ** -0.5, mask=to_np(mask).astype(np.float64))
    got = to_np(w).astype(np.float64)
    assert (np.abs(got - want) <= rel * want + 1e-6).all() and (got[..., ::3] == 0).all()


def test_eager_attention_forward_signature():
    """The reference's eager decode attention function (modeling_qwen3sa.py:569-588), as its cache call
    sites use it (:816-870: a slice of the cache, mask None): output equal to the SDPA variant's,
    probabilities consistent with it (weights @ V reproduces the output)."""
    import ksa_amd
    dev = torch.device("cuda")
    q, k, v = _mk(2, 8, 2, 1, 128, 500, seed=123)
    q, k, v = q.to(dev), k.to(dev), v.to(dev)

    class M:
        num_key_value_groups = 4
    out, w = ksa_amd.eager_attention_forward(M(), q, k[:, :, 7:444], v[:, :, 7:444], None, scaling=128 ** -0.5)
    ref, none = ksa_amd.decode_attention_forward(M(), q, k[:, :, 7:444], v[:, :, 7:444], None, scaling=128 ** -0.5)
    assert none is None and torch.equal(out, ref)
    assert w.shape == (2, 8, 1, 437)
    vv = v[:, :, 7:444].float().repeat_interleave(4, dim=1)           # [b, Hq, L, D]
    recon = torch.matmul(w.float(), vv).transpose(1, 2)                # [b, 1, Hq, D]
    assert (recon - out.float()).abs().max().item() <= 2e-2
    with pytest.raises(NotImplementedError):
        ksa_amd.eager_attention_forward(M(), q, k, v, torch.zeros(1, device=dev), scaling=1.0)


@pytest.mark.parametrize("D,dtype,g", [(128, torch.bfloat16, 4), (128, torch.float16, 1), (64, torch.bfloat16, 2),
                                       (256, torch.bfloat16, 4)])
@pytest.mark.parametrize("nsplit", [1, 3, None])
def test_decode_boundary_equals_two_decodes(D, dtype, g, nsplit):
    """The chunk-boundary form (text token over its range, the S summary tokens over theirs, one launch)
    against the two separate launches it stands for - bit for bit at the same split count - and
    against the oracle; per-sequence text ranges as device tensors with a scalar summary range (the
    small-window layer of a replayed step), per-sequence ranges for both (large window), and scalars."""
    import ksa_amd
    dev = torch.device("cuda")
    Bz, Hkv, S, C, rows = 3, 2, 8, 128, 1200
    q, k, v = _mk(Bz, Hkv * g, Hkv, 1 + S, D, rows, seed=17 + D + g, dtype=dtype)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    t0, t1 = np.array([136 - 5, 136 - 128, 136 - 77], np.int32), np.array([1100, 1100, 900], np.int32)
    cases = [((torch.as_tensor(t0, device=dev), torch.as_tensor(t1, device=dev)), (0, S + C), t0, t1, np.zeros(3, np.int32), np.full(3, S + C, np.int32))]
    s0, s1 = np.array([700, 650, 820], np.int32), np.array([836, 786, 956], np.int32)
    cases.append(((torch.as_tensor(np.zeros(3, np.int32), device=dev), torch.as_tensor(s1 - S, device=dev)),
                  (torch.as_tensor(s0, device=dev), torch.as_tensor(s1, device=dev)), np.zeros(3, np.int32), s1 - S, s0, s1))
    cases.append(((10, 1111), (0, 136), np.full(3, 10, np.int32), np.full(3, 1111, np.int32), np.zeros(3, np.int32), np.full(3, 136, np.int32)))
    for (ta, tb), (sa, sb), ta_n, tb_n, sa_n, sb_n in cases:
        got = ksa_amd.ksa_decode_boundary(qd, kd, vd, ta, tb, sa, sb, nsplit=nsplit)
        assert got.shape == (Bz, 1 + S, Hkv * g, D)
        want_t = c_oracle.decode(to_np(q[:, :, :1]), to_np(k), to_np(v), ta_n, tb_n)
        want_s = c_oracle.decode(to_np(q[:, :, 1:]), to_np(k), to_np(v), sa_n, sb_n)
        want = np.concatenate([want_t, want_s], axis=1)
        err = np.abs(to_np(got) - want).max()
        assert err <= ATOL and err <= RTOL_INF * np.abs(want).max(), err
        if nsplit is not None:
            two = torch.cat([ksa_amd.ksa_decode(qd[:, :, :1], kd, vd, ta, tb, nsplit=nsplit),
                             ksa_amd.ksa_decode(qd[:, :, 1:], kd, vd, sa, sb, nsplit=nsplit)], dim=1)
            assert torch.equal(got, two)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,Hq,Hkv,D,rows,start,end,row,nsplit", [
    (1, 32, 8, 128, 700, 3, 690, 3, None),        # first row of the range (a small window)
    (1, 32, 8, 128, 700, 0, 700, 699, 12),        # last row (a large window), splits without rows
    (1, 32, 8, 128, 5000, 0, 4999, 2500, 64),     # most splits; 40 of them have rows
    (2, 8, 8, 128, 300, 10, 299, 138, 2),         # one query head per kv head; last row of a workgroup's round
    (3, 15, 3, 128, 300, 0, 129, 128, 2),         # group of 5; a slice of one row, the new one
    (4, 32, 1, 128, 260, 1, 258, 33, 3),          # group of 32: several passes over the query rows
    (8, 32, 4, 64, 500, 5, 400, 6, 4),
    (2, 16, 8, 64, 90, 0, 64, 63, 1),             # no split
    (16, 32, 8, 128, 400, 0, 300, 200, 3),
])
def test_decode_qkv_equals_separate_launches(dtype, b, Hq, Hkv, D, rows, start, end, row, nsplit):
    """The attention of a step from the projection's partial sums against the pre-attention step and the decode
    call it stands for: output and caches bit for bit."""
    import ksa_amd
    from ksa_amd import decode, gemm, pre
    g = torch.Generator(device="cuda").manual_seed(b * 1000 + end)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    H = 1536 if D == 128 else 5120                 # 3 or 10 slices of the projection's K
    width = (Hq + 2 * Hkv) * D
    h, w = rnd(b, 1, H).to(dtype), (rnd(width, H) * H ** -0.5).to(dtype)
    qw, kw = (1 + 0.1 * rnd(D)).to(dtype), (1 + 0.1 * rnd(D)).to(dtype)
    ang = rnd(1, 1, D // 2)
    ang = torch.cat((ang, ang), -1)
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    qkv = gemm.linear_rows(h, w, defer=True)
    assert isinstance(qkv, gemm.SplitKPartials)
    caches = [rnd(b, Hkv, rows, D).to(dtype) for _ in range(2)]
    caches[0][:, :, row] = float("nan")            # what the new row overwrites must not be read
    caches[1][:, :, row] = float("nan")
    for device_bounds in (False, True):
        kc, vc = (c.clone() for c in caches)
        kr, vr = (c.clone() for c in caches)
        at = torch.full((b,), row, dtype=torch.int32, device="cuda")
        q, _, _ = pre.pre_attention_partials(qkv, Hq, Hkv, D, qw, kw, cos, sin, 1e-6, k_out=kr[:, :, :1].transpose(1, 2),
                                             v_out=vr[:, :, :1].transpose(1, 2), kv_out_row=at)
        lo, hi, r = start, end, row
        if device_bounds:
            lo, hi, r = (torch.full((b,), x, dtype=torch.int32, device="cuda") for x in (start, end, row))
        want = ksa_amd.ksa_decode(q.transpose(1, 2), kr, vr, lo, hi, nsplit=nsplit)
        got = decode.ksa_decode_qkv(qkv, qw, kw, cos, sin, 1e-6, kc, vc, Hq, r, lo, hi, nsplit=nsplit)
        assert torch.equal(got, want.reshape(b, 1, Hq * D)) and torch.isfinite(got.float()).all()
        assert torch.equal(kc, kr) and torch.equal(vc, vr)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,Hq,Hkv,D", [(5, 32, 8, 128), (6, 8, 4, 64), (17, 4, 2, 128)])
@pytest.mark.parametrize("nsplit", [1, 4, None])
def test_decode_qkv_with_a_range_row_and_position_per_sequence(dtype, b, Hq, Hkv, D, nsplit):
    """Every sequence with its own range, new row and rotary row: the new row first, last, in between and at the
    borders of a workgroup's rounds, long sequences next to ones of few rows (whose later splits are empty).
    Bit for bit the separate launches, and within the usual bound of the oracle."""
    import ksa_amd
    from ksa_amd import decode, gemm, pre
    rows = 1100
    g = torch.Generator(device="cuda").manual_seed(b * 10 + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    forms = [(0, 1100, 1099), (7, 1031, 7), (3, 40, 20), (128, 129, 128), (0, 300, 127), (5, 645, 133), (90, 1000, 511)]
    lo, hi, row = (np.array([forms[i % len(forms)][j] for i in range(b)], np.int32) for j in range(3))
    dev = lambda a: torch.as_tensor(a, device="cuda")
    H, width = 1536, (Hq + 2 * Hkv) * D
    h, w = rnd(b, 1, H).to(dtype), (rnd(width, H) * H ** -0.5).to(dtype)
    qw, kw = (1 + 0.1 * rnd(D)).to(dtype), (1 + 0.1 * rnd(D)).to(dtype)
    ang = rnd(b, 1, D // 2)
    ang = torch.cat((ang, ang), -1)
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    qkv = gemm.linear_rows(h, w, defer=True)
    kc, vc = (rnd(b, Hkv, rows, D).to(dtype) for _ in range(2))
    for i in range(b):                             # what the new rows overwrite must not be read
        kc[i, :, row[i]] = vc[i, :, row[i]] = float("nan")
    kr, vr = kc.clone(), vc.clone()
    q, _, _ = pre.pre_attention_partials(qkv, Hq, Hkv, D, qw, kw, cos, sin, 1e-6, k_out=kr[:, :, :1].transpose(1, 2),
                                         v_out=vr[:, :, :1].transpose(1, 2), kv_out_row=dev(row))
    want = ksa_amd.ksa_decode(q.transpose(1, 2), kr, vr, dev(lo), dev(hi), nsplit=nsplit)
    got = decode.ksa_decode_qkv(qkv, qw, kw, cos, sin, 1e-6, kc, vc, Hq, dev(row), dev(lo), dev(hi), nsplit=nsplit)
    assert torch.equal(got, want.reshape(b, 1, Hq * D))
    assert torch.equal(kc, kr) and torch.equal(vc, vr)
    ref = c_oracle.decode(to_np(q.transpose(1, 2)), to_np(kr), to_np(vr), lo, hi)
    assert np.abs(to_np(got).reshape(ref.shape) - ref).max() <= ATOL * max(1.0, np.abs(ref).max())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,Hq,Hkv,D,N,nsplit", [
    (1, 32, 8, 128, 2560, None),
    (1, 32, 8, 128, 256, 1),       # no split: nothing for the second half of a workgroup to merge
    (1, 16, 2, 128, 144, 39),      # odd count, several requests; the last workgroup has one tile
    (1, 8, 4, 64, 16, 64),         # eight heads of several kv heads in a chunk
    (2, 32, 8, 128, 272, 32),      # a row's splits end with a request
    (3, 8, 8, 64, 128, 21),        # rows 0 and 2 / row 1 over two requests each
    (5, 4, 2, 128, 512, 7),
    (8, 32, 8, 128, 2560, 8),
    (16, 32, 8, 128, 1024, 4),
])
def test_decode_qkv_o_equals_separate_launches(dtype, b, Hq, Hkv, D, N, nsplit):
    """Attention and o projection of a step in one launch against the two launches (three with the merge) it stands for, with
    ranges from one row to all (later splits empty), several launches on one workspace, fresh data each.  The
    splits are merged in another order: a head's output may move by one unit in the last place (2^-8 / 2^-11 of it),
    a random share of which reaches a product of K terms - bound: 2 units x sqrt(K) times the mean term; most are equal."""
    from ksa_amd import _lib, decode, gemm
    rows = 4100 if nsplit is None or nsplit > 16 else 1100
    auto = _lib.lib().ksa_decode_qkv_o_splits(b, Hq, Hkv, D, rows)   # (another count rounds other probabilities)
    g = torch.Generator(device="cuda").manual_seed(b * 10 + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    H, width, K = 1536, (Hq + 2 * Hkv) * D, Hq * D
    wo = (rnd(N, K) * K ** -0.5).to(dtype)
    tiled, ws = gemm.TiledWeight(wo), gemm.MlpRowsWorkspace(N, 64, torch.device("cuda"))
    qw, kw = (1 + 0.1 * rnd(D)).to(dtype), (1 + 0.1 * rnd(D)).to(dtype)
    ang = rnd(b, 1, D // 2)
    ang = torch.cat((ang, ang), -1)
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    w = (rnd(width, H) * H ** -0.5).to(dtype)
    forms = [(0, rows, rows - 1), (7, 1031, 7), (128, 129, 128), (3, 40, 20), (0, 300, 127)]
    dev = lambda v: torch.as_tensor(v, device="cuda", dtype=torch.int32)
    for rep in range(3):
        lo, hi, row = (dev([forms[(i + rep) % len(forms)][j] for i in range(b)]) for j in range(3))
        qkv = gemm.linear_rows(rnd(b, 1, H).to(dtype), w, defer=True)
        caches = [rnd(b, Hkv, rows, D).to(dtype) for _ in range(2)]
        kc, vc = (c.clone() for c in caches)
        kr, vr = (c.clone() for c in caches)
        attn = decode.ksa_decode_qkv(qkv, qw, kw, cos, sin, 1e-6, kr, vr, Hq, row, lo, hi, nsplit=nsplit or auto)
        got = decode.ksa_decode_qkv_o(qkv, qw, kw, cos, sin, 1e-6, kc, vc, Hq, row, lo, hi, tiled, ws, nsplit=nsplit)
        torch.cuda.synchronize()
        assert not ws.failed() and int(ws.step.view(torch.int64).abs().sum().item()) == 0
        assert torch.equal(kc, kr) and torch.equal(vc, vr)
        got = got.workspace.view(torch.float32).view(K // 512, 16, N)[:, :b].sum(0)
        want = attn.view(b, K).double() @ wo.double().t()
        ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        term = (attn.view(b, K).double().square() @ wo.double().t().square() / K).sqrt()
        assert ((got - want).abs() <= 2 * ulp * K ** 0.5 * term + 1e-5 * want.abs().max()).all()
        assert (got - want).square().mean() <= (0.25 * ulp) ** 2 * (K * term.square()).mean()


@pytest.mark.parametrize("scale", [-0.3, 0.0])
def test_decode_scale_that_is_not_positive(scale):
    """Ranges that end inside a tile (hidden rows) with one split and with several; the one-launch step against the oracle
    on the rows that it wrote."""
    from ksa_amd import decode, gemm
    q, k, v = _mk(2, 4, 2, 1, 128, 700, seed=8)
    for nsplit in (1, 3):
        _check(q, k, v, [3, 0], [77, 690], nsplit, scale=scale)
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(9)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    qkv = gemm.linear_rows(rnd(2, 1, 1024), rnd(8 * 128, 1024), defer=True)
    kc, vc, one, zero = k.to(dev), v.to(dev), torch.ones(128, device=dev).bfloat16(), torch.zeros(128, device=dev).bfloat16()
    got = decode.ksa_decode_qkv(qkv, one, one, one, zero, 1e-6, kc, vc, 4, 76, 3, 77, scale=scale)
    x = qkv.workspace.view(torch.float32).view(qkv.ksplit, 16, 1024)[:, :2].sum(0).bfloat16().float().view(2, 8, 128)
    qn = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6))[:, :4, None]
    want = c_oracle.decode(to_np(qn), to_np(kc), to_np(vc), 3, 77, scale=scale)
    assert np.abs(to_np(got).reshape(want.shape) - want).max() <= ATOL * max(1.0, np.abs(want).max())


@pytest.mark.gpu
def test_decode_qkv_o_bounded_wait_gives_up_and_recovers():
    """The give-up path of the wait for the attention, forced from the host: the counts are set far below zero.  The first
    workgroup to exhaust its bounded wait (about a second) sets the status word, the others leave, the launch ends;
    `failed()` reports it and zeroes the words, and the next launch equals one on a fresh workspace."""
    from ksa_amd import decode, gemm
    g = torch.Generator(device="cuda").manual_seed(4)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    qkv = gemm.linear_rows(rnd(2, 1, 1024), rnd(8 * 128, 1024), defer=True)
    kc, vc, tiled = rnd(2, 2, 300, 128), rnd(2, 2, 300, 128), gemm.TiledWeight(rnd(256, 512))
    one, ws = torch.ones(128, device="cuda").bfloat16(), gemm.MlpRowsWorkspace(256, 64, torch.device("cuda"))
    call = lambda w: decode.ksa_decode_qkv_o(qkv, one, one, one, one, 1e-6, kc, vc, 4, 5, 0, 300, tiled, w, nsplit=2)
    ws.step.view(torch.int64)[4 * 64::64] = -(1 << 40)
    torch.cuda.synchronize()
    call(ws)
    assert ws.failed() and not ws.failed()
    assert int(ws.step.view(torch.int64).abs().sum().item()) == 0
    a, b = call(ws), call(gemm.MlpRowsWorkspace(256, 64, torch.device("cuda")))
    assert not ws.failed()
    assert torch.equal(*(t.workspace.view(torch.float32).view(1, 16, 256)[:, :2] for t in (a, b)))


@pytest.mark.parametrize("Hkv,D,nsplit", [(2, 256, None), (4, 256, 64), (2, 256, 33), (1, 128, 100), (1, 64, 150), (2, 256, 32),
                                          (2, 128, 32), (2, 128, 33), (1, 64, 32), (1, 64, 33)])
def test_decode_merge_of_more_splits_than_one_pass_takes(Hkv, D, nsplit):
    """The merge walks more than 32 splits at head_dim 256 (64 at 128, 128 at 64) in several passes; up to 32 it has
    a thread per element, one pass.  Scores that grow along the rows move the maximum in each of them; falling ones leave it in the first; a sequence of few
    rows leaves all but the first splits empty."""
    from ksa_amd import _lib
    b, rows = 3, 64 * 300
    if nsplit is None:
        assert _lib.lib().ksa_decode_splits(b, 2 * Hkv, Hkv, 1, D, rows) > 32
    q, k, v = _mk(b, 2 * Hkv, Hkv, 1, D, rows, seed=D + Hkv)
    ramp = torch.linspace(0.1, 4.0, rows)[:, None]
    k[0], k[1] = (k[0].float() * ramp).bfloat16(), (k[1].float() * ramp.flip(0)).bfloat16()
    _check(q, k, v, np.array([0, 0, 11], np.int32), np.array([rows, rows - 3, 300], np.int32), nsplit)
    _check(q[:1], k[:1], v[:1], 0, rows, nsplit)


@pytest.mark.parametrize("D,nsplit", [(128, 5), (64, 3), (256, 4)])
def test_decode_workspace_on_a_four_byte_border(D, nsplit):
    """A caller of the C entry may put the fp32 workspace anywhere floats go."""
    import ctypes
    import ksa_amd
    from ksa_amd import _lib
    q, k, v = (t.cuda() for t in _mk(2, 8, 2, 1, D, 700, seed=D))
    want = ksa_amd.ksa_decode(q, k, v, 3, 690, nsplit=nsplit)
    L = _lib.lib()
    need = L.ksa_decode_workspace_bytes(2, 8, 2, 1, D, nsplit)
    for shift in (4, 8, 12):
        ws = torch.full((need + 16,), 0xff, dtype=torch.uint8, device="cuda")
        out = torch.empty_like(want)
        strides = [(ctypes.c_int64 * 3)(*t.stride()[:3]) for t in (q, k, v, out)]
        rc = L.ksa_decode_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), None, None, 3, 690, 2, 8, 2, 1, D, 0,
                              *strides, D ** -0.5, nsplit, ws.data_ptr() + shift, need, _lib.stream_ptr(q.device))
        assert rc == 0 and torch.equal(out, want)
        assert (ws[:shift] == 0xff).all() and (ws[shift + need:] == 0xff).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("b,Hq,Hkv,Q,rows,nsplit", [(1, 32, 8, 1, 1, 1), (2, 16, 1, 1, 63, 1), (3, 8, 8, 1, 65, 2), (2, 10, 2, 3, 512, 1),
                                                    (1, 32, 8, 4, 513, 3), (5, 12, 4, 1, 1100, 5), (1, 4, 1, 1, 4500, 64)])
def test_decode_wide_workgroups(dtype, D, b, Hq, Hkv, Q, rows, nsplit):
    """Workgroups of eight waves of 64 rows: one row to several rounds, whole and cut tiles, waves and slices without rows, columns
    up to 16, a range per sequence (an empty one among them) on strided caches, against the oracle."""
    import ksa_amd  # noqa: F401
    g = torch.Generator().manual_seed(rows + D)
    q = torch.randn(b, Q, Hq, D, generator=g).to(dtype)
    kv = torch.randn(b, rows + 3, 2 * Hkv, D, generator=g).to(dtype)
    lo = np.array([(7 * i) % max(1, rows // 2) for i in range(b)], np.int32)
    hi = np.array([max(lo[i] + 1, rows - 61 * i) for i in range(b)], np.int32)
    if b == 5:
        hi[2] = lo[2]
    kvd = kv.cuda().transpose(1, 2)
    k, v = kvd[:, :Hkv, :rows], kvd[:, Hkv:, :rows]
    dev = lambda a: torch.as_tensor(a, device="cuda")
    got = torch.ops.ksa_amd.wide_decode_fwd(q.cuda().transpose(1, 2), k, v, dev(lo), dev(hi), 0, 0, D ** -0.5, nsplit)
    kept = np.maximum(hi, lo + 1)
    want = c_oracle.decode(to_np(q.transpose(1, 2)), to_np(kv.transpose(1, 2)[:, :Hkv]), to_np(kv.transpose(1, 2)[:, Hkv:]), lo, kept)
    if b == 5:
        want[2] = 0
    assert np.abs(to_np(got).reshape(want.shape) - want).max() <= ATOL * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,Hq,Hkv,D,Q,rows,nsplit", [(1, 4, 1, 128, 1, 1, 1), (2, 32, 8, 128, 1, 300, None), (1, 16, 1, 128, 1, 1100, 2),
                                                      (2, 10, 2, 64, 3, 512, 1), (1, 8, 2, 64, 1, 4500, 7), (1, 32, 8, 128, 1, 577, 1)])
def test_decode_wide_infinite_values(dtype, b, Hq, Hkv, D, Q, rows, nsplit):
    """An infinite value of an attended row is the outcome in its column, whatever its row - the first, the last, one in the
    middle of a cut tile - and of no other column; both signs in a column have no sum.  From the projection's sums as well."""
    import ksa_amd
    from ksa_amd import decode, gemm, pre
    g = torch.Generator().manual_seed(rows + D)
    rnd = lambda *s: torch.randn(*s, generator=g)
    q, k, v = rnd(b, Hq, Q, D).to(dtype), rnd(b, Hkv, rows, D).to(dtype), rnd(b, Hkv, rows, D).to(dtype)
    lo, hi = rows // 7, rows - rows // 9
    inf = float("inf")
    for col, row in ((0, lo), (5, hi - 1), (17, (lo + hi) // 2), (D - 1, lo)):
        v[:, :, row, col] = inf
    v[:, -1, hi - 1, 9] = v[:, 0, lo, 33] = -inf
    if hi - lo > 2:
        v[:, :, lo, 40], v[:, :, hi - 1, 40] = inf, -inf
    if rows > 9:
        v[:, :, lo - 1], v[:, :, hi] = inf, float("nan")     # outside of the range
    args = (q.cuda(), k.cuda(), v.cuda())
    got = ksa_amd.ksa_decode(*args, lo, hi) if nsplit is None else \
        torch.ops.ksa_amd.wide_decode_fwd(*args, None, None, lo, hi, D ** -0.5, nsplit)
    rep = lambda t: t[:, :, lo:hi].double().repeat_interleave(Hq // Hkv, 1)
    want = ((q.double() @ rep(k).transpose(-1, -2)) * D ** -0.5).softmax(-1) @ rep(v)
    want = want.transpose(1, 2)
    assert want.isinf().any() and (hi - lo <= 2 or want.isnan().any())
    torch.testing.assert_close(got.double().cpu(), want, rtol=0, atol=ATOL, equal_nan=True)
    if Q > 1:
        return
    # the new row somewhere in the range, its cache row holding what must not be read
    x, w = rnd(b, 1, 1536).to(dtype).cuda(), rnd((Hq + 2 * Hkv) * D, 1536).to(dtype).cuda()
    qkv, one = gemm.linear_rows(x, w, defer=True), torch.ones(D, dtype=dtype, device="cuda")
    cos, sin = (torch.full((1, 1, D), c, dtype=dtype, device="cuda") for c in (0.6, 0.8))
    kc, vc = args[1].clone(), args[2].clone()
    at = (lo + hi) // 2
    kc[:, :, at] = vc[:, :, at] = float("nan")
    kr, vr = kc.clone(), vc.clone()
    qr, _, _ = pre.pre_attention_partials(qkv, Hq, Hkv, D, one, one, cos, sin, 1e-6, k_out=kr[:, :, at:at + 1].transpose(1, 2),
                                          v_out=vr[:, :, at:at + 1].transpose(1, 2))
    n = nsplit or 1
    want = torch.ops.ksa_amd.wide_decode_fwd(qr.transpose(1, 2), kr, vr, None, None, lo, hi, D ** -0.5, n)
    got = decode.ksa_decode_qkv(qkv, one, one, cos, sin, 1e-6, kc, vc, Hq, at, lo, hi, nsplit=n, wide=True)
    torch.testing.assert_close(got.view(want.shape), want, rtol=0, atol=0, equal_nan=True)
    assert rows == 1 or want.isinf().any()


def test_decode_wide_workgroups_refuse_what_they_do_not_take():
    import ksa_amd  # noqa: F401
    from ksa_amd import _lib
    for Hq, D in ((17, 64), (4, 256), (4, 32)):
        q = torch.randn(1, Hq, 1, D, device="cuda").bfloat16()
        k = torch.randn(1, 1, 40, D, device="cuda").bfloat16()
        assert _lib.lib().ksa_decode_wide_splits(1, Hq, 1, 1, D, 40) == 0
        with pytest.raises(_lib.KsaError):
            torch.ops.ksa_amd.wide_decode_fwd(q, k, k, None, None, 0, 40, 0.1, 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,Hq,Hkv,D,N,nsplit", [
    (1, 32, 8, 128, 2560, None), (1, 32, 8, 128, 256, 1), (1, 16, 2, 128, 144, 39), (1, 8, 4, 64, 16, 64), (1, 64, 4, 64, 272, 2),
    (2, 32, 8, 128, 272, 32), (3, 8, 8, 64, 128, 21), (5, 4, 2, 128, 512, 7), (7, 16, 1, 128, 528, 3), (16, 32, 8, 128, 1024, 4),
    (8, 32, 8, 128, 2560, None), (16, 32, 8, 128, 2560, None),
])
def test_decode_qkv_o_wide_equals_separate_launches(dtype, b, Hq, Hkv, D, N, nsplit):
    """The wide form of a step's attention, alone and with the o projection in the launch, with ranges from one row to all (later
    slices empty) and new rows at every place of a tile, several launches on one workspace.  Attention: against the decode call on
    the rows of the pre-attention step, both in wide workgroups and bit for bit; with the o projection: the splits are merged in
    another order, bounds as for the four-wave form."""
    from ksa_amd import decode, gemm, pre
    import ksa_amd._lib as _lib
    rows = 4100 if nsplit is None or nsplit > 16 else 1100
    n = nsplit or _lib.lib().ksa_decode_qkv_o_wide_splits(b, Hq, Hkv, D, N, rows)
    assert n > 0
    g = torch.Generator(device="cuda").manual_seed(b * 10 + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    H, width, K = 1536, (Hq + 2 * Hkv) * D, Hq * D
    wo = (rnd(N, K) * K ** -0.5).to(dtype)
    tiled, ws = gemm.TiledWeight(wo), gemm.MlpRowsWorkspace(N, 64, torch.device("cuda"))
    qw, kw = (1 + 0.1 * rnd(D)).to(dtype), (1 + 0.1 * rnd(D)).to(dtype)
    ang = rnd(b, 1, D // 2)
    ang = torch.cat((ang, ang), -1)
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    w = (rnd(width, H) * H ** -0.5).to(dtype)
    forms = [(0, rows, rows - 1), (7, 1031, 7), (128, 129, 128), (3, 40, 20), (0, 300, 127), (1, 1000, 64 * 9 + 1)]
    dev = lambda v: torch.as_tensor(v, device="cuda", dtype=torch.int32)
    for rep in range(3):
        lo, hi, row = (dev([forms[(i + 2 * rep) % len(forms)][j] for i in range(b)]) for j in range(3))
        qkv = gemm.linear_rows(rnd(b, 1, H).to(dtype), w, defer=True)
        kc, vc = (rnd(b, Hkv, rows, D).to(dtype) for _ in range(2))
        for i in range(b):                             # what the new rows overwrite must not be read
            kc[i, :, row[i]] = vc[i, :, row[i]] = float("nan")
        kr, vr = kc.clone(), vc.clone()
        ko, vo = kc.clone(), vc.clone()
        q, _, _ = pre.pre_attention_partials(qkv, Hq, Hkv, D, qw, kw, cos, sin, 1e-6, k_out=kr[:, :, :1].transpose(1, 2),
                                             v_out=vr[:, :, :1].transpose(1, 2), kv_out_row=row)
        want = torch.ops.ksa_amd.wide_decode_fwd(q.transpose(1, 2), kr, vr, lo, hi, 0, 0, D ** -0.5, n)
        attn = decode.ksa_decode_qkv(qkv, qw, kw, cos, sin, 1e-6, kc, vc, Hq, row, lo, hi, nsplit=n, wide=True)
        assert torch.equal(attn, want.reshape(b, 1, K)) and torch.equal(kc, kr) and torch.equal(vc, vr)
        got = decode.ksa_decode_qkv_o(qkv, qw, kw, cos, sin, 1e-6, ko, vo, Hq, row, lo, hi, tiled, ws, nsplit=nsplit, wide=True)
        torch.cuda.synchronize()
        assert not ws.failed() and int(ws.step.view(torch.int64).abs().sum().item()) == 0
        assert torch.equal(ko, kr) and torch.equal(vo, vr)
        got = got.workspace.view(torch.float32).view(K // 512, 16, N)[:, :b].sum(0)
        want = attn.view(b, K).double() @ wo.double().t()
        ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        term = (attn.view(b, K).double().square() @ wo.double().t().square() / K).sqrt()
        assert ((got - want).abs() <= 2 * ulp * K ** 0.5 * term + 1e-5 * want.abs().max()).all()
        assert (got - want).square().mean() <= (0.25 * ulp) ** 2 * (K * term.square()).mean()


def test_decode_qkv_o_wide_bounded_wait_gives_up_and_recovers():
    """As for the four-wave form: counts set far off from the host, every wait ends, the cleared words serve the next launch."""
    from ksa_amd import decode, gemm
    g = torch.Generator(device="cuda").manual_seed(9)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    qkv = gemm.linear_rows(rnd(2, 1, 1024), rnd(8 * 128, 1024), defer=True)
    kc, vc, tiled = rnd(2, 2, 300, 128), rnd(2, 2, 300, 128), gemm.TiledWeight(rnd(256, 512))
    one, ws = torch.ones(128, device="cuda").bfloat16(), gemm.MlpRowsWorkspace(256, 64, torch.device("cuda"))
    call = lambda w: decode.ksa_decode_qkv_o(qkv, one, one, one, one, 1e-6, kc, vc, 4, 5, 0, 300, tiled, w, nsplit=2, wide=True)
    ws.step.view(torch.int64)[4 * 64::64] = -(1 << 40)
    torch.cuda.synchronize()
    call(ws)
    assert ws.failed() and not ws.failed()
    assert int(ws.step.view(torch.int64).abs().sum().item()) == 0
    a, b = call(ws), call(gemm.MlpRowsWorkspace(256, 64, torch.device("cuda")))
    assert not ws.failed()
    assert torch.equal(*(t.workspace.view(torch.float32).view(1, 16, 256)[:, :2] for t in (a, b)))
