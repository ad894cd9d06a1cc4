"""Fused residual-add + RMSNorm and SiLU-mul kernels against the reference's op sequence.

Oracle: `oracle/cpu_path.add_rmsnorm` / `silu_mul` = the reference's torch ops
(examples/pretrain/hf_template/modeling_qwen3sa.py:64-79, :507-514, :946, :952) on the CPU in the
input dtype.  Pins of the oracle (CPU tests): an fp64 closed form, scale invariance of the norm,
SiLU special values.  GPU tests: bit-identical to the oracle except where the fp32 summation
order / the exponential differ in the last place: at most 0.5 % of the elements, each by one
unit in the last place of the rounded intermediate (at most two of the result).
"""
import pytest
import torch

from oracle import cpu_path


def test_oracle_rmsnorm_closed_form():
    g = torch.Generator().manual_seed(0)
    x = torch.randn(5, 96, generator=g, dtype=torch.float64)
    r = torch.randn(5, 96, generator=g, dtype=torch.float64)
    w = torch.randn(96, generator=g, dtype=torch.float64)
    s, y = cpu_path.add_rmsnorm(x.float(), r.float(), w.float(), 1e-6)
    t = x + r
    exp = w * t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6)
    assert torch.allclose(s.double(), t, atol=1e-6)
    assert torch.allclose(y.double(), exp, atol=1e-5, rtol=1e-5)
    # scale invariance (eps aside): norm(4 x) == norm(x)
    _, y4 = cpu_path.add_rmsnorm(4 * x.float(), None, w.float(), 0.0)
    _, y1 = cpu_path.add_rmsnorm(x.float(), None, w.float(), 0.0)
    assert torch.allclose(y4, y1, atol=1e-5, rtol=1e-5)


def test_oracle_silu_values():
    gate = torch.tensor([0.0, 1.0, -1.0, 20.0, -20.0])
    up = torch.tensor([3.0, 2.0, 2.0, 1.0, 1.0])
    out = cpu_path.silu_mul(gate, up)
    e = torch.tensor(1.0).exp()
    exp = torch.tensor([0.0, 2.0 / (1 + 1 / e), -2.0 / (1 + e), 20.0, -20.0 * torch.tensor(-20.0).exp()])
    assert torch.allclose(out, exp, atol=1e-6, rtol=1e-5)


def _ulp_check(got, exp, max_frac):
    got, exp = got.cpu(), exp.cpu()
    diff = got != exp
    frac = diff.float().mean().item()
    if diff.any():
        a, b = got[diff].float(), exp[diff].float()
        mag = torch.maximum(a.abs(), b.abs())
        emin, mant = (-126, 7) if got.dtype == torch.bfloat16 else (-14, 10)   # subnormals share one spacing
        ulp = torch.exp2(torch.floor(torch.log2(mag.clamp_min(1e-38))).clamp_min(emin) - mant)
        # one unit in the last place of the normalised value can be two of the product with the
        # weight when the product falls into the binade below
        assert ((a - b).abs() <= 2 * ulp * 1.001).all(), "a mismatch larger than two units in the last place"
    assert frac <= max_frac, f"{frac:.4%} of the elements differ"
    return frac


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,H", [(1, 64), (7, 2560), (33, 4096), (5, 8192), (300, 520)])
@pytest.mark.parametrize("with_res", [True, False])
def test_gpu_add_rmsnorm(dtype, rows, H, with_res):
    from ksa_amd.elementwise import add_rmsnorm
    g = torch.Generator().manual_seed(rows * 31 + H)
    x = (torch.randn(2, rows, H, generator=g) * 1.5).to(dtype)
    r = torch.randn(2, rows, H, generator=g).to(dtype) if with_res else None
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(dtype)
    s_exp, y_exp = cpu_path.add_rmsnorm(x, r, w, 1e-6)
    s, y = add_rmsnorm(x.cuda(), r.cuda() if with_res else None, w.cuda(), 1e-6)
    assert torch.equal(s.cpu(), s_exp), "the residual sum must be bit-exact"
    _ulp_check(y, y_exp, 5e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H", [8, 512, 520, 2048, 2056, 2552, 2560, 2568, 4104, 8192])
def test_gpu_add_rmsnorm_row_lengths_in_place(dtype, H):
    """The items of a row are requested together, lanes past its end its last one: lengths around every count of items per
    lane, the sum written over the residual."""
    from ksa_amd import _lib
    rows = 5
    g = torch.Generator().manual_seed(H)
    x = (torch.randn(rows, H, generator=g) * 1.5).to(dtype)
    r = torch.randn(rows, H, generator=g).to(dtype)
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(dtype)
    s_exp, y_exp = cpu_path.add_rmsnorm(x, r, w, 1e-6)
    buf = torch.full((rows + 1, H), 3.0, dtype=dtype, device="cuda")
    buf[:rows] = r
    y = torch.full((rows + 1, H), 3.0, dtype=dtype, device="cuda")
    xd, wd = x.cuda(), w.cuda()
    _lib.check(_lib.lib().ksa_add_rmsnorm(xd.data_ptr(), buf.data_ptr(), wd.data_ptr(), y.data_ptr(), buf.data_ptr(), rows, H, H, H,
                                          H, H, 0 if dtype == torch.bfloat16 else 1, 1e-6, _lib.stream_ptr(xd.device)), "add_rmsnorm")
    assert torch.equal(buf[:rows].cpu(), s_exp)
    assert bool((buf[rows] == 3.0).all()) and bool((y[rows] == 3.0).all())
    _ulp_check(y[:rows], y_exp, 5e-3)


@pytest.mark.gpu
def test_gpu_add_rmsnorm_strided_rows_and_errors():
    from ksa_amd import KsaError
    from ksa_amd.elementwise import add_rmsnorm
    big = torch.randn(6, 3 * 256, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    x = big[:, 256:512]                       # row stride 768
    w = torch.ones(256, dtype=torch.bfloat16, device="cuda")
    _, y = add_rmsnorm(x, None, w)
    _, y_exp = cpu_path.add_rmsnorm(x.cpu(), None, w.cpu())
    _ulp_check(y, y_exp, 5e-3)
    with pytest.raises(KsaError):
        add_rmsnorm(torch.zeros(2, 12, dtype=torch.bfloat16, device="cuda"), None,
                    torch.ones(12, dtype=torch.bfloat16, device="cuda"))      # H not a multiple of 8
    with pytest.raises(KsaError):
        add_rmsnorm(torch.zeros(2, 16384, dtype=torch.bfloat16, device="cuda"), None,
                    torch.ones(16384, dtype=torch.bfloat16, device="cuda"))   # H above the supported size


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,I", [(1, 8), (9, 9728), (130, 2056)])
def test_gpu_silu_mul(dtype, rows, I):
    from ksa_amd.elementwise import silu_mul
    g = torch.Generator().manual_seed(rows + I)
    gu = (torch.randn(rows, 2 * I, generator=g) * 3).to(dtype)
    gate, up = gu[:, :I], gu[:, I:]            # halves of one fused projection output
    exp = cpu_path.silu_mul(gate, up)
    gug = gu.cuda()
    got = silu_mul(gug[:, :I], gug[:, I:])
    _ulp_check(got, exp, 5e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,N", [(8, 151936), (1, 8), (3, 1000), (5, 8192 + 3), (16, 5)])
def test_gpu_argmax_rows(dtype, rows, N):
    """The greedy token choice against torch.argmax on the CPU (first index among equal values:
    16-bit logits tie often), with the row maximum planted at both ends, inside a tail that is
    shorter than one 16-byte item, and doubled."""
    from ksa_amd.elementwise import argmax_rows
    g = torch.Generator().manual_seed(rows * 1000 + N)
    Np = (N + 7) // 8 * 8
    x = torch.randn(rows, Np, generator=g).to(dtype)[:, :N]   # rows start 16-byte aligned
    x[0, N - 1] = 30.0
    if rows > 1:
        x[1, 0] = 30.0
    if rows > 2:
        x[2, N // 2] = 30.0
        x[2, N - 1] = 30.0                                    # the first of two equal maxima wins
    def dev(t):  # same padded row stride on the GPU (a plain .cuda() would pack the rows)
        buf = torch.zeros(rows, Np, dtype=dtype, device="cuda")
        buf[:, :N] = t
        return buf[:, :N]

    got = argmax_rows(dev(x)).cpu()
    want = x.float().argmax(-1)
    assert got.dtype == torch.long and torch.equal(got, want), (got, want)
    if rows > 3 and N > 20:
        x[3, 17] = float("nan")                               # a NaN counts as the largest value
        assert int(argmax_rows(dev(x))[3]) == 17 == int(x.float().argmax(-1)[3])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", [9, 8192, 81920, 81928, 163851])
def test_gpu_argmax_rows_ties_and_special_values(dtype, N):
    """Equal maxima in every place of the scan (batches of 81920 values, items of 8, the values behind the
    last item), rows of one value, -inf, zeros of both signs, and NaNs of both signs: first index, as torch."""
    from ksa_amd.elementwise import argmax_rows
    g = torch.Generator().manual_seed(N)
    Np = (N + 7) // 8 * 8
    x = torch.randn(8, Np, generator=g).to(dtype)
    places = sorted({0, 7, 8, N // 2, N - 2, N - 1, min(N, 81919), min(N - 1, 81920), min(N - 1, 1024 * 8)} & set(range(N)))
    for i, first in enumerate((0, 1, len(places) // 2)):
        x[i, places[first:]] = 40.0
    x[3] = float("-inf")
    x[4] = -1.5
    x[5] = -torch.rand(Np, generator=g).to(dtype) - 1
    x[5, places[1]] = -0.0
    x[5, places[-1]] = 0.0
    x[6, places[-1]] = float("nan")
    x[6, places[1]] = -float("nan")
    x[6, 0] = float("inf")
    x[7, N - 1] = float("inf")
    got = argmax_rows(x.cuda()[:, :N]).cpu()
    assert torch.equal(got, x[:, :N].float().argmax(-1))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,H,vocab,D", [(1, 64, 9, 64), (3, 2560, 1000, 128), (4, 520, 50, 256), (8, 8192, 40, 8),
                                            (129, 4096, 300, 128)])
def test_gpu_embed_rmsnorm_equals_separate_launches(dtype, rows, H, vocab, D):
    """The head of a step against embedding lookup, norm and row choice, bit for bit; a table with padded rows."""
    from ksa_amd.elementwise import add_rmsnorm, embed_rmsnorm
    g = torch.Generator(device="cuda").manual_seed(rows + H)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    table, w, rope = rnd(vocab, H + 8)[:, :H], rnd(H), rnd(70, 2, D)
    ids = torch.randint(-vocab, vocab, (rows, 1), generator=g, device="cuda")
    ids[0], ids[-1] = vocab - 1, -vocab
    for at in (0, 69):
        x, h, r = (torch.full(s, 7.0, dtype=dtype, device="cuda") for s in ((rows, 1, H), (rows, 1, H), (1, 2, D)))
        embed_rmsnorm(table, ids, w, 1e-6, rope, torch.tensor([at], dtype=torch.int32, device="cuda"), x, h, r)
        s, n = add_rmsnorm(table[ids], None, w, 1e-6)
        assert torch.equal(x, s) and torch.equal(h, n) and torch.equal(r[0], rope[at])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gpu_embed_rmsnorm_ids_outside_the_table(dtype):
    """An id outside the table gives a row of NaN, normalised or not, and leaves the other rows alone; a rotary row
    outside of its table is the nearest one of it."""
    from ksa_amd.elementwise import add_rmsnorm, embed_rmsnorm
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    vocab, H, D = 50, 2560, 128
    table, w, rope = rnd(vocab, H), rnd(H), rnd(70, 2, D)
    ids = torch.tensor([[3], [vocab], [-vocab - 1], [49], [2**40], [-2**62], [-50]], device="cuda")
    bad = torch.tensor([False, True, True, False, True, True, False])
    for at, row in ((70, 69), (2**31 - 1, 69), (-1, 0)):
        x, h, r = (torch.full(s, 7.0, dtype=dtype, device="cuda") for s in ((7, 1, H), (7, 1, H), (1, 2, D)))
        embed_rmsnorm(table, ids, w, 1e-6, rope, torch.tensor([at], dtype=torch.int32, device="cuda"), x, h, r)
        assert torch.equal(r[0], rope[row])
        for t in (x, h):
            assert t[bad].isnan().all() and t[~bad].isfinite().all()
        s, n = add_rmsnorm(table[ids[~bad]], None, w, 1e-6)
        assert torch.equal(x[~bad], s) and torch.equal(h[~bad], n)


def test_embed_rmsnorm_argument_checks():
    """What the head-of-step kernel does not take is refused on the host."""
    from ksa_amd import _lib
    base = dict(table=16, vocab=10, stride=64, ids=8, w=16, out=16, norm=16, rows=2, H=64, rope=16, rr=4, rw=16, row=4, ro=16,
                dt=0, eps=1e-6, st=None)
    call = lambda **kw: _lib.lib().ksa_embed_rmsnorm(*{**base, **kw}.values())
    for bad in (dict(table=None), dict(ids=None), dict(row=None), dict(rows=0), dict(H=60), dict(H=8200), dict(vocab=0),
                dict(rr=0), dict(rw=12), dict(table=24), dict(stride=60), dict(ro=8), dict(dt=5), dict(eps=-1.0)):
        assert call(**bad) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ksplit", [1, 8, 9, 19, 20, 21, 40, 41, 64])
@pytest.mark.parametrize("rows,H", [(1, 2560), (17, 4096), (3, 4104)])
def test_gpu_add_rmsnorm_partials_slice_counts(dtype, ksplit, rows, H):
    """Slice counts around the batches in which they are requested: the residual sum is bit for bit that of the
    slices added in order, the norm within one rounding."""
    from ksa_amd.elementwise import add_rmsnorm
    from ksa_amd.gemm import SplitKPartials
    g = torch.Generator().manual_seed(ksplit * 100 + rows)
    part = torch.randn(ksplit, (rows + 15) // 16 * 16, H, generator=g) * ksplit ** -0.5
    acc = torch.zeros(rows, H)
    for s in part:
        acc = acc + s[:rows]
    r = torch.randn(rows, H, generator=g).to(dtype)
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(dtype)
    x = SplitKPartials(part.cuda().view(-1).view(torch.uint8), ksplit, rows, (rows, H), dtype)
    s, y = add_rmsnorm(x, r.cuda(), w.cuda(), 1e-6)
    s_exp, y_exp = cpu_path.add_rmsnorm(acc.to(dtype), r, w, 1e-6)
    assert torch.equal(s.cpu(), s_exp)
    _ulp_check(y, y_exp, 5e-3)
