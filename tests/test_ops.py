"""The helper operators as `torch.ops.ksa_amd.*` (`ksa_amd/ops.py`): registration and shape-only (fake)
kernels on the CPU; on the GPU each operator against the direct call (bit-identical: same kernel),
`torch.library.opcheck`, and a traced layer body (`torch.compile`, graph capture without code
generation) against the same body run eagerly.
"""
import pytest
import torch

H, I, HQ, HKV, D = 256, 512, 4, 2, 64


def _layer_weights(dev, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)

    def r(*shape, s=0.05):
        return (torch.randn(*shape, generator=g) * s).to(dtype).to(dev)

    return {"norm1": 1 + r(H), "norm2": 1 + r(H), "qkv": r((HQ + 2 * HKV) * D, H), "o": r(H, HQ * D),
            "gate_up": r(2 * I, H), "down": r(H, I), "qn": 1 + r(D), "kn": 1 + r(D)}


def _rope(rows, dev, dtype):
    pos = torch.arange(rows, dtype=torch.float32)
    inv = 1.0 / (10000 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    f = torch.outer(pos, inv)
    e = torch.cat((f, f), -1)
    return e.cos().to(dtype).to(dev)[None], e.sin().to(dtype).to(dev)[None]


def test_operators_registered_with_fake_kernels():
    import ksa_amd
    from torch._subclasses.fake_tensor import FakeTensorMode
    ns = torch.ops.ksa_amd
    for name in ksa_amd.ops.OPERATORS:
        assert hasattr(ns, name), name
    ks = ksa_amd.ops.mlp_rows_down_splits(H, I)
    with FakeTensorMode():
        bf = dict(dtype=torch.bfloat16, device="cuda")
        x = torch.empty(2, 4, H, **bf)
        w = torch.empty(H, **bf)
        s, y = ns.add_rmsnorm(x, x, w, 1e-6)
        assert s.shape == x.shape and y.shape == x.shape and y.dtype == torch.bfloat16 and y.device.type == "cuda"
        assert ns.rmsnorm(x, w, 1e-6).shape == x.shape
        qkv = ns.linear_rows(x, torch.empty((HQ + 2 * HKV) * D, H, **bf))
        assert qkv.shape == (2, 4, (HQ + 2 * HKV) * D)
        q = qkv[..., :HQ * D].view(2, 4, HQ, D)
        k = qkv[..., HQ * D:(HQ + HKV) * D].view(2, 4, HKV, D)
        cs = torch.empty(1, 4, D, **bf)
        qo, ko, vo = ns.pre_attention(q, k, k, torch.empty(D, **bf), torch.empty(D, **bf), cs, cs, 1e-6)
        assert qo.shape == q.shape and ko.shape == k.shape and vo.shape == k.shape
        assert ns.gate_up_silu_rows(x, torch.empty(2 * I, H, **bf)).shape == (2, 4, I)
        g = torch.empty(2, 4, I, **bf)
        assert ns.silu_mul(g, g).shape == g.shape
        part = ns.mlp_rows(x, torch.empty(2 * I, H, **bf), torch.empty(H, I, **bf),
                           torch.empty(64, dtype=torch.uint8, device="cuda"))
        assert part.shape == (ks, 16, H) and part.dtype == torch.float32
        s2, y2 = ns.add_rmsnorm_partials(part, x, w, 1e-6)
        assert s2.shape == x.shape and y2.dtype == torch.bfloat16
        am = ns.argmax_rows(torch.empty(2, 4, 1000, **bf))
        assert am.shape == (2, 4) and am.dtype == torch.long


def _layer_body(ka, x, res, W, cos, sin):
    """The element-wise and few-rows steps of one decoder layer around the attention call (which is left
    out: q stands in for its output), through the package-level functions."""
    res, h = ka.add_rmsnorm(x, res, W["norm1"], 1e-6)
    qkv = ka.linear_rows(h, W["qkv"])
    b, S = x.shape[:2]
    q = qkv[..., :HQ * D].view(b, S, HQ, D)
    k = qkv[..., HQ * D:(HQ + HKV) * D].view(b, S, HKV, D)
    v = qkv[..., (HQ + HKV) * D:].view(b, S, HKV, D)
    q, k, v = ka.pre_attention(q, k, v, W["qn"], W["kn"], cos, sin, 1e-6)
    o = ka.linear_rows(q.reshape(b, S, HQ * D), W["o"])
    res, h = ka.add_rmsnorm(o, res, W["norm2"], 1e-6)
    a = ka.silu_mul(ka.linear_rows(h, W["gate_up"]))
    return res, ka.linear_rows(a, W["down"]), k, v


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gpu_traced_layer_body_equals_eager(dtype):
    import ksa_amd
    dev = torch.device("cuda", 0)
    W = _layer_weights(dev, dtype)
    g = torch.Generator().manual_seed(1)
    x = torch.randn(2, 4, H, generator=g).to(dtype).to(dev)
    res = torch.randn(2, 4, H, generator=g).to(dtype).to(dev)
    cos, sin = _rope(4, dev, dtype)
    exp = _layer_body(ksa_amd, x, res, W, cos, sin)
    torch._dynamo.reset()
    seen = []

    def backend(gm, example_inputs):  # graph capture only: the captured graph is run as it is
        seen.extend(str(n.target) for n in gm.graph.nodes if n.op == "call_function")
        return gm.forward

    fn = torch.compile(lambda x, res, cos, sin: _layer_body(ksa_amd, x, res, W, cos, sin), backend=backend,
                       fullgraph=True)
    got = fn(x, res, cos, sin)
    for name in ("add_rmsnorm", "linear_rows", "pre_attention", "silu_mul"):
        assert any("ksa_amd." + name in t or "ksa_amd::" + name in t for t in seen), (name, seen)
    for a, b in zip(got, exp):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_gpu_operators_equal_direct_calls_and_opcheck():
    import ksa_amd
    from ksa_amd import elementwise, gemm, pre
    ns = torch.ops.ksa_amd
    dev = torch.device("cuda", 0)
    dtype = torch.bfloat16
    W = _layer_weights(dev, dtype, seed=2)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(8, H, generator=g).to(dtype).to(dev)
    res = torch.randn(8, H, generator=g).to(dtype).to(dev)
    cases = []
    # residual add + norm, norm alone
    s, y = ns.add_rmsnorm(x, res, W["norm1"], 1e-6)
    es, ey = elementwise.add_rmsnorm(x, res, W["norm1"], 1e-6)
    assert torch.equal(s, es) and torch.equal(y, ey)
    assert torch.equal(ns.rmsnorm(x, W["norm1"], 1e-6), elementwise.add_rmsnorm(x, None, W["norm1"], 1e-6)[1])
    cases.append((ns.add_rmsnorm, (x, res, W["norm1"], 1e-6)))
    cases.append((ns.rmsnorm, (x, W["norm1"], 1e-6)))
    # projections
    assert torch.equal(ns.linear_rows(x, W["qkv"]), gemm.linear_rows(x, W["qkv"]))
    assert torch.equal(ns.gate_up_silu_rows(x, W["gate_up"]), gemm.gate_up_silu_rows(x, W["gate_up"]))
    cases.append((ns.linear_rows, (x, W["qkv"])))
    cases.append((ns.gate_up_silu_rows, (x, W["gate_up"])))
    gu = gemm.linear_rows(x, W["gate_up"])
    assert torch.equal(ns.silu_mul(gu[:, :I], gu[:, I:]), elementwise.silu_mul(gu))
    cases.append((ns.silu_mul, (gu[:, :I], gu[:, I:])))
    # q/k norm + rotary
    qkv = gemm.linear_rows(x, W["qkv"]).view(2, 4, -1)
    q = qkv[..., :HQ * D].view(2, 4, HQ, D)
    k = qkv[..., HQ * D:(HQ + HKV) * D].view(2, 4, HKV, D)
    v = qkv[..., (HQ + HKV) * D:].view(2, 4, HKV, D)
    cos, sin = _rope(4, dev, dtype)
    for a, b in zip(ns.pre_attention(q, k, v, W["qn"], W["kn"], cos, sin, 1e-6),
                    pre.pre_attention(q, k, v, W["qn"], W["kn"], cos, sin, 1e-6)):
        assert torch.equal(a, b)
    cases.append((ns.pre_attention, (q, k, v, W["qn"], W["kn"], cos, sin, 1e-6)))
    # one-launch MLP and the norm that adds its partial sums: against the separate launches
    ws = ksa_amd.ops.mlp_rows_workspace(H, I, dev)
    part = ns.mlp_rows(x, W["gate_up"], W["down"], ws)
    s2, y2 = ns.add_rmsnorm_partials(part, res, W["norm2"], 1e-6)
    down = gemm.linear_rows(gemm.gate_up_silu_rows(x, W["gate_up"]), W["down"])
    es2, ey2 = elementwise.add_rmsnorm(down, res, W["norm2"], 1e-6)
    # (the partial sums are added in fp32 and rounded once, the separate launches round the product first)
    assert (s2.float() - es2.float()).abs().max() <= 2 ** -6 * es2.float().abs().max()
    assert (y2.float() - ey2.float()).abs().max() <= 2 ** -5 * ey2.float().abs().max()
    logits = torch.randn(8, 1000, generator=g).to(dtype).to(dev)
    assert torch.equal(ns.argmax_rows(logits), torch.argmax(logits, dim=-1))
    cases.append((ns.argmax_rows, (logits,)))
    for op, args in cases:
        torch.library.opcheck(op, args, test_utils=("test_schema", "test_faketensor"))
    # the workspace argument is declared as written to
    torch.library.opcheck(ns.mlp_rows, (x, W["gate_up"], W["down"], ws), test_utils=("test_schema", "test_faketensor"))
    assert int(ws[ksa_amd._lib.lib().ksa_mlp_rows_status_offset():][:8].view(torch.int64).item()) == 0


@pytest.mark.gpu
def test_direct_calls_step_aside_for_modes_and_subclasses():
    """`_lib.direct` decides whether an attention call goes past the dispatcher: not under a dispatch mode,
    not for tensor subclasses, not while gradients are asked for."""
    from torch.utils._python_dispatch import TorchDispatchMode

    import ksa_amd
    from ksa_amd import _lib

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    q = torch.randn(1, 40, 4, 64, device="cuda", dtype=torch.bfloat16)
    k, v = q[:, :, :2].contiguous(), q[:, :, 2:].contiguous()
    plain, _ = ksa_amd.summary_attn_func(q, k, v, 32, 4, 1)
    with Seen() as mode:
        assert not _lib.direct(q)
        moded, _ = ksa_amd.summary_attn_func(q, k, v, 32, 4, 1)
    assert any("summary_attn_fwd" in n for n in mode.names)
    assert torch.equal(plain, moded)
    assert _lib.direct(q, None) and not _lib.direct(torch.nn.Parameter(q))
    with torch.no_grad():
        assert _lib.direct(q.detach().requires_grad_())
    assert not _lib.direct(q.detach().requires_grad_())


@pytest.mark.gpu
def test_prefill_operators_refuse_what_they_do_not_take():
    """The operator of the block index knows the shapes of the library and no other, the one of the chunk tiles takes no
    built prefix and no layout outside of the library's rule; a call through each equals the direct call."""
    import ksa_amd
    from ksa_amd import _lib, prefill
    ns = torch.ops.ksa_amd
    g = torch.Generator(device="cuda").manual_seed(1)
    C, S, W, n = 128, 8, 1, 3 * 136 + 70
    q, k, v = (torch.randn(1, n, h, 64, generator=g, device="cuda").bfloat16() for h in (4, 2, 2))
    pos = torch.arange(n, device="cuda") % (C + S) >= C
    built = [torch.cat((t[:, pos], t), dim=1) for t in (k, v)]
    idx = prefill.compute_block_sparsity(n, n + 3 * S, C, S, W)
    for bad in (128, 1, -1):
        with pytest.raises(_lib.KsaError):
            ns.summary_attn_fwd(q, *built, *idx, C, S, W, 3 * S, False, True, 0.125, False, bad)
        with pytest.raises(_lib.KsaError):
            ksa_amd.summary_attn_func(q, *built, C, S, W, workgroup_shape=bad)
    with pytest.raises(AssertionError):
        ns.summary_attn_chunks_fwd(q, *built, C, S, W, False, 0.125, False)
    with pytest.raises(_lib.KsaError):
        ns.summary_attn_chunks_fwd(q, k, v, 100, S, W, False, 0.125, False)
    args = (q, k, v, C, S, W, False, 0.125, True)
    for got, want in zip(ns.summary_attn_chunks_fwd(*args), ksa_amd.summary_attn_func(*args[:6], pos, return_lse=True)):
        assert torch.equal(got, want)
    torch.library.opcheck(ns.summary_attn_chunks_fwd, args, test_utils=("test_schema", "test_faketensor"))


def test_direct_calls_step_aside_for_transforms_and_negative_views():
    """... nor inside `torch.func` transforms and function modes, nor for views whose negative bit is set."""
    from torch.overrides import TorchFunctionMode

    from ksa_amd import _lib

    seen = []

    def ask(a):
        seen.append(_lib.direct(a))
        return a * 1

    x = torch.randn(2, 3)
    torch.func.vmap(ask)(x)
    torch.func.jvp(ask, (x,), (x,))
    torch.func.functionalize(ask)(x)
    torch.func.grad(lambda a: ask(a).sum())(x)
    assert seen == [False] * 4

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not _lib.direct(x)
    assert _lib.direct(x)
    neg = torch.complex(x, x).conj().imag
    assert neg.is_neg() and not _lib.direct(neg)


def test_direct_calls_step_aside_for_profilers():
    """Operators are seen by name in a profiler's trace."""
    from ksa_amd import _lib
    x = torch.randn(2, 3)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        assert not _lib.direct(x)
    with torch.autograd.profiler.profile():
        assert not _lib.direct(x)
    assert _lib.direct(x)


def test_direct_calls_step_aside_for_tensors_without_memory():
    """Wrappers and zero tensors have the plain type and no memory that a kernel could be given."""
    from ksa_amd import _lib
    x = torch.randn(2, 3)
    assert not _lib.direct(torch._to_functional_tensor(x))
    assert not _lib.direct(x, torch._efficientzerotensor((2, 3)))
    assert _lib.direct(x, x)


def test_calls_without_torchs_private_functions(monkeypatch):
    """Where torch lacks one of the private functions in use, every call takes the dispatcher."""
    from ksa_amd import _lib
    x = torch.randn(2, 3)
    assert _lib.direct(x)
    with monkeypatch.context() as m:
        m.delattr(torch._C, "_len_torch_function_stack")
        assert _lib._private("_C._len_torch_dispatch_stack", "_C._len_torch_function_stack") is None
        m.setattr(_lib, "_WATCHERS", None)
        assert not _lib.direct(x)
    assert _lib.direct(x)


@pytest.mark.gpu
@pytest.mark.parametrize("known", [True, False])
def test_stream_and_device_without_torchs_private_functions(monkeypatch, known):
    """The handle of the current stream, and no device to change to, with and without the private functions."""
    from ksa_amd import _lib
    if not known:
        monkeypatch.setattr(_lib, "_GPU", None)
    for s in (torch.cuda.current_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(s):
            for device in (torch.device("cuda"), torch.device("cuda", 0)):
                assert _lib.stream_ptr(device) == s.cuda_stream
                with _lib.on_device(device):
                    assert torch.cuda.current_device() == 0


@pytest.mark.gpu
def test_decode_row_ranges_that_are_wrappers():
    """A row range of a subclass reaches the operator like the other inputs."""
    import ksa_amd

    class Ranges(torch.Tensor):
        names = []

        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            Ranges.names.append(str(func))
            return super().__torch_function__(func, types, args, kwargs or {})

    q = torch.randn(2, 4, 1, 64, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(2, 2, 300, 64, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    lo, hi = (torch.full((2,), n, dtype=torch.int32, device="cuda") for n in (3, 290))
    got = ksa_amd.ksa_decode(q, k, v, lo.as_subclass(Ranges), hi)
    assert any("decode_fwd" in n for n in Ranges.names)
    assert torch.equal(got.as_subclass(torch.Tensor), ksa_amd.ksa_decode(q, k, v, lo, hi))


@pytest.mark.gpu
def test_prefill_under_vmap():
    """Attention calls inside `torch.func.vmap` equal one call per slice."""
    import ksa_amd
    q = torch.randn(2, 1, 40, 4, 64, device="cuda", dtype=torch.bfloat16)
    k, v = q[:, :, :, :2].contiguous(), q[:, :, :, 2:].contiguous()
    f = lambda a, b, c: ksa_amd.summary_attn_func(a, b, c, 32, 4, 1)[0]
    got = torch.func.vmap(f)(q, k, v)
    assert torch.equal(got, torch.stack([f(q[i], k[i], v[i]) for i in range(2)]))


class _Front:
    """`_lib.fast` with a record of which calls it took (`general`: takes none)."""

    def __init__(self, real, general=False):
        self.real, self.general, self.took = real, general, []

    def __getattr__(self, name):
        def call(*args):
            out = None if self.general else getattr(self.real, name)(*args)
            self.took.append(out is not None)
            return out
        return call


def _front_calls():
    """(name, whether the native front takes the call, the call) over the forms of the four functions."""
    import ksa_amd
    g = torch.Generator(device="cuda").manual_seed(0)
    rnd = lambda dt, *s: torch.randn(*s, generator=g, device="cuda").to(dt)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    for dt in (torch.bfloat16, torch.float16):
        for D, taken in ((64, True), (128, True), (256, True), (72, False)):
            q, kc, vc = rnd(dt, 3, 8, 1, D), rnd(dt, 3, 2, 300, D), rnd(dt, 3, 2, 300, D)
            q9 = rnd(dt, 3, 9, 8, D).transpose(1, 2)
            wide = rnd(dt, 3, 300, 4, D).transpose(1, 2)   # rows and heads in the other order, keys next to values
            dec = ksa_amd.ksa_decode
            yield "decode", taken, lambda: dec(q, kc, vc)
            yield "decode ints", taken, lambda: dec(q, kc, vc, 7, 233)
            yield "decode views", taken, lambda: dec(q9, wide[:, :2, 5:299], wide[:, 2:, 5:299], scale=0.1)
            yield "decode ranges", taken, lambda: dec(q, kc, vc, i32(0, 3, 299), i32(300, 4, 300), nsplit=3)
            yield "decode one range", False, lambda: dec(q, kc, vc, None, i32(300, 4, 17))
            yield "decode strided range", False, lambda: dec(q, kc, vc, i32(0, 9, 3, 9, 2, 9)[::2], i32(300, 4, 17))
            yield "decode long range", False, lambda: dec(q, kc, vc, i32(0, 3, 2).long(), i32(300, 4, 17))
            yield "decode scale", False, lambda: dec(q, kc, vc, scale=-0.1)
            yield "decode int scale", False, lambda: dec(q, kc, vc, scale=1)
            yield "decode strided q", False, lambda: dec(q.repeat(1, 1, 1, 2)[..., ::2], kc, vc)
            n = 3 * 136 + 71
            pos = torch.arange(n, device="cuda") % 136 >= 128
            odd = pos.roll(1)
            qkv = rnd(dt, 2, n, 8, D)
            a = (qkv[:, :, :4], qkv[:, :, 4:6], qkv[:, :, 6:])
            own = tuple(t.contiguous() for t in a)
            sa = ksa_amd.summary_attn_func
            yield "prefill", taken, lambda: sa(*a, 128, 8, 1, pos, return_lse=True)
            yield "prefill own", taken, lambda: sa(*own, 128, 8, 2, summary_pos=pos, skip_old_summary=True)
            yield "prefill no prefix", taken, lambda: sa(*own, 128, 8, 2, softmax_scale=0.2)
            yield "prefill other chunk", False, lambda: sa(*own, 64, 8, 2)
            yield "prefill grid", False, lambda: sa(*own, 128, 8, 2, pos, chunk_tiles=False)
            yield "prefill shape", False, lambda: sa(*own, 128, 8, 2, pos, workgroup_shape=32)
            yield "prefill other mask", False, lambda: sa(*own, 128, 8, 2, odd)
            yield "prefill strides", False, lambda: sa(a[0], a[1], own[2], 128, 8, 2, pos)
            yield "prefill built prefix", False, lambda: sa(own[0], *(torch.cat((t[:, pos], t), 1) for t in own[1:]), 128, 8, 2)
            if D in (64, 128):
                w = [torch.nn.Parameter(rnd(dt, D)) for _ in range(2)]
                cos, sin = rnd(dt, 1, n, D), rnd(dt, 1, n, D)
                pre = ksa_amd.pre_attention
                cache = lambda: [torch.zeros(2, 2, n + 9, D, dtype=dt, device="cuda") for _ in range(2)]

                def into(rows, S):
                    c = cache()
                    o = [t[:, :, :S].transpose(1, 2) for t in c]
                    return pre(*(t[:, :S] for t in a), *w, cos[:, :S].contiguous(), sin[:, :S].contiguous(), 1e-5, k_out=o[0],
                               v_out=o[1], kv_out_row=rows)[:1] + tuple(c)
                yield "pre", True, lambda: pre(*a, *w, cos, sin)
                yield "pre rope per sequence", True, lambda: pre(*own, *w, cos.repeat(2, 1, 1), sin.repeat(2, 1, 1), 1e-4)
                yield "pre rows", True, lambda: into(i32(3, 0), 5)
                yield "pre row per token", True, lambda: into(i32(3, 0, 9, 5, 5, 1, 2, 7).view(2, 4)[:, :3].contiguous(), 3)
                yield "pre into", True, lambda: into(None, n)
                yield "pre 2-d rope", False, lambda: pre(*a, *w, cos[0], sin[0])
                yield "pre fp32 rope", False, lambda: pre(*a, *w, cos.float(), sin)
    for args in ((400, 400, 128, 8, 2), (409, 433, 128, 8, 0, True), (1000, 1056, 100, 7, 3, False, 64, 32)):
        yield "index", True, lambda: ksa_amd.compute_block_sparsity(*args)
    yield "index device", False, lambda: ksa_amd.compute_block_sparsity(400, 400, 128, 8, 2, device="cuda:0")


@pytest.mark.gpu
def test_native_front_equals_general_way(monkeypatch):
    """Every form of the four calls: taken where it should be, and the same tensors (values, shapes, strides) either way."""
    from ksa_amd import _lib
    real = _lib.fast
    flat = lambda o: [t for t in (o if isinstance(o, tuple) else (o,)) if t is not None]
    for name, taken, call in _front_calls():
        front = _Front(real)
        monkeypatch.setattr(_lib, "fast", front)
        got = flat(call())
        assert front.took == [True] if taken else not any(front.took), name
        monkeypatch.setattr(_lib, "fast", _Front(real, general=True))
        want = flat(call())
        assert len(got) == len(want), name
        for x, y in zip(got, want):
            assert torch.equal(x, y) and x.stride() == y.stride() and x.dtype == y.dtype, name


@pytest.mark.gpu
def test_native_front_steps_aside():
    """... for everybody whom `_lib.direct` steps aside for, for other devices and types, and for arguments out of range."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from ksa_amd import _lib
    q = torch.randn(2, 4, 1, 64, device="cuda", dtype=torch.bfloat16)
    kc, vc = (torch.randn(2, 2, 40, 64, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    ask = lambda a=q, k=kc, v=vc, *r: _lib.fast.decode(a, k, v, *(r or (None, None, None, None))) is not None
    assert ask()
    assert not ask(q.cpu()) and not ask(q.float()) and not ask(q.half()) and not ask(torch.nn.Parameter(q)) and not ask(q[0])
    assert not ask(q.detach().requires_grad_()) and not ask(q, kc[:, :, :39]) and not ask(q, kc[:1], vc[:1])
    assert not ask(q[:, :3]) and not ask(q[:0], kc[:0], vc[:0])
    with torch.no_grad():
        assert ask(q.detach().requires_grad_())
    for r in ((-1, 9, None, None), (9, 9, None, None), (0, 41, None, None), (0.0, 9, None, None), (None, None, 0.0, None),
              (None, None, float("nan"), None), (None, None, None, -1), (None, None, None, 0)):
        assert not ask(q, kc, vc, *r), r
    seen = []

    def note(a):
        seen.append(ask(a))
        return a * 1
    torch.func.vmap(lambda a: (seen.append(_lib.fast.decode(a, kc, vc, None, None, None, None) is not None), a)[1])(q[None])
    torch.func.jvp(note, (q,), (q,))
    torch.func.functionalize(note)(q)
    torch.func.grad(lambda a: note(a).sum())(q)
    with torch.autograd.forward_ad.dual_level():
        note(torch.autograd.forward_ad.make_dual(q, q))

    class Fn(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Op(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    for context in (Fn(), Op(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]),
                    torch.autograd.profiler.profile()):
        with context:
            note(q)
    note(torch._to_functional_tensor(q))
    note(torch._efficientzerotensor((2, 4, 1, 64), dtype=q.dtype, device="cuda"))
    assert len(seen) == 11 and not any(seen), seen
    assert ask()


@pytest.mark.gpu
@pytest.mark.parametrize("code", [-5, -1])
def test_native_front_never_launches_twice(code):
    """An error that the library reports behind a launch (-5) is raised: the kernel may have run, on outputs that may be the
    inputs, so the general way must not run it again.  What the library refuses in front of its launch goes that way."""
    import ctypes

    import ksa_amd
    from ksa_amd import _lib
    L = _lib.lib()
    rnd = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    q, kc, vc = rnd(2, 8, 1, 64), rnd(2, 2, 300, 64), rnd(2, 2, 300, 64)
    p, k, v, w, rope = rnd(1, 200, 8, 128), rnd(1, 200, 2, 128), rnd(1, 200, 2, 128), rnd(128), rnd(1, 200, 128)
    qo, ko, vo = (torch.zeros_like(t) for t in (p, k, v))
    calls = {
        "ksa_decode_wide_fwd": lambda: ksa_amd.ksa_decode(q, kc, vc),
        "ksa_decode_fwd": lambda: ksa_amd.ksa_decode(q, kc, vc, nsplit=2),
        "ksa_prefill_chunks_fwd": lambda: ksa_amd.summary_attn_func(p, k, v, 128, 8, 1)[0],
        "ksa_pre_attention": lambda: ksa_amd.pre_attention(p, k, v, w, w, rope, rope, q_out=qo, k_out=ko, v_out=vo)[0],
        "ksa_block_index": lambda: ksa_amd.compute_block_sparsity(400, 400, 128, 8, 2)[1],
    }
    address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
    seen = []

    @ctypes.CFUNCTYPE(ctypes.c_int)
    def stub():                       # (launches nothing; its arguments are the caller's to clear)
        seen.append(code)
        return code
    for name, call in calls.items():
        want = call().clone()
        qo.zero_()
        seen.clear()
        _lib.fast.bind(_lib.check, *(address(stub if n == name else getattr(L, n)) for n in _lib._FAST))
        try:
            if code == -5:
                with pytest.raises(_lib.KsaError, match=name):
                    call()
                assert not qo.any()
            else:
                assert torch.equal(call(), want)
        finally:
            _lib.fast.bind(_lib.check, *(address(getattr(L, n)) for n in _lib._FAST))
        assert seen == [code], name
        assert torch.equal(call(), want)


@pytest.mark.gpu
def test_native_front_allocates_nothing_for_what_it_leaves():
    """Calls that the library refuses - addresses and strides off the 16-byte grid, head dimensions, arguments out
    of range - are left to the general way in front of the first allocation."""
    from ksa_amd import _lib
    rnd = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    shifted = lambda *s: rnd(torch.Size(s).numel() + 4)[4:].view(s)          # 8 bytes off
    odd = lambda *s: rnd(*s[:-1], s[-1] + 4)[..., :s[-1]]                    # rows 8 bytes off each other
    q, kc, vc = rnd(2, 4, 1, 64), rnd(2, 2, 40, 64), rnd(2, 2, 40, 64)
    f = _lib.fast
    dec = lambda a=q, k=kc, v=vc, n=None: f.decode(a, k, v, None, None, None, n)
    p, k, v = rnd(1, 200, 4, 64), rnd(1, 200, 2, 64), rnd(1, 200, 2, 64)
    pre_ = lambda a=p, k=k, v=v, w=rnd(64), c=rnd(1, 200, 64), e=1e-6, o=None: f.pre_attention(a, k, v, w, w, c, c, e, o, None, None, None)
    sa = lambda a=p, k=k, v=v: f.prefill(a, k, v, 128, 8, 1, False, None, False, None, None)
    p256 = [rnd(1, 200, n, 256) for n in (4, 2, 2)]
    w256, c256 = rnd(256), rnd(1, 200, 256)
    args = [shifted(2, 4, 1, 64), odd(2, 4, 1, 64), shifted(2, 2, 40, 64), odd(2, 2, 40, 64), shifted(1, 200, 4, 64), odd(1, 200, 4, 64),
            shifted(1, 200, 2, 64), odd(1, 200, 2, 64), shifted(64), shifted(1, 200, 64)]
    for call in (dec, pre_, sa, lambda: f.block_index(400, 400, 128, 8, 2, False, 128, 64)):
        assert call() is not None
    left = [lambda: dec(args[0]), lambda: dec(args[1]), lambda: dec(k=args[2]), lambda: dec(v=args[3]), lambda: dec(n=0),
            lambda: sa(args[4]), lambda: sa(args[5]), lambda: sa(k=args[6], v=args[6]), lambda: sa(k=args[7], v=args[7]),
            lambda: pre_(args[4]), lambda: pre_(args[5]), lambda: pre_(k=args[6]), lambda: pre_(v=args[7]), lambda: pre_(w=args[8]),
            lambda: pre_(c=args[9]), lambda: pre_(e=-1.0), lambda: pre_(e=float("nan")), lambda: pre_(o=args[4]),
            lambda: pre_(*p256, w=w256, c=c256), lambda: f.block_index(400, 400, 0, 8, 2, False, 128, 64),
            lambda: f.block_index(400, 400, 128, 8, -1, False, 128, 64)]
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    for i, call in enumerate(left):
        before = count()
        assert call() is None and count() == before, i
