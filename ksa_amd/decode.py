"""Decode attention over the contiguous ring-buffer KV slice on MI355X.

`decode_attention_forward` has the signature of the reference's `_decode_attn_fn`
(examples/pretrain/hf_template/modeling_qwen3sa.py:591-612 `_sdpa_attention_forward`,
selected at :643-646 and called at :820-830, :844-870): un-masked, non-causal
soft-max attention of `query [b, Hq, q_len, D]` over `key/value [b, Hkv, L, D]`
(strided views of the cache), GQA by `module.num_key_value_groups`, returning
`(attn_output [b, q_len, Hq, D], None)`.  `ksa_decode` is the lower-level form that
takes the whole cache tensor and per-sequence row ranges, which the reference cannot
express (its cache counters are shared by the batch, :753-754).
"""
from __future__ import annotations

import ctypes
from typing import Optional, Tuple

import torch

from . import _lib
from .prefill import fold_scale, kernel_head_dim, pad_head_dim

_DTYPES = {torch.bfloat16: 0, torch.float16: 1}


def _launch_decode(q, kcache, vcache, start, end, start0, end0, scale, nsplit, wide=False):
    b, Hq, Q, D = q.shape
    Hkv = kcache.shape[1]
    dev = q.device
    lib = _lib.lib()
    out = torch.empty((b, Q, Hq, D), dtype=q.dtype, device=dev)
    ws = None
    ws_bytes = 0
    if nsplit > 1:
        ws_bytes = lib.ksa_decode_workspace_bytes(b, Hq, Hkv, Q, D, nsplit)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    dims = (0, 1, 2)
    with _lib.on_device(dev):
        rc = (lib.ksa_decode_wide_fwd if wide else lib.ksa_decode_fwd)(
            q.data_ptr(), kcache.data_ptr(), vcache.data_ptr(), out.data_ptr(),
            start.data_ptr() if start is not None else None,
            end.data_ptr() if end is not None else None, start0, end0,
            b, Hq, Hkv, Q, D, _DTYPES[q.dtype],
            _lib.strides3(q, dims), _lib.strides3(kcache, dims), _lib.strides3(vcache, dims), _lib.strides3(out, dims),
            scale, nsplit, ws.data_ptr() if ws is not None else None, ws_bytes, _lib.stream_ptr(dev))
    if rc:
        _lib.check(rc, "ksa_decode_wide_fwd" if wide else "ksa_decode_fwd")
    return out


def _launch_wide_decode(q, kcache, vcache, start, end, start0, end0, scale, nsplit):
    return _launch_decode(q, kcache, vcache, start, end, start0, end0, scale, nsplit, wide=True)


@torch.library.custom_op("ksa_amd::decode_fwd", mutates_args=())
def _decode_fwd(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                start: Optional[torch.Tensor], end: Optional[torch.Tensor], start0: int, end0: int,
                scale: float, nsplit: int) -> torch.Tensor:
    return _launch_decode(q, kcache, vcache, start, end, start0, end0, scale, nsplit)


@_decode_fwd.register_fake
def _(q, kcache, vcache, start, end, start0, end0, scale, nsplit):
    b, Hq, Q, D = q.shape
    return q.new_empty((b, Q, Hq, D))


@torch.library.custom_op("ksa_amd::wide_decode_fwd", mutates_args=())
def _wide_decode_fwd(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                     start: Optional[torch.Tensor], end: Optional[torch.Tensor], start0: int, end0: int,
                     scale: float, nsplit: int) -> torch.Tensor:
    return _launch_wide_decode(q, kcache, vcache, start, end, start0, end0, scale, nsplit)


@_wide_decode_fwd.register_fake
def _(q, kcache, vcache, start, end, start0, end0, scale, nsplit):
    b, Hq, Q, D = q.shape
    return q.new_empty((b, Q, Hq, D))


def _wide_splits(b, Hq, Hkv, Q, D, max_rows) -> int:
    """Split count of a call that names none, if it takes the workgroups of eight waves (`ksa_decode_wide_fwd`); else 0."""
    return _lib.lib().ksa_decode_wide_splits(b, Hq, Hkv, Q, D, max_rows)


def _bound(v, default: int, b: int, device) -> torch.Tensor:
    """A row bound as the int32 [b] device tensor that the kernels read."""
    if isinstance(v, torch.Tensor) and v.dtype == torch.int32 and v.device == device and v.shape == (b,) and v.stride(0) == 1:
        return v
    return torch.as_tensor(default if v is None else v, device=device).to(torch.int32).expand(b).contiguous()


def ksa_decode(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
               start=None, end=None, scale: Optional[float] = None,
               nsplit: Optional[int] = None) -> torch.Tensor:
    """q [b, Hq, Q, D]; kcache/vcache [b, Hkv, rows, D] (any batch/head/row strides);
    rows [start, end) are attended: ints for every sequence, or int32 device tensors [b]
    per sequence; default is the whole row axis.  Returns [b, Q, Hq, D]."""
    if not torch.compiler.is_compiling():
        out = _lib.fast.decode(q, kcache, vcache, start, end, scale, nsplit)
        if out is not None:
            return out
    assert q.is_cuda and kcache.is_cuda and vcache.is_cuda, "inputs must be on a GPU"
    assert q.dtype in _DTYPES and q.dtype == kcache.dtype == vcache.dtype, "inputs must share a 16-bit float dtype"
    assert q.dim() == 4 and kcache.dim() == 4 and kcache.shape == vcache.shape
    b, Hq, Q, D = q.shape
    assert kcache.shape[0] == b and kcache.shape[3] == D and Hq % kcache.shape[1] == 0
    if q.stride(-1) != 1:
        q = q.contiguous()
    assert kcache.stride(-1) == 1 and vcache.stride(-1) == 1, "cache rows must be contiguous"
    rows = kcache.shape[2]
    t_start = t_end = None
    s0, e0 = 0, rows
    if isinstance(start, torch.Tensor) or isinstance(end, torch.Tensor):
        t_start, t_end = _bound(start, 0, b, q.device), _bound(end, rows, b, q.device)
        max_rows = rows
    else:
        s0 = 0 if start is None else int(start)
        e0 = rows if end is None else int(end)
        assert 0 <= s0 < e0 <= rows, "row range out of bounds"
        max_rows = e0 - s0
    scale = float(D) ** -0.5 if scale is None else float(scale)
    if scale <= 0:
        q, scale = fold_scale(q, scale)
    wide = False
    if nsplit is None:
        with _lib.on_device(q.device):
            nsplit = _wide_splits(b, Hq, kcache.shape[1], Q, kernel_head_dim(D), max_rows)
            wide = nsplit > 0
            if not wide:
                nsplit = _lib.lib().ksa_decode_splits(b, Hq, kcache.shape[1], Q, D, max_rows)
    op = torch.ops.ksa_amd.wide_decode_fwd if wide else torch.ops.ksa_amd.decode_fwd
    Dk = kernel_head_dim(D)
    if Dk != D:
        # A head dimension without a kernel of its own (the kernels are built for 64 / 128 / 256): the
        # attended rows are copied into zero-padded buffers for this call.  Correct, but it moves the
        # rows twice; a cache that stores its rows at a kernel size avoids it.
        assert D % 8 == 0, "head dimension must be a multiple of 8"
        if t_start is not None:
            lo, hi = int(t_start.min().item()), int(t_end.max().item())
            t_start, t_end = t_start - lo, t_end - lo
        else:
            lo, hi, s0, e0 = s0, e0, 0, e0 - s0
        kcache, vcache = pad_head_dim(kcache[:, :, lo:hi], Dk), pad_head_dim(vcache[:, :, lo:hi], Dk)
        out = op(pad_head_dim(q, Dk), kcache, vcache, t_start, t_end, s0, e0,
                                           scale, int(nsplit))
        return out[..., :D].contiguous()
    direct = _lib.direct(q, kcache, vcache, t_start, t_end)
    forward = (_launch_wide_decode if wide else _launch_decode) if direct else op
    return forward(q, kcache, vcache, t_start, t_end, s0, e0, scale, int(nsplit))


def decode_qkv_supported(Hq: int, Hkv: int, D: int) -> bool:
    return D in (64, 128) and Hq % Hkv == 0 and Hq // Hkv <= 32


def _qkv_splits(b: int, Hq: int, Hkv: int, D: int, max_rows: int) -> Tuple[int, bool]:
    """(splits, whether in workgroups of eight waves) of a `ksa_decode_qkv` call that names no count, on the current GPU."""
    L = _lib.lib()
    n = L.ksa_decode_qkv_wide_splits(b, Hq, Hkv, D, max_rows)
    return (n, True) if n else (L.ksa_decode_splits(b, Hq, Hkv, 1, D, max_rows), False)


def decode_qkv_pays(kcache: torch.Tensor, Hq: int, start, end) -> bool:
    """Whether `ksa_decode_qkv` takes the place of `pre_attention_partials` and `ksa_decode`: where all its workgroups
    run at once (two per CU, one of the wide ones).  A workgroup that starts later pays for its query rows behind the others' loads:
    a decode step of 4 layers, 8 kv heads, separate -> one launch: 1 / 16 / 32 / 64 sequences
    402 -> 393 / 563 -> 552 / 597 -> 589 / 800 -> 774 us, but 24 (576 workgroups) 577 -> 582 and 48 (768) 684 -> 702.
    The two calls alone over 200 to 4000 rows of 1 to 32 sequences, in time of the separate launches: head_dim 64, 32 / 8 heads
    0.69 to 0.86, 14 / 2 0.85 to 1.02; head_dim 128, 16 / 2 heads 0.72 to 0.94, 8 / 8 0.77 to 0.92, 32 / 1 0.72 to 0.96."""
    b, Hkv, rows, D = kcache.shape
    if not decode_qkv_supported(Hq, Hkv, D):
        return False
    L = _lib.lib()
    device = isinstance(start, torch.Tensor) or isinstance(end, torch.Tensor)
    with _lib.on_device(kcache.device):
        n, wide = _qkv_splits(b, Hq, Hkv, D, rows if device else max(1, int(end) - int(start)))
        return wide or b * Hkv * n <= 2 * max(1, L.ksa_device_cu_count())


def _qkv_arguments(qkv, q_norm_weight, k_norm_weight, cos, sin, kcache, vcache, Hq, row, start, end, scale):
    """What the two forms of the one-launch step share: the checked arguments, and the longest range.  (The queries are
    linear in their norm weight, which takes the sign of the scale.)"""
    from .gemm import SplitKPartials
    assert isinstance(qkv, SplitKPartials) and qkv.dtype in _DTYPES and qkv.dtype == kcache.dtype == vcache.dtype
    b, Hkv, rows, D = kcache.shape
    dev = qkv.device
    assert qkv.shape == (b, 1, (Hq + 2 * Hkv) * D) and vcache.shape == kcache.shape and decode_qkv_supported(Hq, Hkv, D)
    assert kcache.stride(-1) == 1 and vcache.stride(-1) == 1, "cache rows must be contiguous"
    dt = qkv.dtype
    cos, sin = (t.to(dt).reshape(-1, D).contiguous() for t in (cos, sin))
    qw, kw = q_norm_weight.to(dt).contiguous(), k_norm_weight.to(dt).contiguous()
    scale = float(D) ** -0.5 if scale is None else float(scale)
    if scale <= 0:
        qw, scale = fold_scale(qw, scale)
    assert cos.shape == sin.shape and cos.shape[0] in (1, b) and qw.shape == (D,) and kw.shape == (D,)
    t_row = t_start = t_end = None
    s0, e0, r0 = 0, 1, 0
    if isinstance(start, torch.Tensor) or isinstance(end, torch.Tensor):
        t_start, t_end = _bound(start, 0, b, dev), _bound(end, rows, b, dev)
        max_rows = rows
    else:
        s0, e0 = int(start), int(end)
        assert 0 <= s0 < e0 <= rows, "row range out of bounds"
        max_rows = e0 - s0
    if isinstance(row, torch.Tensor):
        t_row = _bound(row, 0, b, dev)
    else:
        r0 = int(row)
        assert 0 <= r0 < rows and (t_start is not None or s0 <= r0 < e0), "the new row must lie in the attended range"
    return cos, sin, qw, kw, t_row, r0, t_start, t_end, s0, e0, max_rows, scale


def ksa_decode_qkv(qkv, q_norm_weight: torch.Tensor, k_norm_weight: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                   eps: float, kcache: torch.Tensor, vcache: torch.Tensor, Hq: int, row, start, end,
                   scale: Optional[float] = None, nsplit: Optional[int] = None, wide: bool = False) -> torch.Tensor:
    """`pre_attention_partials` + `ksa_decode` of one new token per sequence in one launch (`ksa_decode_qkv_fwd`).

    qkv: the deferred q | k | v projection (`SplitKPartials` [b, 1, (Hq + 2 Hkv) D]); cos / sin [1 or b, 1, D].  The
    token's key and value go to `row` of the caches and are attended with the rest of [start, end), which has
    to hold that row (each an int, or an int32 GPU tensor [b]).  `wide`: a named count of splits is one of workgroups of eight
    waves (`ksa_decode_qkv_wide_fwd`).  Returns [b, 1, Hq D]."""
    cos, sin, qw, kw, t_row, r0, t_start, t_end, s0, e0, max_rows, scale = _qkv_arguments(
        qkv, q_norm_weight, k_norm_weight, cos, sin, kcache, vcache, Hq, row, start, end, scale)
    b, Hkv, _, D = kcache.shape
    dev, dt = qkv.device, qkv.dtype
    L = _lib.lib()
    ptr = lambda t: None if t is None else t.data_ptr()
    with _lib.on_device(dev):
        if nsplit is None:
            nsplit, wide = _qkv_splits(b, Hq, Hkv, D, max_rows)
        ws = None
        ws_bytes = L.ksa_decode_workspace_bytes(b, Hq, Hkv, 1, D, nsplit)
        if nsplit > 1:
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        out = torch.empty((b, 1, Hq, D), dtype=dt, device=dev)
        dims = (0, 1, 2)
        rc = (L.ksa_decode_qkv_wide_fwd if wide else L.ksa_decode_qkv_fwd)(
            qkv.workspace.data_ptr(), qkv.ksplit, qw.data_ptr(), kw.data_ptr(), cos.data_ptr(), sin.data_ptr(),
            D if cos.shape[0] > 1 else 0, float(eps), kcache.data_ptr(), vcache.data_ptr(), out.data_ptr(), ptr(t_row), r0,
            ptr(t_start), ptr(t_end), s0, e0, b, Hq, Hkv, D, _DTYPES[dt], _lib.strides3(kcache, dims),
            _lib.strides3(vcache, dims), _lib.strides3(out, dims),
            scale, nsplit, ptr(ws), ws_bytes, _lib.stream_ptr(dev))
    _lib.check(rc, "ksa_decode_qkv_fwd")
    return out.view(b, 1, Hq * D)


def decode_qkv_o_supported(kcache: torch.Tensor, Hq: int, N: int) -> bool:
    b, Hkv, _, D = kcache.shape
    return (b <= 16 and Hkv <= 128 and decode_qkv_supported(Hq, Hkv, D) and Hq * D % 512 == 0 and Hq * D <= 32768
            and N % 16 == 0)


def decode_qkv_o_pays(kcache: torch.Tensor, Hq: int, N: int, start, end) -> bool:
    """Whether `ksa_decode_qkv_o` is the faster way (`ksa_decode_qkv_o_wide_pays`, or `ksa_decode_qkv_o_pays` where the wide form is not
    taken, as for groups of more than 16 heads; by the longest possible range where the ranges are on the device)."""
    b, Hkv, rows, D = kcache.shape
    if not (isinstance(start, torch.Tensor) or isinstance(end, torch.Tensor)):
        rows = max(1, int(end) - int(start))
    with _lib.on_device(kcache.device):
        L = _lib.lib()
        wide = L.ksa_decode_qkv_o_wide_splits(b, Hq, Hkv, D, N, rows) > 0
        return (L.ksa_decode_qkv_o_wide_pays if wide else L.ksa_decode_qkv_o_pays)(b, Hq, Hkv, D, N, rows) != 0


def ksa_decode_qkv_o(qkv, q_norm_weight: torch.Tensor, k_norm_weight: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                     eps: float, kcache: torch.Tensor, vcache: torch.Tensor, Hq: int, row, start, end, o_weight, ws,
                     scale: Optional[float] = None, nsplit: Optional[int] = None, wide: bool = False):
    """`ksa_decode_qkv` and the o projection behind it (modeling_qwen3sa.py:879) in one launch
    (`ksa_decode_qkv_o_fwd`), for at most 16 sequences: o_weight a `gemm.TiledWeight` [N, Hq D], ws the step's
    `gemm.MlpRowsWorkspace`.  `wide`: in workgroups of eight waves where they take the call (`ksa_decode_qkv_o_wide_fwd`).  Returns the product's `SplitKPartials` [b, 1, N]."""
    from .gemm import SplitKPartials, TiledWeight
    cos, sin, qw, kw, t_row, r0, t_start, t_end, s0, e0, max_rows, scale = _qkv_arguments(
        qkv, q_norm_weight, k_norm_weight, cos, sin, kcache, vcache, Hq, row, start, end, scale)
    b, Hkv, _, D = kcache.shape
    dev, dt = qkv.device, qkv.dtype
    N = o_weight.shape[0]
    assert isinstance(o_weight, TiledWeight) and o_weight.shape == (N, Hq * D) and o_weight.dtype == dt
    L = _lib.lib()
    ptr = lambda t: None if t is None else t.data_ptr()
    with _lib.on_device(dev):
        if nsplit is None and wide:
            nsplit = L.ksa_decode_qkv_o_wide_splits(b, Hq, Hkv, D, N, max_rows) or None
            wide = nsplit is not None
        if nsplit is None:
            nsplit = L.ksa_decode_qkv_o_splits(b, Hq, Hkv, D, max_rows)
        ws_bytes = L.ksa_decode_qkv_o_workspace_bytes(b, Hq, Hkv, D, nsplit)
        sums = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        ks = Hq * D // 512
        part = torch.empty(ks * 16 * N, dtype=torch.float32, device=dev)
        dims = (0, 1, 2)
        rc = (L.ksa_decode_qkv_o_wide_fwd if wide else L.ksa_decode_qkv_o_fwd)(
            qkv.workspace.data_ptr(), qkv.ksplit, qw.data_ptr(), kw.data_ptr(), cos.data_ptr(), sin.data_ptr(),
            D if cos.shape[0] > 1 else 0, float(eps), kcache.data_ptr(), vcache.data_ptr(), ptr(t_row), r0,
            ptr(t_start), ptr(t_end), s0, e0, b, Hq, Hkv, D, _DTYPES[dt], _lib.strides3(kcache, dims),
            _lib.strides3(vcache, dims), scale, nsplit, o_weight.data_ptr(),
            part.data_ptr(), N, sums.data_ptr(), ws_bytes, ws.step.data_ptr(), ws.step.numel(), _lib.stream_ptr(dev))
    _lib.check(rc, "ksa_decode_qkv_o_fwd")
    return SplitKPartials(part.view(torch.uint8), ks, b, (b, 1, N), dt)


def ksa_decode_boundary(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor, text_start, text_end,
                        sum_start, sum_end, scale: Optional[float] = None,
                        nsplit: Optional[int] = None) -> torch.Tensor:
    """The attention of a chunk-boundary step in one launch (modeling_qwen3sa.py:831-876: two calls of
    the decode attention function and a `torch.cat`): q [b, Hq, 1 + S, D]; query token 0 attends the
    cache rows [text_start, text_end), the S summary tokens attend [sum_start, sum_end); each bound
    an int or an int32 GPU tensor [b].  Returns [b, 1 + S, Hq, D]."""
    assert q.is_cuda and q.dtype in _DTYPES and q.dtype == kcache.dtype == vcache.dtype
    b, Hq, Q, D = q.shape
    Hkv, rows = kcache.shape[1], kcache.shape[2]
    assert Q >= 2 and kcache.shape == vcache.shape and kcache.shape[0] == b and kcache.shape[3] == D and Hq % Hkv == 0
    assert D in (64, 128, 256), "the boundary form has no padded path: head_dim 64, 128 or 256"
    if q.stride(-1) != 1:
        q = q.contiguous()
    assert kcache.stride(-1) == 1 and vcache.stride(-1) == 1, "cache rows must be contiguous"

    def pair(lo, hi):
        if torch.is_tensor(lo) or torch.is_tensor(hi):
            tl = torch.as_tensor(lo, device=q.device).to(torch.int32).expand(b).contiguous()
            th = torch.as_tensor(hi, device=q.device).to(torch.int32).expand(b).contiguous()
            return tl, th, 0, 1
        assert 0 <= int(lo) < int(hi) <= rows, "row range out of bounds"
        return None, None, int(lo), int(hi)
    ts, te, ts0, te0 = pair(text_start, text_end)
    ss, se, ss0, se0 = pair(sum_start, sum_end)
    scale = float(D) ** -0.5 if scale is None else float(scale)
    if scale <= 0:
        q, scale = fold_scale(q, scale)
    lib = _lib.lib()
    if nsplit is None:   # (the count by the slices: ksa_decode_splits is for one range, not for two of different lengths)
        nsplit = lib.ksa_decode_auto_splits(b, Hkv, rows if ts is not None else te0 - ts0)
    out = torch.empty((b, Q, Hq, D), dtype=q.dtype, device=q.device)
    ws, ws_bytes = None, 0
    if nsplit > 1:
        ws_bytes = lib.ksa_decode_boundary_workspace_bytes(b, Hq, Hkv, Q, D, nsplit)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=q.device)
    ptr = lambda t: t.data_ptr() if t is not None else None
    with _lib.on_device(q.device):
        rc = lib.ksa_decode_boundary_fwd(
            q.data_ptr(), kcache.data_ptr(), vcache.data_ptr(), out.data_ptr(), ptr(ts), ptr(te), ts0, te0,
            ptr(ss), ptr(se), ss0, se0, b, Hq, Hkv, Q, D, _DTYPES[q.dtype], _lib.strides3(q, (0, 1, 2)),
            _lib.strides3(kcache, (0, 1, 2)), _lib.strides3(vcache, (0, 1, 2)), _lib.strides3(out, (0, 1, 2)),
            scale, int(nsplit), ptr(ws), ws_bytes, _lib.stream_ptr(q.device))
    _lib.check(rc, "ksa_decode_boundary_fwd")
    return out


def ksa_decode_weights(q: torch.Tensor, kcache: torch.Tensor, start=None, end=None,
                       scale: Optional[float] = None, mask: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The attention probabilities of `ksa_decode`: softmax(q K^T * scale (+ mask)) over the rows
    [start, end) of every sequence, computed in fp32 and rounded to q's dtype, [b, Hq, Q, L] with
    L = the longest range; positions past a shorter sequence's range hold 0.  `mask`, if given, is
    additive, of q's dtype and broadcastable to [b, Hq, Q, L] (the `attention_mask` of the
    reference's eager_attention_forward, modeling_qwen3sa.py:569-588)."""
    assert q.is_cuda and kcache.is_cuda and q.dtype in _DTYPES and q.dtype == kcache.dtype
    assert q.dim() == 4 and kcache.dim() == 4
    b, Hq, Q, D = q.shape
    Hkv, rows = kcache.shape[1], kcache.shape[2]
    assert kcache.shape[0] == b and kcache.shape[3] == D and Hq % Hkv == 0
    if q.stride(-1) != 1:
        q = q.contiguous()
    assert kcache.stride(-1) == 1, "cache rows must be contiguous"
    t_start = t_end = None
    s0, e0 = 0, rows
    if isinstance(start, torch.Tensor) or isinstance(end, torch.Tensor):
        t_start = torch.as_tensor(start if start is not None else 0, device=q.device).to(torch.int32).expand(b).contiguous()
        t_end = torch.as_tensor(end if end is not None else rows, device=q.device).to(torch.int32).expand(b).contiguous()
        L = int((t_end - t_start).max().item())
    else:
        s0 = 0 if start is None else int(start)
        e0 = rows if end is None else int(end)
        assert 0 <= s0 < e0 <= rows, "row range out of bounds"
        L = e0 - s0
    assert L > 0
    Dk = kernel_head_dim(D)
    if scale is None:
        scale = float(D) ** -0.5
    if Dk != D:   # zero-padded copies of the attended rows, as in `ksa_decode`
        assert D % 8 == 0, "head dimension must be a multiple of 8"
        if t_start is not None:
            lo, hi = int(t_start.min().item()), int(t_end.max().item())
            t_start, t_end = t_start - lo, t_end - lo
        else:
            lo, hi, s0, e0 = s0, e0, 0, e0 - s0
        q, kcache = pad_head_dim(q, Dk), pad_head_dim(kcache[:, :, lo:hi], Dk)
    m_strides = None
    if mask is not None:
        assert mask.dtype == q.dtype and mask.is_cuda
        mask = mask.expand(b, Hq, Q, L)
        m_strides = (ctypes.c_int64 * 4)(*mask.stride())
    lib = _lib.lib()
    out = torch.empty((b, Hq, Q, L), dtype=q.dtype, device=q.device)
    ws_bytes = lib.ksa_decode_weights_workspace_bytes(b, Hq, Q, L)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=q.device)
    with _lib.on_device(q.device):
        rc = lib.ksa_decode_weights(
            q.data_ptr(), kcache.data_ptr(), out.data_ptr(), mask.data_ptr() if mask is not None else None,
            t_start.data_ptr() if t_start is not None else None, t_end.data_ptr() if t_end is not None else None,
            s0, e0, b, Hq, Hkv, Q, Dk, _DTYPES[q.dtype], L, _lib.strides3(q, (0, 1, 2)),
            _lib.strides3(kcache, (0, 1, 2)), m_strides, float(scale), ws.data_ptr(), ws_bytes,
            _lib.stream_ptr(q.device))
    _lib.check(rc, "ksa_decode_weights")
    return out


def eager_attention_forward(module, query: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                            attention_mask: Optional[torch.Tensor] = None, scaling: Optional[float] = None,
                            dropout: float = 0.0, **kwargs) -> Tuple[torch.Tensor, torch.Tensor]:
    """Drop-in for the reference's `eager_attention_forward` (modeling_qwen3sa.py:569-588), the decode
    attention function it selects when `config._attn_implementation == "eager"` (:643-646): returns
    `(attn_output [b, q_len, Hq, D], attn_weights [b, Hq, q_len, L])`.  The output comes from the
    decode kernel, the probabilities from `ksa_decode_weights` (a second pass over K).  The cache
    call sites pass no mask (:820-870); one is refused here, because the output kernel has no masked
    form."""
    if dropout:
        raise NotImplementedError("decode attention is inference-only (dropout must be 0)")
    if attention_mask is not None:
        raise NotImplementedError("the decode kernels take no attention mask (the reference's cache call sites pass None)")
    g = query.shape[1] // key.shape[1]
    assert getattr(module, "num_key_value_groups", g) == g, "module.num_key_value_groups does not match the tensor shapes"
    return ksa_decode(query, key, value, scale=scaling), ksa_decode_weights(query, key, scale=scaling)


def decode_attention_forward(module, query: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                             attention_mask: Optional[torch.Tensor] = None,
                             scaling: Optional[float] = None, dropout: float = 0.0,
                             **kwargs) -> Tuple[torch.Tensor, None]:
    """Drop-in for `Qwen3Attention._decode_attn_fn`.  `attention_mask` is ignored exactly
    as the reference's SDPA variant ignores it (it passes attn_mask=None); dropout must be 0."""
    if dropout:
        raise NotImplementedError("decode attention is inference-only (dropout must be 0)")
    g = query.size(1) // key.size(1)
    mg = getattr(module, "num_key_value_groups", g)
    assert mg == g, "module.num_key_value_groups does not match the tensor shapes"
    return ksa_decode(query, key, value, scale=scaling), None
