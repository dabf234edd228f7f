"""Tensor-level wrappers of include/e2h_seq.h: the kernels of layers that carry per-sequence state, and of mixtures of experts.

PyTorch owns the memory and the stream; the arithmetic is in libe2h_seq.so.  Inputs live on the GPU, there is no CPU
implementation behind these functions.  Activations are bfloat16 or float32; norms, biases, gate constants and state are
float32.
"""

import ctypes

import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from . import _lib
from .ops import _current_device, _need_gpu, _OnDevice, _stream

_DTYPES = {torch.bfloat16: _lib.SEQ_BF16, torch.float32: _lib.SEQ_F32}


def _dtype(t, what):
    if t.dtype not in _DTYPES:
        raise TypeError(f"{what}: bfloat16 or float32 activations expected, got {t.dtype}")
    return _DTYPES[t.dtype]


def _lib_for(t):
    lib = _lib.load_seq()
    return lib if t.get_device() == _current_device() else _OnDevice(lib, t.device)


def _p(t):
    return None if t is None else t.data_ptr()


def _vec(t, n, what):
    """data pointer of a float32 vector of n values (None stays None)"""
    if t is None:
        return None
    if t.dtype != torch.float32 or t.numel() != n or not t.is_contiguous() or not t.is_cuda:
        raise TypeError(f"{what}: float32 [{n}] on the GPU expected, got {t.dtype} {tuple(t.shape)} on {t.device}")
    return t.data_ptr()


def _positions(input_pos, first, batch, seqlen, what):
    if input_pos.dtype != torch.int64 or not input_pos.is_cuda or input_pos.numel() != seqlen:
        raise TypeError(f"{what}: input_pos must be int64 [{seqlen}] on the GPU")
    if first is not None and (first.dtype != torch.int64 or not first.is_cuda or first.numel() != batch or not first.is_contiguous()):
        raise TypeError(f"{what}: left padding must be int64 [{batch}] on the GPU")
    return _p(input_pos), _p(first)


def _rows(t, batch, seqlen, what, width=None):
    if t.dim() != 2 or t.shape[0] != batch * seqlen or not t.is_contiguous() or (width is not None and t.shape[1] != width):
        raise RuntimeError(f"{what}: contiguous [{batch * seqlen}, {width if width is not None else '*'}] expected, got {tuple(t.shape)}")


def _check_tail(tails, batch, taps, channels, dtype, what):
    for t in tails:
        if t.dtype != dtype or t.dim() != 3 or t.shape[0] < batch or tuple(t.shape[1:]) != (taps, channels) or not t.is_contiguous() or not t.is_cuda:
            raise RuntimeError(f"{what}: convolution ring must be {dtype} [>= {batch}, {taps}, {channels}], got {t.dtype} {tuple(t.shape)}")


def norm_conv(x, batch, seqlen, eps, dtype, delta=None, delta_weight=None, delta_offset=0.0, norm_weight=None, norm_offset=0.0, conv=None,
              tails=None, input_pos=None, first=None, want_x=True, want_out=True, layer_norm=False, delta_bias=None, norm_bias=None, terms=None,
              term_weights=None):
    """x + norm(delta), its norm and the norm's convolution over time (each optional) in one pass; x float32 [rows, width],
    conv float32 [taps, width].  The norms are RMS norms, or with layer_norm layer norms with optional biases.  terms
    [rows * n, width] with term_weights float32 [rows, n] add a weighted sum to delta (or stand for it).  For one token per sequence delta may be linear_sums' float32 [slices, rows, width].  Returns (x_out float32 or x itself when there is no delta, out in `dtype` or None)."""
    _need_gpu(x)
    width = x.shape[-1]
    if x.dtype != torch.float32:
        raise TypeError("norm_conv: the residual stream is float32")
    _rows(x, batch, seqlen, "norm_conv", width)
    a = _lib.NormConvArgs(dtype=_DTYPES[dtype], batch=batch, seqlen=seqlen, width=width, eps=eps, delta_offset=delta_offset, norm_offset=norm_offset,
                          x=_p(x), norm_kind=int(layer_norm))
    x_out, sums = x, None
    if delta is not None and delta.dim() == 3:
        _need_gpu(delta)
        if delta.dtype != torch.float32 or not delta.is_contiguous() or tuple(delta.shape[1:]) != (batch * seqlen, width):
            raise TypeError(f"norm_conv: sums must be float32 [slices, {batch * seqlen}, {width}], got {delta.dtype} {tuple(delta.shape)}")
        sums = delta
    elif delta is not None:
        _need_gpu(delta)
        _rows(delta, batch, seqlen, "norm_conv delta", width)
        if delta.dtype != dtype:
            raise TypeError(f"norm_conv: delta is {delta.dtype}, expected {dtype}")
        a.delta = _p(delta)
    if terms is not None:
        _need_gpu(terms, term_weights)
        n = terms.shape[0] // (batch * seqlen)
        if terms.dtype != dtype or tuple(terms.shape) != (batch * seqlen * n, width) or not terms.is_contiguous():
            raise TypeError(f"norm_conv: terms must be {dtype} [{batch * seqlen} * n, {width}], got {terms.dtype} {tuple(terms.shape)}")
        a.terms, a.term_weights, a.n_terms = _p(terms), _vec(term_weights, batch * seqlen * n, "norm_conv term_weights"), n
    if delta is not None or terms is not None:
        a.delta_weight = _vec(delta_weight, width, "norm_conv delta_weight")
        a.delta_bias = _vec(delta_bias, width, "norm_conv delta_bias")
        if want_x:
            x_out = torch.empty_like(x)
            a.x_out = _p(x_out)
    a.norm_weight = _vec(norm_weight, width, "norm_conv norm_weight")
    a.norm_bias = _vec(norm_bias, width, "norm_conv norm_bias")
    if conv is not None:
        taps = conv.shape[0]
        a.taps, a.conv = taps, _vec(conv, width * taps, "norm_conv conv")
        a.input_pos, a.first = _positions(input_pos, first, batch, seqlen, "norm_conv")
        if taps > 1:
            _check_tail(tails, batch, taps, width, torch.float32, "norm_conv")
            a.tail_in, a.tail_out = _p(tails[0]), _p(tails[1])
    out = torch.empty((batch * seqlen, width), dtype=dtype, device=x.device) if want_out else None
    a.out = _p(out)
    if sums is not None:
        _lib.check_seq(_lib_for(x).e2h_seq_norm_conv_sums(ctypes.byref(a), _p(sums), sums.shape[0], _stream(x)), "e2h_seq_norm_conv_sums")
    else:
        _lib.check_seq(_lib_for(x).e2h_seq_norm_conv(ctypes.byref(a), _stream(x)), "e2h_seq_norm_conv")
    return x_out, out


def square_relu_(x):
    """max(x, 0)^2 in place."""
    _need_gpu(x)
    assert x.is_contiguous()
    _lib.check_seq(_lib_for(x).e2h_seq_square_relu(_dtype(x, "square_relu_"), _p(x), _p(x), x.numel(), _stream(x)), "e2h_seq_square_relu")
    return x


def softcap_(x, cap):
    """cap * tanh(x / cap) in place."""
    _need_gpu(x)
    assert x.is_contiguous()
    _lib.check_seq(_lib_for(x).e2h_seq_softcap(_dtype(x, "softcap_"), _p(x), _p(x), x.numel(), cap, _stream(x)), "e2h_seq_softcap")
    return x


ACT_NONE, ACT_SQUARE_RELU, ACT_SOFTCAP = 0, 1, 2


STREAMED_ROWS = 64


_PLAIN_TYPES = (torch.Tensor, torch.nn.Parameter)


def watched(*tensors):
    """True where something besides autograd's graph follows what happens to the tensors and would lose sight of it in a launch through
    ctypes: subclasses, forward-mode derivatives, function transforms (vmap, jvp, ..), dispatch modes, torch.jit traces.  (The two last
    do not look through a compiler's trace: that records the registered op.)"""
    if any(type(t) not in _PLAIN_TYPES for t in tensors) or forward_ad._current_level >= 0 or torch._C._are_functorch_transforms_active():
        return True
    return not torch.compiler.is_compiling() and (torch._C._len_torch_dispatch_stack() > 0 or torch._C._get_tracing_state() is not None)


def function_modes():
    """True where somebody intercepts torch functions (a default device does so too, but only looks at factories)."""
    return bool(torch._C._len_torch_function_stack()) and any(type(m) is not DeviceContext for m in torch.overrides._get_current_function_mode_stack())


def intercepted(*tensors):
    """watched(*tensors) or function_modes(): for launches in the place of torch's own functions."""
    return function_modes() or watched(*tensors)


def linear_streams(x, weight):
    """True where `linear` takes x [.., k] and weight [n, k]: bfloat16 on the GPU, up to 64 rows, no gradients, nobody watching."""
    k = weight.shape[1]
    if not 0 < x.numel() <= STREAMED_ROWS * k:
        return False
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or not x.is_cuda or weight.device != x.device or x.shape[-1] != k:
        return False
    if torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad):
        return False
    return k % 8 == 0 and k < 1 << 22 and not torch.is_autocast_enabled() and not watched(x, weight)


def linear(x, weight, act=ACT_NONE, cap=0.0):
    """act(x weight^T) of a decode batch, see e2h_seq_linear; x is copied if it is not 16-byte aligned or not contiguous.  A weight that
    is not takes the library's product, which reads it where it lies."""
    _need_gpu(x, weight)
    n, k = weight.shape
    rows = x.numel() // k
    lib = _lib_for(x)
    need = lib.e2h_seq_linear_scratch_bytes(rows, n, k)
    if need < 0:
        _lib.check_seq(need, "e2h_seq_linear")
    if not weight.is_contiguous() or weight.data_ptr() % 16:
        y = torch.nn.functional.linear(x, weight)
        return square_relu_(y) if act == ACT_SQUARE_RELU else softcap_(y, cap) if act == ACT_SOFTCAP else y
    x2d = x if x.is_contiguous() else x.contiguous()  # the kernel reads it as [rows, k]
    if x2d.data_ptr() % 16:
        x2d = x2d.clone()
    y = torch.empty((*x.shape[:-1], n), dtype=x.dtype, device=x.device)
    scratch = torch.empty((need,), dtype=torch.uint8, device=x.device) if need > 0 else None
    _lib.check_seq(lib.e2h_seq_linear(_p(x2d), _p(weight), _p(y), rows, n, k, act, cap, _p(scratch), need, _stream(x)), "e2h_seq_linear")
    return y


def _product(x, weight, what):
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or weight.dim() != 2 or x.dim() < 1 or x.shape[-1] != weight.shape[1]:
        raise TypeError(f"{what}: bfloat16 [.., k] and [n, k] expected, got {x.dtype} {tuple(x.shape)} and {weight.dtype} {tuple(weight.shape)}")


def linear_sums(x, weight):
    """linear(x, weight) as the float32 sums of its slices of K [slices, rows, n], which norm_conv adds, or None where it has none."""
    _need_gpu(x, weight)
    _product(x, weight, "linear_sums")
    n, k = weight.shape
    rows = x.numel() // k
    if _lib.load_seq().e2h_seq_linear_scratch_bytes(rows, n, k) <= 0 or not (x.is_contiguous() and weight.is_contiguous()) or (x.data_ptr() | weight.data_ptr()) % 16:
        return None
    sums = torch.empty((4, rows, n), dtype=torch.float32, device=x.device)
    _lib.check_seq(_lib_for(x).e2h_seq_linear_sums(_p(x), _p(weight), _p(sums), rows, n, k, _stream(x)), "e2h_seq_linear_sums")
    return sums


def linear_rows_pay(x, weight, act, cap=0.0):
    """True where linear_rows takes x [.., k] and weight [n, k], more rows than a decode step has, and is expected to be faster than the library's product and a pass over its
    result: bfloat16 on the GPU, 16-byte aligned, no gradients, nobody watching."""
    if torch.compiler.is_compiling():
        return False
    n, k = weight.shape
    rows = x.numel() // k if k else 0
    if rows <= STREAMED_ROWS or x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or not x.is_cuda or weight.device != x.device or x.shape[-1] != k:
        return False
    if torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad):
        return False
    if not (x.is_contiguous() and weight.is_contiguous()) or x.data_ptr() % 16 or weight.data_ptr() % 16 or torch.is_autocast_enabled():
        return False
    return bool(_lib.load_seq().e2h_seq_linear_rows_pays(rows, n, k, act, cap)) and not intercepted(x, weight)


def linear_rows(x, weight, act, cap=0.0):
    """act(x weight^T) over many rows in one launch, see e2h_seq_linear_rows (linear_rows_pay)."""
    _need_gpu(x, weight)
    _product(x, weight, "linear_rows")
    if not (x.is_contiguous() and weight.is_contiguous()):
        raise RuntimeError("linear_rows: contiguous x and weight expected")
    n, k = weight.shape
    y = torch.empty((*x.shape[:-1], n), dtype=x.dtype, device=x.device)
    _lib.check_seq(_lib_for(x).e2h_seq_linear_rows(_p(x), _p(weight), _p(y), x.numel() // k, n, k, act, cap, _stream(x)), "e2h_seq_linear_rows")
    return y


def embed_rows(table, tokens, want_rows=True):
    """table[tokens] as float32 and (want_rows) as it is, in one launch; table bfloat16 [vocab, width], tokens int64 [rows] -> (x [rows, width], h or None)."""
    _need_gpu(table, tokens)
    if table.dtype != torch.bfloat16 or tokens.dtype != torch.int64 or not (table.is_contiguous() and tokens.is_contiguous()):
        raise TypeError("embed_rows: a contiguous bfloat16 table and int64 tokens expected")
    rows, width = tokens.numel(), table.shape[1]
    x = torch.empty((rows, width), dtype=torch.float32, device=table.device)
    h = torch.empty((rows, width), dtype=table.dtype, device=table.device) if want_rows else None
    _lib.check_seq(_lib_for(table).e2h_seq_embed_rows(_p(table), _p(tokens), _p(x), _p(h), rows, width, table.shape[0], _stream(table)), "e2h_seq_embed_rows")
    return x, h


def gelu_gate_rows(gate, table, tokens, column):
    """gelu_tanh(gate) * table[tokens, column : column + dim]; gate [rows, dim], tokens int64 [rows]."""
    _need_gpu(gate, table, tokens)
    rows, dim = gate.shape
    if table.dtype != gate.dtype or table.dim() != 2 or not table.is_contiguous() or not gate.is_contiguous():
        raise TypeError("gelu_gate_rows: gate and table must be contiguous and of one dtype")
    if tokens.dtype != torch.int64 or tokens.numel() != rows or not tokens.is_contiguous():
        raise TypeError("gelu_gate_rows: one int64 token per row expected")
    y = torch.empty_like(gate)
    _lib.check_seq(_lib_for(gate).e2h_seq_gelu_gate_rows(_dtype(gate, "gelu_gate_rows"), _p(gate), _p(table), _p(tokens), _p(y), rows, dim,
                                                         table.shape[1], column, table.shape[0], _stream(gate)), "e2h_seq_gelu_gate_rows")
    return y


def linear_gelu_gate(x, weight, table, tokens, column):
    """gelu_gate_rows(linear(x, weight), table, tokens, column) of a decode batch, in one launch where there is one for the sizes."""
    _need_gpu(x, weight, table, tokens)
    n, k = weight.shape
    rows = x.numel() // k
    fits = (weight.is_contiguous() and x.is_contiguous() and not (weight.data_ptr() | x.data_ptr()) % 16 and x.dtype == weight.dtype == table.dtype == torch.bfloat16 and table.dim() == 2
            and table.is_contiguous() and tokens.dtype == torch.int64 and tokens.numel() == rows and tokens.is_contiguous() and column + n <= table.shape[1])
    if not fits or _lib.load_seq().e2h_seq_linear_scratch_bytes(rows, n, k) != 0:
        return gelu_gate_rows(linear(x, weight), table, tokens, column)
    y = torch.empty((*x.shape[:-1], n), dtype=x.dtype, device=x.device)
    _lib.check_seq(_lib_for(x).e2h_seq_linear_gelu_gate(_p(x), _p(weight), _p(table), _p(tokens), _p(y), rows, n, k, table.shape[1], column, table.shape[0], _stream(x)),
                   "e2h_seq_linear_gelu_gate")
    return y


def rotary_table(turns, input_pos, first, batch, seqlen):
    """(cos, sin) of position * turns for every row and rotated pair, float32 [batch * seqlen, pairs, 2]; turns float64 [pairs]
    in whole turns per position."""
    _need_gpu(turns)
    if turns.dtype != torch.float64 or turns.dim() != 1 or not turns.is_contiguous():
        raise TypeError("rotary_table: turns must be float64 [pairs]")
    table = torch.empty((batch * seqlen, turns.numel(), 2), dtype=torch.float32, device=turns.device)
    pos, pad = _positions(input_pos, first, batch, seqlen, "rotary_table")
    _lib.check_seq(_lib_for(turns).e2h_seq_rotary_table(_p(turns), pos, pad, _p(table), batch, seqlen, turns.numel(), _stream(turns)), "e2h_seq_rotary_table")
    return table


def window_attention(proj, batch, seqlen, heads, kv_heads, dim, vdim, offsets, biases, cache, input_pos, first, window, keep_first, scale,
                     out, out_off, out_scale=1.0, norms=(None, None), norm_eps=0.0, rotary=None, sink=None):
    """Softmax attention over a window and the first `keep_first` positions (window 0: all positions), with projection biases
    and output gate; see e2h_seq_window_attention.  offsets = columns of (q, k, v, gate or -1) in proj, biases = (q, k, v)
    float32 or None, cache a state.KVCache.  norms = float32 weights of the RMS norms of query and key heads or None, rotary = a
    rotary_table, sink float32 [heads].  Appends the new keys and values (k and v at -1: the cache is another layer's, which has
    appended them) and writes out[:, out_off : ...]."""
    _need_gpu(proj, out)
    _rows(proj, batch, seqlen, "window_attention proj")
    _rows(out, batch, seqlen, "window_attention out")
    kc, vc = cache.k_cache, cache.v_cache
    if kc.dtype != proj.dtype or vc.dtype != proj.dtype or out.dtype != proj.dtype:
        raise TypeError("window_attention: projections, caches and output must have one dtype")
    if kc.shape[0] < batch or tuple(kc.shape[1::2]) != (kv_heads, dim) or tuple(vc.shape) != (*kc.shape[:3], vdim):
        raise RuntimeError(f"window_attention: cache shapes {tuple(kc.shape)}, {tuple(vc.shape)} do not fit")
    a = _lib.WindowAttentionArgs(dtype=_dtype(proj, "window_attention"), batch=batch, seqlen=seqlen, heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim,
                                 cache_len=kc.shape[2], proj=_p(proj), ld=proj.shape[1], q_off=offsets[0], k_off=offsets[1], v_off=offsets[2],
                                 g_off=offsets[3], k_cache=_p(kc), v_cache=_p(vc), window=window, keep_first=keep_first, scale=scale,
                                 out_scale=out_scale, out=_p(out), ld_out=out.shape[1], out_off=out_off)
    a.q_bias = _vec(biases[0], heads * dim, "window_attention q bias")
    a.k_bias = _vec(biases[1], kv_heads * dim, "window_attention k bias")
    a.v_bias = _vec(biases[2], kv_heads * vdim, "window_attention v bias")
    a.q_norm, a.k_norm, a.norm_eps = _vec(norms[0], dim, "window_attention q norm"), _vec(norms[1], dim, "window_attention k norm"), norm_eps
    if rotary is not None:
        a.rotary, a.rot_pairs = _vec(rotary, batch * seqlen * rotary.shape[-2] * 2, "window_attention rotary"), rotary.shape[-2]
    a.sink = _vec(sink, heads, "window_attention sink")
    a.input_pos, a.first = _positions(input_pos, first, batch, seqlen, "window_attention")
    lib = _lib_for(proj)
    n = max(0, lib.e2h_seq_window_attention_scratch_bytes(ctypes.byref(a))) if seqlen == 1 else 0  # a refused call is refused below
    scratch = torch.empty((n,), dtype=torch.uint8, device=proj.device) if n else None
    _lib.check_seq(lib.e2h_seq_window_attention_split(ctypes.byref(a), _p(scratch), n, _stream(proj)), "e2h_seq_window_attention")


def _scratch(args, query, like):
    n = query(ctypes.byref(args))
    if n < 0:
        _lib.check_seq(int(n), query.__name__ if hasattr(query, "__name__") else "scratch query")
    if n == 0:
        return None
    buf = torch.empty((n,), dtype=torch.uint8, device=like.device)
    args.scratch, args.scratch_bytes = _p(buf), n
    return buf


def _check_state(state, batch, heads, dim, vdim, what):
    if state.dtype != torch.float32 or state.shape[0] < batch or tuple(state.shape[1:]) != (heads, dim, vdim) or not state.is_contiguous() or not state.is_cuda:
        raise RuntimeError(f"{what}: state must be float32 [>= {batch}, {heads}, {dim}, {vdim}], got {state.dtype} {tuple(state.shape)}")


def hgrn2(proj, batch, seqlen, heads, dim, vdim, offsets, f_bias, lower, norm_weight, eps, state, input_pos, first, out, out_off, out_scale=1.0):
    """HGRN2 recurrence with RMS-normed heads; see e2h_seq_hgrn2.  offsets = columns of (q, f, v) in proj; state float32
    [B, heads, dim, vdim], updated in place; writes out[:, out_off : out_off + heads * vdim]."""
    _need_gpu(proj, out, state)
    _rows(proj, batch, seqlen, "hgrn2 proj")
    _rows(out, batch, seqlen, "hgrn2 out")
    _check_state(state, batch, heads, dim, vdim, "hgrn2")
    if out.dtype != proj.dtype:
        raise TypeError("hgrn2: projections and output must have one dtype")
    a = _lib.Hgrn2Args(dtype=_dtype(proj, "hgrn2"), eps=eps, batch=batch, seqlen=seqlen, heads=heads, dim=dim, vdim=vdim, proj=_p(proj), ld=proj.shape[1],
                       q_off=offsets[0], f_off=offsets[1], v_off=offsets[2], f_bias=_vec(f_bias, heads * dim, "hgrn2 f_bias"),
                       lower=_vec(lower, heads * dim, "hgrn2 lower"), norm_weight=_vec(norm_weight, vdim, "hgrn2 norm"), state=_p(state),
                       out_scale=out_scale, out=_p(out), ld_out=out.shape[1], out_off=out_off)
    a.input_pos, a.first = _positions(input_pos, first, batch, seqlen, "hgrn2")
    lib = _lib_for(proj)
    scratch = _scratch(a, lib.e2h_seq_hgrn2_scratch_bytes, proj)
    _lib.check_seq(lib.e2h_seq_hgrn2(ctypes.byref(a), _stream(proj)), "e2h_seq_hgrn2")
    del scratch


def gated_delta(proj, batch, seqlen, heads, kv_heads, dim, vdim, offsets, conv, tails, a_log, dt_bias, norm_weight, eps, state, input_pos, first,
                out, out_off, out_scale=1.0):
    """Gated delta rule with short convolutions and a gated RMS norm; see e2h_seq_delta.  offsets = columns of
    (q, k, v, b, a, gate) in proj; conv float32 [channels, taps] in the order q, k, v; tails = (ring to read, ring to write)."""
    _need_gpu(proj, out, state)
    _rows(proj, batch, seqlen, "gated_delta proj")
    _rows(out, batch, seqlen, "gated_delta out")
    _check_state(state, batch, heads, dim, vdim, "gated_delta")
    if out.dtype != proj.dtype:
        raise TypeError("gated_delta: projections and output must have one dtype")
    channels, taps = 2 * kv_heads * dim + heads * vdim, conv.shape[-1]
    a = _lib.DeltaArgs(dtype=_dtype(proj, "gated_delta"), taps=taps, batch=batch, seqlen=seqlen, heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim,
                       proj=_p(proj), ld=proj.shape[1], q_off=offsets[0], k_off=offsets[1], v_off=offsets[2], b_off=offsets[3], a_off=offsets[4],
                       g_off=offsets[5], conv=_vec(conv, channels * taps, "gated_delta conv"), a_log=_vec(a_log, heads, "gated_delta a_log"),
                       dt_bias=_vec(dt_bias, heads, "gated_delta dt_bias"), norm_weight=_vec(norm_weight, vdim, "gated_delta norm"), state=_p(state),
                       eps=eps, out_scale=out_scale, out=_p(out), ld_out=out.shape[1], out_off=out_off)
    if taps > 1:
        _check_tail(tails, batch, taps, channels, proj.dtype, "gated_delta")
        a.tail_in, a.tail_out = _p(tails[0]), _p(tails[1])
    a.input_pos, a.first = _positions(input_pos, first, batch, seqlen, "gated_delta")
    lib = _lib_for(proj)
    scratch = _scratch(a, lib.e2h_seq_delta_scratch_bytes, proj)
    _lib.check_seq(lib.e2h_seq_delta(ctypes.byref(a), _stream(proj)), "e2h_seq_delta")
    del scratch


def _experts_weight(t, shape, dtype, what):
    if t.dtype != dtype or tuple(t.shape) != shape or not t.is_contiguous() or not t.is_cuda:
        raise RuntimeError(f"{what}: contiguous {dtype} {shape} expected, got {t.dtype} {tuple(t.shape)}")
    return _p(t)


def route(x, router, bias, top):
    """x [rows, width], router [experts, width] in x's dtype, bias float32 [experts] or None -> (chosen int32 [rows, top], weights
    float32 [rows, top]): the largest logits of each row and the softmax over them."""
    _need_gpu(x, router)
    rows, width = x.shape
    experts = router.shape[0]
    if not x.is_contiguous():
        raise RuntimeError("route: contiguous rows expected")
    logits = torch.empty((rows, experts), dtype=torch.float32, device=x.device)
    chosen = torch.empty((rows, top), dtype=torch.int32, device=x.device)
    weights = torch.empty((rows, top), dtype=torch.float32, device=x.device)
    a = _lib.RouteArgs(dtype=_dtype(x, "route"), rows=rows, width=width, experts=experts, top=top, x=_p(x),
                       router=_experts_weight(router, (experts, width), x.dtype, "route router"), bias=_vec(bias, experts, "route bias"),
                       logits=_p(logits), chosen=_p(chosen), weights=_p(weights))
    _lib.check_seq(_lib_for(x).e2h_seq_route(ctypes.byref(a), _stream(x)), "e2h_seq_route")
    return chosen, weights


def experts(x, chosen, up, down, shared_up=None, shared_down=None):
    """Squared-ReLU experts: x [rows, width], chosen int32 [rows, top], up [experts, ff, width], down [experts, width, ff] ->
    (out [rows * top, width], the shared expert's rows [rows, width] or None); nothing is weighted or added here."""
    _need_gpu(x, chosen, up, down)
    rows, width = x.shape
    count, ff = up.shape[0], up.shape[1]
    if not x.is_contiguous() or chosen.dtype != torch.int32 or chosen.dim() != 2 or chosen.shape[0] != rows or not chosen.is_contiguous():
        raise RuntimeError("experts: contiguous rows and int32 choices [rows, top] expected")
    top = chosen.shape[1]
    a = _lib.ExpertsArgs(dtype=_dtype(x, "experts"), rows=rows, width=width, experts=count, top=top, ff=ff, x=_p(x), chosen=_p(chosen),
                         up=_experts_weight(up, (count, ff, width), x.dtype, "experts up"),
                         down=_experts_weight(down, (count, width, ff), x.dtype, "experts down"))
    out = torch.empty((rows * top, width), dtype=x.dtype, device=x.device)
    shared = None
    if shared_up is not None:
        shared_ff = shared_up.shape[0]
        a.shared_ff = shared_ff
        a.shared_up = _experts_weight(shared_up, (shared_ff, width), x.dtype, "experts shared up")
        a.shared_down = _experts_weight(shared_down, (width, shared_ff), x.dtype, "experts shared down")
        shared = torch.empty((rows, width), dtype=x.dtype, device=x.device)
        a.shared_out = _p(shared)
    a.out = _p(out)
    lib = _lib_for(x)
    scratch = _scratch(a, lib.e2h_seq_experts_scratch_bytes, x)
    _lib.check_seq(lib.e2h_seq_experts(ctypes.byref(a), _stream(x)), "e2h_seq_experts")
    del scratch
    return out, shared
