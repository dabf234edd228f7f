"""ctypes bindings of libe2h_quant.so (C ABI: include/e2h_quant.h) and libe2h_seq.so (include/e2h_seq.h).

The libraries are loaded from the package directory.  If one has not been built, loading it raises: there is
no fallback implementation behind these entry points.
"""

import ctypes
import importlib.util
import warnings
from ctypes import c_char_p, c_float, c_int, c_int32, c_int64, c_void_p

import torch

from ._build import CALLS_PATH, LIB_PATH, SEQ_LIB_PATH, build_library, build_seq_library

_P = c_void_p


class RowNorm(ctypes.Structure):
    _fields_ = [("x", _P), ("partials", _P), ("col_scales", _P), ("weight", _P), ("h_out", _P), ("slices", c_int), ("eps", c_float)]


_SIGNATURES = {
    # name: (restype, argtypes)
    "e2h_abi_version": (c_int, []),
    "e2h_status_string": (c_char_p, [c_int]),
    "e2h_set_option": (c_int, [c_char_p, c_int]),
    "e2h_stream_capturing": (c_int, [_P]),
    "e2h_int8_quantize_per_channel": (c_int, [_P, c_int, _P, _P, _P, c_int64, c_int64, _P]),
    "e2h_int4_mm_scratch_bytes": (c_int64, [c_int64, c_int64, c_int64, c_int, c_int]),
    "e2h_int4_mm_scratch": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P, c_int64, _P, c_int64, _P]),
    "e2h_int8_mm_scratch_bytes": (c_int64, [c_int64, c_int64, c_int64]),
    "e2h_int8_mm_scratch": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, _P, c_int64, _P]),
    "e2h_int8_mm": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, _P, c_int64, _P]),
    "e2h_int4_group_qparams": (c_int, [_P, _P, _P, c_int64, c_int64, c_int, _P]),
    "e2h_int4_quantize_from_qparams": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int, _P]),
    "e2h_int4_group_quantize": (c_int, [_P, _P, _P, c_int64, c_int64, c_int, _P]),
    "e2h_int4_pack": (c_int, [_P, _P, c_int64, c_int64, c_int, _P]),
    "e2h_int4_unpack": (c_int, [_P, _P, c_int64, c_int64, c_int, _P]),
    "e2h_int4_quantize_pack": (c_int, [_P, _P, _P, c_int64, c_int64, c_int, c_int, _P]),
    "e2h_int4_dequantize": (c_int, [_P, _P, _P, c_int64, c_int64, c_int, c_int, _P]),
    "e2h_int4_dequantize_codes": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int, _P]),
    "e2h_int4_mm": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P, c_int64, _P]),
    "e2h_workspace_bytes": (c_int64, []),
    "e2h_int4_mm_static_scratch": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P]),
    "e2h_int4_mm_static_scratch_bytes": (c_int64, []),
    "e2h_decode_attention": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_float, _P]),
    "e2h_rmsnorm": (c_int, [_P, _P, _P, c_int64, c_int64, c_float, _P]),
    "e2h_add_rmsnorm": (c_int, [_P, _P, _P, _P, _P, c_int64, c_int64, c_float, _P]),
    "e2h_int4_mm_partial_slices": (c_int, [c_int64, c_int64, c_int64, c_int, c_int]),
    "e2h_int4_mm_partials": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, c_int, _P]),
    "e2h_int8_mm_partial_slices": (c_int, [c_int64, c_int64, c_int64]),
    "e2h_int8_mm_partials": (c_int, [_P, _P, _P, c_int64, c_int64, c_int64, c_int, _P]),
    "e2h_add_rmsnorm_partials": (c_int, [_P, _P, c_int, _P, _P, _P, _P, c_int64, c_int64, c_float, _P]),
    "e2h_rope_kv_write": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, _P]),
    "e2h_prefill_attention": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_float, _P]),
    "e2h_rope_kv_write_seq": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int, _P]),
    "e2h_silu_mul": (c_int, [_P, _P, _P, c_int64, _P]),
    "e2h_int4_mm_rope_kv": (c_int, [_P, _P, _P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int, c_int, _P]),
    "e2h_sample_top_k": (c_int, [_P, c_int64, _P, _P, _P, c_int64, c_int64, c_float, c_int, _P]),
    "e2h_argmax_rows": (c_int, [_P, c_int64, _P, c_int64, c_int64, _P]),
    "e2h_int8_mm_silu_gate": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, _P]),
    "e2h_int8_mm_rope_kv": (c_int, [_P, _P, _P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, _P]),
    "e2h_int8_mm_silu_gate_rows_scratch_bytes": (c_int64, [c_int64, c_int64, c_int64]),
    "e2h_int8_mm_silu_gate_rows": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, _P, c_int64, _P]),
    "e2h_int8_mm_rope_kv_rows_scratch_bytes": (c_int64, [c_int64] * 7),
    "e2h_int8_mm_rope_kv_rows": (c_int, [_P, _P, _P, _P, c_int64, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int, _P, c_int64, _P]),
    "e2h_int4_mm_rope_kv_rows_scratch_bytes": (c_int64, [c_int64] * 7 + [c_int, c_int]),
    "e2h_int4_mm_rope_kv_rows": (c_int, [_P, _P, _P, _P, c_int64, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int, c_int, c_int, _P, c_int64, _P]),
    "e2h_int8_norm_mm_supported": (c_int, [c_int64, c_int64, c_int64]),
    "e2h_int8_norm_mm": (c_int, [ctypes.POINTER(RowNorm), _P, _P, _P, c_int64, c_int64, c_int64, _P]),
    "e2h_int8_norm_mm_silu_gate": (c_int, [ctypes.POINTER(RowNorm), _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, _P]),
    "e2h_int8_norm_mm_rope_kv": (c_int, [ctypes.POINTER(RowNorm), _P, _P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, _P]),
    "e2h_int4_mm_silu_gate_rows_scratch_bytes": (c_int64, [c_int64, c_int64, c_int64, c_int, c_int]),
    "e2h_int4_mm_silu_gate_rows_pays": (c_int, [c_int64, c_int64, c_int64, c_int, c_int]),
    "e2h_int4_mm_silu_gate_rows": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P, c_int64, _P]),
    "e2h_int4_mm_silu_gate": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P]),
    "e2h_int4_staged_bytes": (c_int64, [c_int64, c_int64]),
    "e2h_int4_stage_x": (c_int, [_P, _P, c_int64, c_int64, _P]),
    "e2h_int4_mm_staged_supported": (c_int, [c_int64, c_int64, c_int64, c_int, c_int]),
    "e2h_int4_mm_staged": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, _P]),
    "e2h_int4_mm_staged_argmax_scratch_bytes": (c_int64, [c_int64, c_int64, c_int64, c_int]),
    "e2h_int4_mm_staged_argmax": (c_int, [_P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, _P]),
    "e2h_int4_mm_staged_partial_slices": (c_int, [c_int64, c_int64, c_int64, c_int]),
    "e2h_int4_mm_staged_partials": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P]),
    "e2h_int4_mm_staged_silu_gate": (c_int, [_P, _P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, _P]),
    "e2h_int4_mm_staged_rope_kv": (c_int, [_P, _P, _P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int, _P]),
    "e2h_add_rmsnorm_sums": (c_int, [_P, _P, _P, c_int, _P, _P, _P, _P, c_int64, c_int64, c_int, c_float, _P]),
    "e2h_int4_mm_rows_slices": (c_int, [c_int64, c_int64, c_int64, c_int, c_int]),
    "e2h_int4_mm_rows": (c_int, [_P, _P, _P, _P, c_int, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P]),
    "e2h_int4_mm_silu_gate_rows_sums": (c_int, [_P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int, c_int, _P, c_int64, _P]),
    "e2h_add_rmsnorm_staged": (c_int, [_P, _P, _P, c_int, _P, _P, _P, _P, _P, c_int64, c_int64, c_float, _P]),
    "e2h_stream_read_probe": (c_int, [_P, c_int64, _P, c_int64, _P, _P]),
    "e2h_decode_attention_staged": (c_int, [_P, _P, _P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_float, _P]),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)

# e2h_dtype values of include/e2h_seq.h
SEQ_BF16, SEQ_F32 = 0, 1


class NormConvArgs(ctypes.Structure):
    _fields_ = [("dtype", c_int32), ("taps", c_int32), ("batch", c_int64), ("seqlen", c_int64), ("width", c_int64), ("eps", c_float),
                ("delta_offset", c_float), ("norm_offset", c_float), ("norm_kind", c_int32), ("x", _P), ("delta", _P), ("delta_weight", _P),
                ("x_out", _P), ("norm_weight", _P), ("conv", _P), ("tail_in", _P), ("tail_out", _P), ("out", _P), ("input_pos", _P), ("first", _P),
                ("delta_bias", _P), ("norm_bias", _P), ("terms", _P), ("term_weights", _P), ("n_terms", c_int64)]


class WindowAttentionArgs(ctypes.Structure):
    _fields_ = [("dtype", c_int32), ("pad_", c_int32), ("batch", c_int64), ("seqlen", c_int64), ("heads", c_int64), ("kv_heads", c_int64),
                ("dim", c_int64), ("vdim", c_int64), ("cache_len", c_int64), ("proj", _P), ("ld", c_int64), ("q_off", c_int64),
                ("k_off", c_int64), ("v_off", c_int64), ("g_off", c_int64), ("q_bias", _P), ("k_bias", _P), ("v_bias", _P), ("k_cache", _P),
                ("v_cache", _P), ("input_pos", _P), ("first", _P), ("window", c_int64), ("keep_first", c_int64), ("scale", c_float),
                ("out_scale", c_float), ("out", _P), ("ld_out", c_int64), ("out_off", c_int64), ("q_norm", _P), ("k_norm", _P), ("rotary", _P),
                ("rot_pairs", c_int64), ("sink", _P), ("norm_eps", c_float), ("pad2_", c_int32)]


class Hgrn2Args(ctypes.Structure):
    _fields_ = [("dtype", c_int32), ("eps", c_float), ("batch", c_int64), ("seqlen", c_int64), ("heads", c_int64), ("dim", c_int64),
                ("vdim", c_int64), ("proj", _P), ("ld", c_int64), ("q_off", c_int64), ("f_off", c_int64), ("v_off", c_int64), ("f_bias", _P),
                ("lower", _P), ("norm_weight", _P), ("state", _P), ("input_pos", _P), ("first", _P), ("scratch", _P), ("scratch_bytes", c_int64),
                ("out_scale", c_float), ("pad_", c_int32), ("out", _P), ("ld_out", c_int64), ("out_off", c_int64)]


class DeltaArgs(ctypes.Structure):
    _fields_ = [("dtype", c_int32), ("taps", c_int32), ("batch", c_int64), ("seqlen", c_int64), ("heads", c_int64), ("kv_heads", c_int64),
                ("dim", c_int64), ("vdim", c_int64), ("proj", _P), ("ld", c_int64), ("q_off", c_int64), ("k_off", c_int64), ("v_off", c_int64),
                ("b_off", c_int64), ("a_off", c_int64), ("g_off", c_int64), ("conv", _P), ("tail_in", _P), ("tail_out", _P), ("a_log", _P),
                ("dt_bias", _P), ("norm_weight", _P), ("state", _P), ("input_pos", _P), ("first", _P), ("scratch", _P), ("scratch_bytes", c_int64),
                ("eps", c_float), ("out_scale", c_float), ("out", _P), ("ld_out", c_int64), ("out_off", c_int64)]


class RouteArgs(ctypes.Structure):
    _fields_ = [("dtype", c_int32), ("pad_", c_int32), ("rows", c_int64), ("width", c_int64), ("experts", c_int64), ("top", c_int64), ("x", _P),
                ("router", _P), ("bias", _P), ("logits", _P), ("chosen", _P), ("weights", _P)]


class ExpertsArgs(ctypes.Structure):
    _fields_ = [("dtype", c_int32), ("pad_", c_int32), ("rows", c_int64), ("width", c_int64), ("experts", c_int64), ("top", c_int64),
                ("ff", c_int64), ("shared_ff", c_int64), ("x", _P), ("chosen", _P), ("up", _P), ("down", _P), ("shared_up", _P),
                ("shared_down", _P), ("out", _P), ("shared_out", _P), ("scratch", _P), ("scratch_bytes", c_int64)]


_A = ctypes.POINTER
_SEQ_SIGNATURES = {
    "e2h_seq_abi_version": (c_int, []),
    "e2h_seq_set_option": (c_int, [c_char_p, c_int]),
    "e2h_seq_norm_conv": (c_int, [_A(NormConvArgs), _P]),
    "e2h_seq_square_relu": (c_int, [c_int, _P, _P, c_int64, _P]),
    "e2h_seq_softcap": (c_int, [c_int, _P, _P, c_int64, c_float, _P]),
    "e2h_seq_gelu_gate_rows": (c_int, [c_int, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, _P]),
    "e2h_seq_embed_rows": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, _P]),
    "e2h_seq_linear_gelu_gate": (c_int, [_P, _P, _P, _P, _P, c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, _P]),
    "e2h_seq_norm_conv_sums": (c_int, [_A(NormConvArgs), _P, c_int, _P]),
    "e2h_seq_linear_sums": (c_int, [_P, _P, _P, c_int64, c_int64, c_int64, _P]),
    "e2h_seq_linear_scratch_bytes": (c_int64, [c_int64, c_int64, c_int64]),
    "e2h_seq_linear": (c_int, [_P, _P, _P, c_int64, c_int64, c_int64, c_int, c_float, _P, c_int64, _P]),
    "e2h_seq_linear_rows_pays": (c_int, [c_int64, c_int64, c_int64, c_int, c_float]),
    "e2h_seq_linear_rows": (c_int, [_P, _P, _P, c_int64, c_int64, c_int64, c_int, c_float, _P]),
    "e2h_seq_rotary_table": (c_int, [_P, _P, _P, _P, c_int64, c_int64, c_int64, _P]),
    "e2h_seq_window_attention": (c_int, [_A(WindowAttentionArgs), _P]),
    "e2h_seq_window_attention_scratch_bytes": (c_int64, [_A(WindowAttentionArgs)]),
    "e2h_seq_window_attention_split": (c_int, [_A(WindowAttentionArgs), _P, c_int64, _P]),
    "e2h_seq_hgrn2_scratch_bytes": (c_int64, [_A(Hgrn2Args)]),
    "e2h_seq_hgrn2": (c_int, [_A(Hgrn2Args), _P]),
    "e2h_seq_delta_scratch_bytes": (c_int64, [_A(DeltaArgs)]),
    "e2h_seq_delta": (c_int, [_A(DeltaArgs), _P]),
    "e2h_seq_route": (c_int, [_A(RouteArgs), _P]),
    "e2h_seq_experts_scratch_bytes": (c_int64, [_A(ExpertsArgs)]),
    "e2h_seq_experts": (c_int, [_A(ExpertsArgs), _P]),
}

SEQ_EXPORTED_SYMBOLS = tuple(_SEQ_SIGNATURES)

_lib = None
_seq_lib = None


class E2HLibraryError(RuntimeError):
    pass


def _open(path, build, build_if_missing, signatures, version_symbol, expected=1):
    if not path.exists():
        if not build_if_missing:
            raise E2HLibraryError(
                f"{path} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'` "
                "(there is no fallback path for its kernels)"
            )
        build()
    lib = ctypes.CDLL(str(path))
    for name, (restype, argtypes) in signatures.items():
        fn = getattr(lib, name)  # AttributeError if the symbol is not exported
        fn.restype = restype
        fn.argtypes = argtypes
    version = getattr(lib, version_symbol)()
    if version != expected:
        raise E2HLibraryError(f"{path}: ABI version {version} != {expected}; rebuild the library")
    return lib


def load(build_if_missing=False):
    """Return the loaded libe2h_quant.so.  `build_if_missing` compiles it first when the .so is absent."""
    global _lib
    if _lib is None:
        _lib = _open(LIB_PATH, build_library, build_if_missing, _SIGNATURES, "e2h_abi_version")
    return _lib


def load_seq(build_if_missing=False):
    """Return the loaded libe2h_seq.so.  `build_if_missing` compiles it first when the .so is absent."""
    global _seq_lib
    if _seq_lib is None:
        _seq_lib = _open(SEQ_LIB_PATH, build_seq_library, build_if_missing, _SEQ_SIGNATURES, "e2h_seq_abi_version", 2)
    return _seq_lib


_calls = None


class _PythonCalls:
    """Stands for the extension module where that cannot be used: every call is left to the Python path, which launches the same kernels."""

    @staticmethod
    def int4_linear(*_):
        return None

    int8_linear = int4_rows = int4_linear


def _load_calls(lib):
    if not CALLS_PATH.exists():
        return "is missing"
    from . import ops

    spec = importlib.util.spec_from_file_location(f"{__package__}._calls", CALLS_PATH)
    try:
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
    except ImportError as e:
        return f"cannot be loaded ({e})"
    if module.torch_version != torch.__version__:  # it reads tensors' structures as that torch laid them out
        return f"was built for torch {module.torch_version}, this is {torch.__version__}"
    module.bind(*(ctypes.cast(f, c_void_p).value for f in (lib.e2h_int4_mm, lib.e2h_int8_mm, lib.e2h_stream_capturing)), ops._workspaces, check)
    module.bind_rows(*(ctypes.cast(f, c_void_p).value for f in (lib.e2h_int4_mm_rows, lib.e2h_int4_mm_rows_slices)))
    return module


def calls():
    """The extension module of small calls (csrc/e2h_calls.cpp), bound to libe2h_quant.so and the workspaces of `ops`.  Without one that was built for this torch, a warning
    and a stand-in: such calls then cost the host what they cost through Python."""
    global _calls
    if _calls is None:
        got = _load_calls(load())
        if isinstance(got, str):
            warnings.warn(f"{CALLS_PATH} {got}: small calls of the quantized linears go through Python until it is built with "
                          "`python -c 'import __graft_entry__ as g; g.build()'`", RuntimeWarning, stacklevel=2)
            got = _PythonCalls
        _calls = got
    return _calls


_STATUS_TEXT = {-1: "a required pointer is NULL", -2: "unsupported shape", -5: "pointer not aligned as required", -6: "HIP kernel launch failed",
                -8: "unknown option or value out of range", -9: "scratch memory too small"}


def check_seq(code, what):
    if code != 0:
        raise RuntimeError(f"{what}: {_STATUS_TEXT.get(code, 'unknown status')} (status {code})")


def set_seq_option(name, value):
    check_seq(load_seq().e2h_seq_set_option(name.encode(), int(value)), f"e2h_seq_set_option({name})")


def status_string(code):
    return load().e2h_status_string(code).decode()


def check(code, what):
    if code != 0:
        raise RuntimeError(f"{what}: {status_string(code)} (status {code})")


def set_option(name, value):
    check(load().e2h_set_option(name.encode(), int(value)), f"e2h_set_option({name})")
