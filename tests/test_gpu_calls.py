"""Small calls of the quantized linears in one native call (csrc/e2h_calls.cpp): the same bits as the Python path, and everything out of the ordinary left to it."""

import ctypes

import pytest
import torch

from easy_to_hard_amd import _lib, ops
from easy_to_hard_amd.quantize import WeightOnlyInt4Linear, WeightOnlyInt8Linear, linear_forward_int4

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _linear(mode, n=264, k=512, g=64, ikt=8):
    gen = torch.Generator().manual_seed(n + k)
    w = (torch.randn((n, k), generator=gen) * 0.05).to(torch.bfloat16).to(DEV)
    if mode == "int4":
        lin = WeightOnlyInt4Linear(k, n, bias=False, groupsize=g, inner_k_tiles=ikt, padding=False)
        lin.weight, lin.scales_and_zeros = ops.int4_quantize_pack(w, g, ikt)
    else:
        lin = WeightOnlyInt8Linear(k, n)
        q, scales = ops.int8_quantize_per_channel(w)
        lin.weight, lin.scales = q, scales.to(torch.bfloat16)
    return lin


def _native(lin, x):
    if isinstance(lin, WeightOnlyInt4Linear):
        return _lib.calls().int4_linear(x, lin.weight, lin.scales_and_zeros, lin.groupsize, lin.out_features)
    return _lib.calls().int8_linear(x, lin.weight, lin.scales, lin.out_features)


def _python(lin, x):
    rows = x.reshape(-1, x.shape[-1])
    if isinstance(lin, WeightOnlyInt4Linear):
        y = linear_forward_int4(rows, lin.weight, lin.scales_and_zeros, lin.out_features, lin.groupsize)
    else:
        y = ops.int8_mm_direct(rows, lin.weight, lin.scales)
    return y.reshape(*x.shape[:-1], lin.out_features)


def _x(*shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(shape[0])).to(torch.bfloat16).to(DEV)


@pytest.mark.parametrize("mode,g", [("int4", 32), ("int4", 64), ("int4", 128), ("int4", 256), ("int8", 0)])
@pytest.mark.parametrize("shape", [(1, 512), (512,), (1, 1, 512), (2, 3, 5, 512), (65, 512), (1023, 512)])
def test_native_calls_give_the_python_path_s_bits(mode, g, shape):
    lin, x = _linear(mode, g=g), _x(*shape)
    want = _python(lin, x)  # the first call of a stream makes its workspace
    got = _native(lin, x)
    assert got is not None and got.shape == want.shape and got.dtype == torch.bfloat16 and got.is_contiguous() and not got.requires_grad
    assert torch.equal(got, want) and torch.equal(lin(x), want)


@pytest.mark.parametrize("mode", ["int4", "int8"])
def test_what_is_out_of_the_ordinary_is_left_to_the_python_path(mode):
    lin, x = _linear(mode), _x(4, 512)
    want = lin(x)
    assert _native(lin, x) is not None
    for other in (x.float(), x[:, ::2].repeat(1, 2)[:, ::2], _x(4, 1024)[:, ::2], x[:0], _x(1024, 512), x.cpu(), x[:, :384]):
        assert _native(lin, other) is None
    assert torch.equal(lin(_x(4, 1024)[:, ::2]), lin(_x(4, 1024)[:, ::2].contiguous()))
    assert lin(x[:0]).shape == (0, 264)
    with pytest.raises(RuntimeError):
        lin(x[:, :384])

    class Sub(torch.Tensor):
        pass

    assert _native(lin, x.as_subclass(Sub)) is None
    with torch.utils._python_dispatch.TorchDispatchMode():
        assert _native(lin, x) is None

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert _native(lin, x) is None and torch.equal(lin(x), want)
    inside = []
    try:
        torch.vmap(lambda v: inside.append(_native(lin, v)) or v)(x)
    finally:
        assert inside == [None]
    traced = []
    torch.jit.trace(lambda v: traced.append(_native(lin, v)) or v + 1, (x,), check_trace=False)
    assert traced == [None]
    other = torch.cuda.Stream()  # no workspace yet: the Python path makes it
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        first = _native(lin, x)
        again = lin(x), _native(lin, x)
    torch.cuda.current_stream().wait_stream(other)
    assert first is None and torch.equal(again[0], want) and torch.equal(again[1], want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        none, y = _native(lin, x), lin(x)
    assert none is None
    for _ in range(3):
        y.zero_()
        graph.replay()
        assert torch.equal(y, want)


def test_modules_with_other_forms_of_weights_run_as_before():
    lin, x = _linear("int4", ikt=4), _x(4, 512)
    assert _native(lin, x) is None and lin(x).shape == (4, 264)
    lin = _linear("int4")
    want = lin(x)
    lin.weight = torch.nn.Parameter(lin._buffers.pop("weight"), requires_grad=False)  # not a buffer any more
    assert torch.equal(lin(x), want)
    lin = _linear("int4")
    lin.out_features = 256  # refused where the weight has another number of rows
    with pytest.raises(RuntimeError):
        lin(x)


@pytest.mark.parametrize("mode", ["int4", "int8"])
def test_a_failed_launch_is_reported_and_not_tried_again(mode):
    """The entry point's address is that of a function which launches nothing and returns a status."""
    lin, x = _linear(mode), _x(4, 512)
    want = lin(x)
    lib, calls, asked = _lib.load(), _lib.calls(), []

    def bind(int4, int8):
        calls.bind(*(ctypes.cast(f, ctypes.c_void_p).value for f in (int4, int8, lib.e2h_stream_capturing)), ops._workspaces, _lib.check)

    def answer(real, code):
        return ctypes.CFUNCTYPE(ctypes.c_int, *real.argtypes)(lambda *a: asked.append(code) or code)

    try:
        for code in (-6, -7):
            fakes = answer(lib.e2h_int4_mm, code), answer(lib.e2h_int8_mm, code)
            bind(*fakes)
            with pytest.raises(RuntimeError, match=rf"e2h_{mode}_mm: .*status {code}"):
                lin(x)
        assert asked == [-6, -7]
        fakes = answer(lib.e2h_int4_mm, -5), answer(lib.e2h_int8_mm, -5)  # refused arguments: the Python path's to meet
        bind(*fakes)
        assert torch.equal(lin(x), want) and asked == [-6, -7, -5]
    finally:
        bind(lib.e2h_int4_mm, lib.e2h_int8_mm)
    assert torch.equal(lin(x), want)


@pytest.mark.parametrize("mode,eager,captured", [("int4", (3, 157), (3, 157)), ("int8", (1, 1), (1, 1)), ("int8", (1, 1), (1, 20))])
def test_one_eager_pass_is_enough_for_a_capture(mode, eager, captured):
    """Also where every quantized linear of the pass runs in a launch that has no workspace of its own."""
    from easy_to_hard_amd.model import ModelArgs, random_quantized_transformer

    cfg = ModelArgs(block_size=256, vocab_size=8192, n_layer=1, n_head=32, n_local_heads=32, dim=4096, intermediate_size=5632)
    model = random_quantized_transformer(cfg, mode, device="cuda").requires_grad_(False)
    model.setup_caches(3, 256)
    at = lambda shape: (torch.randint(0, 8192, shape, device="cuda"), torch.arange(shape[1], device="cuda"))
    before = dict(ops._workspaces)
    ops._workspaces.clear()
    try:
        with torch.no_grad():
            model(*at(eager))
            torch.cuda.synchronize()
            assert ("capture", 0) in ops._workspaces
            ids, pos = at(captured)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                logits = model(ids, pos)
            for _ in range(3):
                ids.copy_(at(captured)[0])
                want = model(ids, pos)
                graph.replay()
                assert torch.equal(logits, want)
    finally:
        ops._workspaces.update(before)  # launches recorded earlier use them


def test_products_of_a_prompt_run_in_the_workspace_where_no_memory_is_left():
    lin, x = _linear("int4", n=2048, k=5632, g=128), _x(1000, 5632)
    rows = lambda defer: _lib.calls().int4_rows(x, lin.weight, lin.scales_and_zeros, 128, 2048, None, defer)
    assert ops.int4_rows_slices(1000, 2048, 5632, 128, 8) > 1
    want = lin(x)
    assert torch.equal(rows(False), want) and rows(True).dtype == torch.float32
    spare = lin(x)  # the result's place
    torch.cuda.empty_cache()
    del spare
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    try:
        assert rows(False) is None and rows(True) is None
        assert torch.equal(lin(x), want)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(rows(False), want)
