"""The streamed-weights matmul of decode batches (csrc/e2h_stream.h) at its edges: rows around the tiles of 8 and 16, columns and k that
end inside a tile, a step or a piece, few and many steps per wave.  Operands are small integers, so every float32 sum is exact and
the result has to be the exactly rounded one."""

import pytest
import torch

from easy_to_hard_amd import ops, seq_ops
from easy_to_hard_amd.linear import DecodeLinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROWS = [1, 7, 8, 9, 16, 17, 32, 33, 64]


def ints(shape, seed, dtype, most=4):
    gen = torch.Generator().manual_seed(seed)
    return torch.randint(-most, most + 1, shape, generator=gen).to(dtype).to(DEV)


def exact(x, w):
    """x w^T for integers: sums stay below 2^24, so float64 and float32 agree"""
    return x.double() @ w.double().t()


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("n,k", [(1, 8), (17, 24), (16, 64), (2, 72), (250, 136), (48, 520), (33, 1048), (4103, 256), (4111, 4104), (260, 16384)])
def test_bf16_linear_is_exact_on_integers(rows, n, k):
    x, w = ints((rows, k), rows + k, torch.bfloat16), ints((n, k), n + k, torch.bfloat16)
    want = exact(x, w).to(torch.bfloat16)
    got = seq_ops.linear(x, w)
    assert torch.equal(got, want)
    square = seq_ops.linear(x, w, seq_ops.ACT_SQUARE_RELU)
    assert torch.equal(square, seq_ops.square_relu_(want.clone()))
    capped = seq_ops.linear(x, w, seq_ops.ACT_SOFTCAP, 30.0)
    assert torch.equal(capped, seq_ops.softcap_(want.clone(), 30.0))


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("n,k", [(1, 16), (17, 48), (2, 128), (250, 144), (33, 1040), (4111, 4112), (40, 11008)])
def test_int8_mm_is_exact_on_integers(rows, n, k):
    x, w = ints((rows, k), rows + k, torch.bfloat16), ints((n, k), n + k, torch.int8)
    scales = torch.full((n,), 0.5, dtype=torch.bfloat16, device=DEV)
    want = (exact(x, w).to(torch.bfloat16).float() * 0.5).to(torch.bfloat16)
    assert torch.equal(ops.int8_mm_direct(x, w, scales), want)


@pytest.mark.parametrize("rows", [65, 128, 200])
@pytest.mark.parametrize("n,k", [(1, 128), (16, 384), (17, 256), (48, 4096), (64, 128), (65, 384), (129, 256)])
def test_int8_mm_of_many_rows_and_few_columns_is_exact_on_integers(rows, n, k):
    """one to all four waves of the last workgroup have columns; odd and even numbers of chunks"""
    test_int8_mm_is_exact_on_integers(rows, n, k)


@pytest.mark.parametrize("k", [128, 4096, 4224])
def test_int8_extreme_codes(k):
    """codes -128 and 127 keep their sign and value; the products cancel in pairs"""
    w = torch.tensor([-128, 127], dtype=torch.int8).repeat(24, k // 2).to(DEV)
    x = torch.tensor([127.0, 128.0], dtype=torch.bfloat16).repeat(5, k // 2).to(DEV)
    assert torch.equal(ops.int8_mm_direct(x, w, torch.ones(24, dtype=torch.bfloat16, device=DEV)), torch.zeros((5, 24), dtype=torch.bfloat16, device=DEV))


def test_a_rows_result_depends_on_no_other_row_and_on_no_other_column():
    gen = torch.Generator().manual_seed(3)
    x, w = (torch.randn(s, generator=gen).to(torch.bfloat16).to(DEV) for s in ((64, 4096), (4096, 4096)))
    full = seq_ops.linear(x, w)
    for rows in (1, 8, 16, 31):
        assert torch.equal(seq_ops.linear(x[:rows], w), full[:rows])
    assert torch.equal(seq_ops.linear(x, w[:700].contiguous()), full[:, :700])


def test_module_routes_and_refusals():
    """the module takes its own kernel only for what that is made for, and gives what nn.Linear gives everywhere"""
    gen = torch.Generator().manual_seed(4)
    lin = DecodeLinear(256, 96, bias=False).to(DEV, torch.bfloat16).requires_grad_(False)
    x = torch.randn((3, 5, 256), generator=gen).to(torch.bfloat16).to(DEV)
    ref = torch.nn.functional.linear(x.float(), lin.weight.float())
    assert seq_ops.linear_streams(x, lin.weight)
    for inp in (x, x.transpose(0, 1), torch.cat([x, x], -1)[..., 128:384]):  # other orders and strides
        y, want = lin(inp), torch.nn.functional.linear(inp.float(), lin.weight.float())
        assert y.shape == want.shape and (y.float() - want).abs().max() <= 2 ** -8 * want.abs().max()
    flat = torch.empty((4 * 256 + 1,), dtype=torch.bfloat16, device=DEV)[1:].view(4, 256)  # not 16-byte aligned
    flat.copy_(x[0, :4])
    assert torch.equal(lin(flat), lin(x[0, :4].contiguous()))
    many = x.repeat(1, 5, 1)
    assert not seq_ops.linear_streams(many, lin.weight) and lin(many).shape == (3, 25, 96)
    assert lin(x[:0]).shape == (0, 5, 96)
    xg = x.clone().requires_grad_(True)
    assert not seq_ops.linear_streams(xg, lin.weight)
    lin(xg).float().sum().backward()
    assert xg.grad is not None
    assert not seq_ops.linear_streams(x.float(), lin.weight.float())
    assert (lin.float()(x.float()) - ref).abs().max() <= 1e-4 * ref.abs().max()
    with pytest.raises(RuntimeError):
        seq_ops.linear(torch.zeros((65, 256), dtype=torch.bfloat16, device=DEV), torch.zeros((96, 256), dtype=torch.bfloat16, device=DEV))


def test_module_shows_transforms_and_traces_what_nn_linear_shows():
    """forward-mode derivatives, function transforms, dispatch modes, traces and subclasses see the product: none of them may end in a
    launch that they know nothing of"""
    from torch.autograd import forward_ad
    from torch.utils.flop_counter import FlopCounterMode

    gen = torch.Generator().manual_seed(6)
    lin = DecodeLinear(256, 96, bias=False).to(DEV, torch.bfloat16).requires_grad_(False)
    x, t = (torch.randn((5, 256), generator=gen).to(torch.bfloat16).to(DEV) for _ in range(2))
    assert seq_ops.linear_streams(x, lin.weight)
    want = torch.nn.functional.linear(t, lin.weight)
    with forward_ad.dual_level():
        assert torch.equal(forward_ad.unpack_dual(lin(forward_ad.make_dual(x, t))).tangent, want)
        weight = torch.randn((96, 256), generator=gen).to(torch.bfloat16).to(DEV)
        dual = torch.func.functional_call(lin, {"weight": forward_ad.make_dual(lin.weight, weight)}, (x,))
        assert torch.equal(forward_ad.unpack_dual(dual).tangent, torch.nn.functional.linear(x, weight))
    assert torch.equal(torch.func.jvp(lin, (x,), (t,))[1], want)
    seen = []

    def route(row):
        seen.append(seq_ops.linear_streams(row, lin.weight))
        return row

    torch.func.vmap(route)(x)
    assert seen == [False]
    with FlopCounterMode(display=False) as flops:
        lin(x)
    assert flops.get_total_flops() == 2 * 5 * 96 * 256
    assert torch.equal(torch.jit.trace(lin, x, check_trace=False)(t), want)

    class Named(torch.Tensor):
        pass

    assert type(lin(x.as_subclass(Named))) is Named


@pytest.mark.parametrize("act,cap", [(seq_ops.ACT_NONE, 0.0), (seq_ops.ACT_SQUARE_RELU, 0.0), (seq_ops.ACT_SOFTCAP, 30.0)])
def test_a_weight_that_the_kernel_does_not_read_is_not_copied(act, cap):
    """rows cut out of wider ones and a weight off 16 bytes, as views of a checkpoint's buffer are: integers, so the result is exact"""
    n, k = 4096, 4096
    x = ints((5, k), 1, torch.bfloat16, 1)
    wide = ints((n, k + 8), 2, torch.bfloat16, 1)
    shifted = torch.empty((n * k + 1,), dtype=torch.bfloat16, device=DEV)[1:].view(n, k)
    shifted.copy_(wide[:, :k])
    aligned = shifted.clone()
    want = seq_ops.linear(x, aligned, act, cap)
    for w in (wide[:, :k], shifted, aligned.t().contiguous().t()):
        seq_ops.linear(x, w, act, cap)  # the library's own workspace
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        got = seq_ops.linear(x, w, act, cap)
        assert torch.cuda.max_memory_allocated() - before < n * k
        assert torch.equal(got, want)


@pytest.mark.parametrize("m,k", [(1, 1 << 23), (17, (1 << 23) + 128), (33, 1 << 23), (3, 1 << 25)])
def test_int8_fused_launches_take_very_long_rows(m, k):
    """rows of 2^23 values and more, where a workgroup's tiles have to stay below 2^31 bytes: some 64 values per row of x are not zero, so
    the sums of integers are exact; gate, K halves and the plain form"""
    n = 48
    gen = torch.Generator().manual_seed(k + m)
    x = torch.zeros((m, k), dtype=torch.bfloat16, device=DEV)
    at = torch.unique(torch.cat([torch.randint(0, k, (62,), generator=gen), torch.tensor([0, k - 1])])).to(DEV)
    x[:, at] = ints((m, len(at)), 3, torch.bfloat16)
    w, w3 = (torch.randint(-4, 5, (n, k), dtype=torch.int8, device=DEV, generator=torch.Generator(DEV).manual_seed(s)) for s in (1, 2))
    scales = torch.full((n,), 0.5, dtype=torch.bfloat16, device=DEV)
    want, want3 = (exact(x[:, at], q[:, at]) for q in (w, w3))
    lin, up = ((t.to(torch.bfloat16).float() * 0.5).to(torch.bfloat16) for t in (want, want3))
    assert torch.equal(ops.int8_mm_direct(x, w, scales), lin)
    assert torch.equal(ops.int8_mm_silu_gate(x, w, scales, w3, scales), ops.silu_mul(lin, up))
    sums = ops.int8_mm_partials(x, w, scales, ops._lib.load().e2h_int8_mm_partial_slices(m, n, k)).partials
    assert torch.equal(sums.double().sum(0), want)


def test_sliced_launches_change_a_row_by_float32_rounding_at_most():
    """From 17 rows on K is cut over four workgroups (N <= 4096, K >= 8192): among those a row depends on no other row and no other column;
    beside one workgroup's sum the order differs.  Either is within N 2^-24 A of the exact sum (N <= K / 32 + 12 additions in a chain, A
    the sum of the magnitudes), and rounding to bfloat16 adds 2^-8 of the value."""
    gen = torch.Generator().manual_seed(8)
    k = 8192
    x, w = (torch.randn(s, generator=gen).to(torch.bfloat16).to(DEV) for s in ((64, k), (4112, k)))
    narrow = w[:4096]
    full = seq_ops.linear(x, narrow)
    for rows in (17, 32, 33):
        assert torch.equal(seq_ops.linear(x[:rows], narrow), full[:rows])
    assert torch.equal(seq_ops.linear(x, w[:700]), full[:, :700])
    bound = 2 * (k / 32 + 12) * 2.0**-24 * (x.double().abs() @ narrow.double().abs().t()) + 2.0**-8 * full.double().abs()
    assert ((seq_ops.linear(x[:16], narrow).double() - full[:16].double()).abs() <= bound[:16]).all()
    assert ((seq_ops.linear(x, w)[:, :4096].double() - full.double()).abs() <= bound).all()
