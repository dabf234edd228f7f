"""The many-row int4 matmul (csrc/e2h_int4_gemm.hip) at its edges: rows around its workgroups of 64 and 128, columns that end inside a
workgroup, odd counts of 128-wide k blocks, K slices, and scales that its running units do not carry.

Operands are chosen so that every product and sum is a small multiple of a power of two (codes, x in -2 .. 2, scales 2^-3 .. 2^3,
zeros in quarters), below 2^24 of its unit in any order: the result has to be the exactly rounded one."""

import pytest
import torch

from easy_to_hard_amd import _lib, ops
from oracle import quant_oracle as qo

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def many_row_kernel():
    _lib.set_option("int4_gemm32_min_rows", 1)
    yield
    _lib.set_option("int4_gemm32_min_rows", 0)
    _lib.set_option("int4_k_slices", 0)
    _lib.set_option("int4_gemm_tile", 0)


def _case(m, n, k, g, seed=5, low=-3, high=3):
    gen = torch.Generator().manual_seed(seed + m + n + k + g)
    codes = torch.randint(0, 16, (n, k), generator=gen, dtype=torch.int32)
    scale = torch.exp2(torch.randint(low, high + 1, (k // g, n), generator=gen).float())
    zero = torch.randint(-8, 9, (k // g, n), generator=gen).float() / 4
    x = torch.randint(-2, 3, (m, k), generator=gen).to(torch.bfloat16).to(DEV)
    return codes, scale, zero, x


def _run(codes, scale, zero, x, g):
    packed = torch.from_numpy(qo.int4_tile_pack(codes.numpy(), 8)).to(DEV)
    sz = torch.stack([scale, zero], dim=-1).to(torch.bfloat16).contiguous().to(DEV)
    n, k = codes.shape
    w = ((codes.double() - 8).view(n, k // g, g) * scale.double().t()[:, :, None] + zero.double().t()[:, :, None]).view(n, k).to(DEV)
    return ops.int4_mm(x, packed, g, sz), x.double() @ w.t()


# slices: at most, as many as there are blocks of 128 k; tile 128: 128 rows per workgroup but at group size 32
@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("slices", [1, 2, 8])
@pytest.mark.parametrize("tile", [0, 128])
@pytest.mark.parametrize("m,n,k", [(65, 8, 128), (64 + 1, 264, 384), (128, 256, 1024), (129, 520, 1152), (471, 1032, 2176)])
def test_exact_on_dyadic_operands(many_row_kernel, g, slices, tile, m, n, k):
    _lib.set_option("int4_k_slices", slices)
    _lib.set_option("int4_gemm_tile", tile)
    got, want = _run(*_case(m, n, k, g), g)
    assert torch.equal(got, want.to(torch.bfloat16))


# slices of an odd number of blocks of 128 k, so that pairs of groups are cut; (256, 513, 12288, 1024) has no room for sums of slices and keeps one
@pytest.mark.parametrize("slices", [0, 1, 2, 4])
@pytest.mark.parametrize("tile", [0, 96, 128])
@pytest.mark.parametrize("g,m,n,k", [(256, 130, 3080, 768), (256, 471, 1032, 2304), (256, 513, 12288, 1024), (128, 470, 12296, 384), (64, 195, 5128, 640), (64, 97, 8200, 1408)])
def test_pairs_of_groups_and_96_row_workgroups_are_exact(many_row_kernel, g, m, n, k, tile, slices):
    _lib.set_option("int4_k_slices", slices)
    _lib.set_option("int4_gemm_tile", tile)
    got, want = _run(*_case(m, n, k, g), g)
    assert torch.equal(got, want.to(torch.bfloat16))


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("slices", [1, 2])
def test_scales_outside_the_running_units(many_row_kernel, g, slices):
    """a scale of zero, and columns of scales that the units do not carry, whose workgroups form every group's sum by itself.  Columns whose
    scales are finite stay exact; a column with an infinite or NaN scale is not finite, its neighbours are untouched."""
    m, n, k = 130, 528, 1024
    _lib.set_option("int4_k_slices", slices)
    codes, scale, zero, x = _case(m, n, k, g)
    scale[0, 3] = 0.0
    zero[:, 5], scale[:, 5] = 0.0, 2.0**-100
    zero[:, 7], scale[:, 7] = 0.0, 2.0**-101
    zero[:, 260], scale[:, 260] = 0.0, 2.0**40
    scale[-1, 300] = float("inf")
    scale[-1, 301] = float("nan")
    got, want = _run(codes, scale, zero, x, g)
    finite = torch.ones(n, dtype=torch.bool)
    finite[[300, 301]] = False
    assert torch.equal(got[:, finite], want[:, finite].to(torch.bfloat16))
    assert not torch.isfinite(got[:, 301]).any() and not torch.isfinite(got[:, 300]).all()


def test_error_is_that_of_the_final_rounding(many_row_kernel):
    """random scales over a wide range and x with a mean: against 64 bits the relative error stays that of rounding to bfloat16,
    at most 2^-9 per value plus the float32 sums' share (K = 4096 terms of up to 31 |x s|, 2^-24 each, far below 2^-12 here)"""
    gen = torch.Generator().manual_seed(9)
    m, n, k, g = 200, 512, 4096, 64
    codes = torch.randint(0, 16, (n, k), generator=gen, dtype=torch.int32)
    scale = torch.exp2(torch.rand((k // g, n), generator=gen) * 16 - 14).to(torch.bfloat16).float()
    zero = torch.randn((k // g, n), generator=gen).to(torch.bfloat16).float()
    x = (torch.randn((m, k), generator=gen) + 1).to(torch.bfloat16).to(DEV)
    got, want = _run(codes, scale, zero, x, g)
    assert (got.double() - want).norm() <= 2**-9 * want.norm()


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("slices", [1, 2])
@pytest.mark.parametrize("tile", [0, 128])
def test_sums_that_only_the_running_units_cannot_hold(many_row_kernel, g, slices, tile):
    """A sum in units of its column's scale may leave float32's range although the sum itself does not: a large zero beside a small scale,
    and rows of x near the end of the type.  All terms of a column are multiples of one power of two below 2^24 of it
    (K * 31 * 2 * 2^6 = 2^22 for the products, and the columns with large zeros have products far below half a unit of the sum), so results are exact."""
    m, n, k = 150, 528, 1024
    _lib.set_option("int4_k_slices", slices)
    _lib.set_option("int4_gemm_tile", tile)
    codes, scale, zero, x = _case(m, n, k, g, low=-20, high=-14)
    zero = zero.mul(4) * 2.0**-20
    for col, z in ((5, 2.0**100), (259, -(2.0**99)), (527, 2.0**110)):
        scale[:, col], zero[:, col] = 2.0**-26, z
    codes[[5, 259, 527]] = 8
    x[0], x[70] = 2.0**114, x[70] * 2.0**112  # a group of products alone stays below 128 * 31 * 2^114 < 2^126
    x[149] = 0
    cols = torch.ones(n, dtype=torch.bool)
    cols[[5, 259, 527]] = False
    got, want = _run(codes, scale, zero, x, g)
    assert want[:, cols].abs().max() < 2.0**127 and want[0, cols].abs().max() > 2.0**100
    assert torch.equal(got[:, cols], want[:, cols].to(torch.bfloat16))
    small = torch.ones(m, dtype=torch.bool)
    small[[0, 70]] = False
    assert torch.equal(got[small][:, ~cols], want[small][:, ~cols].to(torch.bfloat16))


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_a_row_that_is_not_finite_touches_no_other(many_row_kernel, value):
    codes, scale, zero, x = _case(140, 264, 512, 64)
    x[3, 77] = value
    got, want = _run(codes, scale, zero, x, 64)
    rest = torch.arange(140) != 3
    assert not torch.isfinite(got[3]).any()
    assert torch.equal(got[rest], want[rest].to(torch.bfloat16))


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("slices", [1, 2])
@pytest.mark.parametrize("tile", [0, 128])
def test_groups_whose_scale_is_zero_add_nothing(many_row_kernel, g, slices, tile):
    """the first group, the last, neighbours, every second one and all of a column, a negative zero, and scales at the ends of what
    the running units carry; only a row's zero-point term is left where all scales are zero"""
    m, n, k = 150, 528, 1152
    _lib.set_option("int4_k_slices", slices)
    _lib.set_option("int4_gemm_tile", tile)
    codes, scale, zero, x = _case(m, n, k, g)
    scale[0, 3] = scale[-1, 4] = scale[2:5, 5] = 0.0
    scale[::2, 6] = scale[1::2, 7] = 0.0
    scale[:, 8] = 0.0
    scale[:, 300], zero[:, 300] = 0.0, 0.0
    scale[1, 301] = -0.0
    zero[:, 400:402] = 0.0
    scale[:, 400], scale[:, 401] = 2.0**-100, 2.0**13
    scale[1::2, 400] = 0.0
    got, want = _run(codes, scale, zero, x, g)
    assert torch.equal(got, want.to(torch.bfloat16))
    assert not got[:, 300].any()


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("n,k", [(1032, 1024), (4096, 1024), (4096, 4096)])
def test_a_row_differs_by_float32_rounding_at_most_between_row_counts(g, n, k):
    """The kernels for 1 .. 64 rows, 65 and more, many, and every choice of K slices add the same exact products in another order.  A sum
    of N additions is within N 2^-24 A of the exact one, A the sum of the magnitudes added, and rounding to bfloat16 adds 2^-8 of the
    value between two results.  A chain has at most K / 16 products' steps, two additions per group and 16 for the parts that
    meet; the magnitudes are those of 128 + q <= 143 and of z - 136 s.  The same call gives the same bits."""
    m = 1030
    gen = torch.Generator().manual_seed(n + k + g)
    codes = torch.randint(0, 16, (n, k), generator=gen, dtype=torch.int32)
    scale = (torch.rand((k // g, n), generator=gen) * 0.02 + 0.01).to(torch.bfloat16)
    zero = (torch.randn((k // g, n), generator=gen) * 0.02).to(torch.bfloat16)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV)
    packed = torch.from_numpy(qo.int4_tile_pack(codes.numpy(), 8)).to(DEV)
    sz = torch.stack([scale, zero], dim=-1).contiguous().to(DEV)
    full = ops.int4_mm(x, packed, g, sz)
    size = (143 * scale + 136 * scale + zero.abs()).double().to(DEV)  # [K / g, N]
    magnitude = x.double().abs().view(m, k // g, g).sum(-1) @ size
    bound = 2 * (k / 16 + 2 * k / g + 16) * 2.0**-24 * magnitude + 2.0**-8 * full.double().abs()
    for rows in (1, 16, 17, 33, 64, 65, 128, 129, 300, 512, 640):
        part = ops.int4_mm(x[:rows], packed, g, sz)
        assert torch.equal(part, ops.int4_mm(x[:rows], packed, g, sz))
        assert ((part.double() - full[:rows].double()).abs() <= bound[:rows]).all()


# ---- both matrices of a gated feed-forward in one launch --------------------------------------------------------------------------------
# workgroups of 64, 96 and 128 rows (the last three), columns that end inside a wave's 32 and a workgroup's 128, odd counts of 128-wide k blocks; scales up to 2^15
# leave the running units (above 2^13) in some workgroups only
@pytest.mark.parametrize("g", [32, 64, 128, 256])
@pytest.mark.parametrize("high", [-4, 15])
@pytest.mark.parametrize("m,n,k", [(65, 8, 256), (129, 264, 768), (471, 1032, 1280), (190, 12296, 256), (200, 12296, 512), (1000, 2056, 256)])
def test_gated_rows_are_the_two_exact_products_gated(g, high, m, n, k):
    """Dyadic operands as above: both products have to be exactly rounded, and the gate is what ops.silu_mul makes of them."""
    halves = [_case(m, n, k, g, seed=seed, low=-9, high=-4) for seed in (5, 77)]
    halves[1][1][:, 3::97] = 2.0 ** high
    halves[1][2][:, 3::97] = 0.0  # (multiples of 2^15 beside quarters would not fit 24 bits; without them these columns are multiples of their scale below 2^24 of it)
    x = halves[0][3]
    weights = []
    for codes, scale, zero, _ in halves:
        weights += [torch.from_numpy(qo.int4_tile_pack(codes.numpy(), 8)).to(DEV), torch.stack([scale, zero], dim=-1).to(torch.bfloat16).contiguous().to(DEV)]
    got = ops.int4_mm_silu_gate_rows(x, *weights, g)
    assert got is not None  # these sizes are taken
    a, b = (x.double() @ ((c.double() - 8).view(n, k // g, g) * s.double().t()[:, :, None] + z.double().t()[:, :, None]).view(n, k).to(DEV).t() for c, s, z, _ in halves)
    assert torch.equal(got, ops.silu_mul(a.to(torch.bfloat16), b.to(torch.bfloat16)))


@pytest.mark.parametrize("g", [32, 64, 128, 256])
def test_gated_rows_form_what_float32_units_do_not_hold(g):
    """Infinite and NaN scales, sums that leave float32's range only in units of a scale, rows of x that are not finite: as two calls of the kernel give them."""
    m, n, k = 471, 1032, 1280
    gen = torch.Generator().manual_seed(g)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16)
    x[3, 5], x[200, 7] = float("inf"), float("nan")
    w = [ops.int4_quantize_pack((torch.randn((n, k), generator=gen) * 0.02).to(torch.bfloat16).to(DEV), g, 8) for _ in range(2)]
    w[0][1][0, 17, 0], w[0][1][-1, 600, 0], w[1][1][0, 333, 0] = float("inf"), float("nan"), 2.0 ** -20
    w[1][1][0, 333, 1] = 2.0 ** 100
    x = x.to(DEV)
    got = ops.int4_mm_silu_gate_rows(x, *w[0], *w[1], g)
    _lib.set_option("int4_gemm32_min_rows", 1)
    try:
        want = ops.silu_mul(*(ops.int4_mm(x, p, g, sz) for p, sz in w))
    finally:
        _lib.set_option("int4_gemm32_min_rows", 0)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    fine = torch.isfinite(want)
    assert torch.equal(got[~fine & ~torch.isnan(want)], want[~fine & ~torch.isnan(want)])
    # one product may differ by a rounding to bfloat16 (K slices of the two calls), the gate of it by its slope: at most 1.1 in relative size away from its zero
    assert ((got[fine].double() - want[fine].double()).norm() <= 2 ** -8 * want[fine].double().norm()).item()


def test_gated_rows_leave_watched_modules_and_other_forms_to_the_modules():
    from easy_to_hard_amd.model import FeedForward, ModelArgs
    from easy_to_hard_amd.quantize import WeightOnlyInt4QuantHandler, prepare_int4_weight_and_scales_and_zeros

    args = ModelArgs(dim=512, intermediate_size=1024, n_head=4, n_layer=1)
    ff = FeedForward(args)
    WeightOnlyInt4QuantHandler(ff, groupsize=64).convert_for_runtime()
    gen = torch.Generator().manual_seed(1)
    for lin in (ff.w1, ff.w2, ff.w3):
        w = (torch.randn((lin.out_features, lin.in_features), generator=gen) * 0.05).to(torch.bfloat16).to(DEV)
        lin.weight, lin.scales_and_zeros = prepare_int4_weight_and_scales_and_zeros(w, 64, 8)
    x = torch.randn((3, 40, 512), generator=gen).to(torch.bfloat16).to(DEV)
    whole = ff(x)
    assert ff._gate_rows(x).shape == (3, 40, 1024)
    seen = []
    handle = ff.w3.register_forward_hook(lambda *_: seen.append(1))
    assert ff._gate_rows(x) is None
    assert seen == [] and (ff(x).double() - whole.double()).norm() <= 2 ** -7 * whole.double().norm() and seen == [1]
    handle.remove()
    assert ff._gate_rows(x[:, :20]) is None  # 60 rows: the decode launch
    assert ff._gate_rows(x.float()) is None and ff._gate_rows(x[..., :384]) is None
    strided = x.transpose(0, 1)
    assert torch.equal(ff._gate_rows(strided), ff._gate_rows(x).transpose(0, 1))


def test_gated_rows_are_left_to_calls_that_are_faster():
    """Group size 256 on small weights, whose products run on 16 x 16 tiles."""
    from easy_to_hard_amd.model import FeedForward, ModelArgs
    from easy_to_hard_amd.quantize import WeightOnlyInt4QuantHandler, prepare_int4_weight_and_scales_and_zeros

    ff = FeedForward(ModelArgs(dim=1024, intermediate_size=1408, n_head=8, n_layer=1))
    WeightOnlyInt4QuantHandler(ff, groupsize=128).convert_for_runtime()
    gen = torch.Generator().manual_seed(2)
    for lin in (ff.w1, ff.w3):
        lin.groupsize = 256
    for lin in (ff.w1, ff.w2, ff.w3):
        w = (torch.randn((lin.out_features, lin.in_features), generator=gen) * 0.05).to(torch.bfloat16).to(DEV)
        lin.weight, lin.scales_and_zeros = prepare_int4_weight_and_scales_and_zeros(w, lin.groupsize, 8)
    x = torch.randn((2, 64, 1024), generator=gen).to(torch.bfloat16).to(DEV)
    assert ff._gate_rows(x) is None
    assert torch.equal(ff(x), ff.w2(ops.silu_mul(ff.w1(x), ff.w3(x))))


# ---- weights unpacked to float16 first (csrc/e2h_unpacked_gemm.hip) ---------------------------------------------------------------------

def _unpacked(codes, scale, zero, x, g, flag=None):
    """(with scratch memory, without, bytes of it), through the C interface; flag: a list that is given the scratch memory's first number, not zero where the other
    kernel was asked for"""
    lib = _lib.load()
    packed = torch.from_numpy(qo.int4_tile_pack(codes.numpy(), 8)).to(DEV)
    sz = torch.stack([scale, zero], dim=-1).to(torch.bfloat16).contiguous().to(DEV)
    (m, k), n, ws = x.shape, codes.shape[0], ops._workspace(x.device)
    need = lib.e2h_int4_mm_scratch_bytes(m, n, k, g, 8)
    scratch = torch.full((max(need, 16),), 255, dtype=torch.uint8, device=DEV)  # a NaN wherever it is read unwritten
    out = []
    for given in (need, 0):
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        rc = lib.e2h_int4_mm_scratch(ops._ptr(x), ops._ptr(packed), ops._ptr(sz), ops._ptr(y), m, n, k, g, 8, ops._ptr(ws), ws.numel(), ops._ptr(scratch), given, ops._stream(x))
        assert rc == 0
        if flag is not None and given:
            flag.append(int(scratch[:4].view(torch.int32)))
        out.append(y)
    return (*out, need)


def _double(codes, scale, zero, x, g, rows):
    n, k = codes.shape
    w = ((codes.double() - 8).view(n, k // g, g) * scale.double().t()[:, :, None] + zero.double().t()[:, :, None]).view(n, k).to(DEV)
    return x[rows].double() @ w.t()


UNPACKED = [(70000, 264, 256), (70000, 8, 256), (66049, 520, 512)]  # the shortest K, few and ragged columns, a last tile of one row


@pytest.mark.parametrize("g", [32, 64, 128, 256])
@pytest.mark.parametrize("m,n,k", UNPACKED)
def test_unpacked_weights_are_exact_on_dyadic_operands(m, n, k, g):
    case = _case(m, n, k, g)
    got, other, need = _unpacked(*case, g)
    assert need > 0 and torch.equal(got, other)
    rows = torch.cat([torch.arange(0, 300), torch.arange(m - 300, m)]).to(DEV)
    assert torch.equal(got[rows], _double(*case, g, rows).to(torch.bfloat16))


@pytest.mark.parametrize("g", [32, 128, 256])
def test_unpacked_weights_round_once(g):
    """Rows in units from 2^-60 to 2^60 with values 2^-28 .. 1 of them, scales over 2^-20 .. 1 in one column, zeros: all held without rounding, so the error is that of
    the result's rounding (half a unit of eight significant bits: 2^-8 of the value at most) and of float32 sums of K = 512 terms (2^-24 each)."""
    m, n, k = 66049, 264, 512
    gen = torch.Generator().manual_seed(3)
    codes = torch.randint(0, 16, (n, k), generator=gen, dtype=torch.int32)
    scale = torch.exp2(torch.rand((k // g, n), generator=gen) * 20 - 20).to(torch.bfloat16).float()
    zero = (torch.randn((k // g, n), generator=gen) * 8 * scale).to(torch.bfloat16).float()
    zero[zero.abs() < 2.0**-30 * torch.maximum(8 * scale, 128 * zero.abs()).max(0).values] = 0.0  # smaller ones send the call to the other kernel
    x = torch.exp2(torch.randint(-28, 1, (m, k), generator=gen).float() + torch.randint(-60, 61, (m, 1), generator=gen).float()).to(torch.bfloat16)
    x = (x * (torch.randint(0, 2, (m, k), generator=gen) * 2 - 1)).to(DEV)
    x[5] = 0
    got, _, need = _unpacked(codes, scale, zero, x, g)
    rows = torch.cat([torch.arange(0, 512), torch.arange(m - 512, m)]).to(DEV)
    want = _double(codes, scale, zero, x, g, rows)
    err, size = (got[rows].double() - want).abs(), want.abs()
    terms = (x[rows].double().abs() @ ((codes.double() - 8).abs().view(n, k // g, g) * scale.double().t()[:, :, None] + zero.double().abs().t()[:, :, None]).view(n, k).to(DEV).t())
    assert need > 0 and bool((err <= 2**-8 * size + 2**-15 * terms).all()) and bool((got[5] == 0).all())
    assert (err / terms.clamp(min=1e-300)).mean() < 2**-9


@pytest.mark.parametrize("count", [14, 15])
def test_unpacked_x_keeps_what_its_float16_values_lack(count):
    """Values of x far below their row's largest, which meets a group whose scale and zero are zero in the first columns: there they alone are the result.  One to fourteen of
    them in one and two groups, which with the groups' sums a row's list of sixteen holds, and fifteen in three, which it does not; up to 2^-174 of the largest.  2^-31 of it
    is held by the float16 values themselves.  Every sum is of at most 16 multiples of one power of two, so the result is the exactly rounded one."""
    m, n, k, g = 66049, 264, 512, 128
    codes, scale, zero, x = _case(m, n, k, g)
    scale[0, :130], zero[0, :130] = 0.0, 0.0
    special = {0: (2.0**110, 2.0**-64, 10), 77: (1.0, 2.0**-40, 1), 300: (-1.0, -(2.0**-31), 16), 4097: (2.0**40, 3 * 2.0**-20, count), m - 1: (2.0**-30, 2.0**-70, 5)}
    for row, (largest, small, n_small) in special.items():
        x[row] = 0
        x[row, row % g] = largest
        x[row, k - 1 - 19 * torch.arange(n_small)] = small
    flag = []
    got, _, need = _unpacked(codes, scale, zero, x, g, flag)
    rows = torch.tensor(list(special) + [1, 78, 4096, m - 2], device=DEV)
    assert need > 0 and (flag[0] != 0) == (count > 14)
    assert torch.equal(got[rows][:, :130], _double(codes, scale, zero, x, g, rows)[:, :130].to(torch.bfloat16))


@pytest.mark.parametrize("what", ["scale ratio", "infinite scale", "NaN zero", "tiny zero", "large scales", "small scales", "infinite x", "NaN x", "small x"])
def test_what_float16_does_not_hold_is_left_to_the_other_kernel(what):
    """bit for bit what the call without scratch memory gives, wherever in x or the weights it stands"""
    m, n, k, g = 70000, 264, 256, 128
    codes, scale, zero, x = _case(m, n, k, g)
    if what == "scale ratio":
        scale[1, 77], zero[1, 77] = 2.0**-40, 0.0
    elif what == "infinite scale":
        scale[0, 263] = float("inf")
    elif what == "NaN zero":
        zero[1, 0] = float("nan")
    elif what == "tiny zero":
        zero[0, 100] = 2.0**-60
    elif what == "large scales":
        scale[:, 3], zero[:, 3] = 2.0**50, 0.0
    elif what == "small scales":
        scale[:, 3], zero[:, 3] = 2.0**-70, 0.0
    elif what == "infinite x":
        x[m - 1, 255] = float("inf")
    elif what == "NaN x":
        x[0, 0] = float("nan")
    else:
        x[12345] = 2.0**-50
        x[12345, 9] = 1.0
    got, other, need = _unpacked(codes, scale, zero, x, g)
    assert need > 0
    same = torch.where(torch.isnan(other), torch.isnan(got), got == other)
    assert bool(same.all())


@pytest.mark.parametrize("exponent,held", [(-50, False), (-49, True), (41, True), (42, False)])
def test_units_of_columns_on_both_sides_of_their_ends(exponent, held):
    """A column of scales 2^-49 .. 2^41 (8 s from 2^-46 to below 2^45) has a unit, one beyond sends the call to the other kernel; exact either way."""
    m, n, k, g = 66049, 264, 512, 128
    codes, scale, zero, x = _case(m, n, k, g)
    scale[:, 3], zero[:, 3] = 2.0**exponent, 0.0
    flag = []
    got, _, need = _unpacked(codes, scale, zero, x, g, flag)
    assert need > 0 and (flag[0] == 0) == held
    rows = torch.tensor([0, 255, 4097, m - 1], device=DEV)
    assert torch.equal(got[rows], _double(codes, scale, zero, x, g, rows).to(torch.bfloat16))


@pytest.mark.parametrize("g", [32, 128])
def test_rows_of_an_unpacked_call_stand_alone(g):
    """Rows that the float16 form does not take (a NaN, an infinity, values over 2^60) leave every other row as it is without them, bit for bit, first, last and
    neighbours of them included, with operands whose sums are rounded.  The wide rows are as exact as float32 sums are: K = 512 terms, each within 2^-15 of the magnitudes added."""
    m, n, k = 66049, 264, 512
    gen = torch.Generator().manual_seed(g)
    codes = torch.randint(0, 16, (n, k), generator=gen, dtype=torch.int32)
    scale = (torch.rand((k // g, n), generator=gen) * 0.02 + 0.01).to(torch.bfloat16).float()
    zero = (torch.randn((k // g, n), generator=gen) * 0.02).to(torch.bfloat16).float()
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV)
    flag = []
    plain, _, need = _unpacked(codes, scale, zero, x, g, flag)
    wide = [1, 128, 40000, *range(512, 768)]  # a whole block of the product's rows among them
    odd = [0, 127, 4100, m - 1]
    for row in wide:
        x[row] *= torch.exp2(torch.randint(-60, 1, (k,), generator=gen).float()).to(torch.bfloat16).to(DEV)
    x[0, 3] = x[127, 511] = float("nan")
    x[4100, 7] = x[m - 1, 0] = float("inf")
    got, _, _ = _unpacked(codes, scale, zero, x, g, flag)
    assert need > 0 and flag == [0, 2]
    rest = torch.ones(m, dtype=torch.bool)
    rest[wide + odd] = False
    assert torch.equal(got[rest], plain[rest])
    assert not torch.isfinite(got[odd]).any()
    w = torch.tensor(wide, device=DEV)
    want = _double(codes, scale, zero, x, g, w)
    size = ((codes.double() + 24).view(n, k // g, g) * scale.double().t()[:, :, None] + zero.double().abs().t()[:, :, None]).view(n, k).to(DEV)
    assert bool(((got[w].double() - want).abs() <= 2**-8 * want.abs() + 2**-15 * (x[w].double().abs() @ size.t())).all())


@pytest.mark.parametrize("g,m,n,k", [(64, 470, 12296, 640), (128, 470, 12296, 384), (256, 470, 12296, 768)])
def test_odd_scales_in_96_row_workgroups(many_row_kernel, g, m, n, k):
    """Five rows of workgroups, the last of 86 rows; the plain loop walks pairs of row tiles, of which the last holds one, and stores nothing of the next workgroup's rows"""
    _lib.set_option("int4_gemm_tile", 96)
    codes, scale, zero, x = _case(m, n, k, g)
    zero[:, 5], scale[:, 5] = 0.0, 2.0**-101
    zero[:, 12290], scale[:, 12290] = 0.0, 2.0**40
    scale[-1, 300] = float("nan")
    got, want = _run(codes, scale, zero, x, g)
    finite = torch.ones(n, dtype=torch.bool)
    finite[300] = False
    assert torch.equal(got[:, finite], want[:, finite].to(torch.bfloat16)) and not torch.isfinite(got[:, 300]).any()


# ---- the gated launch on unpacked operands ------------------------------------------------------------------------------------------------
def _gate_of(a, b):
    """silu(a) * b with the rounding points of stock ops on bfloat16 tensors, from products in float64"""
    a, b = a.to(torch.bfloat16), b.to(torch.bfloat16)
    return ((a.double() / (1 + torch.exp(-a.double()))).to(torch.bfloat16).double() * b.double()).to(torch.bfloat16)


def _check_gate(got, want):
    """A gate within three units in the last place of float32 rounds to another bfloat16 in about one value of 4000, by a unit of 2^-7 of it at most; the product's own
    rounding makes that two units at most.  Below -88.7, where exp(-a) leaves float32, gates are zero for at most 2^-121 in size and their products (|b| < 2^30) for 2^-91."""
    got, want = got.double(), want.double()
    assert torch.isfinite(got).all()
    assert ((got - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -91).all()
    assert ((got != want) & (want.abs() > 2.0 ** -90)).double().mean() <= 2e-3


@pytest.mark.parametrize("g", [32, 64, 128, 256])
@pytest.mark.parametrize("m,n,k", [(70000, 8, 256), (66049, 264, 512), (66100, 1032, 512)])  # ragged columns of a tile's 128, a last tile of 112 rows, of one and of 52
def test_gated_unpacked_rows_are_the_two_exact_products_gated(g, m, n, k):
    halves = [_case(m, n, k, g, seed=seed) for seed in (5, 77)]
    x = halves[0][3]
    weights = []
    for codes, scale, zero, _ in halves:
        weights += [torch.from_numpy(qo.int4_tile_pack(codes.numpy(), 8)).to(DEV), torch.stack([scale, zero], dim=-1).to(torch.bfloat16).contiguous().to(DEV)]
    lib = _lib.load()
    assert lib.e2h_int4_mm_silu_gate_rows_scratch_bytes(m, n, k, g, 8) >= lib.e2h_int4_mm_scratch_bytes(m, 2 * n, k, g, 8) > 0
    got = ops.int4_mm_silu_gate_rows(x, *weights, g)
    rows = torch.cat([torch.arange(0, 300), torch.arange(m - 300, m)]).to(DEV)
    _check_gate(got[rows], _gate_of(*(_double(c, s, z, x, g, rows) for c, s, z, _ in halves)))


def test_gates_of_a_tile_round_as_the_pass_does_for_every_bfloat16():
    """All 65536 gates as they are and times column scales up to where they overflow, beside ups of both signs: bit for bit two calls and silu_mul, NaN and infinities included."""
    k = 256
    x = torch.zeros((65536, k), dtype=torch.bfloat16)
    x[:, 0] = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x[:, 1] = 1.0
    x = x.to(DEV)
    q = torch.zeros((2, 8, k), dtype=torch.int8, device=DEV)
    q[0, :, 0] = torch.tensor([1, -1, 3, 7, 1, 1, 101, 1])
    q[1, :, 1] = torch.tensor([1, 3, -1, 1, 1, 5, 1, -7])
    s = torch.tensor([[1, 1, 0.37, 2.0 ** -20, 2.0 ** 100, 2.0 ** -100, 0.0113, 1.7], [1, 0.3, 1, 2.0 ** 60, 1, 1, 2.0 ** -60, 1]], dtype=torch.bfloat16, device=DEV)
    got = ops.int8_mm_silu_gate_rows(x, q[0], s[0], q[1], s[1])
    a, b = (ops.int8_mm(x, w, t) for w, t in zip(q, s))
    want = ops.silu_mul(a, b)
    assert torch.isinf(a).any() and torch.isinf(want).any() and torch.isnan(want).any()
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan) and torch.equal(got[~nan].view(torch.int16), want[~nan].view(torch.int16))


@pytest.mark.parametrize("g,m,n,k", [(32, 66049, 1032, 512), (128, 8190, 11000, 4096)])
def test_gated_unpacked_rows_are_the_two_calls_on_unpacked_operands_bit_for_bit(g, m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(g)
    x = torch.randn((m, k), generator=gen, device=DEV).to(torch.bfloat16)
    w = [ops.int4_quantize_pack((torch.randn((n, k), generator=gen, device=DEV) * 0.05).to(torch.bfloat16), g, 8) for _ in range(2)]
    lib = _lib.load()
    assert lib.e2h_int4_mm_silu_gate_rows_scratch_bytes(m, n, k, g, 8) > 0 and lib.e2h_int4_mm_scratch_bytes(m, n, k, g, 8) > 0
    want = ops.silu_mul(*(ops.int4_mm(x, p, g, sz) for p, sz in w))
    assert torch.equal(ops.int4_mm_silu_gate_rows(x, *w[0], *w[1], g), want)


def test_gated_unpacked_rows_leave_what_float16_lacks_to_the_other_kernel():
    """A row that is not finite, a row of small values beside a large one, and a scale that float16 does not hold in the second matrix: as two calls give them."""
    m, n, k, g = 66049, 264, 512, 128
    gen = torch.Generator().manual_seed(4)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16)
    x[7, 5], x[300, 9] = float("inf"), float("nan")
    x[900, 1:40] *= 2.0 ** -40
    x = x.to(DEV)
    w = [ops.int4_quantize_pack((torch.randn((n, k), generator=gen) * 0.02).to(torch.bfloat16).to(DEV), g, 8) for _ in range(2)]
    for plant in (False, True):
        if plant:
            w[1][1][0, 33, 0] = float("inf")
        got = ops.int4_mm_silu_gate_rows(x, *w[0], *w[1], g)
        a, b = (ops.int4_mm(x, p, g, sz) for p, sz in w)
        want = torch.nn.functional.silu(a.double()).to(torch.bfloat16).double() * b.double()
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want.to(torch.bfloat16)))
        fine = torch.isfinite(want)
        # the calls' sums have another order where the other kernel forms them: a product may round to another bfloat16, its gate by 1.1 times that
        assert (got[fine].double() - want[fine]).norm() <= 2.0 ** -7 * want[fine].norm()


@pytest.mark.parametrize("m,n,k", [(1030, 8200, 256), (1500, 5504, 384), (4096, 2056, 512), (70000, 8, 256)])
def test_gated_int8_rows_are_the_two_calls_gated(m, n, k):
    """Whole numbers as operands, so that products are exact whatever the order of their sums."""
    gen = torch.Generator().manual_seed(m + n)
    x = torch.randint(-8, 9, (m, k), generator=gen).to(torch.bfloat16).to(DEV)
    q = [torch.randint(-128, 128, (n, k), generator=gen, dtype=torch.int8).to(DEV) for _ in range(2)]
    s = [(torch.rand((n,), generator=gen) * 0.002).to(torch.bfloat16).to(DEV) for _ in range(2)]
    got = ops.int8_mm_silu_gate_rows(x, q[0], s[0], q[1], s[1])
    assert got is not None
    a, b = (((x.double() @ w.double().t()).to(torch.bfloat16).double() * t.double()).to(torch.bfloat16) for w, t in zip(q, s))
    _check_gate(got, _gate_of(a.double(), b.double()))
    assert ops.int8_mm_silu_gate_rows(x[:1000], q[0], s[0], q[1], s[1]) is None


def test_gated_int8_rows_leave_watched_modules_to_the_modules():
    from easy_to_hard_amd.model import FeedForward, ModelArgs
    from easy_to_hard_amd.quantize import WeightOnlyInt8QuantHandler

    ff = FeedForward(ModelArgs(dim=256, intermediate_size=8200, n_head=4, n_layer=1))
    WeightOnlyInt8QuantHandler(ff).convert_for_runtime()
    gen = torch.Generator().manual_seed(1)
    for lin in (ff.w1, ff.w2, ff.w3):
        lin.weight = torch.randint(-128, 128, (lin.out_features, lin.in_features), generator=gen, dtype=torch.int8).to(DEV)
        lin.scales = torch.full((lin.out_features,), 2.0 ** -11, dtype=torch.bfloat16, device=DEV)
    x = torch.randn((2, 515, 256), generator=gen).to(torch.bfloat16).to(DEV)
    whole = ff(x)
    assert ff._gate_rows(x).shape == (2, 515, 8200)
    seen = []
    handle = ff.w3.register_forward_hook(lambda *_: seen.append(1))
    assert ff._gate_rows(x) is None and seen == []
    assert (ff(x).double() - whole.double()).norm() <= 2.0 ** -7 * whole.double().norm() and seen == [1]
    handle.remove()
    assert ff._gate_rows(x.float()) is None and ff._gate_rows(x[:, :20]) is None


@pytest.mark.parametrize("by_token", [False, True])
@pytest.mark.parametrize("bsz,t,heads,kv_heads,length,d,k", [
    (4141, 17, 2, 2, 40, 64, 256),          # a lane's rows 16 apart lie in as many sequences; two heads per 128 columns, a last tile of 128 columns
    (70, 1003, 4, 2, 1100, 128, 256),       # fewer heads of k and v
    (3, 1000, 32, 32, 1000, 128, 384),      # a last tile of 184 rows
    (41, 1601, 1, 1, 1700, 128, 32768),     # x of more than 4 GB, in two slices of rows
])
def test_int8_projection_that_rotates_and_writes_the_caches(bsz, t, heads, kv_heads, length, d, k, by_token):
    """Whole numbers as operands, so that products are exact whatever the order of their sums and the two ways agree bit for bit; tokens without a place in the cache write nothing."""
    gen = torch.Generator(device=DEV).manual_seed(t + k)
    n = (heads + 2 * kv_heads) * d
    x = torch.empty((bsz, t, k), dtype=torch.bfloat16, device=DEV)
    for row in x:
        row.copy_(torch.randint(-8, 9, (t, k), generator=gen, device=DEV, dtype=torch.int8))
    q = torch.randint(-128, 128, (n, k), generator=gen, device=DEV, dtype=torch.int8)
    s = (torch.rand((n,), generator=gen, device=DEV) * 0.002).to(torch.bfloat16)
    freqs = torch.randn((2000, d // 2, 2), generator=gen, device=DEV).to(torch.bfloat16)
    pos = torch.randperm(t, generator=gen, device=DEV) + (300 if by_token else length - t)
    rows, there = t if by_token else length, torch.ones(t, dtype=torch.bool, device=DEV)
    if not by_token:
        pos[t // 2], pos[t // 3] = length, -1
        there[t // 2] = there[t // 3] = False
    before = [torch.randn((bsz, kv_heads, rows, d), generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2)]
    got, want = [c.clone() for c in before], before
    q_got = ops.int8_mm_rope_kv_rows(x, q, s, freqs, *got, pos, heads, kv_heads, d, by_token)
    assert q_got is not None
    q_want = ops.rope_kv_write_seq(ops.int8_mm(x.view(-1, k), q, s).view(bsz, t, n), freqs, *want, pos, heads, kv_heads, d, by_token)
    assert torch.equal(q_got[:, :, there], q_want[:, :, there]) and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("by_token", [False, True])
@pytest.mark.parametrize("g,bsz,t,heads,kv_heads,length,d,k", [
    (32, 70, 1003, 4, 2, 1100, 128, 256),
    (64, 70, 1003, 4, 2, 1100, 128, 512),
    (128, 4141, 17, 2, 2, 40, 64, 256),
    (256, 32, 256, 32, 32, 300, 128, 4096),
])
def test_int4_projection_that_rotates_and_writes_the_caches(g, bsz, t, heads, kv_heads, length, d, k, by_token):
    """Bit for bit the product and the pass behind it, also with rows and (then) a scale that the other kernel takes."""
    gen = torch.Generator(device=DEV).manual_seed(t + k)
    n, m = (heads + 2 * kv_heads) * d, bsz * t
    x = torch.randn((m, k), generator=gen, device=DEV).to(torch.bfloat16)
    x[7, 5], x[1300, 9] = float("inf"), float("nan")
    x[900, 1:40] *= 2.0 ** -40
    packed, sz = ops.int4_quantize_pack((torch.randn((n, k), generator=gen, device=DEV) * 0.02).to(torch.bfloat16), g, 8)
    freqs = torch.randn((2000, d // 2, 2), generator=gen, device=DEV).to(torch.bfloat16)
    pos = torch.randperm(t, generator=gen, device=DEV) + (300 if by_token else length - t)
    rows, there = t if by_token else length, torch.ones(t, dtype=torch.bool, device=DEV)
    if not by_token:
        pos[t // 2 - 2], pos[3] = length, -1  # (not the planted rows' tokens: what those give is compared, too)
        there[t // 2 - 2] = there[3] = False
    for plant in (False, True):
        if plant:
            sz[0, 33, 0] = float("inf")
        got = torch.randn((2, bsz, kv_heads, rows, d), generator=gen, device=DEV).to(torch.bfloat16)
        want = got.clone()
        q_got = ops.int4_mm_rope_kv_rows(x.view(bsz, t, k), packed, sz, g, freqs, *got, pos, heads, kv_heads, d, by_token)
        assert q_got is not None
        q_want = ops.rope_kv_write_seq(ops.int4_mm(x, packed, g, sz).view(bsz, t, n), freqs, *want, pos, heads, kv_heads, d, by_token)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(), want.nan_to_num()) and torch.isnan(want).any()
        a, b = q_got[:, :, there], q_want[:, :, there]
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a.nan_to_num(), b.nan_to_num())


def test_prompts_with_angles_beyond_32_bits_leave_the_rotation_to_its_pass():
    bsz, t, heads, d, k = 70, 1003, 2, 64, 256
    x, pos = torch.zeros((bsz, t, k), dtype=torch.bfloat16, device=DEV), torch.arange(t, device=DEV)
    q, s = torch.zeros((3 * heads * d, k), dtype=torch.int8, device=DEV), torch.ones((3 * heads * d,), dtype=torch.bfloat16, device=DEV)
    packed, sz = ops.int4_quantize_pack(torch.zeros((3 * heads * d, k), dtype=torch.bfloat16, device=DEV), 32, 8)
    caches = torch.zeros((2, bsz, heads, t, d), dtype=torch.bfloat16, device=DEV)
    most = (2 ** 31 - 1) // 2 // d
    freqs = torch.zeros((most + 1, d // 2, 2), dtype=torch.bfloat16, device=DEV)
    for f, taken in ((freqs[:most], True), (freqs, False)):
        assert (ops.int8_mm_rope_kv_rows(x, q, s, f, *caches, pos, heads, heads, d) is not None) == taken
        assert (ops.int4_mm_rope_kv_rows(x, packed, sz, 32, f, *caches, pos, heads, heads, d) is not None) == taken


def test_int8_prompts_leave_watched_projections_to_the_modules():
    from easy_to_hard_amd.model import Attention, ModelArgs, precompute_freqs_cis
    from easy_to_hard_amd.quantize import WeightOnlyInt8QuantHandler

    att = Attention(ModelArgs(dim=4096, n_head=32, n_local_heads=32, n_layer=1, intermediate_size=64))
    WeightOnlyInt8QuantHandler(att).convert_for_runtime()
    gen = torch.Generator().manual_seed(1)
    for lin in (att.wqkv, att.wo):
        lin.weight = torch.randint(-128, 128, (lin.out_features, lin.in_features), generator=gen, dtype=torch.int8).to(DEV)
        lin.scales = torch.full((lin.out_features,), 2.0 ** -13, dtype=torch.bfloat16, device=DEV)
    att.freqs_table = precompute_freqs_cis(1024, 128, 10000, device=DEV)
    x, pos = torch.randn((3, 1000, 4096), generator=gen).to(torch.bfloat16).to(DEV), torch.arange(1000, device=DEV)
    k, v = torch.empty((2, 3, 32, 1000, 128), dtype=torch.bfloat16, device=DEV)
    with torch.no_grad():
        assert att._rope_rows(x, k, v, pos, True).shape == (3, 32, 1000, 128)
        whole, seen = att(x, None, None, pos, True), []
        handle = att.wqkv.register_forward_hook(lambda *_: seen.append(1))
        assert att._rope_rows(x, k, v, pos, True) is None and seen == []
        assert torch.equal(att(x, None, None, pos, True), whole) and seen == [1]
        handle.remove()
        assert att._rope_rows(x[:, :20], k, v, pos[:20], True) is None and att._rope_rows(x, k.transpose(0, 1), v.transpose(0, 1), pos, True) is None


# ---- prompts whose norms leave the group sums and add the slices -----------------------------------------------------------------------

@pytest.mark.parametrize("g,m,n,k", [(128, 471, 4096, 4096), (32, 65, 12288, 1024), (64, 129, 12296, 1152), (256, 1023, 3080, 2304), (128, 471, 2048, 5632)])
def test_group_sums_of_a_norm_serve_the_products_behind_it(g, m, n, k):
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    randn = lambda *shape: torch.randn(shape, generator=gen, device=DEV).to(torch.bfloat16)
    x, delta, w = randn(m, k), randn(m, k), randn(k)
    lins = [ops.int4_quantize_pack(randn(n, k) * 0.02, g, 8) for _ in range(2)]
    part = torch.randn((2, m, k), generator=gen, device=DEV)
    for term, (h, want) in ((None, (x, ops.rmsnorm(x, w, 1e-5))), (delta, ops.add_rmsnorm(x, delta, w, 1e-5)), (part, ops.add_rmsnorm(x, part, w, 1e-5))):
        h2, y, sums = ops.add_rmsnorm_sums(x, term, w, 1e-5, g)
        assert torch.equal(h2, h) and torch.equal(y, want)
    own = y.double().view(m, -1, min(g, 128)).sum(-1).t()
    assert (sums[:, :m].double() - own).abs().max() <= min(g, 128) * 2.0 ** -24 * y.double().abs().view(m, -1, min(g, 128)).sum(-1).max()  # float32 sums in any order
    packed, sz = lins[0]
    slices = ops.int4_rows_slices(m, n, k, g, 8)
    assert slices > 0
    want = ops.int4_mm(y, packed, g, sz)
    rows = lambda *rest: _lib.calls().int4_rows(y, packed, sz, g, n, *rest)
    assert torch.equal(rows(sums, False), want) and torch.equal(rows(None, False), want)
    left = rows(sums, True)
    assert rows(sums[:, 64:], True) is None and rows(sums.double(), True) is None and _lib.calls().int4_rows(y[:64], packed, sz, g, n, None, False) is None
    if slices == 1:
        assert torch.equal(left, want)
    else:
        assert tuple(left.shape) == (slices, m, n) and left.dtype == torch.float32
        assert (left.double().sum(0) - want.double()).abs().max() <= 2.0 ** -8 * want.double().abs().max()
        wide = (torch.randn((n,), generator=gen, device=DEV).to(torch.bfloat16), torch.randn((m, n), generator=gen, device=DEV).to(torch.bfloat16)) if n % 128 == 0 else None
        if wide:
            assert all(torch.equal(a, b) for a, b in zip(ops.add_rmsnorm_sums(wide[1], left, wide[0], 1e-5, 128), ops.add_rmsnorm(wide[1], want, wide[0], 1e-5)))
    eight = torch.randn((8, m, k), generator=gen, device=DEV)
    pairs = eight[0::2] + eight[1::2]
    pairs = pairs[0::2] + pairs[1::2]
    assert all(torch.equal(a, b) for a, b in zip(ops.add_rmsnorm_sums(x, eight, w, 1e-5, g), ops.add_rmsnorm(x, (pairs[0] + pairs[1]).to(torch.bfloat16), w, 1e-5)))
    if ops.int4_gate_rows_pay(m, n, k, g):
        assert torch.equal(ops.int4_mm_silu_gate_rows(y, *lins[0], *lins[1], g, sums), ops.int4_mm_silu_gate_rows(y, *lins[0], *lins[1], g))
    assert slices == (4 if n == 2048 else 2 if n == 4096 else 1)
    assert ops.int4_rows_slices(64, n, k, g, 8) == 0 and ops.int4_rows_slices(1024, n, k, g, 8) == 0


def test_a_prompt_with_group_sums_from_its_norms_equals_the_modules(monkeypatch):
    from easy_to_hard_amd import generate
    from easy_to_hard_amd.model import ModelArgs, Transformer
    from easy_to_hard_amd.quantize import WeightOnlyInt4QuantHandler

    torch.manual_seed(0)
    model = Transformer(ModelArgs(block_size=512, vocab_size=8192, n_layer=2, n_head=16, n_local_heads=16, dim=2048, intermediate_size=5632)).to(torch.bfloat16)
    for p in model.parameters():
        if p.dim() == 2:
            p.data.normal_(0.0, 0.02)
    handler = WeightOnlyInt4QuantHandler(model.to(DEV), groupsize=64)
    state = handler.create_quantized_state_dict()
    model = handler.convert_for_runtime()
    model.load_state_dict(state, assign=True)
    model = model.to(DEV).eval().requires_grad_(False)
    model.setup_caches(3, 200)
    ids, pads = torch.randint(0, 8192, (3, 157), device=DEV), torch.tensor([0, 40, 7], device=DEV)
    calls, real = [], ops.add_rmsnorm_sums
    monkeypatch.setattr(ops, "add_rmsnorm_sums", lambda *a: calls.append(1) or real(*a))
    caches = lambda: [t.clone() for b in model.layers for t in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache)]
    with torch.no_grad():
        got, kept = generate.extend(model, ids, 0, pads), caches()
        assert len(calls) == 5
        watched = [m.register_forward_hook(lambda *a: None) for m in (*(b.attention_norm for b in model.layers), model.norm)]
        want = generate.extend(model, ids, 0, pads)
        assert len(calls) == 5
    for hook in watched:
        hook.remove()
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(kept, caches()))


@pytest.mark.parametrize("watch", [None, "first", "second"])
def test_slices_of_a_prompt_are_added_in_one_order_by_every_norm_behind_them(watch):
    """A head that is no int4 linear, or small, and blocks that somebody watches take the plain norm, which has to add the slices of the block before as the matmul does: bit for bit the modules."""
    from easy_to_hard_amd.model import ModelArgs, random_quantized_transformer

    cfg = ModelArgs(block_size=256, vocab_size=2048, n_layer=2, n_head=16, n_local_heads=16, dim=2048, intermediate_size=5632)
    model = random_quantized_transformer(cfg, "int4", groupsize=128, device=DEV).requires_grad_(False)
    model.setup_caches(3, 200)
    assert ops.int4_rows_slices(471, 2048, 5632, 128, 8) == 4 and ops.int4_rows_slices(471, 2048, 2048, 128, 8) == 0
    gen = torch.Generator(device=DEV).manual_seed(4)
    ids, pos = torch.randint(0, 2048, (3, 157), generator=gen, device=DEV), torch.arange(157, device=DEV)
    watched = [] if watch is None else [model.layers[watch == "second"].ffn_norm.register_forward_hook(lambda *a: None)]
    with torch.no_grad():
        got = model(ids, pos)
        watched += [m.register_forward_hook(lambda *a: None) for b in model.layers for m in (b.attention_norm, b.ffn_norm)]
        want = model(ids, pos)
    for hook in watched:
        hook.remove()
    assert torch.equal(got, want)


def test_steps_of_many_sequences_and_scoring_passes_of_some_hundred_rows(monkeypatch):
    """A step of 80 sequences keeps the steps' own attention, whose products read no group sums: none are formed but the head's.  Without a cache (scoring) they serve as in a prompt."""
    from easy_to_hard_amd.model import ModelArgs, random_quantized_transformer

    cfg = ModelArgs(block_size=64, vocab_size=12288, n_layer=2, n_head=32, n_local_heads=32, dim=4096, intermediate_size=5632)
    model = random_quantized_transformer(cfg, "int4", groupsize=128, device=DEV).requires_grad_(False)
    model.setup_caches(80, 64)
    assert all(ops.int4_rows_slices(m, 12288, 4096, 128, 8) > 0 for m in (80, 300))
    calls, real = [], ops.add_rmsnorm_sums
    monkeypatch.setattr(ops, "add_rmsnorm_sums", lambda *a: calls.append(1) or real(*a))
    gen = torch.Generator(device=DEV).manual_seed(1)
    for shape, fully_causal, count in (((80, 1), False, 1), ((5, 60), True, 5)):
        ids, pos = torch.randint(0, 12288, shape, generator=gen, device=DEV), torch.arange(shape[1], device=DEV) + (7 if shape[1] == 1 else 0)
        for b in model.layers:
            for cache in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache):
                cache.normal_(generator=gen)
        calls.clear()
        with torch.no_grad():
            got = model(ids, pos, fully_causal=fully_causal)
            assert len(calls) == count
            watched = [m.register_forward_hook(lambda *a: None) for m in (*(b.attention_norm for b in model.layers), model.norm)]
            want = model(ids, pos, fully_causal=fully_causal)
            assert len(calls) == count
        for hook in watched:
            hook.remove()
        assert torch.equal(got, want)
