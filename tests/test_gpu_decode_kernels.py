"""GPU checks of the decode-step kernels around the linears (RMSNorm, SiLU*mul, RoPE + KV write, single-query
attention) against the stock torch ops the harness otherwise uses, through the C ABI."""

import copy

import pytest
import torch
import torch.nn.functional as F

import easy_to_hard_amd.model as model_mod
from easy_to_hard_amd import ops
from easy_to_hard_amd.generate import decode_one_token, prefill
from easy_to_hard_amd.model import Transformer, apply_rotary_emb, init_random_, precompute_freqs_cis
from tests.helpers import randn_bf16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rmsnorm_reference(x, w, eps):
    """RMSNorm with the reference's rounding points (models/model.py:363-377) on stock ops.  mean(x^2) depends on the
    summation order in its last float32 bit, and where x * rsqrt(..) sits next to a bfloat16 rounding boundary that bit
    flips the first rounding and, through the multiplication by w, up to two ulps of the result (a whole row of 4096
    can do so when rsqrt(..) happens to be close to a short binary fraction): hence two ulps of tolerance and an
    "almost everywhere identical" check rather than equality."""
    xf = x.float()
    return (xf * torch.rsqrt(torch.mean(xf * xf, dim=-1, keepdim=True) + eps)).to(torch.bfloat16) * w


def test_rmsnorm_matches_stock_ops():
    for rows, dim in [(32, 4096), (5, 256), (1, 8192), (70, 512), (2, 16384), (600, 4096), (3, 20480)]:
        x = randn_bf16((rows, dim), std=1.5, seed=rows).to(DEV)
        w = (1 + 0.1 * randn_bf16((dim,), seed=dim).float()).to(torch.bfloat16).to(DEV)
        ref = _rmsnorm_reference(x, w, 1e-5)
        y = ops.rmsnorm(x, w, 1e-5)
        assert torch.allclose(y.float(), ref.float(), rtol=2 ** -6, atol=1e-6)
        assert (y == ref).float().mean() > 0.99


def test_add_rmsnorm_matches_stock_ops():
    for rows, dim in [(32, 4096), (3, 256), (2, 16384), (600, 4096), (3, 20480)]:
        x = randn_bf16((rows, dim), std=1.5, seed=rows).to(DEV)
        d = randn_bf16((rows, dim), std=0.7, seed=rows + 1).to(DEV)
        w = (1 + 0.1 * randn_bf16((dim,), seed=dim).float()).to(torch.bfloat16).to(DEV)
        h_ref = x + d
        ref = _rmsnorm_reference(h_ref, w, 1e-5)
        h, y = ops.add_rmsnorm(x, d, w, 1e-5)
        assert torch.equal(h, h_ref)
        assert torch.allclose(y.float(), ref.float(), rtol=2 ** -6, atol=1e-6)
        assert (y == ref).float().mean() > 0.99


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("slices", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("rows,dim", [(1, 4096), (2, 4104), (33, 8192), (2, 8200), (1, 20480), (600, 4104), (5, 512)])
def test_norm_of_slices_equals_the_norm_of_their_sum(rows, dim, slices, scaled):
    """Rows of one piece per thread, of a piece beyond, of the re-read rest; slices within and beyond those requested at once; rows of both block sizes."""
    gen = torch.Generator().manual_seed(rows + dim + slices)
    x = torch.randn((rows, dim), generator=gen).to(torch.bfloat16).to(DEV)
    w = (1 + 0.1 * torch.randn((dim,), generator=gen)).to(torch.bfloat16).to(DEV)
    parts = torch.randn((slices, rows, dim), generator=gen).to(DEV)
    scales = torch.rand((dim,), generator=gen).to(torch.bfloat16).to(DEV) if scaled else None
    total = parts[0].clone()
    for i in range(1, slices):
        total += parts[i]
    delta = total.to(torch.bfloat16)
    if scaled:
        delta = delta * scales
    h, y = ops.add_rmsnorm(x, ops.ScaledPartials(parts, scales) if scaled else parts, w, 1e-5)
    want_h, want_y = ops.add_rmsnorm(x, delta, w, 1e-5)
    assert torch.equal(h, want_h) and torch.equal(h, x + delta) and torch.equal(y, want_y)


@pytest.mark.parametrize("slices", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("rows,dim", [(2, 8), (3, 2048), (3, 2056), (256, 4608), (257, 4608), (300, 8200), (512, 4104), (513, 4608)])
def test_norm_of_slices_on_both_sides_of_its_lines(rows, dim, slices):
    """Rows of one piece and of two, waves without a second piece, and row counts that change the workgroup."""
    test_norm_of_slices_equals_the_norm_of_their_sum(rows, dim, slices, False)
    x = randn_bf16((rows, dim), std=1.5, seed=rows).to(DEV)
    w = (1 + 0.1 * randn_bf16((dim,), seed=dim).float()).to(torch.bfloat16).to(DEV)
    assert torch.allclose(ops.rmsnorm(x, w, 1e-5).float(), _rmsnorm_reference(x, w, 1e-5).float(), rtol=2 ** -6, atol=1e-6)


def test_silu_mul_matches_stock_ops():
    a = randn_bf16((32, 11008), std=2.0, seed=1).to(DEV)
    b = randn_bf16((32, 11008), std=1.0, seed=2).to(DEV)
    ref = F.silu(a) * b
    y = ops.silu_mul(a, b)
    assert torch.allclose(y.float(), ref.float(), rtol=2 ** -7, atol=1e-6)
    assert (y == ref).float().mean() > 0.99


@pytest.mark.parametrize("n_head,n_kv,d", [(32, 32, 128), (64, 8, 128), (4, 4, 64), (8, 2, 64)])
def test_rope_kv_write_and_attention_match_stock_ops(n_head, n_kv, d):
    bsz, s_max, pos = 3, 96, 41
    gen = torch.Generator().manual_seed(n_head + d)
    qkv = (torch.randn((bsz, (n_head + 2 * n_kv) * d), generator=gen)).to(torch.bfloat16).to(DEV)
    kc = (torch.randn((bsz + 1, n_kv, s_max, d), generator=gen)).to(torch.bfloat16).to(DEV)
    vc = (torch.randn((bsz + 1, n_kv, s_max, d), generator=gen)).to(torch.bfloat16).to(DEV)
    freqs = precompute_freqs_cis(s_max, d, 10000, device=DEV)
    input_pos = torch.tensor([pos], device=DEV)
    # stock path
    kc_ref, vc_ref = kc.clone(), vc.clone()
    q, k, v = qkv.view(bsz, 1, -1).split([n_head * d, n_kv * d, n_kv * d], dim=-1)
    fc = freqs[input_pos]
    q_ref = apply_rotary_emb(q.view(bsz, 1, n_head, d), fc).transpose(1, 2)
    k_rot = apply_rotary_emb(k.view(bsz, 1, n_kv, d), fc).transpose(1, 2)
    kc_ref[:bsz].index_copy_(2, input_pos, k_rot)
    vc_ref[:bsz].index_copy_(2, input_pos, v.view(bsz, 1, n_kv, d).transpose(1, 2))
    # fused kernel
    q_out = ops.rope_kv_write(qkv, freqs, kc, vc, input_pos, n_head, n_kv, d)
    assert torch.equal(q_out, q_ref.squeeze(2))
    assert torch.equal(kc, kc_ref) and torch.equal(vc, vc_ref)
    # attention over positions 0..pos, with and without a left-padding mask
    for left_pad in (None, torch.tensor([0, 7, 41], device=DEV)):
        mask = (torch.arange(s_max, device=DEV) <= pos)[None, None, None, :]
        if left_pad is not None:
            vis = torch.arange(s_max, device=DEV).view(1, -1) >= left_pad.view(-1, 1)
            mask = torch.logical_and(mask, vis[:, None, None, :])
            mask = torch.logical_or(mask, (torch.arange(s_max, device=DEV) == pos)[None, None, None, :])
        rep = n_head // n_kv
        kk = kc_ref[:bsz].repeat_interleave(rep, dim=1).float()
        vv = vc_ref[:bsz].repeat_interleave(rep, dim=1).float()
        ref = F.scaled_dot_product_attention(q_ref.float(), kk, vv, attn_mask=mask).squeeze(2)
        y = ops.decode_attention(q_out, kc, vc, input_pos, left_pad)
        assert y.shape == (bsz, n_head, d)
        err = (y.float() - ref).abs().max() / ref.abs().max()
        assert err < 1e-2, err


def test_fused_decode_step_matches_stock_decode_step():
    model = Transformer.from_name("tiny-gqa-test")
    init_random_(model, seed=5, std=0.05)
    model = model.to(device=DEV, dtype=torch.bfloat16).eval()
    bsz, t = 3, 9
    prompt = torch.randint(0, 512, (bsz, t), generator=torch.Generator().manual_seed(2)).to(DEV)
    logits = {}
    for fused in (False, True):
        model_mod.FUSED_DECODE = fused
        try:
            model.max_seq_length = -1
            model.setup_caches(bsz, 32)
            cur = prefill(model, prompt, torch.arange(0, t, device=DEV))
            out = []
            for i in range(4):
                pos = torch.tensor([t + i], device=DEV)
                lg = model(cur, pos)
                out.append(lg[:, -1].float())
                cur = torch.argmax(lg[:, -1].float(), dim=-1, keepdim=True)
            logits[fused] = torch.stack(out)
        finally:
            model_mod.FUSED_DECODE = True
    err = (logits[True] - logits[False]).abs().max() / logits[False].abs().max()
    assert err < 2e-2, err


@pytest.mark.parametrize("n_head,n_kv,d", [(4, 4, 64), (8, 2, 128)])
@pytest.mark.parametrize("by_token", [False, True])
def test_rope_kv_write_seq_matches_stock_ops(n_head, n_kv, d, by_token):
    """Many tokens per sequence: q comes back head-major and rotated, k / v land in the cache rows of their positions
    (or in token order for a cache-less pass) with exactly the bits of apply_rotary_emb + KVCache.update."""
    bsz, t, s_max = 2, 7, 24
    gen = torch.Generator().manual_seed(n_head * 3 + d)
    qkv = torch.randn((bsz, t, (n_head + 2 * n_kv) * d), generator=gen).to(torch.bfloat16).to(DEV)
    freqs = precompute_freqs_cis(s_max, d, 10000, device=DEV)
    input_pos = torch.arange(5, 5 + t, device=DEV)
    rows = t if by_token else s_max
    kc0 = torch.randn((bsz + 1, n_kv, rows, d), generator=gen).to(torch.bfloat16).to(DEV)
    vc0 = torch.randn((bsz + 1, n_kv, rows, d), generator=gen).to(torch.bfloat16).to(DEV)
    kc, vc = kc0.clone(), vc0.clone()
    q_out = ops.rope_kv_write_seq(qkv, freqs, kc, vc, input_pos, n_head, n_kv, d, rows_by_token=by_token)
    q, k, v = qkv.split([n_head * d, n_kv * d, n_kv * d], dim=-1)
    fc = freqs[input_pos]
    q_ref = apply_rotary_emb(q.view(bsz, t, n_head, d), fc).transpose(1, 2)
    k_ref = apply_rotary_emb(k.view(bsz, t, n_kv, d), fc).transpose(1, 2)
    v_ref = v.view(bsz, t, n_kv, d).transpose(1, 2)
    assert q_out.shape == (bsz, n_head, t, d) and torch.equal(q_out, q_ref)
    kc_ref, vc_ref = kc0.clone(), vc0.clone()
    dest = torch.arange(t, device=DEV) if by_token else input_pos
    kc_ref[:bsz].index_copy_(2, dest, k_ref)
    vc_ref[:bsz].index_copy_(2, dest, v_ref)
    assert torch.equal(kc, kc_ref) and torch.equal(vc, vc_ref)


@pytest.mark.parametrize("fully_causal", [False, True])
def test_fused_prefill_matches_stock_prefill(fully_causal):
    model = Transformer.from_name("tiny-gqa-test")
    init_random_(model, seed=6, std=0.05)
    model = model.to(device=DEV, dtype=torch.bfloat16).eval()
    bsz, t = 3, 11
    ids = torch.randint(0, 512, (bsz, t), generator=torch.Generator().manual_seed(4)).to(DEV)
    out = {}
    for fused in (False, True):
        model_mod.FUSED_DECODE = fused
        try:
            model.max_seq_length = -1
            model.setup_caches(bsz, 32, kv_cache=not fully_causal)
            with torch.no_grad():
                out[fused] = model(ids, torch.arange(0, t, device=DEV), fully_causal=fully_causal).float()
        finally:
            model_mod.FUSED_DECODE = True
    err = (out[True] - out[False]).abs().max() / out[False].abs().max()
    assert err < 2e-2, err


@pytest.mark.parametrize("n_head,n_kv", [(16, 4), (64, 8), (32, 2), (12, 2)])
@pytest.mark.parametrize("s_max,pos", [(96, 0), (96, 31), (96, 32), (96, 41), (640, 575), (300, 299)])
def test_grouped_query_attention_on_matrix_cores_matches_sdpa_and_vector_kernel(n_head, n_kv, s_max, pos):
    """4 .. 16 query heads per kv head at head_dim 128 take the MFMA kernel (both cache lengths: 4 and 8 waves): against
    stock SDPA on the same cache, with and without left padding, and against the float32 vector kernel (the two differ
    by the bfloat16 rounding of the softmax weights only)."""
    from easy_to_hard_amd import _lib

    d, bsz = 128, 3
    rep = n_head // n_kv
    gen = torch.Generator().manual_seed(n_head * 7 + pos)
    q = torch.randn((bsz, n_head, d), generator=gen).to(torch.bfloat16).to(DEV)
    kc = torch.randn((bsz, n_kv, s_max, d), generator=gen).to(torch.bfloat16).to(DEV)
    vc = torch.randn((bsz, n_kv, s_max, d), generator=gen).to(torch.bfloat16).to(DEV)
    input_pos = torch.tensor([pos], device=DEV)
    for left_pad in (None, torch.tensor([0, min(7, pos), pos], device=DEV)):
        mask = (torch.arange(s_max, device=DEV) <= pos)[None, None, None, :]
        if left_pad is not None:
            vis = torch.arange(s_max, device=DEV).view(1, -1) >= left_pad.view(-1, 1)
            mask = torch.logical_and(mask, vis[:, None, None, :])
            mask = torch.logical_or(mask, (torch.arange(s_max, device=DEV) == pos)[None, None, None, :])
        kk = kc.repeat_interleave(rep, dim=1).float()
        vv = vc.repeat_interleave(rep, dim=1).float()
        ref = F.scaled_dot_product_attention(q.float()[:, :, None, :], kk, vv, attn_mask=mask).squeeze(2)
        y = ops.decode_attention(q, kc, vc, input_pos, left_pad)
        scale = float(ref.abs().max())
        assert (y.float() - ref).abs().max() < 1e-2 * scale
        if rep in (4, 8):  # the vector kernel is instantiated for 1, 2, 4 and 8 heads per kv head
            _lib.set_option("attention_no_mfma", 1)
            try:
                y_vec = ops.decode_attention(q, kc, vc, input_pos, left_pad)
            finally:
                _lib.set_option("attention_no_mfma", 0)
            assert (y.float() - y_vec.float()).abs().max() < 1e-2 * scale


@pytest.mark.parametrize("h,hkv,d", [(4, 4, 128), (8, 2, 64), (5, 1, 128), (6, 3, 64)])
@pytest.mark.parametrize("t,start,s_len", [(16, 0, 16), (127, 0, 136), (129, 40, 200), (300, 64, 600)])
def test_prefill_attention_against_float64(h, hkv, d, t, start, s_len):
    """Blocks of 128 queries and tiles of 64 keys that end inside, a prompt behind cached tokens, unequal padding (none, inside the prompt, more than all of it), positions
    in any order, and tokens that stand at their index.  Rows in front of a sequence are their own value.  Cache rows nobody sees hold NaN.  Error against 64 bits: at most that of
    the stock kernel on the same inputs (both round weights and results to bfloat16), with a margin for single inputs."""
    gen = torch.Generator().manual_seed(t + h)
    b = 3
    q = torch.randn((b, h, t, d), generator=gen).to(torch.bfloat16).to(DEV)
    k, v = (torch.randn((b + 1, hkv, s_len, d), generator=gen).to(torch.bfloat16).to(DEV) for _ in range(2))
    pads = torch.tensor([0, min(start + t - 1, 70), start + t + 3], device=DEV)
    order = torch.arange(start, start + t, device=DEV)
    for pos, pad in ((order, None), (order, pads), (order[torch.randperm(t, generator=gen).to(DEV)], pads), (None, None)):
        at = torch.arange(t, device=DEV) if pos is None else pos
        key = torch.arange(s_len, device=DEV)
        mask = (key[None, None] <= at[None, :, None]).expand(b, t, s_len)
        if pad is not None:
            mask = (mask & (key[None, None] >= pad[:, None, None])) | (key[None, None] == at[None, :, None])
        kn, vn = k.clone(), v.clone()
        far = int(at.max()) + 64 - int(at.max()) % 64  # tiles behind the last visible key; in a tile that is seen in part, a value meets a weight of zero
        kn[:, :, far:], vn[:, :, far:] = float("nan"), float("nan")
        got = ops.prefill_attention(q, kn, vn, pos, pad)
        rep = lambda c: c[:b].repeat_interleave(h // hkv, dim=1)  # noqa: E731
        scores = (q.double() @ rep(k).double().transpose(-1, -2).contiguous()) * d ** -0.5
        want = (scores.masked_fill(~mask[:, None], float("-inf")).softmax(-1) @ rep(v).double()).transpose(1, 2).reshape(b, t, h * d)
        stock = torch.nn.functional.scaled_dot_product_attention(q, rep(k), rep(v), attn_mask=mask[:, None]).transpose(1, 2).reshape(b, t, h * d)
        err, err_stock = ((x.double() - want).norm() / want.norm() for x in (got, stock))
        assert err <= 1.05 * err_stock, (err, err_stock)
        if pad is not None:
            for i in range(b):
                front = (at < pad[i]).nonzero().flatten()
                assert torch.equal(got[i, front], rep(v)[i][:, at[front]].transpose(0, 1).reshape(len(front), h * d))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("t,start", [(40, 0), (200, 70)])
@pytest.mark.parametrize("sign", [-1, 1])
def test_prefill_attention_of_scores_far_from_zero(d, t, start, sign):
    """Every score near -2^109 or 2^109: the softmax of what a query sees is as it is anywhere else, the largest score's value (the mean of several alike, rounded to bfloat16: 2^-8
    of values below 8), and no masked key takes part."""
    gen = torch.Generator().manual_seed(d)
    b, h, s_len = 2, 3, start + t
    q = torch.full((b, h, t, d), 2.0**51).to(torch.bfloat16).to(DEV)
    k = (sign * 2.0**52 * (1 + torch.randint(0, 64, (b, h, s_len, 1), generator=gen) / 64)).expand(b, h, s_len, d).to(torch.bfloat16).contiguous().to(DEV)
    v = torch.randn((b, h, s_len, d), generator=gen).to(torch.bfloat16).to(DEV)
    pos, pad = torch.arange(start, s_len, device=DEV), torch.tensor([0, start + 9], device=DEV)
    key = torch.arange(s_len, device=DEV)
    mask = ((key[None, None] <= pos[None, :, None]) & (key[None, None] >= pad[:, None, None])) | (key[None, None] == pos[None, :, None])
    scores = (q.double() @ k.double().transpose(-1, -2).contiguous()) * d ** -0.5
    want = (scores.masked_fill(~mask[:, None], float("-inf")).softmax(-1) @ v.double()).transpose(1, 2).reshape(b, t, h * d)
    assert ((ops.prefill_attention(q, k, v, pos, pad).double() - want).abs() <= 2**-5).all()


def test_prompts_of_a_watched_attention_are_shown_the_mask():
    """A hook on one attention keeps the stock operator and its mask for the whole model, and both give the same logits up to
    the rounding of two layers."""
    model = Transformer(model_mod.ModelArgs(block_size=128, vocab_size=256, n_layer=2, n_head=4, n_local_heads=2, dim=256, intermediate_size=512))
    init_random_(model, seed=3)
    model = model.to(device=DEV, dtype=torch.bfloat16).eval()
    model.setup_caches(3, 64)
    ids, pos, pads = torch.randint(0, 256, (3, 40), generator=torch.Generator().manual_seed(5)).to(DEV), torch.arange(40, device=DEV), torch.tensor([0, 7, 39], device=DEV)
    with torch.no_grad():
        plain = model(ids, pos, pads).float()
        seen = []
        handle = model.layers[1].attention.register_forward_pre_hook(lambda m, args: seen.append(args[2]))
        watched = model(ids, pos, pads).float()
        handle.remove()
        assert torch.equal(model(ids, pos, pads).float(), plain)
    assert len(seen) == 1 and seen[0].dtype == torch.bool and tuple(seen[0].shape) == (3, 1, 40, 64)
    assert (plain - watched).norm() <= 2e-2 * watched.norm()


@pytest.mark.parametrize("b,t,h,s_len,masked,own", [(32, 16, 32, 16, True, False), (32, 47, 32, 56, True, False), (32, 48, 32, 56, True, True), (32, 16, 32, 64, True, True),
                                                     (31, 16, 32, 16, True, True), (32, 16, 32, 16, False, True), (1, 15, 4, 64, True, False), (1, 16, 4, 16, True, True)])
def test_where_prompts_take_the_own_attention(b, t, h, s_len, masked, own):
    k = torch.empty((b, h, s_len, 64), dtype=torch.bfloat16, device=DEV)
    assert ops.prefill_attention_fits(b, t, h, k, k, masked) == own


@pytest.mark.parametrize("how", ["written", "replaced", "copied", "written after a copy"])
def test_a_prompt_reads_masks_that_were_changed(how):
    """A prompt whose first ten tokens see each other, by the model's own mask tensor: the first token's logits change, and go back with the mask.  A copy of a model keeps
    what its masks are."""
    model = Transformer(model_mod.ModelArgs(block_size=128, vocab_size=256, n_layer=2, n_head=4, n_local_heads=2, dim=256, intermediate_size=512))
    init_random_(model, seed=3)
    model = model.to(device=DEV, dtype=torch.bfloat16).eval()
    model.setup_caches(2, 64)
    ids, pos = torch.randint(0, 256, (2, 40), generator=torch.Generator().manual_seed(5)).to(DEV), torch.arange(40, device=DEV)
    with torch.no_grad():
        plain = model(ids, pos).float()
        assert model._masks_by_position(model.tok_embeddings(ids), pos, None)
        if how == "written after a copy":
            model = copy.deepcopy(model)
            assert model._masks_by_position(model.tok_embeddings(ids), pos, None) and torch.equal(model(ids, pos).float(), plain)
        if how == "replaced":
            model.causal_mask = model.causal_mask.clone()
            model.causal_mask[:10, :10] = True
        else:
            model.causal_mask[:10, :10] = True
        if how == "copied":
            model = copy.deepcopy(model)
        changed = model(ids, pos).float()
        model.causal_mask[:10, :10] = torch.ones(10, 10, device=DEV).tril().bool()
        back = model(ids, pos).float()
    assert (changed[:, 0] - plain[:, 0]).norm() > 5e-2 * plain[:, 0].norm()
    assert (back - plain).norm() <= 2e-2 * plain.norm()


@pytest.mark.parametrize("pads,same", [([2.5, 39.25, 0.0], [3, 40, 0]), ([2**32, 2**40 + 5, 0], [64, 64, 0]), ([-(2**32) + 9, -1, 70], [0, 0, 64])])
def test_padding_of_any_number(pads, same):
    """Positions that lie between two tokens, and such as no 32 bits hold, mask what they mask as numbers: the prompt's logits are those of the whole number that masks the
    same (of the stock operator for fractions, up to the rounding of two layers)."""
    model = Transformer(model_mod.ModelArgs(block_size=128, vocab_size=256, n_layer=2, n_head=4, n_local_heads=2, dim=256, intermediate_size=512))
    init_random_(model, seed=3)
    model = model.to(device=DEV, dtype=torch.bfloat16).eval()
    model.setup_caches(3, 64)
    ids, pos = torch.randint(0, 256, (3, 40), generator=torch.Generator().manual_seed(5)).to(DEV), torch.arange(40, device=DEV)
    with torch.no_grad():
        got, want = (model(ids, pos, torch.tensor(p, device=DEV)).float() for p in (pads, same))
    if isinstance(pads[0], int):
        assert torch.equal(got, want)
    else:
        assert (got - want).norm() <= 1.5e-2 * want.norm()
        with torch.no_grad():
            assert (model(ids, pos, torch.tensor(pads, device=DEV).long()).float() - want).norm() > 5e-2 * want.norm()  # what cutting them off would give


@pytest.mark.parametrize("fully_causal", [False, True])
def test_prompts_use_the_stock_attention_where_it_is_watched_or_chosen(monkeypatch, fully_causal):
    """A function mode sees every layer's attention, and a choice among the operator's backends is kept; a default device is neither."""
    model = Transformer(model_mod.ModelArgs(block_size=128, vocab_size=256, n_layer=2, n_head=4, n_local_heads=2, dim=256, intermediate_size=512))
    init_random_(model, seed=3)
    model = model.to(device=DEV, dtype=torch.bfloat16).eval()
    model.setup_caches(3, 64, kv_cache=not fully_causal)
    ids, pos = torch.randint(0, 256, (3, 40), generator=torch.Generator().manual_seed(5)).to(DEV), torch.arange(40, device=DEV)
    pads = None if fully_causal else torch.tensor([0, 7, 39], device=DEV)
    own, seen, launch = [], [], ops.prefill_attention

    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            if func is torch.nn.functional.scaled_dot_product_attention:
                seen.append(func)
            return func(*args, **(kwargs or {}))

    monkeypatch.setattr(ops, "prefill_attention", lambda *a: own.append(None) or launch(*a))
    run = lambda: model(ids, pos, pads, fully_causal=fully_causal).float()  # noqa: E731
    with torch.no_grad():
        plain = run()
        with torch.device(DEV):
            assert torch.equal(run(), plain)
        assert len(own) == 4
        with Watch():
            watched = run()
        assert len(seen) == 2
        with torch.nn.attention.sdpa_kernel(torch.nn.attention.SDPBackend.MATH):
            chosen = run()
        assert len(own) == 4
    for other in (watched, chosen):
        assert (plain - other).norm() <= 2e-2 * other.norm()


def test_a_prompt_keeps_its_padding_while_another_call_runs():
    """A call of the same model without padding, made between the layers of a padded prompt (as another thread's may be), leaves the
    prompt's logits as they are: the second layer still sees this call's padding."""
    model = Transformer(model_mod.ModelArgs(block_size=128, vocab_size=256, n_layer=2, n_head=4, n_local_heads=2, dim=256, intermediate_size=512))
    init_random_(model, seed=3)
    model = model.to(device=DEV, dtype=torch.bfloat16).eval()
    model.setup_caches(3, 64)
    ids, pos, pads = torch.randint(0, 256, (3, 40), generator=torch.Generator().manual_seed(5)).to(DEV), torch.arange(40, device=DEV), torch.tensor([0, 7, 39], device=DEV)
    inner = []

    def between(*_):
        if not inner:
            inner.append(None)
            inner[0] = model(ids, pos)

    with torch.no_grad():
        plain = model(ids, pos, pads)
        handle = model.layers[0].feed_forward.register_forward_pre_hook(between)
        got = model(ids, pos, pads)
        handle.remove()
    assert torch.equal(got, plain) and not torch.equal(inner[0], plain)
