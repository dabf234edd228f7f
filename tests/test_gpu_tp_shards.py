"""Shard views (tp.apply_tp_linear, reference models/tp.py:122-195) on one GPU: the column shards of a quantized
linear concatenate to the full layer's output and the row shards sum to it (the sum stands in for the all-reduce)."""

import copy

import pytest
import torch
import torch.nn as nn

import easy_to_hard_amd as e2h
from easy_to_hard_amd import _lib
from easy_to_hard_amd.tp import apply_tp_linear
from tests.helpers import randn_bf16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _quantized(kind, n, k, g=64):
    lin = nn.Linear(k, n, bias=False)
    lin.weight.data = randn_bf16((n, k), std=0.05, seed=n + k).float()
    holder = nn.Sequential(lin).to(torch.bfloat16)
    if kind == "int4":
        h = e2h.WeightOnlyInt4QuantHandler(holder, groupsize=g, inner_k_tiles=8, padding=False)
    else:
        h = e2h.WeightOnlyInt8QuantHandler(holder)
    sd = h.create_quantized_state_dict()
    h.convert_for_runtime()
    holder.load_state_dict(sd, assign=True)
    return holder[0].to(DEV)


@pytest.mark.parametrize("kind", ["int4", "int8"])
@pytest.mark.parametrize("world", [2, 4])
def test_column_shards_concatenate_to_the_full_output(kind, world):
    n, k = 512, 1024
    full = _quantized(kind, n, k)
    x = randn_bf16((5, k), seed=3).to(DEV)
    _lib.set_option("int4_k_slices", 1)   # same accumulation order whatever the shard's width (int8 has one order)
    try:
        y = full(x)
        parts = []
        for r in range(world):
            shard = copy.deepcopy(full)
            apply_tp_linear(shard, "colwise", r, world)
            assert shard.out_features == n // world and shard.weight.shape[0] == full.weight.shape[0] // world
            parts.append(shard(x))
    finally:
        _lib.set_option("int4_k_slices", 0)
    assert torch.equal(torch.cat(parts, dim=-1), y)


@pytest.mark.parametrize("kind", ["int4", "int8"])
@pytest.mark.parametrize("world", [2, 4])
def test_row_shards_sum_to_the_full_output(kind, world):
    n, k = 256, 2048
    full = _quantized(kind, n, k)
    x = randn_bf16((7, k), seed=4).to(DEV)
    y = full(x).float()
    total = torch.zeros_like(y)
    for r in range(world):
        shard = copy.deepcopy(full)
        apply_tp_linear(shard, "rowwise", r, world)
        assert shard.in_features == k // world
        total += shard(x[:, r * (k // world):(r + 1) * (k // world)]).float()   # what the all-reduce adds up
    # every shard rounds its partial result to bf16 once more than the full layer does
    assert (total - y).abs().max() <= 2.0 ** -6 * y.abs().max()


@pytest.mark.parametrize("kind", ["int4", "int8"])
def test_fused_qkv_is_sharded_part_by_part(kind):
    dim, kv, world = 256, 128, 2
    full = _quantized(kind, dim + 2 * kv, 512)
    x = randn_bf16((3, 512), seed=5).to(DEV)
    _lib.set_option("int4_k_slices", 1)
    try:
        q, k_, v = full(x).split([dim, kv, kv], dim=-1)
        for r in range(world):
            shard = copy.deepcopy(full)
            apply_tp_linear(shard, "colwise", r, world, weight_splits=[dim, kv, kv])
            qs, ks, vs = shard(x).split([dim // world, kv // world, kv // world], dim=-1)
            assert torch.equal(qs, q[:, r * dim // world:(r + 1) * dim // world])
            assert torch.equal(ks, k_[:, r * kv // world:(r + 1) * kv // world])
            assert torch.equal(vs, v[:, r * kv // world:(r + 1) * kv // world])
    finally:
        _lib.set_option("int4_k_slices", 0)


def test_uneven_shards_are_refused():
    full = _quantized("int4", 512, 1024)
    with pytest.raises(AssertionError):
        apply_tp_linear(copy.deepcopy(full), "colwise", 0, 3)
    with pytest.raises(AssertionError):
        apply_tp_linear(copy.deepcopy(full), "diagonal", 0, 2)
