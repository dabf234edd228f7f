"""The Gekapel decoder: windowed attention with normalised and rotated queries and keys and a sink per head, some layers reading
the keys and values of an earlier one, and mixtures of squared-ReLU experts with a shared expert.

Per layer, with n(.) the layer norm:
    x = x + n1(attention(x))
    x = x + n2(experts(x))                              (absent when the layer has no feed-forward)
The residual stream is float32 and the sublayers read it unnormalised.  Each "x + n(y)" is one pass that also rounds the new x
for the next sublayer; the one behind a mixture of experts adds up the experts' weighted rows as it reads them, and the last
one applies the final norm.
"""

from dataclasses import dataclass, field
from typing import List

import torch
import torch.nn as nn

from . import seq_ops
from .decoder import StatefulDecoder, embedded
from .feed_forward import ExpertMixture
from .linear import DecodeLinear
from .mixers import TokenMixer, WindowAttention
from .state import StatePlan


@dataclass
class GekapelArgs:
    vocab_size: int
    dim: int
    layers: List[dict] = field(default_factory=list)  # per layer: {"type", "mixer", "mlp"} as in config.json
    norm_eps: float = 1e-6
    block_size: int = 1 << 20  # positions do not enter any layer's weights; the caches are sized by setup_caches

    @staticmethod
    def model_class():
        return Gekapel

    @classmethod
    def from_config(cls, config: dict) -> "GekapelArgs":
        for i, layer in enumerate(config["layers"]):
            if layer["type"] != "attention":
                raise ValueError(f"layer {i}: unknown mixer type {layer['type']!r}")
            source = layer["mixer"].get("kv_from")
            if source is not None and not (0 <= source < i and config["layers"][source]["mixer"].get("kv_from") is None):
                raise ValueError(f"layer {i}: layer {source} has no keys and values to share")
            mlp = layer.get("mlp")
            if mlp is not None and mlp.get("kind", "moe") != "moe":
                raise ValueError(f"layer {i}: unknown feed-forward kind {mlp['kind']!r}")
        return cls(vocab_size=config["vocab"], dim=config["width"], layers=config["layers"], norm_eps=config["norm"]["eps"])


def _vector(n):
    return nn.Parameter(torch.zeros((n,), dtype=torch.float32), requires_grad=False)


class GekapelLayer(nn.Module):
    def __init__(self, plan: StatePlan, args: GekapelArgs, index: int, earlier):
        super().__init__()
        layer, w = args.layers[index], args.dim
        m, source = layer["mixer"], layer["mixer"].get("kv_from")
        self.mixer = TokenMixer(w, [WindowAttention(
            plan, w, m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["scale"], (m.get("mask") or {}).get("size", 0), 0, biases=False, gate=False,
            norm_eps=args.norm_eps, rotary=m.get("rot"), sink=True, kv_of=None if source is None else earlier[source].mixer.branches[0])], [""])
        self.norm1, self.norm1_bias = _vector(w), _vector(w)
        self.feed_forward = None
        if layer.get("mlp") is not None:
            mlp = layer["mlp"]
            self.feed_forward = ExpertMixture(w, mlp["router"]["experts"], mlp["router"]["top"], mlp["expert"]["ff"], (mlp.get("shared") or {}).get("ff"))
            self.norm2, self.norm2_bias = _vector(w), _vector(w)

    def from_checkpoint(self, get, prefix: str, linear_dtype) -> dict:
        sd = {f"mixer.{k}": v for k, v in self.mixer.from_checkpoint(get, prefix + ".mix", linear_dtype).items()}
        norms = ["norm1"]
        if self.feed_forward is not None:
            norms.append("norm2")
            sd.update({f"feed_forward.{k}": v for k, v in self.feed_forward.from_checkpoint(get, prefix + ".mlp", linear_dtype).items()})
        for n in norms:
            sd[n], sd[n + "_bias"] = get(f"{prefix}.{n}").float(), get(f"{prefix}.{n}.b").float()
        return sd


class Gekapel(StatefulDecoder):
    def __init__(self, config: GekapelArgs):
        super().__init__(config)
        self.tok_embeddings = nn.Embedding(config.vocab_size, config.dim)
        self.layers = nn.ModuleList()
        for i in range(len(config.layers)):
            self.layers.append(GekapelLayer(self.plan, config, i, self.layers))
        self.norm, self.norm_bias = _vector(config.dim), _vector(config.dim)
        self.output = DecodeLinear(config.dim, config.vocab_size, bias=False)
        self.add_rotations()

    @classmethod
    def from_config(cls, config: dict) -> "Gekapel":
        return cls(GekapelArgs.from_config(config))

    def state_dict_from_checkpoint(self, get, linear_dtype=torch.bfloat16) -> dict:
        """This module's state dict from a checkpoint's tensors (`get(name)`), linears in `linear_dtype`, vectors in float32."""
        sd = {"tok_embeddings.weight": get("embed").to(linear_dtype), "norm": get("final.norm").float(), "norm_bias": get("final.norm.b").float(),
              "output.weight": get("head").to(linear_dtype), **self.rotation_state()}
        for i, layer in enumerate(self.layers):
            sd.update({f"layers.{i}.{k}": v for k, v in layer.from_checkpoint(get, f"l{i}", linear_dtype).items()})
        return sd

    def init_random_(self, seed: int = 1234, std: float = 0.02, dtype=torch.bfloat16, device=None) -> "Gekapel":
        """Random weights in place (also of a model built on the meta device): linears, experts, routers and embeddings N(0, std) in
        `dtype`, norms at one, biases and sinks at zero."""
        device = device if device is not None else self.tok_embeddings.weight.device
        gen = torch.Generator(device=device).manual_seed(seed)
        state = self.rotation_state(device)
        for name, p in self.state_dict().items():
            leaf = name.rsplit(".", 1)[-1]
            if name in state:
                continue
            if leaf in ("weight", "up", "down", "router"):
                t = torch.empty(p.shape, dtype=dtype, device=device)
                state[name] = t.normal_(0.0, std, generator=gen)
            else:
                state[name] = torch.full(p.shape, 1.0 if leaf in ("norm", "norm1", "norm2", "q_norm", "k_norm") else 0.0, device=device)
        self.load_state_dict(state, assign=True)
        return self.eval().requires_grad_(False)

    def _hidden(self, idx, bsz, seqlen, state, input_pos, first):
        dtype, eps = self.dtype, self.config.norm_eps
        x, h = embedded(self.tok_embeddings, idx.view(-1))
        rotary = self.rotary_tables(bsz, seqlen, input_pos, first)
        pending = {}  # the sublayer output that has not been added to x yet, with its norm

        def add(x, pending, **kw):
            return seq_ops.norm_conv(x, bsz, seqlen, eps, dtype, layer_norm=True, **pending, **kw)

        for layer in self.layers:
            if pending:
                x, h = add(x, pending)
            pending = {"delta": layer.mixer(h, bsz, seqlen, state, input_pos, first, rotary), "delta_weight": layer.norm1, "delta_bias": layer.norm1_bias}
            if layer.feed_forward is not None:
                x, h = add(x, pending)
                shared, terms, weights = layer.feed_forward(h)
                pending = {"delta": shared, "terms": terms, "term_weights": weights, "delta_weight": layer.norm2, "delta_bias": layer.norm2_bias}
        state.commit(bsz, seqlen)
        _, h = add(x, pending, norm_weight=self.norm, norm_bias=self.norm_bias, want_x=False)
        return h.view(bsz, seqlen, -1)
