"""What decoders with per-sequence state have in common: the state's memory and the step function.

The interface is model.Transformer's: setup_caches, then forward(idx, input_pos) over any number of new tokens.  A subclass
builds `tok_embeddings`, its layers (which register their state with `plan`) and `output`, and gives `_hidden`.
"""

from typing import Optional

import torch
import torch.nn as nn
from torch import Tensor

from . import ops, seq_ops
from .linear import DecodeLinear, fusable, unwatched
from .state import SequenceState, StatePlan, rotary_turns


# torch's embedding stops at a token outside the table where its kernels were built with assertions; where they were not it reads past the table, and the launch here makes a row of NaN instead
EMBEDDING_UNCHECKED = "USE_ROCM_KERNEL_ASSERT=OFF" in torch.__config__.show()


def embedded(emb: nn.Module, tokens: Tensor, want_rows: bool = True):
    """emb(tokens) in float32, where the residual stream starts, and (want_rows) as it is; tokens [rows]."""
    w = emb.weight
    if (EMBEDDING_UNCHECKED and not torch.compiler.is_compiling() and type(emb) is nn.Embedding and emb.max_norm is None and w.dtype == torch.bfloat16 and w.is_cuda and w.device == tokens.device
            and tokens.numel() > 0 and tokens.dtype == torch.int64 and w.is_contiguous() and tokens.is_contiguous() and w.shape[1] % 8 == 0 and w.data_ptr() % 16 == 0 and not (w.requires_grad and torch.is_grad_enabled())
            and unwatched(emb) and not seq_ops.intercepted(w, tokens)):
        return seq_ops.embed_rows(w, tokens, want_rows)
    h = emb(tokens)
    return h.float(), h


class StatefulDecoder(nn.Module):
    returns_greedy_token = True  # forward(..., greedy_token=True) yields the token itself
    logit_softcap: Optional[float] = None

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.plan = StatePlan()
        self.state: Optional[SequenceState] = None
        self.max_batch_size = self.max_seq_length = -1

    def add_rotations(self):
        """Once the layers are built: the turns per position of every rotation that they registered."""
        self.rotations = nn.ParameterList(
            nn.Parameter(torch.zeros((r["dims"] // 2,), dtype=torch.float64), requires_grad=False) for r in self.plan.rotations)

    def rotation_state(self, device="cpu") -> dict:
        """State-dict entries of the rotations; they follow from the configuration, not from a checkpoint."""
        return {f"rotations.{i}": rotary_turns(**r).to(device) for i, r in enumerate(self.plan.rotations)}

    def rotary_tables(self, bsz, seqlen, input_pos, first):
        return [seq_ops.rotary_table(turns, input_pos, first, bsz, seqlen) for turns in self.rotations]

    @property
    def dtype(self):
        return self.tok_embeddings.weight.dtype

    def _new_state(self, max_batch_size, max_seq_length):
        w = self.tok_embeddings.weight
        return SequenceState(self.plan, max_batch_size, max_seq_length, w.dtype, w.device)

    def setup_caches(self, max_batch_size, max_seq_length, kv_cache=True):
        """Memory for the state of `max_batch_size` sequences; kv_cache=False (scoring passes) keeps none."""
        if not kv_cache:
            return
        if self.state is not None and self.max_seq_length >= max_seq_length and self.max_batch_size >= max_batch_size:
            return
        self.max_seq_length, self.max_batch_size = (max_seq_length + 7) // 8 * 8, max_batch_size
        self.state = self._new_state(self.max_batch_size, self.max_seq_length)

    def forward(self, idx: Tensor, input_pos: Optional[Tensor] = None, left_pad_mask_pos: Optional[Tensor] = None, fully_causal: bool = False,
                greedy_token: bool = False) -> Tensor:
        """idx [B, S] token ids at consecutive positions input_pos [S] -> logits [B, S, vocab], or with greedy_token int64
        [B, 1], the arg-max of the last position.  left_pad_mask_pos [B]: positions before it are padding.  fully_causal:
        a pass over whole sequences from position 0 that keeps no state."""
        bsz, seqlen = idx.shape
        idx = idx.to(torch.int64).contiguous()
        if fully_causal:
            assert left_pad_mask_pos is None, "Invalid mask"
            state = self._new_state(bsz, seqlen)
            input_pos = torch.arange(seqlen, device=idx.device)
        else:
            assert self.state is not None, "Caches must be initialized first"
            assert bsz <= self.max_batch_size
            state = self.state
            input_pos = input_pos.to(torch.int64).contiguous()
        first = None if left_pad_mask_pos is None else left_pad_mask_pos.to(torch.int64).contiguous()
        h = self._hidden(idx, bsz, seqlen, state, input_pos, first)
        h = h[:, -1:] if greedy_token else h
        if self.logit_softcap is not None and fusable(self.output, h):
            logits = seq_ops.linear(h, self.output.weight, seq_ops.ACT_SOFTCAP, self.logit_softcap)
        elif (self.logit_softcap is not None and type(self.output) is DecodeLinear and self.output.bias is None and unwatched(self.output)
              and seq_ops.linear_rows_pay(h, self.output.weight, seq_ops.ACT_SOFTCAP, self.logit_softcap)):
            logits = seq_ops.linear_rows(h, self.output.weight, seq_ops.ACT_SOFTCAP, self.logit_softcap)
        else:
            logits = self.output(h)
            if self.logit_softcap is not None:
                logits = seq_ops.softcap_(logits.contiguous(), self.logit_softcap)
        if not greedy_token:
            return logits
        last = logits[:, -1]
        if last.dtype == torch.bfloat16:
            return ops.argmax_rows(last)
        return torch.argmax(last, dim=-1, keepdim=True)

    def _hidden(self, idx, bsz, seqlen, state, input_pos, first) -> Tensor:
        """Normalised output of the last layer, [B, S, dim] in the model's dtype."""
        raise NotImplementedError
