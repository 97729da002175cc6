r"""Top-k of a linear layer (fmoe/gates/naive_gate.py)."""
import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from .. import fmoe_cuda
from ..functions import topk_softmax
from .base_gate import BaseGate


class NaiveGate(BaseGate):
    r"""logits = Linear(d_model, experts); the k largest logits pick the experts
    and their softmax gives the combine weights.  Returns `(idx [..., k] int64,
    score [T, k])`, plus the full logits when `return_all_scores`."""

    def __init__(self, d_model, num_expert, world_size, top_k=2, gate_bias=True):
        super().__init__(num_expert, world_size)
        self.gate = nn.Linear(d_model, self.tot_expert, bias=gate_bias)
        self.top_k = top_k

    def is_plain(self, x) -> bool:
        r"""Whether running this module on the 2-d tensor `x` is exactly Linear -> top-k ->
        softmax in one dtype, with nobody watching and no `forward` set on an instance: a
        layer may then fold the gate into its own autograd node."""
        lin = self.gate
        return (type(self).forward is NaiveGate.forward and type(lin) is nn.Linear
                and "forward" not in self.__dict__ and "forward" not in lin.__dict__
                and lin.weight.dtype == x.dtype and lin.weight.is_cuda
                and self.top_k <= fmoe_cuda.MAX_GATE_TOP_K
                and lin.weight.shape[0] <= fmoe_cuda.MAX_EXPERTS   # (its gradients are routed)
                and torch.get_default_dtype() == torch.float32
                and not torch.is_autocast_enabled()
                and not _has_any_global_hook()
                and not (self._forward_hooks or self._forward_pre_hooks or self._backward_hooks
                         or self._backward_pre_hooks or lin._forward_hooks
                         or lin._forward_pre_hooks or lin._backward_hooks
                         or lin._backward_pre_hooks))

    def native_balance(self, logits):
        r"""The extension where its balance-gate node takes these logits, else None."""
        if (logits.is_cuda and logits.dim() == 2 and logits.shape[0] > 0
                and 2 <= logits.shape[1] <= 512 and logits.shape[1] == self.tot_expert
                and self.world_size == 1
                and logits.dtype in (torch.float32, torch.float16, torch.bfloat16)):
            return fmoe_cuda.native()
        return None

    def forward(self, inp, return_all_scores=False):
        native = fmoe_cuda.native() if not return_all_scores else None
        if native is not None and inp.dim() == 2 and inp.is_cuda and self.is_plain(inp):
            top_idx, score = native.plain_gate(inp, self.gate.weight, self.gate.bias, self.top_k)
            self.set_loss(torch.zeros(1, device=inp.device, requires_grad=True))
            return top_idx, score
        logits = self.gate(inp)
        top_idx, score = topk_softmax(logits, self.top_k)
        # idx keeps the leading dimensions of the input, score is [tokens, k]
        # (naive_gate.py:31-38: topk over dim -1, then view(-1, top_k) of the values)
        top_idx = top_idx.view(*logits.shape[:-1], self.top_k)
        # a zero loss so training loops can always call get_loss(); created on the
        # device (no host-to-device copy, so the forward can sit in a HIP graph)
        self.set_loss(torch.zeros(1, device=inp.device, requires_grad=True))
        if return_all_scores:
            return top_idx, score, logits
        return top_idx, score
