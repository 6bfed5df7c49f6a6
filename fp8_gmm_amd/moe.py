"""Top-k routed MoE layers built on the grouped FP8 modules.

Same classes and data flow as the two FP8 layers of the reference's example (fp8_gmm/example.py:
``Fp8LinearModule`` :72-103, ``Fp8MlpModule`` :106-130): a bf16 gating linear, softmax + top-k, grouping of the
(token, choice) pairs by expert, ``gather`` into expert order, the grouped expert computation, and the weighted
``scatter`` back to token order.  The routing operators come from :mod:`fp8_gmm_amd.moe_ops` instead of
megablocks.  Experts that receive no token are allowed (the reference's modules assert against them,
grouped_linear.py:205, grouped_mlp.py:348).
"""
import numpy as np
import torch

from . import moe_ops
from .grouped_linear import GroupedLinear
from .grouped_mlp import GroupedMlp
from .native import Route, route


def _own(module, cls):
    """Whether what a routed layer calls its experts with is the class's own."""
    return type(module).experts is cls.experts and "experts" not in module.__dict__


class _RoutedModule(torch.nn.Module):
    def __init__(self, n_embd, n_inner, n_experts, top_k, dtype, device):
        super().__init__()
        self.n_embd = n_embd
        self.n_inner = n_inner
        self.n_experts = n_experts
        self.top_k = top_k
        self.sort_end_bit = max(int(np.ceil(np.log2(n_experts))), 1)
        self.gating_network = torch.nn.Linear(n_embd, n_experts, bias=False).to(dtype).to(device)
        self._counts_host = None    # page-locked landing place of the per-expert counts, and the event of its copy
        self._counts_ready = None

    def experts(self, x, batch_sizes):
        raise NotImplementedError

    def start_experts(self):
        """Enqueue what the experts' pass can do before the host knows the split (nothing, by default)."""

    def takes_routed_rows(self, x):
        """Whether ``experts_on_routed_rows`` takes the place of gather, ``experts`` and scatter; asked behind ``start_experts``."""
        return False

    def experts_on_routed_rows(self, x, batch_sizes, indices, inverse, weights, top_k):
        """``scatter(experts(gather(x)))`` in passes that fetch the rows and hand them back themselves."""
        raise NotImplementedError

    def compute(self, x, tokens_per_expert, indices, bin_ids, expert_weights, bins, top_k, inverse=None):
        return self._compute(x, tokens_per_expert, indices, bin_ids, expert_weights, bins, top_k, inverse, False)

    def _compute(self, x, tokens_per_expert, indices, bin_ids, expert_weights, bins, top_k, inverse, sorted_here, counts=None):
        x = x.view(-1, x.size(-1))
        # Rows that the experts' own casts can fetch are not gathered: the mover would write bf16 rows that the cast reads.  Of
        # lists that are surely a permutation and its inverse.
        routed = sorted_here and moe_ops.routed_rows_fit(x, indices, inverse, expert_weights, top_k)
        # The host needs the split to plan the expert launches.  Its copy is enqueued ahead of the gather and of the
        # experts' weight casts, which need nothing from the host: the GPU has that work to do while the host waits
        # for the counts and plans the launches.
        if counts is None:
            if self._counts_host is None or self._counts_host.numel() != tokens_per_expert.numel():
                self._counts_host = torch.empty(tokens_per_expert.shape, dtype=tokens_per_expert.dtype, pin_memory=True)
                self._counts_ready = torch.cuda.Event()
            self._counts_host.copy_(tokens_per_expert, non_blocking=True)
            self._counts_ready.record()
        if not routed:
            x = moe_ops.gather(x, indices, bin_ids, bins, top_k, inverse)
        self.start_experts()
        if routed and not self.takes_routed_rows(x):
            routed = False
            x = moe_ops.gather(x, indices, bin_ids, bins, top_k, inverse)   # ahead of the wait as well
        if counts is not None:   # on their way since the sort
            batch_sizes = torch.tensor(counts.wait(), dtype=torch.long)
        else:
            self._counts_ready.synchronize()
            batch_sizes = self._counts_host.to(torch.long, copy=True)   # the page-locked buffer is reused by the next step
        if routed:
            return self.experts_on_routed_rows(x, batch_sizes, indices, inverse, expert_weights, top_k)
        out = self.experts(x, batch_sizes)
        return moe_ops.scatter(out, indices, bin_ids, expert_weights, bins, top_k, inverse)

    def forward(self, input):
        input = input.view(-1, input.size(-1))
        # Another compute, of a subclass or set on the module, is called as ever: on the rows themselves, which it may change in
        # place where nothing else needs them, and without the inverse.
        own = getattr(self.compute, "__func__", None) is _RoutedModule.compute
        routing_logits, input = moe_ops.gating(self.gating_network, input) if own else (self.gating_network(input), input)
        if own and moe_ops.router_fits(routing_logits, self.top_k, self.n_experts):
            expert_weights, indices, bin_ids, bins, tokens_per_expert, inverse, counts = route(routing_logits, self.top_k)
            return self._compute(input, tokens_per_expert, indices, bin_ids, expert_weights, bins, self.top_k, inverse, True, counts)
        weights0, selected_experts = moe_ops.topk(routing_logits, self.top_k)
        expert_weights = weights0.flatten()
        top_experts = selected_experts.flatten()
        with torch.no_grad():
            indices, bin_ids, bins, tokens_per_expert, inverse = moe_ops.indices_bins_and_inverse(
                top_experts, self.n_experts)
        if own:
            return self._compute(input, tokens_per_expert, indices, bin_ids, expert_weights, bins, self.top_k, inverse, True)
        return self.compute(input, tokens_per_expert, indices, bin_ids, expert_weights, bins, self.top_k)


class Fp8LinearModule(_RoutedModule):
    """Two ``GroupedLinear`` layers with an (erf) GELU between them (fp8_gmm/example.py:72-103)."""

    def __init__(self, n_embd, n_inner, n_experts, top_k, dtype=torch.bfloat16, cutlass=False, device="cuda"):
        super().__init__(n_embd, n_inner, n_experts, top_k, dtype, device)
        self.grouped_linear1 = GroupedLinear(n_embd, n_inner, n_experts, dtype=dtype, cutlass=cutlass, device=device)
        self.grouped_linear2 = GroupedLinear(n_inner, n_embd, n_experts, dtype=dtype, cutlass=cutlass, device=device)
        self.act = torch.nn.GELU()

    def start_experts(self):
        self.grouped_linear1.cast_weights_ahead()
        self.grouped_linear2.cast_weights_ahead()

    def experts(self, x, batch_sizes):
        return self.grouped_linear2(self.act(self.grouped_linear1(x, batch_sizes)), batch_sizes)

    def takes_routed_rows(self, x):
        first, second = self.grouped_linear1, self.grouped_linear2
        return (_own(self, Fp8LinearModule) and type(first) is GroupedLinear and type(second) is GroupedLinear
                and first._takes_routed_rows(x))

    def experts_on_routed_rows(self, x, batch_sizes, indices, inverse, weights, top_k):
        first, second = self.grouped_linear1, self.grouped_linear2
        rows = self.act(first._routed(x, batch_sizes, Route(indices, inverse, None, top_k, True, False)))
        if second._takes_routed_rows(rows):
            return second._routed(rows, batch_sizes, Route(indices, inverse, weights, top_k, False, True))
        return moe_ops.scatter(second(rows, batch_sizes), indices, None, weights, None, top_k, inverse)


class Fp8MlpModule(_RoutedModule):
    """One ``GroupedMlp`` (tanh-GELU fused into the first GEMM) as the experts (fp8_gmm/example.py:106-130)."""

    def __init__(self, n_embd, n_inner, n_experts, top_k, dtype=torch.bfloat16, device="cuda"):
        super().__init__(n_embd, n_inner, n_experts, top_k, dtype, device)
        self.grouped_mlp = GroupedMlp(n_embd, n_inner, n_experts, dtype=dtype, device=device)

    def start_experts(self):
        self.grouped_mlp.cast_weights_ahead()

    def experts(self, x, batch_sizes):
        return self.grouped_mlp(x, batch_sizes)

    def takes_routed_rows(self, x):
        return _own(self, Fp8MlpModule) and type(self.grouped_mlp) is GroupedMlp and self.grouped_mlp._takes_routed_rows(x)

    def experts_on_routed_rows(self, x, batch_sizes, indices, inverse, weights, top_k):
        return self.grouped_mlp._routed(x, batch_sizes, Route(indices, inverse, weights, top_k, True, True))
