"""Token routing around the grouped expert layers: sort by expert, histogram, gather, scatter.

The reference's example MoE layers take these operators from the megablocks package
(``megablocks.ops`` in fp8_gmm/example.py:4,15-32,52,59,88,94,115,119).  megablocks is not part of the
reference tree and no version of it is pinned there; this module provides the operators under the same names,
argument order and meaning, on HIP kernels of this package's library (csrc/router.hip):

    sort(x, end_bit)                                   -> (sorted x, original positions), stable
    histogram(x, num_bins)                             -> entries per value
    inclusive_cumsum(x, dim)
    gather(x, indices, bin_ids, bins, top_k)           -> x[indices // top_k]               (autograd)
    scatter(x, indices, bin_ids, weights, bins, top_k) -> sum_k weights * rows, token order (autograd)

plus ``indices_and_bins`` and ``topk`` of the example itself (example.py:15-32), the former as ONE library call.
Differences, stated where they matter: the weighted sum of ``scatter`` is accumulated in fp32 and rounded to bf16
once (megablocks rounds every weighted row to the output type before adding), and ids outside ``[0, 2**end_bit)``
are clamped into the range instead of being undefined.
"""
import torch

from . import _lib, native
from .backend import _fail, _stream, _timed

MAX_EXPERTS = 4096  # size of the on-chip expert table of the sort kernels


def _check_ids(x):
    if not x.is_cuda:
        _fail("fp8_gmm_amd: expected GPU tensors (the HIP path has no CPU fallback)")
    if x.dtype != torch.int32 or x.dim() != 1 or not x.is_contiguous():
        _fail("fp8_gmm_amd: expert ids must be a contiguous 1-D int32 tensor")


def _check_experts(num_experts):
    if not 1 <= num_experts <= MAX_EXPERTS:
        _fail(f"fp8_gmm_amd: between 1 and {MAX_EXPERTS} experts are supported, got {num_experts}")


def _route(sort_ids, top_expert, num_experts, want_sort, want_inverse, want_counts):
    n, dev = top_expert.numel(), top_expert.device

    def new(count):
        return torch.empty(count, dtype=torch.int32, device=dev)

    bin_ids = new(n) if want_sort else None
    indices = new(n) if want_sort else None
    inverse = new(n) if want_inverse else None
    counts = new(num_experts) if want_counts else None
    bins = new(num_experts) if want_counts else None
    work = torch.empty(_lib.load().fp8gmm_route_workspace_bytes(n, num_experts), dtype=torch.uint8, device=dev)

    def ptr(t):
        return t.data_ptr() if t is not None and t.numel() else None

    with torch.cuda.device(dev):
        rc = sort_ids(ptr(top_expert), n, num_experts, ptr(bin_ids), ptr(indices), ptr(inverse), ptr(counts), ptr(bins),
                      ptr(work), _stream(dev))
    _lib.check(rc)
    return bin_ids, indices, inverse, counts, bins


def route(top_expert, num_experts, want_sort=True, want_inverse=False, want_counts=True):
    """One pass over the expert ids: ``(bin_ids, indices, inverse, tokens_per_expert, bins)``, None where not asked for."""
    _check_ids(top_expert)
    _check_experts(num_experts)
    return _route(_lib.load().fp8gmm_route_sort, top_expert, num_experts, want_sort, want_inverse, want_counts)


def sort(x, end_bit=None):
    """Stable ascending sort of non-negative int32 ids below ``2**end_bit`` (all of 0..4095 when None): returns
    ``(sorted ids, positions they came from)`` like ``megablocks.ops.sort``."""
    num = MAX_EXPERTS if end_bit is None else 1 << int(end_bit)
    bin_ids, indices, _, _, _ = route(x, num, want_counts=False)
    return bin_ids, indices


def histogram(x, num_bins):
    """Number of entries of every value in ``[0, num_bins)``, int32 (``megablocks.ops.histogram``)."""
    return route(x, int(num_bins), want_sort=False)[3]


def inclusive_cumsum(x, dim):
    """``megablocks.ops.inclusive_cumsum``: running sum along ``dim`` in the dtype of ``x``."""
    if x.dim() == 0:
        return x.clone()
    return torch.cumsum(x, dim).to(x.dtype)


def indices_and_bins(top_expert, sort_end_bit, n_experts):
    """``(indices, bin_ids, bins, tokens_per_expert)`` as the example's helper of the same name returns them
    (fp8_gmm/example.py:26-32), from one library call instead of three operators."""
    del sort_end_bit  # the counting sort needs the expert count, not a bit count
    indices, bin_ids, bins, tokens_per_expert, _ = indices_bins_and_inverse(top_expert, n_experts, False)
    return indices, bin_ids, bins, tokens_per_expert


def indices_bins_and_inverse(top_expert, n_experts, want_inverse=True):
    """The four of ``indices_and_bins`` and the inverse of ``indices``, for ``gather`` and ``scatter``."""
    if top_expert.dtype == torch.int64 and top_expert.is_cuda and top_expert.dim() == 1:
        # the router's choices as they are, without a conversion in front
        _check_experts(n_experts)
        bin_ids, indices, inverse, tokens_per_expert, bins = _route(
            _lib.load().fp8gmm_route_sort_selected, top_expert.contiguous(), n_experts, True, want_inverse, True)
    else:
        bin_ids, indices, inverse, tokens_per_expert, bins = route(top_expert.int().contiguous(), n_experts,
                                                                   want_inverse=want_inverse)
    return indices, bin_ids, bins, tokens_per_expert, inverse


MAX_GATING_EXPERTS = 128


def _aligned(t):
    """``t``, or a copy of it that is contiguous and starts on 16 bytes (what a saved-tensor or gradient hook returned
    may be anything)."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone(memory_format=torch.contiguous_format)


class _Gating(torch.autograd.Function):
    """``(x weight^T, x)``: the logits, and x once more for what follows, so that its two gradients meet here and one
    kernel adds them."""

    @staticmethod
    def forward(ctx, x, weight):
        ctx.set_materialize_grads(False)
        # what torch's linear would keep: with a frozen weight the caller may change the rows in place afterwards
        ctx.save_for_backward(x if ctx.needs_input_grad[1] else None, weight if ctx.needs_input_grad[0] else None)
        ctx.hidden = x.shape[1]
        return torch.nn.functional.linear(x, weight), x

    @staticmethod
    def backward(ctx, grad, grad_in):
        if grad is None:
            return grad_in, None
        x, weight = ctx.saved_tensors
        want_x, want_weight = ctx.needs_input_grad
        (tokens, experts), hidden, dev = grad.shape, ctx.hidden, grad.device

        def as_saved(t, rows):
            return t.dtype == torch.bfloat16 and t.device == dev and t.shape == (rows, hidden)

        # a graph of the backward pass is asked for, or a saved-tensor hook returned what the kernels do not read: torch's products
        if torch.is_grad_enabled() or want_weight and not as_saved(x, tokens) or want_x and not as_saved(weight, experts):
            grad_x = grad_weight = None
            if want_x:
                grad_x = grad @ weight if grad_in is None else grad_in + grad @ weight
            if want_weight:
                grad_weight = grad.t() @ x
            return grad_x, grad_weight
        return _gating_gradients(grad, x if want_weight else None, weight if want_x else None, grad_in)


def _gating_gradients(grad, x, weight, grad_in):
    """``(grad_x, grad_weight)``: the first where the weight is given, the second where the rows are."""
    want_x, want_weight = weight is not None, x is not None
    (tokens, experts), dev = grad.shape, grad.device
    hidden = (x if want_weight else weight).shape[1]
    grad = _aligned(grad)
    x = _aligned(x) if want_weight else None
    weight = weight.contiguous() if want_x else None
    grad_in = _aligned(grad_in) if grad_in is not None else None
    L = _lib.load()
    grad_x = torch.empty(tokens, hidden, dtype=grad.dtype, device=dev) if want_x else None
    grad_weight = work = None
    if want_weight:
        grad_weight = torch.empty(experts, hidden, dtype=grad.dtype, device=dev)
        work = torch.empty(L.fp8gmm_gating_workspace_bytes(tokens, hidden, experts), dtype=torch.uint8, device=dev)
    with torch.cuda.device(dev), _timed("gating_backward", lambda: 2 * tokens * hidden * (want_weight + 2 * want_x)):
        rc = L.fp8gmm_gating_backward(grad.data_ptr(), x.data_ptr() if want_weight else None,
                                      weight.data_ptr() if want_x else None,
                                      grad_in.data_ptr() if grad_in is not None else None,
                                      grad_x.data_ptr() if want_x else None,
                                      grad_weight.data_ptr() if want_weight else None, tokens, hidden, experts,
                                      work.data_ptr() if want_weight and work.numel() else None, _stream(dev))
    _lib.check(rc)
    return grad_x, grad_weight


def _unwatched():
    """Nothing that looks at the autograd functions one by one: the native host path has nodes of its own."""
    return (torch._C._functorch.peek_interpreter_stack() is None
            and torch._C._autograd._top_saved_tensors_default_hooks(True) is None and not torch.jit.is_tracing()
            and not torch.compiler.is_compiling())


def _plain_linear(module):
    """A ``torch.nn.Linear`` that is nothing but its product: no bias, hook, parametrisation or replaced forward."""
    return (type(module) is torch.nn.Linear and module.bias is None and "forward" not in module.__dict__
            and type(module._parameters.get("weight")) is torch.nn.Parameter
            and not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks
                     or module._backward_pre_hooks) and not torch.nn.modules.module._has_any_global_hook())


def _gating_is_faster(tokens, hidden, experts, trained):
    """Whether fp8gmm_gating_backward is ahead of the library's products and torch's addition (csrc/gating.hip has both sides).
    Up to 64 experts it is.  Beyond, a row of gradients whose bytes are no multiple of 16 is loaded in pieces of 2 or 4, which
    the input gradient alone does not make up for; the weight gradient's time goes with the columns too, the library's with
    the tokens only.  Short batches wait for the library's launches."""
    if experts <= 64 or tokens * hidden <= 1 << 21:
        return True
    whole = experts % 8 == 0
    return hidden <= (4096 if whole or tokens >= 8192 else 2048) if trained else whole


def _gating_takes(x, weight):
    """What fp8gmm_gating_backward computes, where it is faster; the general path is torch's linear and its gradients.  The
    forward product stays torch's, whose bits decide the routing."""
    tokens, hidden = x.shape
    return (x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and x.is_cuda and weight.device == x.device
            and type(x) in (torch.Tensor, torch.nn.Parameter) and weight.dim() == 2 and weight.shape[1] == hidden
            and 1 <= weight.shape[0] <= MAX_GATING_EXPERTS and 1 <= tokens <= 1 << 20 and 8 <= hidden <= 1 << 16
            and hidden % 8 == 0 and x.is_contiguous() and weight.is_contiguous() and x.data_ptr() % 16 == 0
            and _gating_is_faster(tokens, hidden, weight.shape[0], weight.requires_grad))


def gating(module, x):
    """``(module(x), x)`` for a gating linear of a routed layer (fp8_gmm/example.py:47-50,84-86,112-113), to be followed by
    a use of the returned ``x``: with gradients wanted for the rows, one backward pass on this package's kernels takes the
    gradient of the logits and that of the returned rows together.  Where the module is more than a product, or the rows
    are not what the kernels take, the module is called."""
    if torch.is_grad_enabled() and x.requires_grad and _plain_linear(module) and not torch.is_autocast_enabled("cuda") \
            and not torch.jit.is_tracing() and _gating_takes(x, module.weight):
        return native.gating(x, module.weight) if _unwatched() else _Gating.apply(x, module.weight)
    return module(x), x


MAX_TOP_K = 8


class _TopK(torch.autograd.Function):
    """softmax over the experts + the top_k largest in one launch, and the chain back to the scores in another."""

    @staticmethod
    def forward(ctx, scores, top_k):
        tokens, experts = scores.shape
        probs = torch.empty(tokens, experts, dtype=torch.float32, device=scores.device)
        weights = torch.empty(tokens, top_k, dtype=torch.float32, device=scores.device)
        selected = torch.empty(tokens, top_k, dtype=torch.int64, device=scores.device)
        _lib.check(_lib.load().fp8gmm_route_topk(scores.data_ptr(), int(scores.dtype == torch.bfloat16), tokens,
                                                experts, top_k, probs.data_ptr(), weights.data_ptr(),
                                                selected.data_ptr(), _stream(scores.device)))
        ctx.save_for_backward(probs, selected)
        ctx.dtype = scores.dtype
        ctx.mark_non_differentiable(selected)
        return weights, selected

    @staticmethod
    def backward(ctx, grad_weights, _):
        probs, selected = ctx.saved_tensors
        tokens, experts = probs.shape
        grad_weights = grad_weights.contiguous().float()
        grad = torch.empty(tokens, experts, dtype=ctx.dtype, device=probs.device)
        _lib.check(_lib.load().fp8gmm_route_topk_backward(probs.data_ptr(), selected.data_ptr(), grad_weights.data_ptr(),
                                                         tokens, experts, selected.shape[1], grad.data_ptr(),
                                                         int(ctx.dtype == torch.bfloat16), _stream(probs.device)))
        return grad, None


def topk(scores, top_k, moe_renorm=False):
    """Softmax over experts in fp32, then the ``top_k`` largest (fp8_gmm/example.py:15-23): weights fp32
    ``[tokens, top_k]`` and expert ids int64.  One kernel for 2-D bf16 / fp32 scores on the GPU with ``top_k`` up to 8
    (equal scores: the lower expert first); torch's operators otherwise."""
    if scores.is_cuda and scores.dim() == 2 and scores.dtype in (torch.bfloat16, torch.float32) \
            and 1 <= top_k <= min(MAX_TOP_K, scores.shape[1]):
        with torch.cuda.device(scores.device):
            multiplier, selected_experts = _TopK.apply(scores.contiguous(), top_k)
    else:
        weights = torch.nn.functional.softmax(scores, dim=1, dtype=torch.float)
        multiplier, selected_experts = torch.topk(weights, top_k)
    if moe_renorm:
        multiplier = multiplier / multiplier.sum(dim=-1, keepdim=True)
    return multiplier, selected_experts


def _check_rows(x, what):
    if not x.is_cuda:
        _fail("fp8_gmm_amd: expected GPU tensors (the HIP path has no CPU fallback)")
    if x.dtype != torch.bfloat16 or x.dim() != 2:
        _fail(f"fp8_gmm_amd: {what} must be a 2-D bfloat16 tensor")


def _check_indices(indices, rows):
    _check_ids(indices)
    if indices.numel() != rows:
        _fail(f"fp8_gmm_amd: expected {rows} indices, got {indices.numel()}")


def _invert(indices):
    inverse = torch.empty_like(indices)
    dev = indices.device
    with torch.cuda.device(dev):
        rc = _lib.load().fp8gmm_route_invert(indices.data_ptr(), indices.numel(), inverse.data_ptr(), _stream(dev))
    _lib.check(rc)
    return inverse


def _gather_rows(x, indices, weights, top_k):
    """out[i] = weights[indices[i]] * x[indices[i] // top_k]"""
    rows, hidden = x.shape[0] * top_k, x.shape[1]
    out = torch.empty(rows, hidden, dtype=x.dtype, device=x.device)
    with torch.cuda.device(x.device), _timed("moe_gather", lambda: 4 * rows * hidden):
        rc = _lib.load().fp8gmm_moe_gather(x.data_ptr(), indices.data_ptr(),
                                           weights.data_ptr() if weights is not None else None, out.data_ptr(),
                                           rows, hidden, top_k, _stream(x.device))
    _lib.check(rc)
    return out


def _scatter_rows(x, inverse, weights, top_k):
    """out[t] = sum_k weights[t * top_k + k] * x[inverse[t * top_k + k]]"""
    tokens, hidden = x.shape[0] // top_k, x.shape[1]
    out = torch.empty(tokens, hidden, dtype=x.dtype, device=x.device)
    with torch.cuda.device(x.device), _timed("moe_scatter", lambda: 2 * (x.shape[0] + tokens) * hidden):
        rc = _lib.load().fp8gmm_moe_scatter(x.data_ptr(), inverse.data_ptr(),
                                            weights.data_ptr() if weights is not None else None, out.data_ptr(),
                                            tokens, hidden, top_k, _stream(x.device))
    _lib.check(rc)
    return out


class _Gather(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, indices, top_k, inverse):
        ctx.save_for_backward(indices if inverse is None else None, inverse)
        ctx.top_k = top_k
        return _gather_rows(x, indices, None, top_k)

    @staticmethod
    def backward(ctx, grad):
        indices, inverse = ctx.saved_tensors
        inverse = _invert(indices) if inverse is None else inverse
        return _scatter_rows(grad.contiguous(), inverse, None, ctx.top_k), None, None, None


class _Scatter(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, indices, weights, top_k, inverse):
        ctx.save_for_backward(x if weights is not None and ctx.needs_input_grad[2] else None, indices, weights)
        ctx.top_k = top_k
        return _scatter_rows(x, _invert(indices) if inverse is None else inverse, weights, top_k)

    @staticmethod
    def backward(ctx, grad):
        x, indices, weights = ctx.saved_tensors
        grad = grad.contiguous()
        if weights is not None and ctx.needs_input_grad[0] and ctx.needs_input_grad[2]:
            # both gradients: one pass that reads every gradient row once
            rows, hidden = x.shape
            grad_x = torch.empty(rows, hidden, dtype=grad.dtype, device=grad.device)
            grad_w = torch.zeros_like(weights)
            with torch.cuda.device(grad.device), _timed("moe_scatter_backward", lambda: 6 * rows * hidden):
                rc = _lib.load().fp8gmm_moe_scatter_backward(x.data_ptr(), grad.data_ptr(), indices.data_ptr(),
                                                             weights.data_ptr(), grad_x.data_ptr(), grad_w.data_ptr(),
                                                             rows, hidden, ctx.top_k, _stream(grad.device))
            _lib.check(rc)
            return grad_x, None, grad_w, None, None
        grad_x = _gather_rows(grad, indices, weights, ctx.top_k) if ctx.needs_input_grad[0] else None
        grad_w = None
        if weights is not None and ctx.needs_input_grad[2]:
            grad_w = torch.zeros_like(weights)
            with torch.cuda.device(grad.device):
                rc = _lib.load().fp8gmm_moe_scatter_wgrad(x.data_ptr(), grad.data_ptr(), indices.data_ptr(),
                                                          grad_w.data_ptr(), x.shape[0], x.shape[1], ctx.top_k,
                                                          _stream(grad.device))
            _lib.check(rc)
        return grad_x, None, grad_w, None, None


def _gathering_is_faster(tokens, hidden, top_k):
    """Whether many narrow rows had better be gathered: of fewer than 256 columns the casts that fetch them keep few lanes busy
    (131072 rows of 128 columns: the gradient's 69 us where the launches that it replaces take 64, the forward one 33 and 45), and the gather
    is what the GPU has to do while the host waits for the counts.  A layer's step, fetched / gathered: 131072 rows of 64 columns 663 /
    624 us with one choice, 568 / 541 with two, 489 / 456 with eight; of 128 659 / 626, 580 / 557 and 502 / 473; of 256 752 / 743, 640 /
    636 and 546 / 548; 65536 rows of 128 435 / 416 with one, but 384 / 407 and 357 / 413; 32768 324 / 403: the host has less to do."""
    return hidden < 256 and (tokens >= 1 << 16 or tokens * top_k > 1 << 16)


def routed_rows_fit(x, indices, inverse, weights, top_k):
    """Whether the experts' casts can fetch and weigh the rows themselves (fp8gmm_routed_rows) in place of ``gather`` and
    ``scatter`` around them: tensors as those two make them, nobody looking on."""
    def plain(t, dtype, dim):
        return type(t) is torch.Tensor and t.dtype == dtype and t.dim() == dim and t.is_contiguous() and t.device == x.device

    if not _unwatched():
        return False
    rows = x.shape[0] * top_k if x.dim() == 2 else -1
    return (x.is_cuda and type(x) in (torch.Tensor, torch.nn.Parameter) and x.dtype == torch.bfloat16 and x.dim() == 2
            and x.is_contiguous() and x.data_ptr() % 16 == 0 and x.shape[1] % 16 == 0
            and plain(indices, torch.int32, 1) and plain(inverse, torch.int32, 1) and plain(weights, torch.float32, 1)
            and indices.numel() == inverse.numel() == weights.numel() == rows and 1 <= top_k <= _lib.ROUTED_MAX_TOP_K
            and not _gathering_is_faster(x.shape[0], x.shape[1], top_k))


def router_fits(scores, top_k, experts):
    """Whether ``native.route`` takes ``topk``, ``indices_bins_and_inverse`` and the copy of the counts in one call."""
    return (type(scores) is torch.Tensor and scores.is_cuda and scores.dim() == 2 and scores.is_contiguous()
            and scores.dtype in (torch.bfloat16, torch.float32) and scores.shape[1] == experts <= MAX_EXPERTS
            and 1 <= top_k <= min(MAX_TOP_K, experts) and _unwatched())


def gather(x, indices, bin_ids, bins, top_k, inverse=None):
    """Rows of ``x[tokens, hidden]`` into expert order: ``out[i] = x[indices[i] // top_k]``, ``[tokens * top_k,
    hidden]`` (``megablocks.ops.gather``; ``bin_ids`` and ``bins`` are accepted for that signature and unused).
    ``inverse``: that of ``indices``, where the caller has it.  Differentiable in ``x``."""
    del bin_ids, bins
    _check_rows(x, "gather input")
    _check_indices(indices, x.shape[0] * top_k)
    if inverse is not None:
        _check_indices(inverse, x.shape[0] * top_k)
    return _Gather.apply(x.contiguous(), indices, int(top_k), inverse)


def scatter(x, indices, bin_ids, weights, bins, top_k, inverse=None):
    """Rows in expert order back to token order, weighted: ``out[t] = sum_k weights[t * top_k + k] * x[pos(t, k)]``
    with ``pos`` the inverse of ``indices``; ``weights`` ``[tokens * top_k]`` in (token, choice) order, or None for
    a plain sum (``megablocks.ops.scatter``).  ``inverse``: that of ``indices``, where the caller has it.
    Differentiable in ``x`` and ``weights``."""
    del bin_ids, bins
    _check_rows(x, "scatter input")
    top_k = int(top_k)
    if x.shape[0] % top_k:
        _fail("fp8_gmm_amd: scatter needs tokens * top_k rows")
    _check_indices(indices, x.shape[0])
    if inverse is not None:
        _check_indices(inverse, x.shape[0])
    if weights is not None:
        if weights.numel() != x.shape[0]:
            _fail(f"fp8_gmm_amd: expected {x.shape[0]} scatter weights, got {weights.numel()}")
        weights = weights.reshape(-1).float().contiguous()  # differentiable; a no-op for the example's fp32 weights
    return _Scatter.apply(x.contiguous(), indices, weights, top_k, inverse)
