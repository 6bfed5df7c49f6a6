"""The work a user of this package has it do, as cases that can be prepared, run and timed one by one.

``listed()`` are the representative calls, from the smallest training step to the largest; ``draw(rng)`` gives more of
the same ranges.  A case names what is called (``kind``) and its sizes; the split of the rows over the experts is drawn
from the seed in ``prepare``, as a router decides it anew for every batch.

Kinds:

* ``linear_step`` / ``mlp_step``     forward + backward of a ``GroupedLinear`` / ``GroupedMlp`` in training, with the
                                     default recipe (an amax history of 1024, as ``fp8_gmm_amd.example`` trains with)
* ``mlp_forward``                    inference of a ``GroupedMlp`` on fp8 weights that were cast once and kept
* ``routed_step``                    forward + backward of a whole routed layer: gating, top-k, gather, experts, scatter
* ``gmm``                            the operand-level entry point ``backend.fp8_gmm``
* ``cast_transpose``                 the operand-level entry point ``backend.multi_cast_transpose``
"""
import numpy as np
import torch

import fp8_gmm_amd as pkg
from fp8_gmm_amd import backend
from fp8_gmm_amd.moe import Fp8LinearModule, Fp8MlpModule

HISTORY = 1024   # DelayedScaling's default amax history


def listed():
    return [
        # the smallest layer: a thousand rows over four experts; launches and host work are all there is
        {"name": "linear_small", "kind": "linear_step", "experts": 4, "hidden": 256, "inner": 512, "tokens": 1000,
         "split": "dirichlet", "cutlass": False},
        # many experts under a skewed router: a quarter of the rows in one expert, others with a handful or none
        {"name": "linear_zipf", "kind": "linear_step", "experts": 64, "hidden": 2048, "inner": 1408, "tokens": 24576,
         "split": "zipf", "cutlass": False},
        # the data flow with the scales applied after the GEMM (cutlass=True), an odd number of rows
        {"name": "linear_cutlass", "kind": "linear_step", "experts": 8, "hidden": 1024, "inner": 4096, "tokens": 4001,
         "split": "dirichlet", "cutlass": True},
        # few wide experts, the headline workload: matrix products dominate
        {"name": "mlp_wide", "kind": "mlp_step", "experts": 8, "hidden": 4096, "inner": 14336, "tokens": 16384,
         "split": "dirichlet", "micro": False},
        # many narrow experts, 512 rows each: short contractions, memory traffic dominates
        {"name": "mlp_many", "kind": "mlp_step", "experts": 128, "hidden": 2048, "inner": 768, "tokens": 65536,
         "split": "uniform", "micro": False},
        # a later micro-batch of an optimizer step: the fp8 weights of the first one are reused
        {"name": "mlp_micro", "kind": "mlp_step", "experts": 16, "hidden": 4096, "inner": 6400, "tokens": 4096,
         "split": "uniform", "micro": True},
        # decoding: 32 sequences, top-2 of 8 experts; the weights are read for a few rows each
        {"name": "mlp_decode", "kind": "mlp_forward", "experts": 8, "hidden": 4096, "inner": 14336, "tokens": 64,
         "split": "uniform"},
        # a prefill batch through many narrow experts
        {"name": "mlp_prefill", "kind": "mlp_forward", "experts": 128, "hidden": 2048, "inner": 768, "tokens": 8200,
         "split": "zipf"},
        # a whole routed layer at the sizes of the example script: 16384 tokens, top-2 of 16 experts
        {"name": "routed_mlp", "kind": "routed_step", "experts": 16, "hidden": 4096, "inner": 6400, "tokens": 16384,
         "top_k": 2, "layer": "mlp"},
        # the routed layer of two GroupedLinear, a short odd batch: routing and host work weigh as much as the experts
        {"name": "routed_linear", "kind": "routed_step", "experts": 16, "hidden": 1024, "inner": 2048, "tokens": 1531,
         "top_k": 2, "layer": "linear"},
        # one grouped product on fp8 operands that the caller keeps
        {"name": "gmm", "kind": "gmm", "experts": 8, "hidden": 4096, "inner": 4096, "tokens": 8192, "split": "dirichlet",
         "fp8": "e4m3", "b_transposed": False},
        # eight activation tensors of ragged heights cast, transposed and padded in one call
        {"name": "cast_transpose", "kind": "cast_transpose", "tensors": 8, "cols": 4096, "max_rows": 8191, "fp8": "e4m3"},
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer of [lo, hi], uniform over its logarithm, a multiple of ``step``."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear_step", "mlp_step", "mlp_forward", "routed_step", "gmm", "cast_transpose"])
    while True:
        case = {"kind": kind}
        if kind == "cast_transpose":
            case.update(tensors=_log_int(rng, 1, 24), cols=_log_int(rng, 64, 8192, 16), max_rows=_log_int(rng, 16, 8191),
                        fp8=rng.choice(["e4m3", "e5m2"]))
            if case["tensors"] * case["cols"] * case["max_rows"] <= 8 * 4096 * 8191:
                return case
            continue
        experts = _log_int(rng, 2, 128)
        hidden, inner = _log_int(rng, 128, 4096, 16), _log_int(rng, 128, 14336, 16)
        case.update(experts=experts, hidden=hidden, inner=inner)
        if kind == "routed_step":
            tokens, rows_per_token = _log_int(rng, 16, 16384), 2
            case.update(experts=max(4, experts), tokens=tokens, top_k=2, layer=rng.choice(["mlp", "linear"]))
        else:
            tokens, rows_per_token = _log_int(rng, 1 if kind == "mlp_forward" else 16, 65536), 1
            case.update(tokens=tokens, split=rng.choice(["uniform", "dirichlet", "zipf"]))
            if kind == "linear_step":
                case["cutlass"] = rng.random() < 0.25
            elif kind == "mlp_step":
                case["micro"] = rng.random() < 0.25
            elif kind == "gmm":
                case.update(fp8=rng.choice(["e4m3", "e5m2"]), b_transposed=rng.random() < 0.5)
        rows = tokens * rows_per_token
        # within the largest listed case: weights, products and activation traffic
        if case["experts"] * hidden * inner <= 8 * 4096 * 14336 and rows * hidden * inner <= 0.5 * 16384 * 4096 * 14336 \
                and rows * (hidden + inner) <= 0.5 * 32768 * (4096 + 6400):
            return case


# ------------------------------------------------------------------------------------------------
# work and tolerances
# ------------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "cast_transpose":   # 2 B in, 1 B out, 1 B out padded to 128 columns
        return {"bytes": case["cols"] * sum(3 * m + (m + 127) // 128 * 128 for m in _rows(case)), "flops": 0}
    e, h, f = case["experts"], case["hidden"], case["inner"]
    rows = case["tokens"] * case.get("top_k", 1)
    weights = e * h * f
    gemm = 2 * rows * h * f
    if kind == "gmm":
        return {"bytes": rows * h + weights + 2 * rows * f, "flops": gemm}
    if kind == "mlp_forward":
        return {"bytes": 2 * rows * h + 2 * weights + 2 * rows * h, "flops": 2 * gemm}
    gemms = 1 if kind == "linear_step" else 2
    state = 8 * HISTORY * 5 * e * gemms                       # amax history of both directions, read and written
    if kind == "linear_step":
        return {"bytes": 4 * rows * (h + f) + 4 * weights + state, "flops": 3 * gemm}
    if kind == "mlp_step":                                    # x, dy in, y, dx out; weights in, their gradients out
        return {"bytes": 8 * rows * h + 2 * weights * ((1 if case["micro"] else 2) + 2) + state, "flops": 6 * gemm}
    tokens = case["tokens"]
    return {"bytes": 8 * tokens * h + 8 * weights + 4 * e * h + state, "flops": 6 * gemm + 6 * tokens * h * e}


def tolerance(case):
    """Casts give the same bytes.  A product of fp8 operands differs from its float64 value by its one rounding to bf16
    (measured 1.7e-3, 1.9e-3 with an fp8 activation in between).  Behind a gradient that is rounded to e5m2 once more, a
    value that sits a bf16 rounding away from a rounding boundary lands on the other code: input gradients and first
    weight gradients differ by 1.6e-2 from the same chain in float64."""
    if case["kind"] == "cast_transpose":
        return "exact"
    return {"rel": 3e-2} if case["kind"] in ("mlp_step", "routed_step") else {"rel": 7e-3}


# ------------------------------------------------------------------------------------------------
# preparation
# ------------------------------------------------------------------------------------------------
def _sizes(split, experts, tokens, seed):
    rng = np.random.default_rng(seed)
    if split == "dirichlet":
        p = rng.dirichlet(np.ones(experts))
    elif split == "zipf":
        p = rng.permutation(1.0 / np.arange(1, experts + 1) ** 1.1)
        p /= p.sum()
    else:
        p = np.full(experts, 1.0 / experts)
    return torch.from_numpy(rng.multinomial(tokens, p).astype(np.int64))


def _rows(case):
    """Heights of the tensors of a cast_transpose case: uniform in [1, max_rows], the case's own."""
    return [int(m) for m in np.random.default_rng(case["max_rows"]).integers(1, case["max_rows"] + 1, size=case["tensors"])]


def _normal(shape, std, gen):
    return torch.randn(shape, generator=gen, dtype=torch.bfloat16, device="cuda").mul_(std)


def _fp8(name):
    return torch.float8_e4m3fn if name == "e4m3" else torch.float8_e5m2


def _state(module):
    """The scaling state a checkpoint holds."""
    return [t for d in ("scaling_fwd", "scaling_bwd") for t in module.fp8_meta[d].state().values()]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    s = {"case": case, "recipe": pkg.DelayedScaling()}
    if kind == "cast_transpose":
        # N(0, 1) activations with a few outliers, scaled to the range of the type
        rows = _rows(case)
        dtype, cols = _fp8(case["fp8"]), case["cols"]
        top = 448.0 if case["fp8"] == "e4m3" else 57344.0
        s["ins"], s["outs"], s["touts"], s["scales"] = [], [], [], []
        for m in rows:
            x = _normal((m, cols), 1.0, gen)
            x.masked_fill_(torch.rand((m, cols), generator=gen, device="cuda") < 1e-3, 200.0)
            s["ins"].append(x)
            s["outs"].append(torch.empty(m, cols, dtype=dtype, device="cuda"))
            s["touts"].append(torch.empty(cols, (m + 127) // 128 * 128, dtype=dtype, device="cuda"))
            s["scales"].append((top / x.abs().max().float()).reshape(1))
        s["amaxes"] = torch.zeros(len(rows), device="cuda")
        return s

    e, h, f = case["experts"], case["hidden"], case["inner"]
    if kind == "routed_step":
        layer = Fp8MlpModule if case["layer"] == "mlp" else Fp8LinearModule
        with torch.random.fork_rng(devices=["cuda"]):
            torch.manual_seed(seed)
            s["module"] = layer(h, f, e, case["top_k"])
        s["experts"] = [m for m in s["module"].modules() if isinstance(m, (pkg.GroupedMlp, pkg.GroupedLinear))]
        s["x"] = _normal((case["tokens"], h), 1.0, gen).requires_grad_()
        s["dy"] = _normal((case["tokens"], h), 1e-2, gen)
        _step(s)   # a running training: scales follow the amaxes of the pass before
        return s

    s["sizes"] = _sizes(case["split"], e, case["tokens"], seed)
    if kind == "gmm":
        dtype = _fp8(case["fp8"])
        s["a"] = _normal((case["tokens"], h), 16.0, gen).to(dtype)
        s["b"] = _normal((e, h, f) if case["b_transposed"] else (e, f, h), 16.0, gen).to(torch.float8_e4m3fn)
        s["a_inv"] = torch.full((e,), 1 / 16, device="cuda")
        s["b_inv"] = torch.full((e,), 0.02 / 16, device="cuda")
        return s

    if kind == "linear_step":
        s["module"] = pkg.GroupedLinear(h, f, e, torch.bfloat16, cutlass=case["cutlass"])
    else:
        s["module"] = pkg.GroupedMlp(h, f, e, torch.bfloat16)
    s["experts"] = [s["module"]]
    for p in s["module"].parameters():
        p.data.copy_(_normal(p.shape, 0.02, gen))
    s["x"] = _normal((case["tokens"], h), 1.0, gen).requires_grad_()
    s["dy"] = _normal((case["tokens"], f if kind == "linear_step" else h), 1e-2, gen)
    s["first"] = None
    _step(s)
    if kind == "mlp_forward":      # scales from a training pass, weights cast once for serving
        _step(s)
        s["x"] = s["x"].detach()
        s["module"].eval()
        for p in s["module"].parameters():
            p.grad = None
        with torch.no_grad(), pkg.fp8_autocast(fp8_recipe=s["recipe"]):
            s["module"](s["x"], s["sizes"], is_first_microbatch=True)
    elif case.get("micro"):
        s["first"] = True
        _step(s)
        s["first"] = False
    return s


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def _step(s):
    module, x = s["module"], s["x"]
    module.zero_grad(set_to_none=True)
    x.grad = None
    with pkg.fp8_autocast(enabled=True, fp8_recipe=s["recipe"]):
        if "sizes" not in s:
            out = module(x)
        elif s["first"] is None:
            out = module(x, s["sizes"])
        else:
            out = module(x, s["sizes"], is_first_microbatch=s["first"])
    out.backward(s["dy"])
    return [out.detach(), x.grad] + [p.grad for p in module.parameters()] + [t for m in s["experts"] for t in _state(m)]


def run(state):
    kind = state["case"]["kind"]
    if kind == "cast_transpose":
        backend.multi_cast_transpose(state["ins"], state["outs"], state["touts"], state["scales"], state["amaxes"])
        return [t.view(torch.uint8) for t in state["outs"] + state["touts"]] + [state["amaxes"]]
    if kind == "gmm":
        return backend.fp8_gmm(state["a"], state["b"], state["sizes"], state["a_inv"], state["b_inv"],
                               b_transposed=state["case"]["b_transposed"])
    if kind == "mlp_forward":
        with torch.no_grad(), pkg.fp8_autocast(fp8_recipe=state["recipe"]):
            return state["module"](state["x"], state["sizes"], is_first_microbatch=False)
    return _step(state)
