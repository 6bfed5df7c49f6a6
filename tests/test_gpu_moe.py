"""Token routing on the GPU (sort / histogram / gather / scatter and their gradients) against the CPU oracle,
and the routed example layers end to end.  Integer results and copied rows are compared bit for bit; scatter's
bf16 output too (the kernel and the oracle follow the same fp32 sequence); only the per-row dot products of
scatter's weight gradient, whose summation order differs, get a tolerance (1e-5 relative to the row norms)."""
import contextlib

import numpy as np
import pytest
import torch

from oracle import moe as orc

pytestmark = pytest.mark.gpu


def _ops():
    from fp8_gmm_amd import moe_ops

    return moe_ops


def _ids(n, e, seed, kind="uniform"):
    rng = np.random.default_rng(seed)
    if kind == "zipf":
        p = 1.0 / np.arange(1, e + 1) ** 1.1
        return rng.choice(e, size=n, p=p / p.sum())
    if kind == "one":
        return np.full(n, e - 1)
    return rng.integers(0, e, size=n)


ROUTE_CASES = [(1, 1, "uniform"), (63, 4, "uniform"), (64, 2, "uniform"), (1000, 4, "uniform"), (1025, 7, "zipf"),
               (32768, 8, "uniform"), (24576, 64, "zipf"), (65536, 128, "uniform"), (70000, 4096, "uniform"),
               (5000, 16, "one"), (0, 8, "uniform")]


@pytest.mark.parametrize("n,e,kind", ROUTE_CASES)
def test_sort_histogram_and_bins(dev, n, e, kind):
    ops = _ops()
    ids = _ids(n, e, 100 + n, kind)
    x = torch.tensor(ids, dtype=torch.int32, device=dev)
    want_indices, want_bin_ids, want_bins, want_counts = orc.indices_and_bins(ids, e)
    indices, bin_ids, bins, counts = ops.indices_and_bins(x, max(int(np.ceil(np.log2(e))), 1), e)
    assert indices.dtype == bin_ids.dtype == bins.dtype == counts.dtype == torch.int32
    assert indices.cpu().tolist() == want_indices.tolist()
    assert bin_ids.cpu().tolist() == want_bin_ids.tolist()
    assert counts.cpu().tolist() == want_counts.tolist()
    assert bins.cpu().tolist() == want_bins.tolist()
    # the single operators give the same answers
    end_bit = max(int(np.ceil(np.log2(e))), 1)
    s_ids, s_idx = ops.sort(x, end_bit)
    assert torch.equal(s_ids, bin_ids) and torch.equal(s_idx, indices)
    assert torch.equal(ops.histogram(x, e), counts)
    assert torch.equal(ops.inclusive_cumsum(counts, 0), bins)
    _, _, inverse, _, _ = ops.route(x, e, want_inverse=True)
    assert inverse.cpu().tolist() == orc.invert(want_indices).tolist()


@pytest.mark.parametrize("n,e", [(1, 512), (1024, 512), (1025, 300), (3062, 16), (8192, 128), (8193, 128), (8192, 513)])
def test_short_lists_and_the_routers_own_ids(dev, n, e):
    """Both sides of the limits of the one-launch sort; int64 ids, some out of range, give what their int32 conversion gives."""
    ops = _ops()
    ids = _ids(n, e, 7 + n, "zipf")
    ids[::97] = -5
    ids[1::89] = e + 3
    want_indices, want_bin_ids, want_bins, want_counts = orc.indices_and_bins(ids.clip(0, e - 1), e)
    for x in (torch.tensor(ids, device=dev), torch.tensor(ids, dtype=torch.int32, device=dev)):
        indices, bin_ids, bins, counts, inverse = ops.indices_bins_and_inverse(x, e)
        assert indices.cpu().tolist() == want_indices.tolist()
        assert bin_ids.cpu().tolist() == want_bin_ids.tolist()
        assert counts.cpu().tolist() == want_counts.tolist()
        assert bins.cpu().tolist() == want_bins.tolist()
        assert inverse.cpu().tolist() == orc.invert(want_indices).tolist()
        assert all(torch.equal(a, b) for a, b in zip(ops.indices_and_bins(x, 1, e), (indices, bin_ids, bins, counts)))


def test_out_of_range_ids_are_clamped(dev):
    ops = _ops()
    x = torch.tensor([5, -3, 2, 9, 0], dtype=torch.int32, device=dev)
    bin_ids, indices = ops.sort(x, 2)          # ids below 4
    assert bin_ids.cpu().tolist() == [0, 0, 2, 3, 3] and indices.cpu().tolist() == [1, 4, 2, 0, 3]
    with pytest.raises(RuntimeError):
        ops.histogram(x, 5000)
    with pytest.raises(RuntimeError):
        ops.sort(x.long())


ROW_CASES = [(1, 1, 8, 1), (37, 2, 256, 4), (128, 2, 4096, 8), (50, 1, 520, 3), (64, 8, 768, 16), (33, 3, 100, 5),
             (16, 2, 6, 2), (0, 2, 64, 4)]


@pytest.mark.parametrize("tokens,top_k,hidden,e", ROW_CASES)
def test_gather_scatter_and_their_gradients(dev, tokens, top_k, hidden, e):
    ops = _ops()
    g = torch.Generator().manual_seed(7 + tokens)
    ids = _ids(tokens * top_k, e, 200 + tokens)
    indices_cpu = orc.sort(ids)[1]
    indices = torch.tensor(indices_cpu, dtype=torch.int32, device=dev)
    x = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16)
    y = torch.randn(tokens * top_k, hidden, generator=g).to(torch.bfloat16)
    w = torch.rand(tokens * top_k, generator=g)
    grad_rows = torch.randn(tokens * top_k, hidden, generator=g).to(torch.bfloat16)
    grad_tok = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16)

    xd = x.to(dev).requires_grad_()
    got = ops.gather(xd, indices, None, None, top_k)
    assert torch.equal(got.cpu().view(torch.int16), orc.gather(x, indices_cpu, top_k).view(torch.int16))
    got.backward(grad_rows.to(dev))
    assert torch.equal(xd.grad.cpu().view(torch.int16),
                       orc.gather_backward(grad_rows, indices_cpu, top_k).view(torch.int16))

    for weights in (w, None):
        yd = y.to(dev).requires_grad_()
        wd = weights.to(dev).requires_grad_() if weights is not None else None
        out = ops.scatter(yd, indices, None, wd, None, top_k)
        assert torch.equal(out.cpu().view(torch.int16), orc.scatter(y, indices_cpu, top_k, weights).view(torch.int16))
        out.backward(grad_tok.to(dev))
        want_gx, want_gw = orc.scatter_backward(grad_tok, y, indices_cpu, top_k, weights)
        assert torch.equal(yd.grad.cpu().view(torch.int16), want_gx.view(torch.int16))
        if weights is not None and tokens:
            idx = torch.as_tensor(indices_cpu.astype(np.int64))
            bound = torch.zeros(tokens * top_k)
            bound[idx] = y.float().norm(dim=1) * grad_tok.float()[idx // top_k].norm(dim=1)
            assert ((wd.grad.cpu() - want_gw).abs() <= 1e-5 * bound + 1e-30).all()


@pytest.mark.parametrize("tokens,e,top_k,dtype", [(1, 1, 1, torch.float32), (1000, 16, 2, torch.bfloat16),
                                                   (16384, 16, 2, torch.bfloat16), (513, 64, 8, torch.float32),
                                                   (300, 200, 3, torch.bfloat16), (77, 4096, 4, torch.float32),
                                                   (0, 8, 2, torch.bfloat16)])
def test_topk_against_the_oracle(dev, tokens, e, top_k, dtype):
    """softmax + top-k in one launch: the chosen experts equal the oracle's (bf16 scores are full of equal values,
    so this also holds the rule for ties), the weights agree to a few ulp of fp32, and the gradient with respect to
    the scores agrees with the oracle's float64 chain to fp32 / bf16 rounding."""
    ops = _ops()
    rng = np.random.default_rng(900 + tokens + e)
    z = torch.from_numpy(rng.standard_normal((tokens, e)).astype(np.float32) * 2).to(dtype)
    zd = z.to(dev).requires_grad_()
    w, sel = ops.topk(zd, top_k)
    assert w.dtype == torch.float32 and sel.dtype == torch.int64 and w.shape == sel.shape == (tokens, top_k)
    want_w, want_sel = orc.topk(z.float().numpy(), top_k)
    assert (sel.cpu().numpy() == want_sel).all()
    np.testing.assert_allclose(w.detach().cpu().numpy(), want_w, rtol=4e-6, atol=1e-30)
    gw = torch.from_numpy(rng.standard_normal((tokens, top_k)).astype(np.float32))
    w.backward(gw.to(dev))
    want_g = orc.topk_backward(z.float().numpy(), want_sel, gw.numpy())
    tol = 1e-2 if dtype == torch.bfloat16 else 1e-5
    assert zd.grad.dtype == dtype
    np.testing.assert_allclose(zd.grad.float().cpu().numpy(), want_g, rtol=tol, atol=tol * 1e-2)


def test_topk_falls_back_to_torch_and_renormalises(dev):
    ops = _ops()
    z = torch.randn(50, 8, device=dev, dtype=torch.float64)    # not a dtype of the kernel: torch's operators
    w, sel = ops.topk(z, 2)
    tw, tsel = torch.topk(torch.softmax(z, dim=1, dtype=torch.float), 2)
    assert torch.equal(sel, tsel) and torch.equal(w, tw)
    w, _ = ops.topk(z.float(), 2, moe_renorm=True)
    assert torch.allclose(w.sum(dim=1), torch.ones(50, device=dev))


@pytest.mark.parametrize("tokens,top_k,hidden,e", [(1000, 2, 256, 4), (513, 1, 4096, 7), (300, 4, 2056, 16),
                                                    (64, 2, 100, 3)])
def test_scatter_backward_in_one_pass_equals_the_two_passes(dev, tokens, top_k, hidden, e):
    """With both gradients wanted scatter's backward pass is one launch; it must write the bits of the two
    single-purpose launches (weighted gather, per-row dot products), which run when only one gradient is wanted -
    also on rows that 16-byte accesses cannot take (hidden = 100)."""
    ops = _ops()
    rng = np.random.default_rng(40 + tokens)
    ids = torch.tensor(rng.integers(0, e, size=tokens * top_k), dtype=torch.int32, device=dev)
    indices, bin_ids, bins, _ = ops.indices_and_bins(ids, 0, e)
    x = torch.from_numpy(rng.standard_normal((tokens * top_k, hidden)).astype(np.float32)).to(torch.bfloat16).to(dev)
    w = torch.from_numpy(rng.random(tokens * top_k).astype(np.float32)).to(dev)
    g = torch.from_numpy(rng.standard_normal((tokens, hidden)).astype(np.float32)).to(torch.bfloat16).to(dev)

    def grads(need_x, need_w):
        xd, wd = x.clone().requires_grad_(need_x), w.clone().requires_grad_(need_w)
        ops.scatter(xd, indices, bin_ids, wd, bins, top_k).backward(g)
        return xd.grad, wd.grad

    both_x, both_w = grads(True, True)
    only_x, _ = grads(True, False)
    _, only_w = grads(False, True)
    assert torch.equal(both_x.view(torch.int16), only_x.view(torch.int16))
    assert torch.equal(both_w.view(torch.int32), only_w.view(torch.int32))


def test_bad_arguments_are_rejected(dev):
    ops = _ops()
    x = torch.zeros(4, 8, dtype=torch.bfloat16, device=dev)
    idx = torch.arange(8, dtype=torch.int32, device=dev)
    with pytest.raises(RuntimeError):
        ops.gather(x.float(), idx, None, None, 2)
    with pytest.raises(RuntimeError):
        ops.gather(x, idx[:5], None, None, 2)
    with pytest.raises(RuntimeError):
        ops.scatter(x, idx[:4], None, torch.ones(3, device=dev), None, 2)
    with pytest.raises(RuntimeError):
        ops.gather(x.cpu(), idx.cpu(), None, None, 2)


@pytest.mark.parametrize("kind", ["mlp", "linear"])
def test_routed_layer_forward_against_the_oracle_composition(dev, kind):
    """Fp8MlpModule / Fp8LinearModule: with the layer's own routing decisions (read back from the GPU) the output
    must be scatter(experts(gather(x))) as the CPU oracle computes it."""
    import fp8_gmm_amd as pkg
    from fp8_gmm_amd import moe
    from helpers import assert_close_multistage
    from oracle import modules as orc_mod

    tokens, h, f, e, top_k = 96, 128, 256, 5, 2
    torch.manual_seed(11)
    layer = (moe.Fp8MlpModule if kind == "mlp" else moe.Fp8LinearModule)(h, f, e, top_k, device=dev)
    x = torch.randn(tokens, h).to(torch.bfloat16)
    with torch.no_grad(), pkg.fp8_autocast(fp8_recipe=pkg.DelayedScaling(amax_history_len=1)):
        out = layer(x.to(dev))
        weights0, selected = layer.gating_network(x.to(dev)), None
        weights0, selected = pkg.moe_ops.topk(weights0, top_k)
    ids = selected.flatten().cpu().numpy()
    w = weights0.flatten().cpu()
    indices, _, _, counts = orc.indices_and_bins(ids, e)
    sizes = counts.tolist()
    xs = orc.gather(x, indices, top_k)
    if kind == "mlp":
        fwd, bwd = orc_mod.Meta(3 * 2 * e, 1), orc_mod.Meta(2 * 2 * e, 1)
        y = orc_mod.grouped_mlp_step(xs, layer.grouped_mlp.fc1_weight.detach().cpu(),
                                     layer.grouped_mlp.fc2_weight.detach().cpu(), sizes,
                                     torch.zeros(tokens * top_k, h, dtype=torch.bfloat16), fwd, bwd)["out"]
    else:
        zeros = torch.zeros(tokens * top_k, f, dtype=torch.bfloat16)
        fwd, bwd = orc_mod.Meta(3 * e, 1), orc_mod.Meta(2 * e, 1)
        mid = orc_mod.grouped_linear_step(xs, layer.grouped_linear1.weight_tensor.detach().cpu(), sizes, zeros, fwd,
                                          bwd)["out"]
        mid = torch.nn.functional.gelu(mid.float()).to(torch.bfloat16)
        fwd, bwd = orc_mod.Meta(3 * e, 1), orc_mod.Meta(2 * e, 1)
        y = orc_mod.grouped_linear_step(mid, layer.grouped_linear2.weight_tensor.detach().cpu(), sizes,
                                        torch.zeros(tokens * top_k, h, dtype=torch.bfloat16), fwd, bwd)["out"]
    want = orc.scatter(y, indices, top_k, w)
    assert_close_multistage(out, want, 1e-2, f"{kind} layer output")


def test_routed_mlp_layer_trains_like_a_dense_fp32_model(dev):
    """Forward + backward of Fp8MlpModule against an fp32 autograd model of the same routed layer (same routing
    decisions): cosine similarity of the output and of every gradient, gating weights included."""
    import fp8_gmm_amd as pkg
    from fp8_gmm_amd import moe

    tokens, h, f, e, top_k = 512, 256, 512, 8, 2
    torch.manual_seed(12)
    layer = moe.Fp8MlpModule(h, f, e, top_k, device=dev)
    x = torch.randn(tokens, h, device=dev).to(torch.bfloat16)
    dy = torch.randn(tokens, h, device=dev).to(torch.bfloat16)
    for _ in range(2):   # the second pass runs with real scales
        xd = x.clone().requires_grad_()
        layer.zero_grad()
        with pkg.fp8_autocast(fp8_recipe=pkg.DelayedScaling(amax_history_len=2)):
            out = layer(xd)
        out.backward(dy)

    xr = x.float().requires_grad_()
    gate = layer.gating_network.weight.detach().float().requires_grad_()
    w1 = layer.grouped_mlp.fc1_weight.detach().float().requires_grad_()
    w2 = layer.grouped_mlp.fc2_weight.detach().float().requires_grad_()
    logits = layer.gating_network(x).float()                  # the layer's own bf16 logits decide the routing
    _, selected = pkg.moe_ops.topk(logits, top_k)
    probs = torch.softmax(xr @ gate.t(), dim=1)
    ref = torch.zeros(tokens, h, device=dev)
    for k in range(top_k):
        ek = selected[:, k]
        hidden = torch.nn.functional.gelu(torch.einsum("th,tfh->tf", xr, w1[ek]), approximate="tanh")
        ref = ref + probs.gather(1, ek[:, None]) * torch.einsum("tf,thf->th", hidden, w2[ek])
    ref.backward(dy.float())

    def cos(a, b):
        a, b = a.detach().float().flatten(), b.detach().float().flatten()
        return (torch.dot(a, b) / (a.norm() * b.norm())).item()

    assert cos(out, ref) > 0.995
    assert cos(xd.grad, xr.grad) > 0.99
    assert cos(layer.grouped_mlp.fc1_weight.grad, w1.grad) > 0.99
    assert cos(layer.grouped_mlp.fc2_weight.grad, w2.grad) > 0.99
    assert cos(layer.gating_network.weight.grad, gate.grad) > 0.98


def test_example_bf16_layer_against_a_dense_fp32_model(dev):
    """The bf16 layer of the example recipe (one vendor GEMM per expert on its row slice, hand-written gradients)
    against an fp32 autograd model of the same routed layer with the same routing decisions."""
    import fp8_gmm_amd as pkg
    from fp8_gmm_amd import example

    tokens, h, f, e, top_k = 384, 128, 256, 6, 2
    torch.manual_seed(21)
    layer = example.Bf16Module(h, f, e, top_k, device=dev)
    x = torch.randn(tokens, h, device=dev).to(torch.bfloat16)
    dy = torch.randn(tokens, h, device=dev).to(torch.bfloat16)
    xd = x.clone().requires_grad_()
    out = layer(xd)
    out.backward(dy)

    xr = x.float().requires_grad_()
    gate = layer.gating_network.weight.detach().float().requires_grad_()
    w1 = layer.w1.detach().float().requires_grad_()
    w2 = layer.w2.detach().float().requires_grad_()
    _, selected = pkg.moe_ops.topk(layer.gating_network(x).float(), top_k)
    probs = torch.softmax(xr @ gate.t(), dim=1)
    ref = torch.zeros(tokens, h, device=dev)
    for k in range(top_k):
        ek = selected[:, k]
        hidden = torch.nn.functional.gelu(torch.einsum("th,tfh->tf", xr, w1[ek]))
        ref = ref + probs.gather(1, ek[:, None]) * torch.einsum("tf,thf->th", hidden, w2[ek])
    ref.backward(dy.float())

    def cos(a, b):
        a, b = a.detach().float().flatten(), b.detach().float().flatten()
        return (torch.dot(a, b) / (a.norm() * b.norm())).item()

    assert cos(out, ref) > 0.9995
    assert cos(xd.grad, xr.grad) > 0.999
    assert cos(layer.w1.grad, w1.grad) > 0.999
    assert cos(layer.w2.grad, w2.grad) > 0.999
    assert cos(layer.gating_network.weight.grad, gate.grad) > 0.995


def test_example_recipe_runs_every_kind_of_layer(dev, capsys):
    """``python -m fp8_gmm_amd.example`` at a small size: four timed kinds, one printed line each."""
    from fp8_gmm_amd import example

    times = example.main(["--tokens", "512", "--hidden", "256", "--inner", "512", "--experts", "8", "--warmup", "1",
                          "--steps", "2"])
    assert list(times) == list(example.KINDS) and all(t > 0 for t in times.values())
    lines = [line for line in capsys.readouterr().out.splitlines() if " run: " in line]
    assert len(lines) == 4 and lines[0].startswith("Bf16Module run: ") and lines[3].startswith("Fp8MlpModule run: ")


@pytest.mark.parametrize("tokens,hidden,experts", [(1, 8, 1), (16, 64, 16), (17, 72, 5), (127, 136, 33), (128, 256, 32),
                                                   (129, 264, 65), (1531, 1024, 16), (4097, 520, 128), (16385, 192, 8)])
def test_gating_gradients_are_exact_on_whole_numbers(dev, tokens, hidden, experts):
    """Edges of the token, column and expert tiles, one slice of tokens and many: sums of products of small whole numbers
    are exact in fp32, so the one rounding to bf16 leaves nothing open.  Each gradient alone gives the same bits."""
    ops = _ops()
    gen = torch.Generator().manual_seed(tokens)
    x, w, g, up = (torch.randint(-3, 4, shape, generator=gen).to(torch.bfloat16) for shape in
                   [(tokens, hidden), (experts, hidden), (tokens, experts), (tokens, hidden)])
    want_x = up.double() + g.double() @ w.double()
    want_w = g.double().t() @ x.double()
    alone_x = g.double() @ w.double()
    linear = torch.nn.Linear(hidden, experts, bias=False, dtype=torch.bfloat16, device=dev)
    linear.weight.data.copy_(w)
    g, up = g.to(dev), up.to(dev)
    for train, rows in ((True, True), (True, False), (False, True)):
        xd = x.to(dev).requires_grad_()
        linear.requires_grad_(train).zero_grad()
        logits, again = ops.gating(linear, xd)
        assert "Gating" in logits.grad_fn.name()
        assert torch.equal(logits, torch.nn.functional.linear(xd, linear.weight)) and torch.equal(again, xd)
        torch.autograd.backward((logits, again) if rows else (logits,), (g, up) if rows else (g,))
        assert torch.equal(xd.grad.cpu(), (want_x if rows else alone_x).to(torch.bfloat16))
        if train:
            assert torch.equal(linear.weight.grad.cpu(), want_w.to(torch.bfloat16))


def test_gating_calls_a_module_that_is_more_than_a_product(dev):
    """Hooks, a bias, another class, rows the kernels do not take and rows without a gradient: the module is called, its
    hooks with it; a graph of the backward pass can be asked for on either path."""
    ops = _ops()
    x = torch.randn(33, 64, device=dev).to(torch.bfloat16)

    def linear(h=64, bias=False, dtype=torch.bfloat16):
        return torch.nn.Linear(h, 6, bias=bias, dtype=dtype, device=dev)

    seen = []
    hooked = linear()
    hooked.register_forward_hook(lambda *a: seen.append(1))
    replaced = linear()
    replaced.forward = lambda v: seen.append(2) or torch.nn.functional.linear(v, replaced.weight)
    odd = torch.randn(33, 65, device=dev).to(torch.bfloat16)
    wide = torch.randn(33, 128, device=dev).to(torch.bfloat16)
    for module, rows in ((hooked, x), (replaced, x), (linear(bias=True), x), (torch.nn.Sequential(linear()), x),
                         (linear(65), odd), (linear(), wide[:, :64]), (linear(dtype=torch.float32), x.float())):
        rows = rows.detach().requires_grad_()
        logits, again = ops.gating(module, rows)
        assert again is rows and "Gating" not in logits.grad_fn.name()
    assert seen == [1, 2]
    logits, again = ops.gating(linear(), x)
    assert again is x and "Gating" not in logits.grad_fn.name()
    plain, xd = linear(), x.detach().requires_grad_()
    logits, again = ops.gating(plain, xd)
    first, = torch.autograd.grad((logits.float() ** 2).sum() + again.float().sum(), xd, create_graph=True)
    second, = torch.autograd.grad(first.float().sum(), xd)
    want = 2 * (plain.weight.float().t() @ plain.weight.float()).sum(0)     # the Hessian of |W x|^2 times ones
    assert torch.allclose(second.float(), want.expand_as(second), rtol=2e-2, atol=2e-2 * want.abs().max().item())


@pytest.mark.parametrize("tokens,hidden,experts,trained,kernels", [
    (1 << 16, 64, 64, False, True), (1 << 15, 72, 63, True, True),                        # up to 64 experts
    (1 << 15, 64, 65, False, True), ((1 << 15) + 1, 64, 65, False, False),                # up to 2^21 values of x
    ((1 << 15) + 1, 64, 72, False, True), ((1 << 15) + 1, 64, 65, True, True),            # whole 16 bytes of gradients a token
    (1025, 2048, 100, True, True), (1025, 2056, 100, True, False), (1025, 2056, 104, True, True),
    (1025, 4104, 104, True, False), (8191, 4096, 127, True, False), (8192, 4096, 127, True, True),
    (8192, 4104, 127, True, False), (8192, 4104, 128, False, True)])
def test_gating_runs_on_the_kernels_where_they_are_faster(dev, tokens, hidden, experts, trained, kernels):
    """Many experts: the general path where the library's products are ahead (both sides in csrc/gating.hip)."""
    linear = torch.nn.Linear(hidden, experts, bias=False, dtype=torch.bfloat16, device=dev).requires_grad_(trained)
    x = torch.zeros(tokens, hidden, dtype=torch.bfloat16, device=dev, requires_grad=True)
    logits, again = _ops().gating(linear, x)
    assert ("Gating" in logits.grad_fn.name()) == kernels == (again is not x)


@pytest.mark.parametrize("layer", ["linear", "mlp"])
def test_rows_may_be_changed_in_place_behind_a_layer_whose_gate_is_frozen(dev, layer):
    """``x += layer(x)``: with a frozen gating weight nothing of the pass needs the rows as they were."""
    from fp8_gmm_amd.moe import Fp8LinearModule, Fp8MlpModule

    rows = torch.randn(70, 64, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).to(dev)
    grads = []
    for in_place in (False, True):
        torch.manual_seed(5)   # a module each: a pass changes its scaling state
        module = (Fp8MlpModule if layer == "mlp" else Fp8LinearModule)(64, 96, 4, 2, device=dev)
        module.gating_network.requires_grad_(False)
        leaf = rows.clone().requires_grad_()
        x = leaf * 1
        out = module(x)
        y = x.add_(out) if in_place else x + out
        y.backward(torch.ones_like(y))
        grads.append(leaf.grad)
    assert torch.isfinite(grads[0].float()).all() and torch.equal(grads[0], grads[1])


def test_a_compute_of_ones_own_may_change_the_rows_in_place(dev):
    """With a frozen gate nothing else needs the rows as they were, and a subclass gets the rows themselves."""
    from fp8_gmm_amd.moe import Fp8MlpModule

    class Doubled(Fp8MlpModule):
        in_place = False

        def compute(self, x, *rest):
            return super().compute(x.mul_(2) if self.in_place else x * 2, *rest)

    rows = torch.randn(70, 64, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).to(dev)
    results = []
    for in_place in (False, True):
        torch.manual_seed(5)
        module = Doubled(64, 96, 4, 2, device=dev)
        module.in_place = in_place
        module.gating_network.requires_grad_(False)
        leaf = rows.clone().requires_grad_()
        y = module(leaf * 1)
        y.backward(torch.ones_like(y))
        results.append((y, leaf.grad))
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_gating_gradients_check_what_saved_tensor_hooks_return(dev):
    """Such a hook may hand the backward pass another type, device or shape: what torch's linear makes of it, an error, and no
    kernel on memory that is not what it reads.  (Gradient hooks that change these are refused by autograd.)"""
    ops = _ops()
    gen = torch.Generator().manual_seed(9)
    x, w, g = (torch.randint(-3, 4, shape, generator=gen).to(torch.bfloat16).to(dev) for shape in [(40, 64), (6, 64), (40, 6)])
    linear = torch.nn.Linear(64, 6, bias=False, dtype=torch.bfloat16, device=dev)
    linear.weight.data.copy_(w)

    def passes(kernels, unpack):
        linear.zero_grad()
        xd = x.clone().requires_grad_()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            logits = ops.gating(linear, xd)[0] if kernels else linear(xd)
        assert ("Gating" in logits.grad_fn.name()) == kernels
        logits.backward(g)
        return xd.grad, linear.weight.grad

    want = passes(False, lambda t: t)
    for same in (lambda t: t, lambda t: t.cpu().to(dev), lambda t: t.t().contiguous().t()):
        assert all(torch.equal(a, b) for a, b in zip(passes(True, same), want))
    for other in (lambda t: t.float(), lambda t: t.cpu(), lambda t: t[:, :32], lambda t: t[:3]):
        for kernels in (False, True):
            with pytest.raises(RuntimeError):
                passes(kernels, other)


def _layer_results(layer, state, x, dy, frozen, steps=2):
    """Outputs, gradients and scaling state of a routed layer over some steps."""
    from fp8_gmm_amd import DelayedScaling, fp8_autocast

    layer.load_state_dict(state)
    for name, p in layer.named_parameters():
        p.requires_grad_(not any(f in name for f in frozen))
        p.grad = None
    results = []
    for step in range(steps):
        xs = (x * (1 + step)).detach().requires_grad_("x" not in frozen)
        with fp8_autocast(fp8_recipe=DelayedScaling(amax_history_len=4)):
            out = layer(xs)
        results.append(out.detach().clone())
        if out.requires_grad:
            out.backward(dy)
            results += [t.grad.clone() for t in [xs] + list(layer.parameters()) if t.grad is not None]
            for p in layer.parameters():
                p.grad = None
    for m in layer.modules():
        if "scaling_fwd" in getattr(m, "fp8_meta", {}):
            results += [t.clone() for d in ("scaling_fwd", "scaling_bwd") for t in m.fp8_meta[d].state().values()]
    return results


@pytest.mark.parametrize("kind,tokens,hidden,inner,experts,top_k,frozen", [
    ("mlp", 300, 256, 512, 8, 2, ()), ("mlp", 37, 2064, 48, 5, 3, ()), ("mlp", 1, 16, 16, 4, 1, ()),
    ("mlp", 65, 4112, 160, 100, 2, ("gating", "x")), ("mlp", 64, 256, 256, 4, 2, ("grouped",)),
    ("mlp", 64, 256, 256, 4, 2, ("grouped", "x")), ("mlp", 64, 256, 256, 4, 2, ("grouped", "x", "gating")),
    ("linear", 301, 1024, 528, 16, 2, ()), ("linear", 5, 48, 2064, 3, 3, ("gating",)), ("linear", 0, 64, 64, 4, 2, ()),
    ("linear", 130, 256, 128, 8, 2, ("grouped_linear1", "x")), ("cutlass", 77, 272, 528, 6, 2, ()),
    ("mlp", 9000, 256, 64, 16, 2, ()), ("mlp", 3000, 64, 64, 300, 8, ()), ("linear", 40, 256, 64, 4, 2, ("nan",)),
    # a wavefront that goes on to a second token (from 16384 rows of one choice, 32768 of two), the last ones with fewer; rows of
    # two pieces, fetched again for the token's second choice (from 16384 rows); NaN in tokens that are not a wavefront's first
    ("mlp", 16411, 64, 48, 16, 2, ()), ("linear", 16411, 64, 48, 5, 1, ()), ("mlp", 8203, 4112, 16, 6, 2, ()),
    ("linear", 8203, 4112, 16, 6, 2, ("nan",)), ("mlp", 16411, 64, 48, 16, 2, ("nan",)), ("mlp", 16411, 4112, 16, 6, 2, ("nan",)),
    ("linear", 12301, 96, 32, 7, 4, ("nan",)), ("mlp", 40, 8224, 32, 3, 2, ("nan",)),
    # wavefronts that begin and end inside a token (from 16384 rows of three choices or more)
    ("mlp", 5501, 64, 48, 7, 3, ("nan",)), ("linear", 5501, 4112, 16, 7, 3, ("nan",)), ("mlp", 5301, 96, 32, 20, 8, ("nan",))])
def test_routed_rows_give_the_bits_of_gather_and_scatter(dev, monkeypatch, kind, tokens, hidden, inner, experts, top_k, frozen):
    """A layer whose experts' casts fetch and weigh their rows themselves against the same layer between moe_ops.gather and
    moe_ops.scatter: outputs, every gradient and the scaling state, bit for bit."""
    ops = _ops()
    from fp8_gmm_amd.moe import Fp8LinearModule, Fp8MlpModule

    torch.manual_seed(tokens + hidden)
    layer = Fp8MlpModule(hidden, inner, experts, top_k) if kind == "mlp" else \
        Fp8LinearModule(hidden, inner, experts, top_k, cutlass=kind == "cutlass")
    twin = Fp8MlpModule(hidden, inner, experts, top_k) if kind == "mlp" else \
        Fp8LinearModule(hidden, inner, experts, top_k, cutlass=kind == "cutlass")
    state = layer.state_dict()
    x = torch.randn(tokens, hidden, device=dev).to(torch.bfloat16)
    dy = (torch.randn(tokens, hidden, device=dev) * 1e-2).to(torch.bfloat16)
    if "nan" in frozen:
        frozen = ()
        x[3, 5], x[7, -56], dy[4, -1], dy[9, 0] = float("nan"), float("inf"), float("nan"), -float("inf")
        if tokens > 8000:
            x[-1, -1], x[5001, 9], dy[-2, -1], dy[6003, 17] = float("nan"), float("inf"), float("nan"), float("inf")
    calls = []
    for name in ("gather", "scatter"):
        monkeypatch.setattr(ops, name, lambda *a, _f=getattr(ops, name), _n=name, **k: (calls.append(_n), _f(*a, **k))[1])
    got = _layer_results(layer, state, x, dy, frozen)
    assert not calls
    monkeypatch.setattr(ops, "routed_rows_fit", lambda *a: False)
    want = _layer_results(twin, state, x, dy, frozen)
    assert calls and len(got) == len(want)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


def test_choices_without_a_place_leave_nothing_behind(dev):
    """An entry of ``inverse`` that is no row of the pass: the choice is left out, as the row movers leave it out, of the experts'
    maxima too, and its weight has a gradient of zero."""
    from fp8_gmm_amd import GroupedLinear, native

    x, dy = torch.randn(8, 64, device=dev).to(torch.bfloat16), torch.randn(8, 32, device=dev).to(torch.bfloat16)
    places = [1, 0, -1, 2, 3, 8, 6, 7]     # of the tokens' choices; the rows 4 and 5 are nobody's
    x[2, 5], x[5, 7] = 1000.0, 2000.0
    dy[2, 3], dy[5, 9] = float("inf"), 500.0
    inverse = torch.tensor(places, dtype=torch.int32, device=dev)
    weights = torch.full((8,), 0.5, device=dev, requires_grad=True)
    layer = GroupedLinear(64, 32, 3, torch.bfloat16, device=dev)
    layer.cast_weights_ahead()
    xi = x.clone().requires_grad_()
    out = layer._routed(xi, torch.tensor([3, 0, 5]), native.Route(inverse.clone(), inverse, weights, 1, True, True))
    out.backward(dy)
    experts = [[t for t, p in enumerate(places) if lo <= p < hi] for lo, hi in ((0, 3), (3, 8))]
    fwd, bwd = layer.fp8_meta["scaling_fwd"].amax_history[0], layer.fp8_meta["scaling_bwd"].amax_history[0]
    for slot, tokens in zip((0, 2), experts):
        assert fwd[3 * slot].item() == x[tokens].abs().max().item()
        assert bwd[2 * slot].item() == (dy[tokens] * 0.5).abs().max().item()
    assert fwd[3].item() == 0 and bwd[2].item() == 0
    assert weights.grad[2] == 0 and weights.grad[5] == 0
    assert not out[[2, 5]].any() and not xi.grad[[2, 5]].any()


def test_routed_rows_are_left_to_gather_where_something_looks_on(dev, monkeypatch):
    """A hook on the experts, a replaced `experts` and saved-tensor hooks see what they saw."""
    ops = _ops()
    from fp8_gmm_amd.moe import Fp8LinearModule, Fp8MlpModule

    calls = []
    gather = ops.gather
    monkeypatch.setattr(ops, "gather", lambda *a, **k: (calls.append("gather"), gather(*a, **k))[1])
    x = torch.randn(64, 256, device=dev).to(torch.bfloat16).requires_grad_()

    def gathers(layer):
        calls.clear()
        layer(x).sum().backward()
        return bool(calls)

    layer = Fp8MlpModule(256, 128, 4, 2)
    assert not gathers(layer)
    seen = []
    handle = layer.grouped_mlp.register_forward_hook(lambda m, i, o: seen.append(i[0].shape))
    assert gathers(layer) and seen == [torch.Size([128, 256])]
    handle.remove()
    assert not gathers(layer)
    layer.experts = lambda rows, sizes: layer.grouped_mlp(rows, sizes)
    assert gathers(layer)
    del layer.experts
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(dev)):
        assert gathers(layer)
    two = Fp8LinearModule(256, 128, 4, 2)
    two.grouped_linear2.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    assert not gathers(two) and seen[-1] == torch.Size([128, 256])   # the first layer fetches, the second is called

    class Rows(Fp8MlpModule):
        def experts(self, rows, sizes):
            return super().experts(rows * 1, sizes)

    assert gathers(Rows(256, 128, 4, 2))


@pytest.mark.parametrize("tokens,hidden,top_k,fetched", [
    (65535, 240, 1, True), (65536, 240, 1, False), (65536, 256, 1, True), (32768, 64, 2, True), (32769, 64, 2, False),
    (32769, 256, 2, True), (8192, 16, 8, True), (8193, 16, 8, False)])
def test_many_narrow_rows_are_gathered(dev, monkeypatch, tokens, hidden, top_k, fetched):
    """Rows of few columns in large numbers, which the casts fetch slower than they are gathered, on either side of the line."""
    ops = _ops()
    from fp8_gmm_amd.moe import Fp8MlpModule

    calls, gather = [], ops.gather
    monkeypatch.setattr(ops, "gather", lambda *a, **k: (calls.append(1), gather(*a, **k))[1])
    x = torch.randn(tokens, hidden, device=dev).to(torch.bfloat16).requires_grad_()
    layer = Fp8MlpModule(hidden, 16, 16, top_k)
    layer(x).sum().backward()
    assert bool(calls) is not fetched and torch.isfinite(x.grad).all()


@pytest.mark.parametrize("kind", ["mlp", "linear"])
def test_routed_passes_cast_the_weights_themselves_where_nobody_did(dev, monkeypatch, kind):
    """A layer that starts nothing ahead of its counts: the routed pass casts the experts' weights as well, behind the scaling
    update that is due, with the bits of gather and scatter."""
    ops = _ops()
    from fp8_gmm_amd.moe import Fp8LinearModule, Fp8MlpModule

    class Late((Fp8MlpModule if kind == "mlp" else Fp8LinearModule)):
        def start_experts(self):
            pass

    x, dy = torch.randn(77, 64, device=dev).to(torch.bfloat16), torch.randn(77, 64, device=dev).to(torch.bfloat16)
    layer, twin, calls, gather = Late(64, 48, 5, 2), Late(64, 48, 5, 2), [], ops.gather
    state = layer.state_dict()
    monkeypatch.setattr(ops, "gather", lambda *a, **k: (calls.append(1), gather(*a, **k))[1])
    got = _layer_results(layer, state, x, dy, (), steps=4)
    assert len(calls) == 1   # of the first step, which has no scaling state yet
    monkeypatch.setattr(ops, "routed_rows_fit", lambda *a: False)
    want = _layer_results(twin, state, x, dy, (), steps=4)
    assert len(calls) == 5 and len(got) == len(want)
    for a, b in zip(got, want):
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.parametrize("kind,launches", [
    ("mlp", {"multi_quantize": 1, "routed_cast": 1, "routed_gradient": 1, "multi_cast_dgelu": 1, "grouped_gemm": 6,
             "moe_scatter": 2, "gating_backward": 1}),
    ("linear", {"multi_quantize": 4, "routed_cast": 1, "routed_gradient": 1, "grouped_gemm": 6, "moe_scatter": 2,
                "gating_backward": 1})])
def test_kernel_timing_of_a_routed_layer_is_that_of_its_launches(dev, monkeypatch, kind, launches):
    """A block of kernel timing around a routed layer's step records the launches that the step makes without it: no gather,
    the casts that fetch their rows, the same bits."""
    ops = _ops()
    from fp8_gmm_amd import DelayedScaling, backend, fp8_autocast
    from fp8_gmm_amd.moe import Fp8LinearModule, Fp8MlpModule

    make = lambda: (Fp8MlpModule if kind == "mlp" else Fp8LinearModule)(256, 128, 4, 2)
    state = make().state_dict()
    x0 = torch.randn(64, 256, device=dev).to(torch.bfloat16)
    dy = torch.randn(64, 256, device=dev).to(torch.bfloat16)
    gathers, gather = [], ops.gather
    monkeypatch.setattr(ops, "gather", lambda *a, **k: (gathers.append(1), gather(*a, **k))[1])

    def steps(timed):
        layer, results = make(), []
        layer.load_state_dict(state)
        for _ in range(3):   # the second and third begin with a scaling update
            x = x0.clone().requires_grad_()
            layer.zero_grad()
            with fp8_autocast(fp8_recipe=DelayedScaling(amax_history_len=4)):
                with backend.kernel_timing() if timed else contextlib.nullcontext() as timing:
                    out = layer(x)
                    out.backward(dy)
            results += [out.detach(), x.grad] + [p.grad.clone() for p in layer.parameters()]
            if timed:
                assert {name: rec["launches"] for name, rec in timing.summary().items()} == launches
        return results

    for a, b in zip(steps(False), steps(True)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert not gathers


def test_gathered_rows_are_gathered_ahead_of_the_wait_for_the_counts(dev, monkeypatch):
    """Where a layer's experts do not fetch their rows themselves, the GPU has the gather to do while the host waits."""
    from fp8_gmm_amd import moe

    ops, order, native = _ops(), [], moe.route
    gather = ops.gather

    class Waits:
        def __init__(self, counts):
            self.counts = counts

        def wait(self):
            order.append("wait")
            return self.counts.wait()

    def route(scores, top_k):
        *lists, counts = native(scores, top_k)
        return (*lists, Waits(counts))

    monkeypatch.setattr(ops, "gather", lambda *a, **k: (order.append("gather"), gather(*a, **k))[1])
    monkeypatch.setattr(moe, "route", route)
    x = torch.randn(64, 256, device=dev).to(torch.bfloat16)
    layer = moe.Fp8MlpModule(256, 128, 4, 2)
    want = layer(x)
    assert order == ["wait"]
    layer.grouped_mlp.register_forward_hook(lambda *a: None)
    got = layer(x)
    assert order == ["wait", "gather", "wait"] and got.shape == want.shape


@pytest.mark.parametrize("tokens,experts,top_k,dtype", [(1, 1, 1, torch.float32), (1531, 16, 2, torch.bfloat16),
                                                         (5000, 128, 8, torch.bfloat16), (33, 600, 3, torch.float32),
                                                         (0, 4, 2, torch.bfloat16)])
def test_native_routing_gives_the_bits_of_the_functions(dev, tokens, experts, top_k, dtype):
    """native.route against topk, the sort and the counts one by one; the gradient of its weights against topk's."""
    ops = _ops()
    from fp8_gmm_amd import native

    g = torch.Generator().manual_seed(tokens + experts)
    scores = torch.randn(tokens, experts, generator=g).to(dtype).to(dev)
    a, b = scores.clone().requires_grad_(), scores.clone().requires_grad_()
    assert ops.router_fits(a, top_k, experts) is (type(a) is torch.Tensor)
    weights, indices, bin_ids, bins, counts, inverse, posted = native.route(a, top_k)
    want_weights, selected = ops.topk(b, top_k)
    want = ops.indices_bins_and_inverse(selected.flatten(), experts)
    for x, y in zip((indices, bin_ids, bins, counts, inverse), want):
        assert x.dtype == y.dtype and torch.equal(x, y)
    assert posted.wait() == counts.cpu().tolist()
    assert torch.equal(weights, want_weights.flatten()) and weights.requires_grad
    grad = torch.randn(tokens * top_k, generator=g).to(dev)
    weights.backward(grad)
    want_weights.flatten().backward(grad)
    assert torch.equal(a.grad, b.grad) and a.grad.dtype == dtype
    with torch.no_grad():
        assert not native.route(a, top_k)[0].requires_grad


def test_native_gating_differentiates_twice_and_is_timed(dev):
    """A graph of the gating gradients is torch's own; a block of kernel timing that opens behind the forward pass sees the
    backward launches, with the same bits."""
    ops = _ops()
    from fp8_gmm_amd import backend
    from fp8_gmm_amd.moe import Fp8MlpModule

    gate = torch.nn.Linear(256, 8, bias=False).to(torch.bfloat16).to(dev)
    x = torch.randn(64, 256, device=dev).to(torch.bfloat16).requires_grad_()
    logits, rows = ops.gating(gate, x)
    assert logits.grad_fn.name() == rows.grad_fn.name() == "GatingBackward"
    assert torch.equal(rows, x) and torch.equal(logits, torch.nn.functional.linear(x, gate.weight))
    up = torch.randn(64, 8, device=dev).to(torch.bfloat16).requires_grad_()
    (gx,) = torch.autograd.grad(logits, x, up, create_graph=True)
    gw, gup = torch.autograd.grad(gx, (gate.weight, up), torch.ones_like(gx))
    assert torch.equal(gx, up.detach() @ gate.weight)
    assert torch.equal(gw, up.detach().t() @ torch.ones_like(gx)) and torch.equal(gup, torch.ones_like(gx) @ gate.weight.t())
    logits, rows = ops.gating(gate, x)   # the rows' gradient alone
    assert torch.equal(torch.autograd.grad(rows, x, torch.ones_like(x))[0], torch.ones_like(x))

    layer = Fp8MlpModule(256, 128, 4, 2)
    twin = Fp8MlpModule(256, 128, 4, 2)
    twin.load_state_dict(layer.state_dict())
    dy = torch.randn(64, 256, device=dev).to(torch.bfloat16)
    grads = []
    for module, timed in ((layer, False), (twin, True)):
        x.grad = None
        out = module(x)
        if timed:
            with backend.kernel_timing() as timing:
                out.backward(dy)
            assert {"routed_gradient", "grouped_gemm", "gating_backward"} <= set(timing.summary())
        else:
            out.backward(dy)
        grads.append([x.grad.clone()] + [p.grad.clone() for p in module.parameters()])
    assert all(torch.equal(a, b) for a, b in zip(*grads))
