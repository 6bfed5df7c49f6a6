"""Host-side logic that needs no GPU: token-split bookkeeping, scaling-metadata slot arithmetic,
the delayed-scaling update rule and the recipe / autocast plumbing.

Expected values are worked out from the reference's formulas (fp8_gmm/utils.py:48-62 and :98-103),
not by calling the code under test twice.
"""
import pytest
import torch

from fp8_gmm_amd import fp8
from fp8_gmm_amd.utils import (
    DType,
    Fp8MetaWrapper,
    Fp8TensorType,
    MetaTensorType,
    cumsum_group_sizes,
    to_tex_dtype,
    to_torch_dtype,
)
from oracle import modules as orc


def test_cumsum_group_sizes_config1():
    # worked by hand: [137, 401, 59, 403] padded to multiples of 16 -> [144, 416, 64, 416]
    e, padded, cums, pcums = cumsum_group_sizes([137, 401, 59, 403], need_padding=True)
    assert (e, padded) == (4, True)
    assert cums == [0, 137, 538, 597, 1000]
    assert pcums == [0, 144, 560, 624, 1040]


def test_cumsum_group_sizes_variants():
    assert cumsum_group_sizes([16, 32, 16], need_padding=True) == (3, False, [0, 16, 48, 64], [0, 16, 48, 64])
    assert cumsum_group_sizes([16, 32, 16]) == (3, False, [0, 16, 48, 64], None)
    assert cumsum_group_sizes([5, 0, 17], need_padding=True) == (3, True, [0, 5, 5, 22], [0, 16, 16, 48])
    assert cumsum_group_sizes([5, 0, 129], True, pad_multiple=128) == (3, True, [0, 5, 5, 134], [0, 128, 128, 384])
    assert cumsum_group_sizes(torch.tensor([3, 4]).tolist(), True)[3] == [0, 16, 32]
    assert cumsum_group_sizes([], True) == (0, False, [0], [0])


def test_dtype_maps():
    assert to_tex_dtype(torch.float8_e4m3fn) == DType.kFloat8E4M3
    assert to_tex_dtype(torch.float8_e5m2) == DType.kFloat8E5M2
    assert to_tex_dtype(torch.bfloat16) == DType.kBFloat16
    for d in DType:
        assert to_tex_dtype(to_torch_dtype(d)) == d
    with pytest.raises(ValueError):
        to_tex_dtype(torch.float16)


class _Meta:
    def __init__(self, slots, hist=2):
        self.scale = torch.arange(slots, dtype=torch.float32) + 1000
        self.scale_inv = torch.arange(slots, dtype=torch.float32) + 2000
        self.amax_history = (torch.arange(hist * slots, dtype=torch.float32) + 3000).reshape(hist, slots)


@pytest.mark.parametrize("e", [1, 4])
def test_meta_wrapper_slot_arithmetic(e):
    """slot = (group * E + i) * stride + weight, stride 3 forward / 2 backward (utils.py:98-103)."""
    fwd, bwd = _Meta(3 * 2 * e), _Meta(2 * 2 * e)
    w = Fp8MetaWrapper(e, {"scaling_fwd": fwd, "scaling_bwd": bwd})
    w.set_forward_scale_inv_cloned()
    expect = {
        Fp8TensorType.kInputGroup1: ("fwd", [3 * i for i in range(e)]),
        Fp8TensorType.kInputGroup2: ("fwd", [3 * (e + i) for i in range(e)]),
        Fp8TensorType.kWeightGroup1: ("fwd", [3 * i + 1 for i in range(e)]),
        Fp8TensorType.kWeightGroup2: ("fwd", [3 * (e + i) + 1 for i in range(e)]),
        Fp8TensorType.kGradOutputGroup1: ("bwd", [2 * i for i in range(e)]),
        Fp8TensorType.kGradOutputGroup2: ("bwd", [2 * (e + i) for i in range(e)]),
        Fp8TensorType.kForwardInputGroup1: ("clone", [3 * i for i in range(e)]),
        Fp8TensorType.kForwardInputGroup2: ("clone", [3 * (e + i) for i in range(e)]),
        Fp8TensorType.kForwardWeightGroup1: ("clone", [3 * i + 1 for i in range(e)]),
        Fp8TensorType.kForwardWeightGroup2: ("clone", [3 * (e + i) + 1 for i in range(e)]),
    }
    for ttype, (which, slots) in expect.items():
        if which == "clone":
            got = w.get_meta_tensors(ttype, MetaTensorType.kScaleInv)
            assert [t.item() for t in got] == [2000.0 + s for s in slots]
            with pytest.raises(AssertionError):
                w.get_meta_tensors(ttype, MetaTensorType.kScale)
            continue
        meta = fwd if which == "fwd" else bwd
        assert [t.item() for t in w.get_meta_tensors(ttype, MetaTensorType.kScale)] == [1000.0 + s for s in slots]
        assert [t.item() for t in w.get_meta_tensors(ttype, MetaTensorType.kScaleInv)] == [2000.0 + s for s in slots]
        assert [t.item() for t in w.get_meta_tensors(ttype, MetaTensorType.kAmax)] == [3000.0 + s for s in slots]
        # views, not copies: the kernels write amax in place; and the pointer form addresses the same slots
        views = w.get_meta_tensors(ttype, MetaTensorType.kAmax)
        ptrs = w.get_meta_pointers(ttype, MetaTensorType.kAmax)
        assert [v.data_ptr() for v in views] == [int(p) for p in ptrs]
        assert views[0].data_ptr() == meta.amax_history.data_ptr() + 4 * slots[0]


def test_forward_scale_inv_clone_is_a_snapshot():
    fwd, bwd = _Meta(3), _Meta(2)
    w = Fp8MetaWrapper(1, {"scaling_fwd": fwd, "scaling_bwd": bwd})
    w.set_forward_scale_inv_cloned()
    fwd.scale_inv.fill_(-1.0)
    assert w.get_meta_tensors(Fp8TensorType.kForwardWeightGroup1, MetaTensorType.kScaleInv)[0].item() == 2001.0
    assert w.get_meta_tensors(Fp8TensorType.kWeightGroup1, MetaTensorType.kScaleInv)[0].item() == -1.0


def test_delayed_scaling_update_rule():
    """amax = max over history; scale = fp8_max / amax / 2^margin where amax is finite and > 0;
    history rolls by one row and row 0 is cleared."""
    meta = fp8.Fp8MetaTensors(4, 3, torch.device("cpu"))
    meta.amax_history.copy_(torch.tensor([[2.0, 0.0, float("inf"), 7.0], [4.0, 0.0, 1.0, 1.0], [1.0, 0.0, 1.0, 28.0]]))
    meta.scale.copy_(torch.tensor([9.0, 9.0, 9.0, 9.0]))
    fp8.amax_and_scale_update(meta, 448.0, fp8.DelayedScaling(margin=1, amax_history_len=3))
    assert meta.scale.tolist() == [448.0 / 4.0 / 2.0, 9.0, 9.0, 448.0 / 28.0 / 2.0]
    assert torch.equal(meta.scale_inv, 1.0 / meta.scale)
    assert meta.amax_history.tolist() == [[0.0, 0.0, 0.0, 0.0], [1.0, 0.0, 1.0, 28.0], [2.0, 0.0, float("inf"), 7.0]]
    # most_recent uses row 0 only
    meta2 = fp8.Fp8MetaTensors(1, 2, torch.device("cpu"))
    meta2.amax_history.copy_(torch.tensor([[2.0], [100.0]]))
    fp8.amax_and_scale_update(meta2, 448.0, fp8.DelayedScaling(amax_history_len=2, amax_compute_algo="most_recent"))
    assert meta2.scale.item() == 224.0
    # history of length 1: no roll, just cleared
    meta3 = fp8.Fp8MetaTensors(1, 1, torch.device("cpu"))
    meta3.amax_history.fill_(8.0)
    fp8.amax_and_scale_update(meta3, 57344.0, fp8.DelayedScaling(amax_history_len=1))
    assert meta3.scale.item() == 7168.0 and meta3.amax_history.item() == 0.0


def test_update_rule_equals_the_oracle_restatement():
    """The oracle's Meta.update is pinned by hand-worked numbers (tests/test_oracle_pins.py::test_meta_update_*);
    the product's rule is then held against the oracle over several updates, for every option."""
    g = torch.Generator().manual_seed(3)
    hist = torch.rand(5, 12, generator=g) * torch.tensor([0.0, 1.0, 10.0] * 4)
    hist[2, 5] = float("inf")
    hist[1, 7] = float("nan")
    for algo, margin, keep in (("max", 0, None), ("most_recent", 0, None), ("max", 2, None), ("max", 0, (3, 1))):
        want = orc.Meta(12, 5)
        want.amax_history = hist.clone()
        got = fp8.Fp8MetaTensors(12, 5, torch.device("cpu"))
        got.amax_history.copy_(hist)
        recipe = fp8.DelayedScaling(amax_history_len=5, amax_compute_algo=algo, margin=margin)
        kept = [s for s in range(12) if keep and s % keep[0] == keep[1]]
        for _ in range(7):
            want.update(448.0, margin=margin, algo=algo, keep_scale_inv=kept)
            fp8.amax_and_scale_update(got, 448.0, recipe, keep_scale_inv=keep)
            assert torch.equal(got.scale, want.scale) and torch.equal(got.scale_inv, want.scale_inv), (algo, margin)
            assert torch.equal(got.amax_history.nan_to_num(nan=-1.0), want.amax_history.nan_to_num(nan=-1.0))
            want.amax_history[0] += 1.5
            got.amax_history[0] += 1.5


def test_recipe_and_autocast():
    r = fp8.DelayedScaling()
    assert (r.margin, r.interval, r.fp8_format, r.amax_compute_algo) == (0, 1, fp8.Format.HYBRID, "max")
    assert fp8.get_fp8_te_dtype(r, True) == DType.kFloat8E4M3
    assert fp8.get_fp8_te_dtype(r, False) == DType.kFloat8E5M2
    assert fp8.get_fp8_te_dtype(fp8.DelayedScaling(fp8_format=fp8.Format.E4M3), False) == DType.kFloat8E4M3
    assert fp8.current_recipe() is None
    with fp8.fp8_autocast(enabled=True, fp8_recipe=r):
        assert fp8.current_recipe() is r
        with fp8.fp8_autocast(enabled=False):
            assert fp8.current_recipe() is None
        assert fp8.current_recipe() is r
    assert fp8.current_recipe() is None
    with pytest.raises(ValueError):
        fp8.DelayedScaling(amax_compute_algo="median")
    assert fp8.recipe.DelayedScaling is fp8.DelayedScaling and fp8.recipe.Format is fp8.Format


def test_prepare_forward_allocates_three_and_two_slots_per_gemm():
    m = fp8.Fp8GroupedModuleBase()
    x = torch.zeros(4, 8)
    with fp8.fp8_autocast(fp8_recipe=fp8.DelayedScaling(amax_history_len=7)):
        with m.prepare_forward(x, None, num_gemms=6):
            pass
    assert m.fp8_meta["scaling_fwd"].scale.shape == (18,)
    assert m.fp8_meta["scaling_bwd"].scale.shape == (12,)
    assert m.fp8_meta["scaling_fwd"].amax_history.shape == (7, 18)
    assert m.fp8_meta["scaling_fwd"].scale.eq(1).all() and m.fp8_meta["scaling_bwd"].scale_inv.eq(1).all()
    # scaling state round-trips through extra_state
    m.fp8_meta["scaling_fwd"].scale.fill_(3.0)
    state = m.get_extra_state()
    m2 = fp8.Fp8GroupedModuleBase()
    m2.set_extra_state(state)
    with fp8.fp8_autocast(fp8_recipe=fp8.DelayedScaling(amax_history_len=7)):
        with m2.prepare_forward(x, None, num_gemms=6):
            pass
    assert m2.fp8_meta["scaling_fwd"].scale.eq(3).all()


def test_reusing_cached_weights_keeps_their_scale_inv():
    """is_first_microbatch=False: the update still moves every scale, but the weights' scale_inv (slot 1 of
    each GEMM's three forward slots) stays what the cached fp8 weights were cast with; True / None update all."""
    m = fp8.Fp8GroupedModuleBase()
    x = torch.zeros(4, 8)
    rec = fp8.DelayedScaling(amax_history_len=1)
    weight_slots = torch.tensor([1, 4])
    other_slots = torch.tensor([0, 2, 3, 5])

    def step(first, amax):
        with fp8.fp8_autocast(fp8_recipe=rec), m.prepare_forward(x, first, num_gemms=2):
            pass
        m.fp8_meta["scaling_fwd"].amax_history[0] = amax   # what the kernels of the pass would record
        m.fp8_meta["scaling_bwd"].amax_history[0] = 1.0

    step(True, 2.0)                       # first pass: no update yet, scales 1
    step(False, 4.0)                      # update from amax 2: scale 224, weights keep scale_inv 1
    fwd = m.fp8_meta["scaling_fwd"]
    assert fwd.scale.eq(224.0).all()
    assert fwd.scale_inv[weight_slots].eq(1.0).all() and fwd.scale_inv[other_slots].eq(1 / 224.0).all()
    assert m.fp8_meta["scaling_bwd"].scale_inv.eq(1 / 57344.0).all()   # the gradient direction has no weights
    step(True, 8.0)                       # update from amax 4: everything follows
    assert fwd.scale.eq(112.0).all() and fwd.scale_inv.eq(1 / 112.0).all()
    step(None, 8.0)
    assert fwd.scale.eq(56.0).all() and fwd.scale_inv.eq(1 / 56.0).all()


def test_weight_cache_bookkeeping():
    cache = fp8.Fp8WeightCache()
    w = torch.zeros(3, 4, 5, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="is_first_microbatch=False"):
        cache.require(False)
    a, a_t = cache.buffers(w, torch.float8_e4m3fn)
    assert a.shape == (3, 4, 5) and a_t.shape == (3, 5, 4) and a.dtype == a_t.dtype == torch.float8_e4m3fn
    b, b_t = cache.buffers(w, torch.float8_e4m3fn)
    assert b is a and b_t is a_t                        # kept, not reallocated
    cache.valid = True
    cache.require(False)
    with pytest.raises(RuntimeError, match="transposes"):
        cache.require(True)
    c, _ = cache.buffers(torch.zeros(3, 4, 6, dtype=torch.bfloat16), torch.float8_e4m3fn)
    assert c is not a and not cache.valid               # a new shape drops the old contents
    # a module drops its caches when the scaling state is replaced
    m = fp8.Fp8GroupedModuleBase()
    m._weight_caches.append(cache)
    cache.valid = cache.valid_t = True
    with fp8.fp8_autocast(fp8_recipe=fp8.DelayedScaling(amax_history_len=3)), m.prepare_forward(w, None, 2):
        pass
    assert not cache.valid and not cache.valid_t


def test_tensor_batch_describes_the_same_memory_as_views():
    """TensorBatch (array form of "per-expert views") must address exactly what the tensor views address."""
    from fp8_gmm_amd.backend import TensorBatch

    x = torch.zeros(10, 6, dtype=torch.bfloat16)
    bounds = [0, 3, 3, 7, 10]
    b = TensorBatch.rows_of(x, bounds)
    views = [x[bounds[i]: bounds[i + 1]] for i in range(4)]
    assert [int(p) for p in b.ptr] == [x.data_ptr() + bounds[i] * 6 * 2 for i in range(4)]
    assert b.rows.tolist() == [v.shape[0] for v in views] and b.cols.tolist() == [6] * 4 and b.contiguous
    assert [int(p) for p, v in zip(b.ptr, views) if v.numel()] == [v.data_ptr() for v in views if v.numel()]

    w = torch.zeros(3, 4, 5, dtype=torch.float8_e4m3fn)
    s = TensorBatch.stack_of(w)
    assert [int(p) for p in s.ptr] == [v.data_ptr() for v in w.unbind(0)]
    assert (s.rows.tolist(), s.cols.tolist()) == ([4] * 3, [5] * 3)

    flat = torch.zeros(12, 6, dtype=torch.float8_e4m3fn)
    pb = [0, 4, 4, 8, 12]
    t = TensorBatch.transposed_blocks_of(flat, pb)
    for i in range(4):
        rows = pb[i + 1] - pb[i]
        if rows:
            v = flat[pb[i]: pb[i + 1]].view(6, rows)  # the reference's reinterpretation (grouped_linear.py:36-52)
            assert int(t.ptr[i]) == v.data_ptr() and (int(t.rows[i]), int(t.cols[i])) == tuple(v.shape)
    both = b + TensorBatch.rows_of(x, [0, 10])
    assert len(both) == 5 and both.rows.tolist() == [3, 0, 4, 3, 10]
    with pytest.raises(RuntimeError):
        TensorBatch.concat([b, s])  # dtypes differ
    with pytest.raises(RuntimeError):
        TensorBatch.rows_of(x.t(), [0, 1])  # not contiguous


def test_the_rule_for_few_rows_is_the_same_in_both_planners():
    """backend._rows_tiles and the pass planner's rows_pay choose the same launches, on either side of every bound."""
    import numpy as np

    from fp8_gmm_amd import _lib, backend

    lib = _lib.load()
    rng = np.random.default_rng(5)
    taken = 0
    for case in range(300):
        experts = int(rng.choice([1, 8, 32, 64, 128]))
        k, n = 16 * int(rng.integers(16, 400)), 16 * int(rng.integers(16, 400))
        sizes = rng.integers(0, int(rng.choice([2, 17, 34, 66, 130])), size=experts).astype(np.int64)
        sizes[rng.random(experts) < 0.2] = 0
        d = _lib.LinearPass()
        d.experts, d.in_features, d.out_features, d.grid, d.stream_k = experts, k, n, 256, 1
        d.tokens, d.group_sizes = int(sizes.sum()), sizes.ctypes.data
        for f in ("x", "x_fp8", "w_fp8", "y", "fwd_scale", "fwd_scale_inv", "fwd_amax"):
            setattr(d, f, 1 << 20)
        plan = _lib.PassPlan()
        assert lib.fp8gmm_plan_linear_forward(d, None, 0, plan) == -8 or d.tokens == 0
        table = np.zeros(experts, dtype=_lib.GEMM_PROBLEM)
        table["m"], table["n"], table["k"] = sizes, n, k
        want = backend._rows_tiles(table)
        if d.tokens:
            assert (plan.launch[1].plan.tile_m == _lib.GEMM_ROWS_TILE_M) == want, (experts, k, n, sizes)
        taken += want
    assert 20 < taken < 280


def test_the_rules_for_tiles_are_the_same_in_both_planners():
    """backend._small_tiles / _dual_tiles and the pass planner choose the same tile for the three launches of a linear
    layer, on either side of every bound."""
    import numpy as np

    from fp8_gmm_amd import _lib, backend

    lib = _lib.load()
    rng = np.random.default_rng(6)
    taken = {}

    def tile_of(plan):
        return (plan.tile_m or plan.tile or 256, plan.tile or 256)

    def want(m, n, k, a_kmajor, layout):
        table = np.zeros(len(m), dtype=_lib.GEMM_PROBLEM)
        table["m"], table["n"], table["k"] = m, n, k
        if not layout and backend._rows_tiles(table):
            return (_lib.GEMM_ROWS_TILE_M, 128)
        if backend._small_tiles(table, a_kmajor, True):
            return (128, 128)
        return (128, 256) if backend._dual_tiles(table, a_kmajor) else (256, 256)

    for case in range(400):
        experts = int(rng.choice([1, 3, 8, 16, 48, 128]))
        k, n = (16 * int(rng.choice([rng.integers(4, 20), rng.integers(16, 130), rng.integers(100, 300)])) for _ in range(2))
        mean = int(rng.choice([40, 150, 500, 1200, 2500]))
        sizes = rng.multinomial(experts * mean, rng.dirichlet(np.full(experts, float(rng.choice([0.4, 1, 1000])))))
        sizes = np.ascontiguousarray(sizes.astype(np.int64))
        d = _lib.LinearPass()
        d.experts, d.in_features, d.out_features, d.grid, d.stream_k = experts, k, n, 256, 1
        d.tokens, d.group_sizes = int(sizes.sum()), sizes.ctypes.data
        d.dgrad = d.wgrad = 1
        for f in ("x", "x_fp8", "w_fp8", "y", "dy", "dy_fp8", "dx", "dw", "fwd_scale", "fwd_scale_inv", "fwd_amax",
                  "bwd_scale", "bwd_scale_inv", "bwd_amax"):
            setattr(d, f, 1 << 20)
        fwd, bwd = _lib.PassPlan(), _lib.PassPlan()
        assert lib.fp8gmm_plan_linear_forward(d, None, 0, fwd) == -8
        assert lib.fp8gmm_plan_linear_backward(d, None, 0, bwd) == -8
        got = [tile_of(fwd.launch[1].plan), tile_of(bwd.launch[1].plan), tile_of(bwd.launch[2].plan)]
        full = np.full(experts, n), np.full(experts, k)
        assert got == [want(sizes, n, k, False, 0), want(full[0], k, sizes, True, 3), want(sizes, k, n, False, 1)], \
            (experts, k, n, sizes)
        for i, g in enumerate(got):
            taken[i, g] = taken.get((i, g), 0) + 1
    assert all(taken.get((i, g), 0) > 10 for i in (0, 2) for g in ((128, 128), (128, 256), (256, 256))), taken
    assert all(taken.get((1, g), 0) > 10 for g in ((128, 128), (256, 256))), taken


def test_tiles_of_weight_gradients_follow_the_split_not_its_size():
    """A split of one skew keeps its tile as the batch grows: the rule asks for the longest contraction in shares of the
    launch.  Even splits take the small tile up to a number of steps, whatever the number of tiles."""
    import numpy as np

    from fp8_gmm_amd import backend

    def small(experts, m, n, sizes):
        table = np.zeros(experts, dtype=backend._lib.GEMM_PROBLEM)
        table["m"], table["n"], table["k"] = m, n, sizes
        return backend._small_tiles(table, True, True)

    zipf = 1.0 / np.arange(1, 65) ** 1.1
    zipf /= zipf.sum()
    # 64 experts, a quarter of the rows in one: 3 to 40 thousand steps
    for rows in (9000, 18000, 24576, 30000, 32768, 40000, 49152, 98304):
        assert small(64, 1408, 2048, np.round(rows * zipf).astype(np.int64)), rows
    # 8 experts: a contraction of more than two shares, 800 to 6000 steps
    first = zipf[:8] / zipf[:8].sum()
    for rows in (3000, 6000, 9000, 12000, 18000, 23000):
        assert small(8, 2048, 1024, np.round(rows * first).astype(np.int64)), rows
    # tiles of one step, 1024 to 8192 of them; as many rows under a long even contraction
    for experts in (16, 64, 128):
        assert small(experts, 2048, 2048, np.full(experts, 100))
    assert not small(64, 2048, 2048, np.full(64, 600))
    # narrow results in many tiles
    assert small(40, 9600, 144, np.full(40, 100)) and not small(125, 9600, 144, np.full(125, 100))


def test_row_sliced_launches_of_nearly_whole_rounds_keep_two_sets_of_accumulators():
    """More than nine K steps: the small tile where the last round of 128 x 256 tiles is half empty, not where it is nearly
    full."""
    import numpy as np

    from fp8_gmm_amd import backend

    def small(experts, rows, n, k):
        table = np.zeros(experts, dtype=backend._lib.GEMM_PROBLEM)
        table["m"], table["n"], table["k"] = rows, n, k
        return backend._small_tiles(table, False, True)

    for k in (1168, 1600, 2048):
        assert small(11, 120, 6144, k) and small(12, 300, 2560, k)           # 1.03 and 1.41 rounds
        assert not small(13, 300, 2816, k) and not small(12, 500, 2560, k)   # 1.68 and 1.88
    assert small(13, 300, 2816, 1024) and small(12, 500, 2560, 1024)


def test_native_passes_refuse_operands_that_do_not_fit():
    """The kernels follow addresses: widths, group counts and scaling slots that do not fit are refused on the host,
    before anything is launched."""
    from fp8_gmm_amd.native import Due, Setup, linear_step, mlp_step

    def setup(experts, gemms):
        f, b = torch.ones(3 * experts * gemms), torch.ones(2 * experts * gemms)
        return Setup(0, 1, 256, f, f, f.reshape(1, -1), b, b, b.reshape(1, -1))

    def bf16(*shape):
        return torch.zeros(shape, dtype=torch.bfloat16)

    with pytest.raises(RuntimeError, match="columns"):
        linear_step(bf16(3, 16), bf16(2, 16, 32), [1, 2], None, True, setup(2, 1), Due())
    with pytest.raises(RuntimeError, match="entries"):
        linear_step(bf16(3, 16), bf16(2, 16, 16), [1, 1, 1], None, True, setup(3, 1), Due())
    with pytest.raises(RuntimeError, match="slots"):
        linear_step(bf16(3, 16), bf16(2, 16, 16), [1, 2], None, True, setup(1, 1), Due())
    with pytest.raises(RuntimeError, match="columns"):
        mlp_step(bf16(3, 32), bf16(2, 32, 16), bf16(2, 16, 32), [1, 2], None, None, True, setup(2, 2), Due())
    with pytest.raises(RuntimeError, match="fc2"):
        mlp_step(bf16(3, 16), bf16(2, 32, 16), bf16(2, 16, 16), [1, 2], None, None, True, setup(2, 2), Due())


def test_native_passes_take_group_sizes_of_any_iterable():
    """As ``cumsum_group_sizes`` does: every entry through ``int``."""
    from fp8_gmm_amd.native import Due, Setup, linear_step

    z = torch.ones(12).reshape(1, -1)
    x, w = torch.zeros(4, 16, dtype=torch.bfloat16), torch.zeros(2, 16, 16, dtype=torch.bfloat16)
    for sizes in ([1, 2], (1, 2), iter([1, 2]), [1.0, 2.0], torch.tensor([1, 2]).numpy(), [torch.tensor(1), 2],
                  torch.tensor([1, 2], dtype=torch.int32)):
        with pytest.raises(RuntimeError, match="must sum"):   # read, and not the input's four rows
            linear_step(x, w, sizes, None, True, Setup(0, 1, 256, z, z, z, z, z, z), Due())


def test_fp8_autocast_as_a_decorator_keeps_every_call_apart():
    """A decorated function may run in two threads at once: each restores what its own thread had before."""
    import threading

    from fp8_gmm_amd.fp8 import _STATE, DelayedScaling, fp8_autocast

    inside, leave, seen = threading.Barrier(2), [threading.Event(), threading.Event()], [None, None]

    @fp8_autocast(enabled=True)
    def body(i):
        inside.wait(30)
        leave[i].wait(30)

    outer = [DelayedScaling(margin=1), DelayedScaling(margin=2)]

    def thread(i):
        with fp8_autocast(fp8_recipe=outer[i]):
            body(i)
            seen[i] = _STATE.recipe

    threads = [threading.Thread(target=thread, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for i in range(2):
        leave[i].set()
        threads[i].join(30)
    assert seen[0] is outer[0] and seen[1] is outer[1]


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("kind", ["linear", "mlp"])
def test_modules_refuse_to_be_traced(kind, grad):
    """A tracer sees the allocation of a pass's result and none of the launches that write it: the recorded graph would
    return uninitialised memory.  With and without gradients, before anything of the module has changed."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from fp8_gmm_amd import GroupedLinear, GroupedMlp

    module = (GroupedLinear if kind == "linear" else GroupedMlp)(16, 32, 2, torch.bfloat16, device="cpu")
    x = torch.zeros(3, 16, dtype=torch.bfloat16, requires_grad=grad)
    module._ahead = ahead = ()   # what cast_weights_ahead() leaves for the next forward pass
    with torch.set_grad_enabled(grad):
        with pytest.raises(RuntimeError, match="cannot be traced"):
            torch.jit.trace(module, (x, torch.tensor([1, 2])), check_trace=False)
        with pytest.raises(RuntimeError, match="cannot be traced"):
            make_fx(lambda t: module(t, [1, 2]))(x)
    assert module._fp8_steps == 0 and module._ahead is ahead


def _native_module_on_the_cpu(monkeypatch, kind):
    """A module that takes the native path with CPU tensors: good for calls that are refused before any launch."""
    from fp8_gmm_amd import GroupedLinear, GroupedMlp, _lib

    cls = GroupedLinear if kind == "linear" else GroupedMlp
    monkeypatch.setattr(cls, "_native", lambda self, *tensors: True)
    monkeypatch.setattr(_lib, "device_grid", lambda index: 256)
    return cls(16, 32, 2, torch.bfloat16, device="cpu")


@pytest.mark.parametrize("kind", ["linear", "mlp"])
def test_a_refused_first_microbatch_leaves_no_valid_weight_cache(monkeypatch, kind):
    """A first micro-batch that raises has cast nothing: the next one must not compute with what the buffer holds, neither
    uninitialised memory nor the weights of the step before."""
    module = _native_module_on_the_cpu(monkeypatch, kind)
    x = torch.zeros(3, 16, dtype=torch.bfloat16)
    for earlier in (False, True):
        for cache in module._weight_caches:
            cache.valid = earlier
        with pytest.raises(RuntimeError, match="must sum"):
            module(x, [1, 1], is_first_microbatch=True)
        with pytest.raises(RuntimeError, match="no earlier pass"):
            module(x, [1, 2], is_first_microbatch=False)


@pytest.mark.parametrize("reuse", [False, True])
@pytest.mark.parametrize("kind", ["linear", "mlp"])
def test_a_refused_native_pass_keeps_its_scaling_update(monkeypatch, kind, reuse):
    """The update that is due in front of a pass has taken its turn (``interval`` counts passes): where the pass is refused
    it is run all the same, once, as it is in front of the other paths."""
    module = _native_module_on_the_cpu(monkeypatch, kind)
    x = torch.zeros(3, 16, dtype=torch.bfloat16)
    recipe = fp8.DelayedScaling(amax_history_len=3, interval=2)
    passes = [(1.0, 1.0, [0.0, 0.0, 0.0]), (1.0, 1.0, [2.0, 0.0, 0.0]), (224.0, 28672.0, [0.0, 0.0, 2.0]),
              (224.0, 28672.0, [2.0, 0.0, 2.0])]   # due in front of the third pass alone
    for want in passes:
        with fp8.fp8_autocast(fp8_recipe=recipe), pytest.raises(RuntimeError, match="no earlier pass" if reuse else "must sum"):
            module(x, [1, 1], is_first_microbatch=False if reuse else None)
        fwd, bwd = module.fp8_meta["scaling_fwd"], module.fp8_meta["scaling_bwd"]
        assert (fwd.scale[0].item(), bwd.scale[0].item(), fwd.amax_history[:, 0].tolist()) == want
        fwd.amax_history[0] = bwd.amax_history[0] = 2.0


def test_cutlass_products_need_their_factors():
    """``multi_scale_mul`` refuses a missing factor, and the form that scales in the GEMM's epilogue does too."""
    from fp8_gmm_amd import backend

    a = torch.zeros(3, 16, dtype=torch.uint8).view(torch.float8_e4m3fn)
    b = torch.zeros(2, 16, 16, dtype=torch.uint8).view(torch.float8_e4m3fn)
    ones = torch.ones(2)
    for sa, sb in ((None, ones), (ones, None)):
        with pytest.raises(RuntimeError, match="needs a_scale_invs"):
            backend.fp8_gmm(a, b, [1, 2], sa, sb, cutlass=True)
    with pytest.raises(RuntimeError, match="entries"):
        backend.fp8_gmm(a, b, [1, 2], ones, ones.reshape(1, 2), cutlass=True)
