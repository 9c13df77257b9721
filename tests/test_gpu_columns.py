"""Small convolution calls as columns and matrix products (csrc/conv_columns.hip) against the
oracle in float64 accumulation, and the tile kernels at the same sizes.

The tile kernels are reached at small sizes by turning the route off for the thread (the
tile_kernels fixture); the plan tests then run on them.
"""
import numpy as np
import pytest
import torch

import test_gpu_conv_plans as plans
from conftest import runs_by_columns

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    import _spherical_distortion_ext._ops as o
    return o


@pytest.fixture(scope="module")
def oracle():
    from oracle import oracle as o
    return o


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
@pytest.mark.parametrize("tc", plans.CASES, ids=lambda t: "x".join(map(str, t)))
def test_tile_kernels_at_small_sizes(ops, oracle, tile_kernels, tc, mode):
    plans.test_planned_calls_match_plain_calls_and_the_oracle(ops, oracle, tc, mode)


# (batch, Cin, Cout, H, W, OH, OW, K, P, interp): one tile and one over its edges (64 x 64 tiles,
# reduction steps of 32, splits of the pixels), widths that are no multiple of eight, one pixel,
# one sample, the most points a weighted sample may have on the route
SIZES = [
    (1, 5, 1, 1, 1, 1, 1, 1, 0, 0),
    (1, 8, 64, 8, 8, 8, 8, 4, 0, 1),
    (2, 9, 65, 9, 15, 5, 13, 9, 0, 1),
    (1, 64, 7, 16, 20, 8, 8, 1, 0, 2),
    (3, 33, 40, 12, 25, 6, 11, 25, 0, 1),
    (2, 7, 130, 10, 18, 13, 20, 9, 0, 2),
    (1, 12, 17, 10, 14, 10, 14, 3, 8, 1),
    (2, 16, 24, 11, 13, 9, 10, 7, 2, 0),
    (5, 40, 72, 20, 31, 10, 16, 9, 0, 0),
]


def _arrays(tc):
    B, Cin, Cout, H, W, OH, OW, K, P, interp = tc
    rng = np.random.default_rng(sum(tc))
    shape = (OH, OW, K) + ((P,) if P else ())
    ys = rng.uniform(-2, H + 1, shape)      # some samples outside the image
    xs = rng.uniform(-2, W + 1, shape)
    ys[0, 0, 0], xs[0, 0, 0] = -9, -9       # ... one with no tap in it
    m = np.stack([xs, ys], -1).astype(np.float32)
    iw = rng.uniform(0.1, 1, shape).astype(np.float32) if P else None
    f = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    return (m, iw, f(B, Cin, H, W), f(Cout, Cin, K), f(Cout), f(B, Cout, OH, OW), f(Cin))


def _rel(a, b):
    d = np.linalg.norm(np.asarray(a, np.float64) - b)
    return d / max(np.linalg.norm(np.asarray(b, np.float64)), 1e-30)


@pytest.mark.parametrize("mode", ["native", "split", "bf16"])
@pytest.mark.parametrize("tc", SIZES, ids=lambda t: "x".join(map(str, t)))
def test_columns_route_matches_the_oracle(ops, oracle, tc, mode):
    from _spherical_distortion_ext import _capi
    B, Cin, Cout, H, W, OH, OW, K, P, interp = tc
    for transposed in (0, 1) if Cout >= 5 else (0,):
        taken = _capi.load().sdk_mapped_conv_by_columns(
            B, Cout if transposed else Cin, Cin if transposed else Cout, H, W, OH, OW, K, P,
            interp, _capi.SDK_F32, 0, transposed)
        assert taken == 1
    m, iw, x, w, b, g, bt = _arrays(tc)
    t = lambda a: None if a is None else torch.from_numpy(a).to(DEV)  # noqa: E731
    with ops.conv_compute(mode):
        y = ops.ops.mapped_conv_forward(t(x), t(m), t(iw), t(w), t(b), K, interp)
        gi, gw, gb = ops.ops.mapped_conv_backward(t(g), t(m), t(iw), t(x), t(w), t(b), K, interp)
        yt = ops.ops.mapped_transposed_conv_forward(t(g), t(m), t(iw), t(w), t(bt), H, W, K, interp)
    # float32: sums of at most Cin * K (or pixels) terms, random signs: eps * sqrt(n) < 5e-6;
    # bf16 operands: 2^-9 each, so 2^-8 of the norm at most
    tol = 4e-3 if mode == "bf16" else 5e-6
    assert _rel(y.cpu().numpy(), oracle.mapped_conv_forward(x, m, w, b, K, interp, iw)) <= tol
    wi, ww, wb = oracle.mapped_conv_backward(g, m, x, w, b, K, interp, iw)
    for have, want in ((gi, wi), (gw, ww), (gb, wb)):
        assert _rel(have.cpu().numpy(), want) <= tol
    want = oracle.mapped_transposed_conv_forward(g, m, w, bt, H, W, K, interp, iw)
    assert _rel(yt.cpu().numpy(), want) <= tol


def test_the_inverted_map_is_built_by_the_first_backward(ops):
    """A forward builds nothing; results do not depend on which call comes first, and a replayed
    capture whose entry is not built gives the eager result."""
    m, iw, x, w, b, g, _ = _arrays((2, 16, 24, 11, 13, 9, 10, 9, 0, 1))
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    tx, tw, tb, tg, K = t(x), t(w), t(b), t(g), 9
    args = lambda tm: (tg, tm, None, tx, tw, tb, K, 1)  # noqa: E731
    want = [o.cpu() for o in ops.ops.mapped_conv_backward(*args(t(m)))]
    tm = t(m)
    before = ops.plan_cache_size()
    ops.ops.mapped_conv_forward(tx, tm, None, tw, tb, K, 1)
    assert ops.plan_cache_size() == before
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        outs = [torch.empty_like(o, device=DEV) for o in want]
        with torch.cuda.graph(graph, stream=side):
            for o, r in zip(outs, ops.ops.mapped_conv_backward(*args(tm))):
                o.copy_(r)
    for _ in range(3):
        for o in outs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        eager = ops.ops.mapped_conv_backward(*args(tm))
        for o, e, r in zip(outs, eager, want):
            assert torch.equal(o.cpu(), r) and torch.equal(e.cpu(), r)


def test_calls_that_read_no_plan_leave_the_cache_alone(ops):
    """Forwards on pictures of new sizes (columns, first layers) neither push out a plan nor keep
    a map."""
    t = lambda a: None if a is None else torch.from_numpy(a).to(DEV)  # noqa: E731
    shapes = [(2, 16, 24, 11, 13, 9, 10, 9, 0, 1), (2, 3, 24, 20, 36, 16, 24, 9, 0, 1)]

    def forward(tc):
        m, _, x, w, b, _, _ = _arrays(tc)
        ops.ops.mapped_conv_forward(t(x), t(m), None, t(w), t(b), tc[7], tc[9])

    ops.set_conv_plan_cache(False)
    ops.set_conv_plan_cache(True, max_entries=2)
    try:
        for h in (12, 13):      # two training maps with their inverted maps
            m, _, x, w, b, g, _ = _arrays((2, 16, 24, 11, 13, h, 10, 9, 0, 1))
            ops.ops.mapped_conv_backward(t(g), t(m), None, t(x), t(w), t(b), 9, 1)
        assert ops.plan_cache_size() == 2
        held = torch.cuda.memory_allocated()
        for tc in shapes * 2:
            forward(tc)
        assert ops.plan_cache_size() == 2
        assert torch.cuda.memory_allocated() == held     # (a plan let go, a map kept would show)
    finally:
        ops.set_conv_plan_cache(True, max_entries=16)


def test_columns_layers_keep_their_lists_alone(ops):
    """64 -> 64 channels at 1 x 128 x 256 keep 10 MB of lists, not room for a plan of 100; a layer on
    the same map that runs on a plan shares the map's entry."""
    from _spherical_distortion_ext import _capi
    lib = _capi.load()
    size = (128, 256, 128, 256, 9, 0, 1, _capi.SDK_F32)
    m, _, x, w, b, g, _ = _arrays((1, 64, 64, 128, 256, 128, 256, 9, 0, 1))
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    args = (t(g), t(m), None, t(x), t(w), t(b), 9, 1)
    ops.ops.mapped_conv_backward(t(g), t(m), None, t(x), t(w), t(b), 9, 1)     # (side streams' memory)
    ops.set_conv_plan_cache(False)
    ops.set_conv_plan_cache(True)
    try:
        before = torch.cuda.memory_allocated()
        ops.ops.mapped_conv_backward(*args)
        held = torch.cuda.memory_allocated() - before
        assert 0 < held <= lib.sdk_mapped_conv_columns_bytes(*size) + 1024 < 11e6
        assert ops.plan_cache_size() == 1
        lib.sdk_mapped_conv_columns_enable(0)
        ops.ops.mapped_conv_backward(*args)
        lib.sdk_mapped_conv_columns_enable(1)
        assert ops.plan_cache_size() == 1
        assert torch.cuda.memory_allocated() - before >= lib.sdk_mapped_conv_plan_bytes(*size)
        ops.ops.mapped_conv_backward(*args)
    finally:
        lib.sdk_mapped_conv_columns_enable(1)


def test_every_buffer_a_columns_call_may_be_given(ops):
    """No plan, the inverted map alone, a plan with it (built whole, or that part of it) and one
    without: the same gradient; the inverted map alone is refused by calls of the tile kernels."""
    from _spherical_distortion_ext import _capi
    lib = _capi.load()
    B, Cin, Cout, H, W, K = 1, 40, 48, 40, 64, 9
    m, _, x, w, _, g, _ = _arrays((B, Cin, Cout, H, W, H, W, K, 0, 1))
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    tm, tg, tw = t(m), t(g), t(w)
    size = (H, W, H, W, K, 0, 1, _capi.SDK_F32)
    plain, both, alone = (int(f(*size)) for f in (
        lib.sdk_mapped_conv_plan_bytes, lib.sdk_mapped_conv_plan_bytes_columns,
        lib.sdk_mapped_conv_columns_bytes))
    assert plain % 256 == both % 256 == 0 and alone % 256 == 128 and alone < both - plain + 256
    nws = lib.sdk_mapped_conv_workspace_bytes(B, Cin, Cout, H, W, H, W, K, 0, 1, _capi.SDK_F32, 0)
    ws = torch.empty(nws, dtype=torch.uint8, device=DEV)
    p, stream = (lambda a: a.data_ptr()), torch.cuda.current_stream().cuda_stream  # noqa: E731

    def call(plan):
        out = torch.empty(B, Cin, H, W, device=DEV)
        rc = lib.sdk_mapped_conv_backward_input_planned(
            p(tg), p(tm), None, p(tw), p(out), p(ws), nws, None if plan is None else p(plan),
            0 if plan is None else plan.numel(), B, Cin, H, W, Cout, H, W, K, 0, 1, _capi.SDK_F32, 0,
            stream)
        return rc, out

    want = call(None)[1]
    for build, n in (("sdk_mapped_conv_plan_build_columns", alone), ("sdk_mapped_conv_plan_build", plain),
                     ("sdk_mapped_conv_plan_build_columns", both), ("sdk_mapped_conv_plan_build", both)):
        plan = torch.empty(n, dtype=torch.uint8, device=DEV)
        assert getattr(lib, build)(p(tm), None, p(plan), n, *size, stream) == 0
        rc, out = call(plan)
        assert rc == 0 and torch.equal(out, want), (build, n)
    plan = torch.empty(alone, dtype=torch.uint8, device=DEV)
    assert lib.sdk_mapped_conv_plan_build_columns(p(tm), None, p(plan), alone - 128, *size, stream) == -3
    assert lib.sdk_mapped_conv_plan_build(p(tm), None, p(plan), alone, *size, stream) == -3
    lib.sdk_mapped_conv_columns_enable(0)
    try:
        nws = lib.sdk_mapped_conv_workspace_bytes(B, Cin, Cout, H, W, H, W, K, 0, 1, _capi.SDK_F32, 0)
        ws = torch.empty(nws, dtype=torch.uint8, device=DEV)
        assert call(plan)[0] == -3 and b"inverted map alone" in lib.sdk_last_error()
    finally:
        lib.sdk_mapped_conv_columns_enable(1)


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("columns", [0, 1])
def test_a_backward_captured_after_a_forward_finds_its_plan(ops, columns, transposed):
    """Nothing is built under capture: a forward whose input requires a gradient builds what the
    input's gradient reads, and the replays rebuild nothing."""
    from _spherical_distortion_ext import _capi
    import spherical_distortion.nn as snn
    H, W, C = (40, 64, 40) if columns else (256, 256, 16)
    m, _, x, _, _, _, _ = _arrays((1, C, C, H, W, H, W, 9, 0, 1))
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    cls = snn.MappedTransposedConvolution if transposed else snn.MappedConvolution
    layer, tx = cls(C, C, 9).to(DEV), t(x).requires_grad_()
    args = lambda tm: (H, W, tm) if transposed else (tm,)  # noqa: E731
    name = "mapped_transposed_conv_backward" if transposed else "mapped_conv_backward"
    w, b, g = layer.weight.detach(), layer.bias.detach(), t(x)
    lib = _capi.load()
    lib.sdk_mapped_conv_columns_enable(columns)
    times = {}
    try:
        want = getattr(ops.ops, name)(g, t(m), None, tx.detach(), w, b, 9, 1)
        for warm in ("nothing", "forward", "step"):
            tm = t(m)
            if warm != "nothing":
                y = layer(tx, *args(tm))
                if warm == "step":
                    torch.autograd.grad(y, [tx], g)
            outs = [torch.empty_like(o) for o in want]
            graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                with torch.cuda.graph(graph, stream=side):
                    for o, r in zip(outs, getattr(ops.ops, name)(g, tm, None, tx.detach(), w, b, 9, 1)):
                        o.copy_(r)
            times[warm] = 1e9
            for _ in range(8):
                for o in outs:
                    o.zero_()
                start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                start.record()
                graph.replay()
                end.record()
                torch.cuda.synchronize()
                times[warm] = min(times[warm], start.elapsed_time(end))
                for o, r in zip(outs, want):
                    assert _rel(o.cpu().numpy(), r.cpu().numpy()) <= 2e-6
    finally:
        lib.sdk_mapped_conv_columns_enable(1)
    print(times)
    # (the columns' gathers read no plan: nothing to rebuild in the backward of a transposed layer)
    assert times["forward"] <= 1.15 * times["step"]
    assert (columns and transposed) or times["forward"] <= 0.97 * times["nothing"]


def test_plan_parts_are_built_by_the_calls_that_read_them(ops, tile_kernels):
    """A convolution's forward builds what it gathers by, its backward the inverse; results are those
    of a plan built at once, whichever call comes first, and of no plan."""
    m, iw, x, w, b, g, bt = _arrays((2, 40, 72, 16, 24, 16, 24, 9, 0, 1))
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    tx, tw, tb, tg, tbt, K = t(x), t(w), t(b), t(g), t(bt), 9
    calls = {
        "forward": lambda tm: [ops.ops.mapped_conv_forward(tx, tm, None, tw, tb, K, 1)],
        "weights": lambda tm: list(ops.ops.mapped_conv_backward_select(
            tg, tm, None, tx, tw, K, 1, False, False, True))[1:],
        "transposed": lambda tm: [ops.ops.mapped_transposed_conv_forward(tg, tm, None, tw, tbt, 16, 24, K, 1)],
        "backward": lambda tm: list(ops.ops.mapped_conv_backward(tg, tm, None, tx, tw, tb, K, 1)),
    }
    ops.set_conv_plan_cache(False)
    want = {n: f(t(m)) for n, f in calls.items()}
    ops.set_conv_plan_cache(True)
    for order in (list(calls), list(calls)[::-1], ["transposed", "forward", "backward", "weights"]):
        tm = t(m)
        for n in order:
            for have, ref in zip(calls[n](tm), want[n]):
                assert _rel(have.cpu().numpy(), ref.cpu().numpy()) <= 1e-6, (order, n)


@pytest.mark.parametrize("shape", [
    (2, 3, 24, 20, 36, 16, 24, 9, 0, 1),    # a first layer reads no plan
    (1, 4, 128, 20, 36, 16, 24, 9, 0, 1),   # ... nor with two blocks of columns
    (1, 4, 100, 13, 17, 24, 30, 25, 0, 1),  # its weight gradient does: too many accumulators
    (2, 16, 24, 40, 72, 16, 24, 9, 0, 0),   # the scatter by the product route
])
def test_layers_on_a_shared_map_build_what_each_reads(ops, tile_kernels, shape):
    """Layers of different widths on one map, in both orders: the parts one of them left out are
    there for the next; results are those without plans."""
    m, iw, x, w, b, g, bt = _arrays(shape)
    K, interp = shape[7], shape[9]
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    wide = _arrays(shape[:1] + (40, 72) + shape[3:])

    def step(tm, arrays):
        _, _, x, w, b, g, bt = (None if a is None else t(a) for a in arrays)
        return [ops.ops.mapped_conv_forward(x, tm, None, w, b, K, interp),
                *ops.ops.mapped_conv_backward(g, tm, None, x, w, b, K, interp)]

    layers = [(m, iw, x, w, b, g, bt), wide]
    ops.set_conv_plan_cache(False)
    want = [step(t(m), a) for a in layers]
    ops.set_conv_plan_cache(True)
    for order in ((0, 1, 0), (1, 0, 1)):
        tm = t(m)
        for i in order:
            for have, ref in zip(step(tm, layers[i]), want[i]):
                assert _rel(have.cpu().numpy(), ref.cpu().numpy()) <= 2e-6, (order, i)


@pytest.mark.parametrize("mode", ["native", "split"])
def test_weight_gradient_keeps_the_bits_of_its_sums(ops, mode):
    """7500 pixels: added one after the other within a split, the float32 sums were 4.5e-7 from
    float64 in the norm, the tile kernels' 2.1e-7."""
    tc = (6, 96, 160, 50, 100, 25, 50, 9, 0, 1)
    assert runs_by_columns(*tc)
    m, _, x, w, b, g, _ = _arrays(tc)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    with ops.conv_compute(mode):
        gw = ops.ops.mapped_conv_backward(t(g), t(m), None, t(x), t(w), t(b), 9, 1)[1]
    d = lambda a: t(a).double()  # noqa: E731
    want = ops.ops.mapped_conv_backward(d(g), d(m), None, d(x), d(w), d(b), 9, 1)[1]
    assert _rel(gw.cpu().numpy(), want.cpu().numpy()) <= 2.6e-7


@pytest.mark.parametrize("tc", [
    # reductions of two steps and fewer (operands split late, or by a small forward early), in few tiles and
    # in more than are at work at once, and of more steps; weight gradients in runs of 64 pixels and of 128
    (1, 8, 8, 16, 31, 1), (1, 64, 8, 20, 40, 1), (1, 8, 70, 24, 40, 9), (4, 8, 9, 112, 113, 1),
    (2, 7, 65, 50, 100, 3), (1, 65, 72, 30, 61, 1),
], ids=lambda t: "x".join(map(str, t)))
def test_split_products_early_and_late_are_exact(ops, oracle, tc):
    """Integers of four bits and samples at halves: every product and sum is a float32 number."""
    B, Cin, Cout, H, W, K = tc
    assert runs_by_columns(B, Cin, Cout, H, W, H, W, K, 0, 1)
    rng = np.random.default_rng(sum(tc))
    y, x, k = np.meshgrid(np.arange(H), np.arange(W), np.arange(K), indexing="ij")
    m = np.stack([x + k % 3 * 0.5 - 0.5, y + k // 3 * 0.5 - 0.5], -1).astype(np.float32)
    f = lambda *s: rng.integers(-4, 5, s).astype(np.float32)  # noqa: E731
    img, w, b, g = f(B, Cin, H, W), f(Cout, Cin, K), f(Cout), f(B, Cout, H, W)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    with ops.conv_compute("split"):
        out = ops.ops.mapped_conv_forward(t(img), t(m), None, t(w), t(b), K, 1)
        grads = ops.ops.mapped_conv_backward(t(g), t(m), None, t(img), t(w), t(b), K, 1)
    assert np.array_equal(out.cpu().numpy(), oracle.mapped_conv_forward(img, m, w, b, K, 1))
    for have, want in zip(grads, oracle.mapped_conv_backward(g, m, img, w, b, K, 1)):
        assert np.array_equal(have.cpu().numpy(), want)
