"""The split fp32 product (kla_linear_f32_fwd) against float64 torch: every tile's
edges, strided and unaligned operands, rows fp16 could not hold, rows with an
infinity or a NaN, and which calls of a module take it."""

import ctypes

import pytest
import torch
import torch.nn.functional as F

from kla.ops.hip import _lib
from kla.ops.hip import linear as lin

pytestmark = pytest.mark.gpu


def _bound(x, w):
    """|error| of one output: with sum |x w| = s, each operand is off by 2^-23 of itself
    and lo lo is left out (2^-22 s together), and an fp32 sum takes three MFMA
    products a 16-wide step of k, each at most 17 roundings of 2^-24 s."""
    k = x.shape[-1]
    s = x.double().abs() @ w.double().abs().t()
    return s * (2.0 ** -21 + 51 * -(-k // 16) * 2.0 ** -24) + 1e-44


def _check(got, x, w, bias=None):
    want = x.double() @ w.double().t() + (0 if bias is None else bias.double())
    assert got.dtype == torch.float32 and got.shape == want.shape
    err = (got.double() - want).abs() / (_bound(x, w) + 2.0 ** -23 * want.abs())
    assert err.max().item() <= 1.0, err.max().item()


# (rows, n, k): single rows and columns, one off each tile (64, 128), the chunk's 32
# and the register-held widths of the split (512, 1024, 2048), and each tile choice.
SIZES = [(1, 1, 1), (1, 300, 31), (63, 65, 32), (64, 64, 33), (65, 129, 511), (255, 1365, 512), (257, 40, 513),
         (300, 2080, 1025), (130, 70, 2049), (1025, 1030, 96), (2049, 2049, 40), (4100, 2100, 64),
         (8100, 4200, 1024)]


@pytest.mark.parametrize("rows,n,k", SIZES)
def test_matches_float64(cuda, rows, n, k):
    print(f"[linear_f32] {rows} x {k} -> {n}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(rows + n + k)
    x = torch.randn(rows, k + 3, device=cuda, generator=g)[:, 1:k + 1]     # unaligned rows
    w = torch.randn(n, k, device=cuda, generator=g) * 0.05
    bias = torch.randn(n, device=cuda, generator=g)
    _check(lin.linear_f32(x, w, bias), x, w, bias)
    _check(lin.linear_f32(x, w), x, w)


def test_scales_of_rows(cuda):
    """Rows from fp32's smallest to its largest magnitudes, rows of zeros, and entries far
    below their row's largest: the error stays relative to each output's own terms,
    plus its own last place (what rows may lose in the planes is held to that)."""
    g = torch.Generator(device=cuda).manual_seed(3)
    x = torch.randn(160, 200, device=cuda, generator=g)
    scale = torch.tensor([1e-42, 1e-38, 1e-20, 1.0, 1e20, 1e37, 0.0, -1.0], device=cuda)
    x = x * scale.repeat(20)[:, None]
    x[3, :100] *= 1e-9
    w = torch.randn(96, 200, device=cuda, generator=g)
    w[5] *= 1e-30
    w[6] = 0
    got = lin.linear_f32(x, w)
    want = x.double() @ w.double().t()
    top = torch.finfo(torch.float32).max
    fits, over = want.abs() < top * (1 - 1e-5), want.abs() > top * (1 + 1e-5)
    err = (got.double() - want).abs() / (_bound(x, w) + 2.0 ** -22 * want.abs() + 2.0 ** -149)
    assert err[fits].max().item() <= 1.0
    assert torch.isinf(got[over]).all() and torch.equal(got[over] > 0, want[over] > 0)


# A size for each tile of split_gemm_launch (W rows x tokens), ragged at both ends, and the
# lengths of its three- or four-deep pipeline: steps of 16 (32 for 64 x 64) with every
# remainder, and the split's widths (held in registers up to 2048, read twice beyond).
TILES = {"64x64": (2040, 510), "128x64": (4090, 1020), "128x128": (4090, 2040), "256x128": (8190, 4090)}


@pytest.mark.parametrize("k", [512, 1024, 1056, 1088, 1365, 2049])
@pytest.mark.parametrize("tile", TILES)
def test_no_tile_is_less_exact_than_the_library(cuda, tile, k):
    """2-norm error against float64 at most the library's fp32 product's on the same
    operands (0.62 to 0.64 of it measured; a product that left out either low half would
    have 500 times it), and each output within _bound."""
    rows, n = TILES[tile]
    print(f"[linear_f32] {tile} {rows} x {k} -> {n}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(n + k)
    x, w = torch.randn(rows, k, device=cuda, generator=g), torch.randn(n, k, device=cuda, generator=g)
    got, want = lin.linear_f32(x, w), x.double() @ w.double().t()
    err, library = ((y.double() - want).norm() / want.norm() for y in (got, F.linear(x, w)))
    assert err <= library and err <= 8e-7, (err.item(), library.item())
    _check(got, x, w)


@pytest.mark.parametrize("what", ["residual", "norm+swiglu", "norm+residual"])
@pytest.mark.parametrize("k", [1024, 1056, 1088])
@pytest.mark.parametrize("tile", ["128x64", "128x128", "256x128"])
def test_folded_options_on_large_tiles(cuda, tile, k, what):
    """The same options against the product and torch's operations apart, with a row and a
    column of non-finite values and rows of wide range inside the tiles."""
    rows, n = TILES[tile]
    if "swiglu" in what:
        n //= 2                     # two rows of W a column
    print(f"[linear_f32] {tile} {what} {rows} x {k} -> {n}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(n + k)

    def rn(*s):
        return torch.randn(*s, device=cuda, generator=g)

    x, w, bias, opts = rn(rows, k), rn(n * (2 if "swiglu" in what else 1), k) * k ** -0.5, rn(n * (2 if "swiglu" in what else 1)), {}
    x[777, 5], w[n - 3, 11] = float("nan"), float("inf")
    x[1500:1504, 3], w[:, 3] = 1e12, 0
    if "norm" in what:
        opts["norm"] = (1 + 0.1 * rn(k), 1e-5)
    if "residual" in what:
        opts["residual"] = rn(rows, n)
    opts["swiglu"] = "swiglu" in what
    got = lin.linear_f32(x, w, bias, **opts)
    want, xd, a = _folded(x, w, bias, opts)
    fin = torch.isfinite(want)
    assert fin.sum() == (rows - 1) * (n - 1) and torch.equal(torch.isfinite(got), fin)
    # Plain: fp32's accuracy (2-norm 3.6e-7 at k = 1024, measured); the norm, silu and the
    # adds round a few times more.
    err = ((got.double() - want)[fin].norm() / want[fin].norm()).item()
    assert err <= 1e-6, err
    part = 1500 if "norm" not in what else 1600     # the wide rows by themselves
    err = ((got.double() - want)[part][fin[part]].norm() / want[part][fin[part]].norm()).item()
    assert err <= 2e-6, err


def _wide(kind, x, w):
    """Operands whose rows span more than two fp16 planes hold, made from x [rows, k], w [n, k]."""
    k = x.shape[1]
    j = k // 3
    if kind.startswith("column"):               # a large feature that the weights ignore
        x[:, j] = float(kind.split()[1])
        w[:, j] = 0
    elif kind == "weights":                     # and the other way round
        w[:, j] = 3e10
        x[:, j] = 0
    elif kind == "halves":                      # half the features large, half the outputs blind to them
        x[:, : k // 2] *= 1e8
        w[: w.shape[0] // 2, : k // 2] = 0
    elif kind == "picked":                      # few small entries, and weights that pick one each
        i = torch.arange(w.shape[0], device=w.device) % k
        w.zero_()[torch.arange(w.shape[0], device=w.device), i] = 1.0
        x[:, ::7] *= 1e-11
    elif kind == "scaled down":                 # small terms that vanish at the large one's scale
        x[:, j] = 1e38
        x[:, j + 1:] *= 1e-12
        w[:, : j + 1] = 0
    elif kind == "magnitudes":                  # log-uniform over 24 decades
        x *= 10.0 ** (24 * torch.rand(x.shape, device=x.device, generator=torch.Generator(device=x.device).manual_seed(1)) - 12)
    return x, w


@pytest.mark.parametrize("kind", ["column 1e7", "column 1.7e9", "column 1e12", "weights", "halves", "picked",
                                  "scaled down", "magnitudes"])
@pytest.mark.parametrize("rows,n,k", [(300, 200, 512), (70, 130, 1030), (2050, 1030, 257)])
def test_rows_of_wide_range_keep_fp32_accuracy(cuda, kind, rows, n, k):
    """Each output as good as fp32's terms allow (_bound, and its own last place), and as
    close to float64 as the library's fp32 product."""
    g = torch.Generator(device=cuda).manual_seed(rows + k)
    x, w = _wide(kind, torch.randn(rows, k, device=cuda, generator=g), torch.randn(n, k, device=cuda, generator=g))
    got, want = lin.linear_f32(x, w), x.double() @ w.double().t()
    err = (got.double() - want).abs()
    assert (err / (_bound(x, w) + 2.0 ** -22 * want.abs())).max().item() <= 1.0
    # By output column, so that columns of large values hide none of small ones: within
    # twice the library's own error (its kernels differ by as much among themselves) and
    # two units of the operands' 2^-23 (where few terms make an output, or few rows are
    # in flight, the library has less to round).
    mine, library = err.norm(dim=0), (F.linear(x, w).double() - want).norm(dim=0)
    worst = (mine / (2 * library + 2.0 ** -22 * want.norm(dim=0))).max().item()
    assert worst <= 1.0


@pytest.mark.parametrize("k", [1, 2, 3, 5, 8, 15, 16, 17, 31, 33, 255, 256, 259, 1025])
@pytest.mark.parametrize("what", ["plain", "norm", "norm+swiglu", "residual"])
def test_outputs_formed_again_match_float64(cuda, what, k):
    """Every output through the plain fp32 path (its rows hold a feature that the weights
    ignore, or for k = 1 and 2 an infinity elsewhere in the tile): lengths at the edges
    of a lane's loads and of its steps of 16, ragged tiles, each epilogue."""
    g = torch.Generator(device=cuda).manual_seed(k)
    rows, n = 71, 70
    x, w, bias = (torch.randn(*s, device=cuda, generator=g) for s in ((rows, k), (n, k), (n,)))
    if k > 2:
        x[:, 1], w[:, 1] = 1e12, 0
    else:
        x[5, 0] = float("inf")
    opts = {"bias": bias}
    if "norm" in what:
        opts["norm"] = (1 + 0.1 * torch.randn(k, device=cuda, generator=g), 1e-5)
        if k > 2:
            opts["norm"][0][1] = 1e14           # (the norm has brought the feature to about 1)
            x[:, 1] = 1.0
    if what == "residual":
        opts["residual"] = torch.randn(rows, n, device=cuda, generator=g)
    opts["swiglu"] = "swiglu" in what
    got = lin.linear_f32(x, w, **opts)
    want, xd, a = _folded(x, w, bias, {key: v for key, v in opts.items() if key != "bias"})
    prod = _bound(xd, w) + (2.0 ** -21 + k * 2.0 ** -25) * (xd.abs() @ w.double().abs().t()) + 2.0 ** -22 * a.abs()
    if opts["swiglu"]:
        h = n // 2
        bound = (1.1 * prod[:, :h] * (a[:, h:].abs() + prod[:, h:]) + F.silu(a[:, :h]).abs() * prod[:, h:]
                 + 2.0 ** -20 * want.abs())
    else:
        bound = prod + 2.0 ** -22 * want.abs()
    ok = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and ok[6:].all()
    assert ((got.double() - want).abs() / (bound + 1e-30))[ok].max().item() <= 1.0


def test_layer_ignores_a_large_feature_its_weights_ignore(cuda):
    """KLALayer on raw inputs: a timestamp column with zero weights changes nothing (fp32
    products keep every entry's own exponent)."""
    from kla import KLAConfig, KLALayer

    torch.manual_seed(0)
    layer = KLALayer(512, KLAConfig(backend="hip")).to(cuda).eval()
    x = torch.randn(2, 300, 512, device=cuda)
    with torch.no_grad():
        layer.in_proj.weight[:, 3] = 0
        x[..., 3] = 0
        want = layer(x)
        x[..., 3] = 1.7e9
        got = layer(x)
    assert (got - want).norm() <= 3e-6 * want.norm()


def test_infinities_and_nans_give_fp32_results(cuda):
    g = torch.Generator(device=cuda).manual_seed(4)
    x = torch.randn(300, 100, device=cuda, generator=g)
    w = torch.randn(200, 100, device=cuda, generator=g)
    x[2, 7], x[150, 0], x[299, 99], w[199, 3], w[64, 7] = float("inf"), float("nan"), -float("inf"), float("inf"), 0.0
    bias = torch.randn(200, device=cuda, generator=g)
    got, want = lin.linear_f32(x, w, bias), x.double() @ w.double().t() + bias.double()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(got)], want[torch.isinf(want)].float())
    ok = torch.isfinite(want)
    err = (got.double() - want).abs() / (_bound(x.nan_to_num(0, 0, 0), w.nan_to_num(0, 0, 0)) + 2.0 ** -23 * want.abs())
    assert err[ok].max().item() <= 1.0


def test_which_calls_take_it(cuda, monkeypatch):
    """plain_linear takes linear_f32 for a bare fp32 nn.Linear without a gradient from
    F32_MIN_ROWS rows on; hooks, subclasses, autocast, a gradient, few rows and other
    dtypes keep the module's own call."""
    calls = []
    orig = lin.linear_f32
    monkeypatch.setattr(lin, "linear_f32", lambda *a, **kw: calls.append(1) or orig(*a, **kw))
    mod = torch.nn.Linear(64, 80).to(cuda)
    x = torch.randn(2, 200, 64, device=cuda)

    def taken(m, t):
        calls.clear()
        out = lin.plain_linear(m, t)
        with torch.autocast("cuda", enabled=False):
            want = F.linear(t.float(), m.weight.float(), m.bias.float())
        assert torch.allclose(out.float(), want, rtol=2e-2, atol=2e-2)
        return bool(calls)

    with torch.no_grad():
        assert taken(mod, x)
        assert taken(mod, x.transpose(0, 1)) and taken(mod, x.expand(3, 2, 200, 64)[1])
        assert not taken(mod, x[:1])
        assert not taken(torch.nn.Linear(64, 80).to(cuda).bfloat16(), x.bfloat16())
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not taken(mod, x)
        handle = mod.register_forward_hook(lambda m, a, out: out)
        assert not taken(mod, x)
        handle.remove()

        class Sub(torch.nn.Linear):
            pass

        assert not taken(Sub(64, 80).to(cuda), x)
    assert not taken(mod, x)
    with pytest.raises(ValueError):
        orig(x, torch.randn(80, 63, device=cuda))
    with pytest.raises(TypeError):
        orig(x.double(), mod.weight)


def test_an_mlp_whose_second_weight_is_no_plain_tensor(cuda):
    """A block's MLP whose w3 the product cannot take (a tensor subclass, another dtype's
    module) runs w3's own call on the folded first product."""
    from kla.layers.common import MLP, RMSNorm

    class Doubling(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            if func is F.linear:
                return 2 * F.linear(args[0], args[1].as_subclass(torch.Tensor), *args[2:])
            return super().__torch_function__(func, types, args, kwargs or {})

    torch.manual_seed(0)
    mlp, norm = MLP(64, 4.0).to(cuda).requires_grad_(False), RMSNorm(64).to(cuda).requires_grad_(False)
    mlp.backend = norm.backend = "hip"
    x = torch.randn(300, 64, device=cuda)
    want = mlp.block_forward_hip(x, norm)
    w = mlp.w3.weight
    del mlp.w3.weight
    mlp.w3.weight = w.detach().as_subclass(Doubling)
    got = mlp.block_forward_hip(x, norm)
    assert torch.allclose((got - x).as_subclass(torch.Tensor), 2 * (want - x), rtol=1e-4, atol=1e-5)

    class Half(torch.nn.Module):
        def __init__(self, weight):
            super().__init__()
            self.weight = torch.nn.Parameter(weight.bfloat16(), requires_grad=False)

        def forward(self, h):
            return F.linear(h, self.weight.float())

    mlp.w3 = Half(w)
    assert torch.allclose(mlp.block_forward_hip(x, norm), want, rtol=2e-2, atol=2e-2)


def test_a_forward_set_on_an_instance_is_called(cuda):
    """A module whose instance carries its own forward keeps that call, wherever the split
    product or a block's folded norms would step past it."""
    from kla import KLAConfig
    from kla.configs import ModelConfig
    from kla.models import Block

    torch.manual_seed(0)
    block = Block(64, KLAConfig(backend="hip"), ModelConfig(d_model=64)).to(cuda)
    x = torch.randn(2, 200, 64, device=cuda)
    with torch.no_grad():
        want = block(x)
        mods = (block.mixer.in_proj, block.mixer.out_proj, block.mlp.w12, block.mlp.w3, block.mixer_norm,
                block.mlp_norm, block.mlp, block.mixer)
        for mod in mods:
            seen, plain = [], mod.forward
            mod.forward = lambda *a, **kw: seen.append(1) or plain(*a, **kw)
            got = block(x)
            del mod.forward
            assert len(seen) == 1, type(mod).__name__
            assert torch.allclose(got, want, rtol=1e-4, atol=1e-5 * want.abs().max().item())


def test_what_watches_a_product_sees_the_module(cuda):
    """Tangents, vmap, dispatch and function modes and tensor subclasses meet F.linear, as
    with any nn.Linear, in MLPs and layers of a hip backend too."""
    from torch.autograd import forward_ad
    from torch.utils.flop_counter import FlopCounterMode

    from kla.layers.common import MLP

    mlp = MLP(64, 2.0, kind="gelu").to(cuda)
    mlp.backend = "hip"
    x, t = (torch.randn(300, 64, device=cuda) for _ in range(2))
    with torch.no_grad():
        want = mlp(x)
        with forward_ad.dual_level():
            out = forward_ad.unpack_dual(mlp(forward_ad.make_dual(x, t)))
        assert out.tangent is not None
        h = 1e-3
        slope = (mlp(x + h * t) - mlp(x - h * t)) / (2 * h)
        assert torch.allclose(out.tangent, slope, rtol=1e-2, atol=1e-2)
        batched = torch.func.vmap(mlp)(torch.stack([x, t]))
        assert torch.allclose(batched[0], want, rtol=1e-4, atol=1e-5)
        with FlopCounterMode(display=False) as flops:
            mlp(x)
        assert flops.get_total_flops() == 2 * 300 * 64 * 2 * mlp.w1.weight.shape[0]
        with torch.overrides.BaseTorchFunctionMode():
            assert not lin.product_ok(mlp.w1, x)
        assert lin.product_ok(mlp.w1, x)

        class Sub(torch.Tensor):
            pass

        assert not lin.product_ok(mlp.w1, x.as_subclass(Sub)) and isinstance(mlp.w1(x.as_subclass(Sub)), Sub)


@pytest.mark.parametrize("k", [1, 4, 16, 31, 32, 40, 64, 100, 512, 1365, 2049])
def test_modules_keep_the_library_accuracy(cuda, k):
    """No module's fp32 inference product is further from float64 (2-norm) than the
    library's: short rows keep it, the others are closer on the matrix cores."""
    g = torch.Generator(device=cuda).manual_seed(k)
    mod = torch.nn.Linear(k, 512, bias=False).to(cuda)
    for gated in (False, True):
        x = torch.randn(1024, k, device=cuda, generator=g)
        if gated:
            x = x * F.silu(torch.randn(1024, k, device=cuda, generator=g))
        with torch.no_grad():
            mod.weight.copy_(torch.randn(512, k, device=cuda, generator=g))
            want = x.double() @ mod.weight.double().t()
            err, library = ((y.double() - want).norm() for y in (lin.plain_linear(mod, x), mod(x)))
        # (The 2-norm of 512 x 1024 nearly independent errors varies by under 1%.)
        assert err <= 1.01 * library, (k, gated, (err / library).item())


def test_under_graph_capture_and_on_two_streams(cuda):
    """Each call's workspace is its own: replays and calls on two streams in turn give
    the eager results."""
    g = torch.Generator(device=cuda).manual_seed(5)
    xs = [torch.randn(512, 160, device=cuda, generator=g) for _ in range(2)]
    w = torch.randn(300, 160, device=cuda, generator=g)
    want = [lin.linear_f32(x, w) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    for _ in range(3):
        got = []
        for s, x in zip(streams, xs):
            with torch.cuda.stream(s):
                got.append(lin.linear_f32(x, w))
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    buf = xs[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = lin.linear_f32(buf, w)
    for i in (1, 0, 1):
        buf.copy_(xs[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[i])
        assert torch.equal(lin.linear_f32(xs[i], w), want[i])


def _folded(x, w, bias, opts):
    """linear_f32's options in float64, and the operand of the product."""
    xd = x.double()
    if "norm" in opts:
        nw, eps = opts["norm"]
        xd = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + eps) * nw.double()
    a = xd @ w.double().t() + bias.double()
    if opts.get("swiglu"):
        h = w.shape[0] // 2
        return F.silu(a[..., :h]) * a[..., h:], xd, a
    return (a if "residual" not in opts else opts["residual"].double() + a), xd, a


@pytest.mark.parametrize("rows,n,k", [(1, 2, 1), (33, 64, 31), (65, 66, 513), (300, 130, 1030), (70, 1366, 2060),
                                      (1030, 2050, 64)])
@pytest.mark.parametrize("what", ["norm", "norm+swiglu", "norm+residual", "swiglu", "residual"])
def test_folded_options_match_float64(cuda, rows, n, k, what):
    print(f"[linear_f32] {what} {rows} x {k} -> {n}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(rows + n + k)

    def rn(*s):
        return torch.randn(*s, device=cuda, generator=g)

    x, w, bias, opts = rn(rows, k), rn(n, k) * k ** -0.5, rn(n), {}
    if "norm" in what:
        opts["norm"] = (1 + 0.1 * rn(k), 1e-5)
    if "residual" in what:
        opts["residual"] = rn(rows, n)
    if "swiglu" in what:
        opts["swiglu"] = True
    got = lin.linear_f32(x, w, bias, **opts)
    want, xd, a = _folded(x, w, bias, opts)
    # The product's bound on the operand formed in fp32: the norm's few roundings
    # (a sum of k squares among them) and hardware exp, 2^-21 of it each element.
    prod = _bound(xd, w) + (2.0 ** -21 + k * 2.0 ** -25) * (xd.abs() @ w.double().abs().t()) + 2.0 ** -22 * a.abs()
    if "swiglu" in opts:
        h = n // 2
        ga, ua = a[:, :h], a[:, h:]
        # silu' <= 1.1; silu itself good to 2^-20 of its value plus its argument's error.
        bound = 1.1 * prod[:, :h] * (ua.abs() + prod[:, h:]) + F.silu(ga).abs() * prod[:, h:] + 2.0 ** -20 * want.abs()
    else:
        bound = prod + 2.0 ** -22 * want.abs()
    assert got.shape == want.shape
    assert ((got.double() - want).abs() / (bound + 1e-30)).max().item() <= 1.0


def test_folded_options_with_infinities_and_nans(cuda):
    g = torch.Generator(device=cuda).manual_seed(8)
    x, w, bias = (torch.randn(*s, device=cuda, generator=g) for s in ((100, 70), (96, 70), (96,)))
    nw, res = torch.ones(70, device=cuda), torch.randn(100, 96, device=cuda, generator=g)
    x[3, 4], x[64, 0], w[9, 2], x[5] = float("inf"), float("nan"), -float("inf"), 1e30
    for opts in ({"norm": (nw, 1e-5), "swiglu": True}, {"norm": (nw, 1e-5), "residual": res}, {"residual": res}):
        got, xw = lin.linear_f32(x, w, bias, **opts), x.clone()
        if "norm" in opts:      # fp32 squares of 1e30 overflow, as torch's do: the row normalises to 0
            xw[5] = 0
        want = _folded(xw, w, bias, opts)[0]
        rows = [i for i in range(100) if i not in (3, 64)]
        cols = [i for i in range(want.shape[1]) if i != 9]
        scale = want[rows][:, cols].abs().amax(1, keepdim=True)
        assert ((got[rows][:, cols].double() - want[rows][:, cols]).abs() <= 1e-4 * scale).all()
        for r in (3, 64):
            assert torch.equal(torch.isfinite(got[r]), torch.isfinite(want[r].float())), (opts.keys(), r)
        assert not torch.isfinite(got[rows, 9]).all()


def _best_ms(f):
    times = []
    for _ in range(3):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    return min(times)


def test_a_batch_of_nans_stays_near_the_library(cuda):
    """Every output formed again in plain fp32: a few times the library product (2.4
    measured), not the hundreds of a serial sum a lane."""
    g = torch.Generator(device=cuda).manual_seed(10)
    x, w = (torch.randn(2048, 1024, device=cuda, generator=g) for _ in range(2))
    x[:, 5] = float("nan")
    assert torch.isnan(lin.linear_f32(x, w)).all()
    F.linear(x, w)
    got, library = _best_ms(lambda: lin.linear_f32(x, w)), _best_ms(lambda: F.linear(x, w))
    print(f"[linear_f32] NaN rows {got:.3f} ms, library {library:.3f} ms", flush=True)
    assert got < 20 * library + 0.2


def _in_place(x, w, bias, res):
    """kla_linear_f32_fwd with the residual add in place (y is res): the returned tensor."""
    lib, p = _lib.lib(), _lib.ptr
    y, (rows, k), n = res.clone(), x.shape, w.shape[0]
    nbytes = lib.kla_linear_f32_workspace_bytes(rows, n, k, _lib.KLA_ROWS_RESIDUAL)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    args = _lib.LinearF32(epilogue=_lib.KLA_ROWS_RESIDUAL, x=p(x), w=p(w), bias=p(bias), res=p(y), y=p(y), ldx=k, ldw=k,
                          ldres=n, ldy=n, rows=rows, n=n, k=k)
    _lib.check("kla_linear_f32_fwd", lib.kla_linear_f32_fwd(ctypes.byref(args), p(ws), nbytes, _lib.stream(x.device)))
    return y


def test_residual_in_place(cuda):
    """y is res: the same values as out of place, rows and columns that hold an infinity or
    a NaN included (their outputs read res where no earlier store has been)."""
    g = torch.Generator(device=cuda).manual_seed(9)
    x, w, bias, res = (torch.randn(*s, device=cuda, generator=g) for s in ((150, 70), (133, 70), (133,), (150, 133)))
    assert torch.equal(_in_place(x, w, bias, res), lin.linear_f32(x, w, bias, residual=res))
    x[3, 4], x[64, 0], w[9, 2], w[128, 1] = float("inf"), float("nan"), -float("inf"), float("nan")
    x[:, 2] = x[:, 2].abs()     # a finite value against W's infinity leaves no 0 * inf
    got, want = _in_place(x, w, bias, res), lin.linear_f32(x, w, bias, residual=res)
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    assert torch.isfinite(want[5, :9]).all() and not torch.isfinite(want[3]).any() and torch.isnan(want[:, 128]).all()
    w[9, 2], w[9, 3] = 0.0, float("inf")
    x[:, 3] = 0.0
    x[7, 3] = 1.0
    got, want = _in_place(x, w, bias, res), lin.linear_f32(x, w, bias, residual=res)
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0)) and got[7, 9] == float("inf")


def test_blocks_fold_their_norms_and_residuals(cuda, monkeypatch):
    """A block's prefill with the folded products against the same modules called one by
    one (hooks on them), with and without a state; a hook keeps its module's own call."""
    from kla import KLAConfig
    from kla.configs import ModelConfig
    from kla.models import Block

    torch.manual_seed(0)
    for cfg in (KLAConfig(backend="hip"), KLAConfig(backend="hip", use_gating=False, value_rank="conv", var_rank="dt"),
                KLAConfig(backend="hip", lambda_skip_mode="vector", gating_activation="gelu", bias=True)):
        block = Block(48, cfg, ModelConfig(d_model=48, mlp_ratio=3.0)).to(cuda)
        x = torch.randn(3, 100, 48, device=cuda)
        folded = []
        orig = lin.linear_f32
        monkeypatch.setattr(lin, "linear_f32", lambda *a, **kw: folded.append(set(kw)) or orig(*a, **kw))
        with torch.no_grad():
            y, st = block(x, return_state=True)
            y2 = block(x)
            assert any("norm" in f for f in folded) and any("swiglu" in f for f in folded)
            assert torch.equal(y, y2)
            folded.clear()
            seen = []
            hooks = [m.register_forward_hook(lambda m, a, o: seen.append(type(m).__name__)) for m in
                     (block.mixer_norm, block.mlp_norm, block.mixer.in_proj, block.mixer.out_proj, block.mlp.w12)]
            want, wst = block(x, return_state=True)
            assert len(seen) == 5 and not any("norm" in f or "swiglu" in f for f in folded)
            for h in hooks:
                h.remove()
            monkeypatch.setattr(lin, "linear_f32", orig)
        # Two fp32 evaluations of one block, a few products deep.
        assert torch.allclose(y, want, rtol=1e-4, atol=1e-5 * want.abs().max().item())
        for a, b in zip((st.conv, *st.ssm), (wst.conv, *wst.ssm)):
            assert torch.allclose(a, b, rtol=1e-4, atol=1e-5 * b.abs().max().item())
