"""The split fp32 product (kla_linear_f32_fwd) against float64 torch: every tile's
edges, strided and unaligned operands, rows fp16 could not hold, rows with an
infinity or a NaN, and which calls of a module take it."""

import pytest
import torch
import torch.nn.functional as F

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
         (300, 2080, 1025), (130, 70, 2049), (1025, 1030, 96), (2049, 2049, 40), (4100, 2100, 64)]


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
    plus what entries 2^17 below the row's largest lose (2^-39 of it each)."""
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
    small = 2.0 ** -39 * (x.double().abs().amax(1)[:, None] * w.double().abs().sum(1)
                          + x.double().abs().sum(1)[:, None] * w.double().abs().amax(1))
    top = torch.finfo(torch.float32).max
    fits, over = want.abs() < top * (1 - 1e-5), want.abs() > top * (1 + 1e-5)
    err = (got.double() - want).abs() / (_bound(x, w) + small + 2.0 ** -23 * want.abs() + 2.0 ** -149)
    assert err[fits].max().item() <= 1.0
    assert torch.isinf(got[over]).all() and torch.equal(got[over] > 0, want[over] > 0)


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
    monkeypatch.setattr(lin, "linear_f32", lambda *a: calls.append(1) or orig(*a))
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
