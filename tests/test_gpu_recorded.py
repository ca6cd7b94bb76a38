"""Recording an op's gradient without the dispatcher (kla.ops.hip._lib._Recorded)
against the dispatched op: the same bits and the same saved tensors in eager
autograd, and the dispatcher wherever something else watches the call."""

import pytest
import torch

from kla import KLAConfig, KLALayer
from kla.ops import kla_scan
from kla.ops.hip import _lib, affine_scan, mobius_scan

pytestmark = pytest.mark.gpu


def _mobius(d, g):
    xs = [torch.rand(2, 40, 9, device=d, generator=g) for _ in range(3)]
    xs += [torch.rand(2, 40, 9, device=d, generator=g) + 0.5, torch.rand(2, 9, device=d, generator=g)]
    return xs, lambda *x: (mobius_scan(*x),)


def _affine(d, g):
    xs = [torch.rand(2, 40, 9, device=d, generator=g).bfloat16() for _ in range(2)]
    return xs + [torch.rand(2, 9, device=d, generator=g)], lambda *x: (affine_scan(*x),)


def _kla(d, g):
    xs = [torch.randn(2, 40, 6, device=d, generator=g), torch.rand(2, 40, 6, device=d, generator=g) + 0.5,
          *(torch.randn(2, 40, 5, device=d, generator=g) for _ in range(2)),
          torch.rand(6, 5, device=d, generator=g) * 0.5 + 0.4, torch.rand(6, 5, device=d, generator=g) * 0.1 + 0.01]

    def f(*x):
        y, y_var, st = kla_scan(*x, backend="hip")
        return y, y_var, *st

    return xs, f


def _layer(d, g):
    torch.manual_seed(0)
    layer = KLALayer(24, KLAConfig(backend="hip", var_rank="dt", clip_value=0.4)).to(d)
    xs = [torch.randn(2, 40, 24, device=d, generator=g), *(p.detach().clone() for p in layer.parameters())]
    names = [n for n, _ in layer.named_parameters()]
    return xs, lambda x, *w: (torch.func.functional_call(layer, dict(zip(names, w)), (x,)),)


@pytest.mark.parametrize("case", [_mobius, _affine, _kla, _layer])
def test_same_gradients_and_saved_tensors_as_dispatched(cuda, monkeypatch, case):
    def run(needs):
        g = torch.Generator(device=cuda).manual_seed(1)
        xs, f = case(cuda, g)
        xs = [x.requires_grad_(n) for x, n in zip(xs, needs)]
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(tuple(t.shape)) or t, lambda t: t):
            outs = f(*xs)
        douts = [torch.randn(o.shape, device=cuda, generator=g).to(o.dtype) for o in outs]
        return list(outs) + list(torch.autograd.grad(outs, [x for x in xs if x.requires_grad], douts)), sorted(packed)

    n = len(case(cuda, torch.Generator(device=cuda))[0])
    for needs in ([True] * n, [True] + [False] * (n - 1), [False, True] + [False] * (n - 2)):
        got, saved = run(needs)
        with monkeypatch.context() as m:
            m.setattr(_lib, "_eager", lambda: False)
            want, want_saved = run(needs)
        assert saved == want_saved
        assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_what_watches_a_call_keeps_the_dispatcher(cuda, monkeypatch):
    """functorch transforms, forward mode, dispatch and function modes: the op itself is
    called (so each behaves as it does for any custom op), not its recorded form."""
    seen = []
    apply = _lib._Recorded.apply
    monkeypatch.setattr(_lib._Recorded, "apply", lambda *a: seen.append(1) or apply(*a))
    xs, f = _mobius(cuda, torch.Generator(device=cuda).manual_seed(2))
    x0 = xs[0].clone().requires_grad_(True)

    def loss(a):
        return f(a, *xs[1:])[0].square().sum()

    torch.autograd.grad(loss(x0), x0)
    assert seen
    seen.clear()
    with pytest.raises(RuntimeError, match="functorch"):   # torch refuses custom ops' autograd there
        torch.func.grad(loss)(xs[0])
    assert not seen

    class Count(torch.utils._python_dispatch.TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    with Count() as mode:
        loss(x0)
    assert any("mobius_scan" in n for n in mode.names) and not seen
    with torch.overrides.BaseTorchFunctionMode():
        loss(x0)
    assert not seen
    with torch.autograd.forward_ad.dual_level():
        loss(x0)
    assert not seen


def test_checkpointed_and_retained_backward(cuda):
    xs, f = _kla(cuda, torch.Generator(device=cuda).manual_seed(3))
    xs = [x.requires_grad_(True) for x in xs]
    want = torch.autograd.grad(f(*xs)[0].sum(), xs)
    y = torch.utils.checkpoint.checkpoint(lambda *x: f(*x)[0], *xs, use_reentrant=False)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y.sum(), xs, retain_graph=True), want))
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y.sum(), xs), want))
