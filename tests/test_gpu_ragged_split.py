"""The time split at lengths that equal chunks do not divide (kla_fused_split_fwd,
kla_fused_split_bwd): chunks of whole checkpoint blocks with a shorter last one,
against the float64 filter and its autograd, and the plan that picks them."""

import ctypes

import pytest
import torch

from kla.ops import KLAState, kla_scan
from kla.ops.hip import _lib, fused
from test_gpu_backend import _projection, _views, check_scan, make_inputs, oracle, random_state


def test_ragged_plan():
    plan = fused.ragged_chunk
    # 64 workgroups: eight chunks of 128 steps, the last one of 125.
    assert plan(1, 1021, 1024, 16, 256, 1, False) == 128
    assert plan(1, 301, 1024, 16, 256, 1, False) == 0        # two chunks gain less than their launches
    assert plan(1, 501, 1024, 16, 256, 1, False) == 128      # four do: 3 x 128 + 117
    assert plan(1, 191, 1024, 16, 256, 1, False) == 0        # one chunk
    assert plan(1, 2500, 8, 16, 256, 4, False) == 128        # four equal chunks leave the grid small
    assert plan(2, 389, 1000, 16, 256, 1, False) == 0        # 126 workgroups: the second pass is not free
    assert plan(3, 1501, 1000, 16, 256, 1, False) == 0
    assert plan(2, 1021, 1000, 16, 256, 1, True) == 208      # with gradients
    assert plan(1, 643, 1000, 16, 256, 1, True) == 0         # gains less than its launches take of the host
    assert plan(2, 500, 768, 16, 256, 1, True) == plan(3, 1501, 1000, 16, 256, 1, True) == 0
    assert plan(4, 1023, 1024, 16, 256, 1, False) == 0       # one workgroup per CU already
    assert plan(1, 1024, 1024, 16, 256, 8, False) == 0       # equal chunks serve
    assert plan(0, 1021, 1024, 16, 256, 1, False) == plan(1, 1021, 0, 16, 256, 1, True) == 0
    for L in range(1, 3000, 7):
        for train in (False, True):
            for M in (64, 700, 2000):
                steps = plan(1, L, M, 16, 256, 1, train)
                assert steps == 0 or (steps % 16 == 0 and fused.MIN_CHUNK <= steps < L)


# (B, L, M, S), steps: a last chunk of one step, of one step under a block, of half a
# block, and a channel spanning waves.
CASES = [((2, 33, 9, 16), 32), ((1, 95, 70, 4), 48), ((3, 200, 5, 24), 96), ((1, 50, 2, 128), 16), ((2, 47, 3, 256), 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,steps", CASES)
@pytest.mark.parametrize("with_state,prior", [(False, False), (True, True)])
def test_forced_ragged_split_matches_float64(cuda, monkeypatch, shape, steps, with_state, prior):
    B, L, M, S = shape
    print(f"[ragged split] {shape} steps={steps} state={with_state} prior={prior}", flush=True)
    calls = []
    monkeypatch.setattr(fused, "ragged_chunk", lambda *a: calls.append(a) or steps)
    ins = make_inputs(B, L, M, S, seed=31)
    st = random_state(B, M, S, seed=5) if with_state else None
    wy, wv, wl, we = oracle(ins, st, prior)
    state = None if st is None else KLAState(st.lam.to(cuda), st.eta.to(cuda))
    y, y_var, fin = kla_scan(*(t.to(cuda) for t in ins), backend="hip_fused", decode_from_prior=prior,
                             initial_state=state)
    assert calls
    for name, got, want in (("y", y, wy), ("y_var", y_var, wv), ("lam", fin.lam, wl), ("eta", fin.eta, we)):
        check_scan(name, got, want)

    # Gradients, the final state's among them, against the same call in one piece.
    g = torch.Generator(device=cuda).manual_seed(6)

    def grads():
        xs = [t.to(cuda).requires_grad_(True) for t in ins]
        s0 = None if state is None else KLAState(*(t.clone().requires_grad_(True) for t in state))
        out = kla_scan(*xs, backend="hip_fused", decode_from_prior=prior, initial_state=s0)
        flat = (out[0], out[1], *out[2])
        g.manual_seed(6)
        return torch.autograd.grad(flat, xs + ([] if s0 is None else list(s0)),
                                   [torch.randn(t.shape, device=cuda, generator=g) for t in flat])

    split = grads()
    monkeypatch.setattr(fused, "ragged_chunk", lambda *a: 0)
    monkeypatch.setattr(fused, "train_chunks", lambda *a: 1)
    for got, want in zip(split, grads()):
        # Two fp32 evaluations of one sum: each within 1e-5 of the tensor's scale.
        assert torch.allclose(got, want, rtol=2e-5, atol=2e-5 * want.abs().max().item())


@pytest.mark.gpu
def test_unforced_ragged_lengths_match_float64(cuda):
    for B, L, M, S in ((1, 1021, 64, 16), (2, 771, 40, 8)):
        ins = make_inputs(B, L, M, S, seed=33)
        cus = fused._cus(cuda.index or 0)
        assert fused.ragged_chunk(B, L, M, S, cus, fused.time_chunks(B, L, M, S, cus), False)
        y, y_var, fin = kla_scan(*(t.to(cuda) for t in ins), backend="hip_fused")
        for name, got, want in zip(("y", "y_var", "lam", "eta"), (y, y_var, *fin), oracle(ins, None, False)):
            check_scan(name, got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape,steps", CASES)
@pytest.mark.parametrize("prior,with_var", [(False, False), (True, True)])
def test_forced_ragged_split_of_the_sensor_route(cuda, monkeypatch, shape, steps, prior, with_var, dtype):
    """As a layer runs it: v and log sigma^2 as column slices of a projection, fp32 and
    bf16, forward and every gradient, against the same call in one piece."""
    B, L, M, S = shape
    print(f"[ragged split] sensors {shape} steps={steps} {dtype}", flush=True)
    _, _, k, q, a, p = make_inputs(B, L, M, S, seed=41)
    st = random_state(B, M, S, seed=6)
    g = torch.Generator(device=cuda).manual_seed(7)
    proj = _projection(B, L, M, S, seed=9).to(cuda, dtype)

    def run():
        xs = [t.detach().to(cuda).requires_grad_(True) for t in (proj, k, q, a, p, st.lam, st.eta)]
        out = fused.kla_scan_fused_sensors(*_views(xs[0], M), *xs[1:], obs_var_min=1e-4, obs_var_max=1.5,
                                           decode_from_prior=prior, with_var=with_var)
        out = [t for t in out if t is not None]
        g.manual_seed(7)
        return [t.detach() for t in out] + list(torch.autograd.grad(
            out, xs, [torch.randn(t.shape, device=cuda, generator=g) for t in out]))

    calls = []
    monkeypatch.setattr(fused, "ragged_chunk", lambda *a: calls.append(a) or steps)
    split = run()
    assert len(calls) == 2
    monkeypatch.setattr(fused, "ragged_chunk", lambda *a: 0)
    monkeypatch.setattr(fused, "train_chunks", lambda *a: 1)
    for got, want in zip(split, run()):
        # Two fp32 evaluations of one sum, each within 1e-5 of the tensor's scale; bf16
        # gradients are those values rounded once (2^-8).
        tol = 2e-5 if got.dtype == torch.float32 else 2.0 ** -8
        assert got.dtype == want.dtype
        assert torch.allclose(got.float(), want.float(), rtol=tol, atol=2e-5 * want.abs().max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("prior,with_var", [(False, False), (True, True)])
def test_adjoint_maps_and_ends_match_the_split_backward(cuda, prior, with_var):
    """kla_fused_adjoint_maps, kla_adjoint_ends and the backward of every chunk from there,
    call by call on the [B nc, L / nc] view, against kla_fused_split_bwd's one call over the
    same chunks: the same kernels on the same numbers, so the same bits."""
    B, L, M, S, nc = 2, 96, 5, 16, 3
    lib, pt, f32 = _lib.lib(), _lib.ptr, dict(dtype=torch.float32, device=cuda)
    v, lv, k, q, a, p = (t.to(cuda) for t in make_inputs(B, L, M, S, seed=51))
    g = torch.Generator(device=cuda).manual_seed(8)
    dy, dyv, dlam, deta = (torch.randn(*s, device=cuda, generator=g) for s in ((B, L, M), (B, L, M), (B, M, S), (B, M, S)))
    dyv = dyv if with_var else None
    sn, stream = fused._dense_sensors(v, lv), _lib.stream(cuda)
    y, yv, lf, ef = torch.empty(B, L, M, **f32), torch.empty(B, L, M, **f32), torch.empty(B, M, S, **f32), torch.empty(B, M, S, **f32)
    ckl, cke = torch.empty(B, L // 16, M, S, **f32), torch.empty(B, L // 16, M, S, **f32)
    _lib.check("fwd", lib.kla_fused_scan_sensors_fwd(
        ctypes.byref(sn), pt(k), pt(q), pt(a), pt(p), None, None, pt(y), pt(yv), pt(lf), pt(ef), pt(ckl), pt(cke),
        int(prior), B, L, M, S, stream))

    def grads():
        return [torch.empty_like(t) for t in (v, lv, k, q, a, p)]

    one, d0 = grads(), [torch.empty(B, M, S, **f32) for _ in range(2)]
    nbytes = lib.kla_fused_split_workspace_bytes(B, L, M, S, L // nc, 1)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=cuda)
    _lib.check("split", lib.kla_fused_split_bwd(
        pt(dy), pt(dyv), pt(dlam), pt(deta), ctypes.byref(sn), pt(k), pt(q), pt(a), pt(p), pt(ckl), pt(cke),
        *(pt(t) for t in one), *(pt(t) for t in d0), int(prior), B, L, M, S, L // nc, pt(ws), nbytes, stream))

    two, maps = grads(), torch.empty(B * nc, M, S, 8, **f32)
    _lib.check("maps", lib.kla_fused_adjoint_maps(
        pt(dy), pt(dyv), ctypes.byref(sn), pt(k), pt(q), pt(a), pt(p), pt(ckl), pt(cke), pt(maps), int(prior), B * nc,
        L // nc, M, S, stream))
    ends = [torch.empty(B, nc, M, S, **f32) for _ in range(4)]
    _lib.check("ends", lib.kla_adjoint_ends(pt(maps), pt(dlam), pt(deta), pt(ends[0]), pt(ends[1]), B, nc, M, S, stream))
    nbytes = lib.kla_fused_workspace_bytes(B * nc, L // nc, M, S)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=cuda)
    _lib.check("bwd", lib.kla_fused_scan_sensors_bwd(
        pt(dy), pt(dyv), pt(ends[0]), pt(ends[1]), ctypes.byref(sn), pt(k), pt(q), pt(a), pt(p), pt(ckl), pt(cke),
        *(pt(t) for t in two), pt(ends[2]), pt(ends[3]), int(prior), B * nc, L // nc, M, S, pt(ws), nbytes, stream))
    for got, want in zip(one + d0, two + [ends[2][:, 0], ends[3][:, 0]]):
        assert torch.equal(got, want)
