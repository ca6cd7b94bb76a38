"""The time split at lengths that equal chunks do not divide (kla_fused_split_fwd,
kla_fused_split_bwd): chunks of whole checkpoint blocks with a shorter last one,
against the float64 filter and its autograd, and the plan that picks them."""

import pytest
import torch

from kla.ops import KLAState, kla_scan
from kla.ops.hip import fused
from test_gpu_backend import check_scan, make_inputs, oracle, random_state


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
