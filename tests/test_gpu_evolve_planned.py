"""The ragged update's chunks in one library call each, against the same update launched call by call.

Both run the same kernels in the same order on each stream with the same rounding points, so what
may differ between them is the order of the split sums of the slow-weight products: the bound is
that of bf16 rows at another batch size (2e-2 on the weights, relative on the surprise).  The row
counts step down one by one, by several at once and not at all; the last chunks are ragged; the
per-chunk gate and a chunk without valid tokens run too.
"""
import pytest
import torch

from test_gpu_model import DEV, NAMES, build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths, gate", [
    ([5], 0.0), ([16, 16, 16], 0.0), ([80, 64, 48, 33, 17, 1], 0.0), ([97, 1, 1, 96, 2], 0.0), ([70, 31, 15, 64], 1.0),
])
def test_planned_update_matches_call_by_call(lengths, gate, monkeypatch):
    from utttcompanion_amd import FastWeightState, evolve
    model, oracle = build(dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(len(lengths))
    ids = [torch.randint(6, 256, (n,), generator=g).to(DEV) for n in lengths]
    masks = [torch.ones(n) for n in lengths]
    if lengths[0] > 48:
        masks[0][16:32] = 0
    states = []
    for i in range(len(lengths)):
        st = oracle.init_state(1)
        st.w_up.add_(0.02 * torch.randn(st.w_up.shape, generator=g))
        states.append(FastWeightState(*(getattr(st, n).clone().to(DEV) for n in NAMES), st.ln_weight.to(DEV),
                                      st.ln_bias.to(DEV), i, 0.0, []))
    before = [st.w_up.clone() for st in states]
    planned = []
    run = evolve._run_planned
    monkeypatch.setattr(evolve, "_run_planned", lambda *a: (planned.append(1), run(*a)))
    print("planned ragged update", lengths, gate, flush=True)
    got = evolve.ragged_test_time_update(model, ids, states, masks, min_chunk_surprise=gate)
    torch.cuda.synchronize()
    assert planned
    monkeypatch.setattr(evolve, "plan_supported", lambda *a: False)
    want = evolve.ragged_test_time_update(model, ids, states, masks, min_chunk_surprise=gate)
    torch.cuda.synchronize()
    assert len(planned) == 1
    for i, ((a, sa, la), (b, sb, lb)) in enumerate(zip(got, want)):
        worst = max((getattr(a, n) - getattr(b, n)).abs().max().item() for n in NAMES)
        print(i, worst, sa, sb, flush=True)
        assert worst <= 2e-2 and abs(sa - sb) <= 2e-2 * max(1.0, abs(sb))
        assert a.step == b.step and len(la) == len(lb)
        assert torch.equal(states[i].w_up, before[i])
