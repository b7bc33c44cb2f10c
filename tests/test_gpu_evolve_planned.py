"""The ragged update's chunks in one library call each, against the same update launched call by call.

Both run the same kernels in the same order on each stream with the same rounding points, so what
may differ between them is the order of the sums of the slow-weight products (library products
there, uttt_linear here), which now and then turns the bf16 rounding of an activation the other way.
The row counts step down one by one, by several at once and not at all; the last chunks are ragged; the
per-chunk gate and a chunk without valid tokens run too.
"""
import pytest
import torch

from test_gpu_evolve import _chunk_row_means, to_state
from test_gpu_model import DEV, NAMES, build

pytestmark = pytest.mark.gpu

LENGTHS = [[5], [16, 16, 16], [80, 64, 48, 33, 17, 1], [97, 1, 1, 96, 2], [70, 31, 15, 64]]
# An activation that rounds the other way is off by 2^-8 of itself at most; of independent ones a share
# of the elements, at each of some ten rounding points a layer, and what was written from it is read by the
# chunks after: five times 2^-8 of the written part.  A chunk that is lost is 1 / 7 of it and more, one of
# the wrong row or the wrong momentum all of it.
REL = 0.02


def make(lengths):
    model, oracle = build(dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(len(lengths))
    ids = [torch.randint(6, 256, (n,), generator=g) for n in lengths]
    masks = [torch.ones(n) for n in lengths]
    if lengths[0] > 48:
        masks[0][16:32] = 0
    ostates = []
    for i in range(len(lengths)):
        st = oracle.init_state(1)
        st.w_up.add_(0.02 * torch.randn(st.w_up.shape, generator=g))
        st.s_down.add_(1e-3 * torch.randn(st.s_down.shape, generator=g))
        st.step = i
        ostates.append(st)
    return model, oracle, ids, masks, ostates


def written(state, before, name):
    return getattr(state, name).double().cpu() - getattr(before, name).double()


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("lengths", LENGTHS)
def test_planned_update_matches_call_by_call(lengths, gated, monkeypatch):
    from utttcompanion_amd import evolve
    model, oracle, ids, masks, ostates = make(lengths)
    gate = 0.0
    if gated:  # in the widest gap of the middle of the chunks' losses
        _, means = _chunk_row_means(oracle, ids, masks, ostates, 0.0)
        vals = torch.sort(means[means > 0]).values
        lo, hi = len(vals) // 4, max(len(vals) // 4 + 1, 3 * len(vals) // 4)
        j = lo + int(torch.argmax((vals[1:] - vals[:-1])[lo:hi]))
        gate = float((vals[j] + vals[j + 1]) / 2)
        _, seen = _chunk_row_means(oracle, ids, masks, ostates, gate)
        seen = seen[seen > 0]
        margin = float((seen - gate).abs().min() / gate)
        print("gate", gate, "margin", margin, "of", len(seen), "skipped", int((seen < gate).sum()), flush=True)
        assert bool((seen < gate).any()) and bool((seen >= gate).any())
    planned = []
    real = evolve._run_planned
    monkeypatch.setattr(evolve, "_run_planned", lambda *a: (planned.append(1), real(*a)))

    def run(min_chunk_surprise):
        states = [to_state(st) for st in ostates]
        out = evolve.ragged_test_time_update(model, [t.to(DEV) for t in ids], states, masks,
                                             min_chunk_surprise=min_chunk_surprise)
        torch.cuda.synchronize()
        for st, ost in zip(states, ostates):  # the caller's states are untouched
            assert all(torch.equal(getattr(st, n).cpu(), getattr(ost, n)) for n in NAMES)
        return out

    print("planned ragged update", lengths, gate, flush=True)
    got, again, plain = run(gate), run(gate), run(0.0)
    assert len(planned) == 3
    monkeypatch.setattr(evolve, "plan_supported", lambda *a: False)
    want = run(gate)
    assert len(planned) == 3
    changed = False
    for i, ((a, sa, la), (b, sb, lb), (a2, s2, l2), (p, _, _)) in enumerate(zip(got, want, again, plain)):
        assert sa == s2 and la == l2 and a.step == b.step == a2.step
        assert len(la) == len(lb) == len(model.layers)
        assert all(abs(x - y) <= 1e-2 * max(abs(y), 1e-6) for x, y in zip(la + [sa], lb + [sb])), (i, la, lb)
        for n in NAMES:
            assert torch.equal(getattr(a, n), getattr(a2, n)), (i, n)
            da, db = written(a, ostates[i], n), written(b, ostates[i], n)
            rel = float((da - db).norm() / db.norm().clamp_min(1e-30))
            print(i, n, "written", float(db.norm()), "off by", rel, flush=True)
            assert gated or float(db.norm()) > 0.0
            assert rel <= REL, (i, n)
            changed |= float((written(p, ostates[i], n) - da).norm()) > 2 * REL * float(da.norm())
    assert changed == gated  # the gate kept some chunk out that is written without it


def test_planned_update_above_every_loss_writes_nothing():
    from utttcompanion_amd import evolve
    model, _, ids, masks, ostates = make(LENGTHS[2])
    got = evolve.ragged_test_time_update(model, [t.to(DEV) for t in ids], [to_state(st) for st in ostates], masks,
                                         min_chunk_surprise=1e30)
    for (cand, _, _), ost in zip(got, ostates):
        assert all(torch.equal(getattr(cand, n).cpu(), getattr(ost, n)) for n in NAMES)
