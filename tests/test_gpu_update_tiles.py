"""The bf16 chunk update against float64 at the edges of its tiles: one token to several token
blocks, the smallest and ragged widths, reads through the cursor's own weights (one matrix of K and Q
rows), through other weights and through shared ones, masks, in place and into unaligned outputs."""
import pytest
import torch

from oracle import uttt_math as om

pytestmark = pytest.mark.gpu

CASES = [
    # rows, tokens, d_model, d_ff, read, masked, clip
    (1, 1, 64, 64, "own", False, 1.0),
    (3, 63, 128, 192, "own", True, 1.0),
    (2, 64, 192, 64, "other", False, 0.01),   # the clip is active
    (1, 64, 576, 1088, "own", False, 0.0),    # no clip
    (5, 65, 128, 128, "other", True, 0.01),   # two token blocks, rows not a power of two
    (2, 129, 64, 320, "shared", False, 0.01), # three token blocks
    (1, 300, 256, 192, "own", True, 0.01),    # five
    (8, 37, 320, 256, "shared", True, 1.0),
    (2, 40, 64, 8256, "own", True, 0.01),     # 129 norm partials, one past the straight loads
    # the larger tiles, by the plan's rule (H's, Z's); K and Q rows of one matrix meet inside a tile
    (16, 190, 512, 1024, "own", True, 1.0),   # 256 x 256, 64 x 128; three token blocks
    (16, 300, 512, 1024, "own", False, 0.01), # 256 x 256, 128 x 128; five
    (36, 300, 320, 256, "own", True, 1.0),    # 256 x 256 both; ragged columns
    (36, 300, 320, 256, "other", False, 1.0), # 128 x 128 both, a matrix each
    (26, 300, 512, 256, "shared", False, 1.0),# 256 x 256 both, a matrix each
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("out", ["new", "in_place", "unaligned"])
def test_update_matches_float64(case, out):
    from utttcompanion_amd import kernels as K
    b, c, d, f, read, masked, clip = case
    print(f"update {case} {out}", flush=True)
    g = torch.Generator().manual_seed(sum(case[:4]))
    unit = lambda: torch.nn.functional.rms_norm(torch.randn(b, c, d, generator=g), (d,)).bfloat16()
    q, k, v = unit(), unit(), unit()
    eta = (0.015 * torch.rand(b, c, 1, generator=g)).bfloat16()
    alpha = (0.005 * torch.rand(b, c, 1, generator=g)).bfloat16()
    weights = lambda n: [torch.randn(n, d, f, generator=g) / d ** 0.5, torch.randn(n, d, f, generator=g) / d ** 0.5,
                         torch.randn(n, f, d, generator=g) * 0.1 / f ** 0.5]
    w = weights(b)
    s = [1e-4 * t for t in weights(b)]
    rd = None if read == "own" else weights(1 if read == "shared" else b)
    ln = [1 + 0.1 * torch.randn(d, generator=g), 0.1 * torch.randn(d, generator=g)]
    mask = None
    if masked:
        mask = (torch.arange(c)[None] < torch.randint(0, c + 1, (b, 1), generator=g)).float()
        mask[0] = 0.0  # a row without tokens
    dev = lambda ts: [t.cuda() for t in ts]
    state = dev(w) + dev(s)
    outs = None
    if out == "in_place":
        outs = state
    elif out == "unaligned":  # one float past an aligned address
        outs = [torch.empty(t.numel() + 1, device="cuda")[1:].view(t.shape) for t in state]
    res = K.chunk_update(*dev([q, k, v, eta, alpha]), *state, *dev(ln), None if mask is None else mask.cuda(), 0.9,
                         clip, True, 1e-5, *(dev(rd) if rd else (None,) * 3), out_state=outs)
    rd64 = None if rd is None else [t.bfloat16().double().expand(b, -1, -1) for t in rd]
    w16 = [t.bfloat16().double() for t in w]  # the operands of the matrix units
    ref = om.fused_chunk_ttt_step(q.double(), k.double(), v.double(), eta.double(), alpha.double(), *w16,
                                  *(t.double() for t in s), *(t.double() for t in ln),
                                  None if mask is None else mask.double(), 0.9, clip, True, 1e-5,
                                  *(rd64 or w16))
    decay = 1.0 - (alpha[..., 0].double().mean(1) if mask is None else
                   (alpha[..., 0].double() * mask.double()).sum(1) / mask.double().sum(1).clamp_min(1)).view(-1, 1, 1)
    live = torch.ones(b, 1, 1) if mask is None else mask.any(1).view(-1, 1, 1).float()
    # H, dZ, dU and dG are rounded once (2^-9 relative at most): a gradient sums products of two of
    # them or of one and K, so its norm is off by at most about 2 * 2^-9; doubled for the clip factor
    for i in range(3):
        step = ref[4 + i] - 0.9 * s[i].double() * live - s[i].double() * (1 - live)
        got = res[4 + i].double().cpu() - 0.9 * s[i].double() * live - s[i].double() * (1 - live)
        floor = 1e-6 * float(s[i].double().norm())  # the fp32 momentum's own rounding
        assert float((got - step).norm()) <= 2.0 ** -7 * float(step.norm()) + floor, ("s", i)
        new_w = torch.where(live.bool(), decay * w[i].double() + res[4 + i].double().cpu(), w[i].double())
        assert float((res[1 + i].double().cpu() - new_w).abs().max()) <= 4 * 2.0 ** -24 * float(new_w.abs().max()), ("w", i)
    # the readout as in the frozen one: the LayerNorm pair enters in the activation type; output rounding, and
    # H's through the LayerNorm (with the pair in 64 bits, its own rounding, up to 2^-8 of LN(z) and of the bias,
    # used the bound up at one of the 1.6 million elements of 16 x 190 x 512)
    r = rd64 or w16
    z = (torch.nn.functional.silu(q.double() @ r[1]) * (q.double() @ r[0])) @ r[2]
    out64 = q.double() + torch.nn.functional.layer_norm(z, (d,), *(t.bfloat16().double() for t in ln), 1e-5)
    assert float((out64 - ref[0]).abs().max()) <= 2.0 ** -8 * float((out64 - q.double()).abs().max() + ln[1].abs().max())
    bound = 2.0 ** -8 * out64.abs() + 7 * 2.0 ** -9 / 3 ** 0.5 * 2.0
    assert bool(((res[0].double().cpu() - out64).abs() <= bound).all())
    assert abs(float(res[7]) - float(ref[7])) <= 2.0 ** -8 * abs(float(ref[7]))


@pytest.mark.parametrize("tokens", [37, 64, 129])
@pytest.mark.parametrize("noise", [1.0, 0.1, 0.01, 0.0])
def test_clip_factor_of_similar_tokens(tokens, noise):
    """The applied clip factor against the norm of the gradient itself, read back from an update without
    clipping (S' = -g from S = 0), where a chunk's keys are nearly one token and their errors nearly cancel:
    the norm is then a small difference of large sums unless its terms are squares."""
    from utttcompanion_amd import kernels as K
    b, d, f, eps = 2, 320, 256, 1e-5
    print(f"clip factor {tokens} tokens, noise {noise}", flush=True)
    g = torch.Generator().manual_seed(tokens)
    k = torch.nn.functional.rms_norm(torch.randn(b, 1, d, generator=g) + noise * torch.randn(b, tokens, d, generator=g),
                                     (d,)).bfloat16()
    w = [torch.randn(b, d, f, generator=g) / d ** 0.5, torch.randn(b, d, f, generator=g) / d ** 0.5,
         torch.randn(b, f, d, generator=g) / f ** 0.5]
    ln = [1 + 0.1 * torch.randn(d, generator=g), 0.1 * torch.randn(d, generator=g)]
    kd, w16 = k.double(), [t.bfloat16().double() for t in w]
    z = (torch.nn.functional.silu(kd @ w16[1]) * (kd @ w16[0])) @ w16[2]
    sign = torch.tensor([1.0, -1.0]).repeat(tokens)[:tokens] * (1.0 if tokens % 2 == 0 else (torch.arange(tokens) > 0))
    v = (kd + torch.nn.functional.layer_norm(z, (d,), ln[0].double(), ln[1].double(), eps)
         + sign[None, :, None] * torch.randn(b, 1, d, generator=g)).bfloat16()
    eta = torch.full((b, tokens, 1), 0.5).bfloat16()
    args = [t.cuda() for t in (k, k, v, eta, torch.zeros_like(eta), *w, *(torch.zeros_like(t) for t in w), *ln)]
    grad = [t.double() for t in K.chunk_update(*args, None, 0.9, 0.0, False, eps)[4:7]]
    n2 = sum(t.square().sum((1, 2)) for t in grad)
    clip = 0.25 * float(n2.min().sqrt())
    got = [t.double() for t in K.chunk_update(*args, None, 0.9, clip, False, eps)[4:7]]
    # the least squares factor between the two, a mean over their 2^-24 roundings
    factor = sum((a * t).sum((1, 2)) for a, t in zip(got, grad)) / n2
    want = clip / (n2 + 1e-8).sqrt()
    print(n2.tolist(), (factor / want - 1).tolist(), flush=True)
    # squares added up in fp32 in chains of at most 12 D / 64 + 20 additions, 2^-24 each; half of it in the
    # root, whose own rounding and the division's are 2^-23
    assert float((factor / want - 1).abs().max()) <= (12 * d / 64 + 20) * 2.0 ** -25 + 2.0 ** -22


def gate_inputs(tokens, masked):
    """Four rows with losses far apart: (chunk_update's first 14 arguments on the GPU, token counts)."""
    b, d, f = 4, 128, 192
    g = torch.Generator().manual_seed(tokens + masked)
    unit = lambda: torch.nn.functional.rms_norm(torch.randn(b, tokens, d, generator=g), (d,))
    q, k, v = unit(), unit(), unit() * torch.tensor([0.3, 1.0, 3.0, 10.0]).view(b, 1, 1)
    eta, alpha = (x * torch.rand(b, tokens, 1, generator=g) for x in (0.015, 0.005))
    w = [torch.randn(b, d, f, generator=g) / d ** 0.5, torch.randn(b, d, f, generator=g) / d ** 0.5,
         torch.randn(b, f, d, generator=g) * 0.1 / f ** 0.5]
    s = [1e-3 * torch.randn(t.shape, generator=g) for t in w]
    ln = [1 + 0.1 * torch.randn(d, generator=g), 0.1 * torch.randn(d, generator=g)]
    mask = None
    if masked:
        mask = torch.ones(b, tokens)
        mask[1, tokens // 2:] = 0
        mask[3, ::3] = 0
    args = [t.bfloat16().cuda() for t in (q, k, v, eta, alpha)] + [t.cuda() for t in w + s + ln]
    return args + [None if mask is None else mask.cuda()], mask.sum(1) if masked else torch.full((b,), float(tokens))


@pytest.mark.parametrize("tokens", [37, 64, 129])  # the row scalars formed in the write, and in a launch of their own
@pytest.mark.parametrize("masked", [False, True])
def test_row_loss_and_inclusive_gate(tokens, masked):
    """The per-row [sum of masked token losses, valid tokens] against float64, and the gate at a row's own
    mean exactly: that row is written there and keeps W and S one float step above."""
    import numpy as np
    from utttcompanion_amd import kernels as K
    args, counts = gate_inputs(tokens, masked)
    print(f"row loss and gate {tokens} tokens, masked {masked}", flush=True)

    def run(gate):
        row_loss = torch.full((4, 2), float("nan"), device="cuda")
        out = K.prepare_chunk_update(*args, 0.9, 1.0, True, 1e-5, row_loss=row_loss, min_row_surprise=gate).launch()
        return [t.clone() for t in out], row_loss.cpu()

    plain, rl = run(0.0)
    assert torch.equal(rl[:, 1], counts)
    means = rl[:, 0] / torch.clamp(rl[:, 1], min=1.0)  # as the kernels form it
    k, v, w = args[1], args[2], args[5:8]
    mask = args[13]
    rows = om.row_surprise(k.double(), v.double(), *(t.bfloat16().double() for t in w), *(t.double() for t in args[11:13]),
                           None if mask is None else mask.double(), True, 1e-5).cpu()
    # H is rounded to bf16 (2^-8 relative at most), so LN(z), of unit size, is off by that a token at most, and a
    # token's loss, half the mean square of an error e, by 2^-8 sqrt(2 loss) (and its square)
    assert bool(((means.double() - rows).abs() <= 2.0 ** -8 * (2 * rows).sqrt() + 2.0 ** -16).all())
    assert all(means[i] < means[i + 1] for i in range(3))
    surprise = float(rl[:, 0].double().sum() / rl[:, 1].double().sum())
    assert abs(float(plain[7]) - surprise) <= 1e-6 * surprise
    start = args[5:11]
    for r in range(4):
        at = float(means[r])
        for gate in (at, float(np.nextafter(np.float32(at), np.float32(np.inf)))):
            got, rl2 = run(gate)
            assert torch.equal(rl2, rl) and torch.equal(got[0], plain[0]) and torch.equal(got[7], plain[7])
            for i in range(4):
                kept = i < r or (i == r and gate > at)
                for a, p, o in zip(got[1:7], plain[1:7], start):
                    assert torch.equal(a[i], o[i] if kept else p[i]), (r, gate, i)
    assert not any(torch.equal(p[i], o[i]) for p, o in zip(plain[1:7], start) for i in range(4))
