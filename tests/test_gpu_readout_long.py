"""The frozen readout over more than one token block: the long-block products against float64 at the
edges of their tiles (tokens around 64, 128 and 256, column remainders of both tile widths, split
down products), with bf16 copies and fp32 masters, per-row and shared weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [
    # rows, tokens, d_model, d_ff
    (1, 65, 64, 64),        # smallest: one step, column tiles mostly past the end
    (3, 129, 192, 320),     # every tile ragged
    (2, 333, 768, 2048),
    (1, 255, 512, 1024),
    (2, 256, 576, 1088),    # whole row tiles, ragged columns
    (4, 1025, 512, 1024),   # the wide tiles, one row past them
    (8, 700, 1024, 2816),   # the wide tiles, ragged rows
    (1, 2048, 2048, 5504),
    (4, 250, 512, 1024),    # fp32 W: the down product in 64 x 64 tiles, at its smallest number of them
    (8, 100, 768, 2048),    # shared W: the rows' tiles next to each other
    (3, 129, 320, 8256),    # the same with ragged columns
]


def _inputs(rows, tokens, d, f, shared, dtype):
    g = torch.Generator().manual_seed(rows * tokens + d)
    n = 1 if shared else rows
    x = torch.randn(rows, tokens, d, generator=g).bfloat16()
    w = [torch.randn(n, d, f, generator=g) / d ** 0.5, torch.randn(n, d, f, generator=g) / d ** 0.5,
         torch.randn(n, f, d, generator=g) / f ** 0.5]
    ln = (1 + 0.1 * torch.randn(d, generator=g), 0.1 * torch.randn(d, generator=g))
    return x.cuda(), [t.to(dtype).cuda() for t in w], [t.cuda() for t in ln]


@pytest.mark.parametrize("rows,tokens,d,f", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shared", [False, True])
def test_long_readout_matches_float64(rows, tokens, d, f, dtype, shared):
    from utttcompanion_amd import kernels as K
    x, w, ln = _inputs(rows, tokens, d, f, shared, dtype)
    if shared:
        w = [t.expand(rows, -1, -1) for t in w]
    out = K.swiglu_readout(x, *w, *ln, 1e-5)
    again = K.swiglu_readout(x, *w, *ln, 1e-5)
    assert torch.equal(out, again)
    xd = x.double()
    wd = [t.bfloat16().double() for t in w]  # the operands of the matrix units, for both weight types
    z = (torch.nn.functional.silu(xd @ wd[1]) * (xd @ wd[0])) @ wd[2]
    lnd = [t.bfloat16().double() for t in ln]  # the readout rounds the LayerNorm pair to the activation type
    ref = xd + torch.nn.functional.layer_norm(z, (d,), *lnd, 1e-5)
    # the output's rounding (half an ulp, 2^-9 relative) doubled, and H's: z sums f terms with independent relative
    # errors of at most 2^-9 (2^-9 / sqrt 3 rms), so LN(z), of unit size, is off by about that rms; seven of them for
    # the largest of up to 2^24 elements
    bound = 2.0 ** -8 * ref.abs() + 7 * 2.0 ** -9 / 3 ** 0.5 * 1.5
    assert bool(((out.double() - ref).abs() <= bound).all())
