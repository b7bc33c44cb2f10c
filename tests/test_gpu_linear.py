"""GPU parity of ``uttt_linear`` (out = x W^T (+ residual), bf16 operands, fp32 accumulation)
against a float32 product of the same bf16 operands rounded once to bf16.

Tolerance (north star, bf16 <= 2e-2 max-abs): per element |gpu - ref| <= 2^-8 |ref| + 1e-3 (one
bf16 rounding of an fp32 sum whose order differs from the reference's).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def ref_linear(x, w, residual=None):
    y = x.float() @ w.float().t()
    if residual is not None:
        y = y + residual.float()
    return y


def check(got, ref):
    err = (got.float() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + 1e-3
    assert bool((err <= bound).all()), f"max err {err.max().item():.3e}"
    assert err.max().item() <= 2e-2


# (m, n, k): config-3 chunk shapes (256 rows of d_model 2048: packed uTTT projections 3 D + 2,
# packed QKV, the output / residual projections), config-2 (512 rows of 768), ragged m and n
SHAPES = [(256, 6146, 2048), (256, 3072, 2048), (256, 2048, 2048), (512, 2306, 768), (512, 768, 768),
          (100, 70, 128), (1, 33, 64), (200, 130, 192), (4096, 256, 512)]


@pytest.mark.parametrize("shape", SHAPES, ids=[f"m{m}-n{n}-k{k}" for m, n, k in SHAPES])
@pytest.mark.parametrize("with_residual", [False, True], ids=["plain", "residual"])
def test_linear_matches_fp32_product(shape, with_residual):
    from utttcompanion_amd import kernels as K
    m, n, k = shape
    print(f"linear m {m} n {n} k {k} residual {with_residual}", flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).bfloat16().to(DEV)
    w = (torch.randn(n, k, generator=g) / k ** 0.5).bfloat16().to(DEV)
    r = torch.randn(m, n, generator=g).bfloat16().to(DEV) if with_residual else None
    got = K.linear(x, w, residual=r)
    torch.cuda.synchronize()
    check(got, ref_linear(x, w, r))


def test_linear_strided_operands_and_in_place_residual():
    """x and W as column slices of wider tensors (row strides > k), out a column slice of a wider
    buffer, the residual the output itself (h += x W^T)."""
    from utttcompanion_amd import kernels as K
    g = torch.Generator().manual_seed(5)
    xb = torch.randn(300, 1088, generator=g).bfloat16().to(DEV)
    wb = (torch.randn(500, 1032, generator=g) / 32).bfloat16().to(DEV)
    x, w = xb[:, 64:1024], wb[:, 8:968]
    hb = torch.randn(300, 520, generator=g).bfloat16().to(DEV)
    h = hb[:, 8:508]
    before = h.clone()
    spare = hb[:, :8].clone(), hb[:, 508:].clone()
    K.linear(x, w, out=h, residual=h)
    torch.cuda.synchronize()
    check(h, ref_linear(x, w, before))
    assert torch.equal(hb[:, :8], spare[0]) and torch.equal(hb[:, 508:], spare[1])


def test_linear_refuses_unsupported_operands():
    from utttcompanion_amd import kernels as K
    x = torch.randn(8, 96, device=DEV).bfloat16()
    w = torch.randn(16, 96, device=DEV).bfloat16()
    assert not K.linear_fits(x, w)
    with pytest.raises(RuntimeError, match="multiple of 64"):
        K.linear(x, w)
    with pytest.raises(ValueError, match="bf16"):
        K.linear(x.float(), w.float())


@pytest.mark.parametrize("m, n, k", [(64, 2048, 2048), (192, 768, 768), (100, 512, 1024)])
def test_linear_adds_its_k_splits_in_order(m, n, k):
    """Each split's partial is one term of 2^24, 1, 1, .., -2^24: added up in their order the ones vanish
    (2^24 + 1 rounds to 2^24) and the sum is 0; started from the last one, whose workgroup may well be
    the one that adds up, it is their number."""
    from utttcompanion_amd import _native as N
    from utttcompanion_amd import kernels as K
    nbytes = N.load_library().uttt_linear_workspace(m, n, k)
    assert nbytes > 0
    s = (nbytes - 4 * 16384) // (4 * 64 * 64 * ((m + 63) // 64) * (n // 64))  # after the counters: 64 x 64 fp32 tiles
    assert s >= 3
    print(f"linear split order m {m} n {n} k {k} splits {s}", flush=True)
    x = torch.zeros(m, k, dtype=torch.bfloat16)
    w = torch.zeros(n, k, dtype=torch.bfloat16)
    for i in range(s):
        first = 64 * (i * (k // 64) // s)  # split i's first column
        x[:, first] = 1.0
        w[:, first] = 2.0 ** 24 if i == 0 else -2.0 ** 24 if i == s - 1 else 1.0
    x, w = x.to(DEV), w.to(DEV)
    for _ in range(20):
        assert not bool(K.linear(x, w).any())


@pytest.mark.parametrize("m, n, k", [(64, 2048, 2048), (448, 768, 768)])
def test_linear_repeats_itself(m, n, k):
    from utttcompanion_amd import kernels as K
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).bfloat16().to(DEV)
    w = torch.randn(n, k, generator=g).bfloat16().to(DEV)
    first = K.linear(x, w)
    for _ in range(20):
        assert torch.equal(K.linear(x, w), first)
