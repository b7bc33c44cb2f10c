"""bf16 prefill attention against float64 where its units, tiles and key splits can go wrong: heads
sharing keys 1 to 8 ways, query blocks of 32 and key tiles of 64 with one more or one fewer, windows
from one key to more than there are, and grids that split the keys or do not."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    # rows, heads, kv heads, queries, keys, head_dim, window
    (1, 1, 1, 1, 1, 64, 1),
    (1, 1, 1, 1, 200, 128, 64),        # one query, window of one tile, split keys
    (2, 3, 1, 33, 97, 64, 40),         # three heads per kv head, window inside a tile and a half
    (1, 6, 2, 64, 64, 128, 64),
    (3, 4, 4, 31, 95, 64, 1),          # window 1: self only
    (1, 8, 1, 65, 300, 64, 257),       # eight heads per kv head
    (2, 2, 1, 129, 129, 128, 1000),    # window past the keys
    (5, 5, 5, 100, 163, 64, 65),       # rows * kv heads not a power of two
    (2, 12, 4, 1500, 1500, 64, 128),   # six-wave workgroups
    (4, 16, 4, 1025, 1100, 128, 333),  # eight-wave workgroups, one query past the blocks
    (2, 16, 16, 700, 700, 64, 96),     # no sharing
]


@pytest.mark.parametrize("case", CASES)
def test_prefill_attention_matches_float64(case):
    from utttcompanion_amd import kernels as K
    b, h, hkv, tq, tkv, hd, win = case
    print(f"prefill attention {case}", flush=True)
    g = torch.Generator().manual_seed(sum(case))
    q = (2.0 * torch.randn(b, tq, h, hd, generator=g)).bfloat16().cuda().transpose(1, 2)
    k = torch.randn(b, hkv, tkv + 7, hd, generator=g).bfloat16().cuda()
    v = torch.randn(b, hkv, tkv + 7, hd, generator=g).bfloat16().cuda()
    k[:, :, tkv:] = float("nan")  # the buffers go on past the keys
    v[:, :, tkv:] = float("nan")
    off = tkv - tq
    got = K.swa_prefill(q, k, v, win, off, kv_len=tkv)
    assert torch.equal(got, K.swa_prefill(q, k, v, win, off, kv_len=tkv))
    kd, vd = (t[:, :, :tkv].double().repeat_interleave(h // hkv, 1) for t in (k, v))
    d = (torch.arange(tq, device="cuda")[:, None] + off) - torch.arange(tkv, device="cuda")
    p = (q.double() @ kd.transpose(-1, -2) / hd ** 0.5).masked_fill((d < 0) | (d >= win), float("-inf")).softmax(-1)
    ref = p @ vd
    # half an ulp of the output (2^-9) and of each weight (2^-9 of sum p |v|), doubled for the fp32
    # score and exponent errors, which are far smaller
    bound = 2.0 ** -8 * (ref.abs() + p @ vd.abs())
    assert bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("spread", [1.0, 2.0, 4.0])
@pytest.mark.parametrize("case", [(2, 4, 2, 700, 1300, 64, 512), (1, 8, 2, 1024, 1024, 128, 1024),
                                  (1, 4, 1, 64, 900, 128, 512)])  # the last one in key splits
def test_heaviest_weight_of_a_query_is_not_rounded(case, spread):
    """Scores with a spread of ``spread``, as trained heads have them: the heaviest key of a query weighs
    1 before the normalisation, so only the other weights are rounded."""
    from utttcompanion_amd import kernels as K
    b, h, hkv, tq, tkv, hd, win = case
    print(f"peaked attention {case} {spread}", flush=True)
    g = torch.Generator().manual_seed(sum(case))
    q = (spread * torch.randn(b, tq, h, hd, generator=g)).bfloat16().cuda().transpose(1, 2)
    k, v = (torch.randn(b, hkv, tkv, hd, generator=g).bfloat16().cuda() for _ in range(2))
    off = tkv - tq
    got = K.swa_prefill(q, k, v, win, off).double()
    kd, vd = (t.double().repeat_interleave(h // hkv, 1) for t in (k, v))
    d = (torch.arange(tq, device="cuda")[:, None] + off) - torch.arange(tkv, device="cuda")
    p = (q.double() @ kd.transpose(-1, -2) / hd ** 0.5).masked_fill((d < 0) | (d >= win), float("-inf")).softmax(-1)
    ref = p @ vd
    # half an ulp of the output (2^-8 relative at most) and of every weight but the heaviest; 2^-14 for
    # the fp32 scores (up to about 30, summed over hd products in fp32) and exponents
    rest = p.masked_fill(p >= p.amax(-1, keepdim=True), 0.0)
    bound = 2.0 ** -8 * (ref.abs() + rest @ vd.abs()) + 2.0 ** -14 * (p @ vd.abs())
    assert bool(((got - ref).abs() <= bound).all())
    # as a whole: the error of weights rounded against the query's own heaviest, and of the rounded output; the
    # kernel rounds against the heaviest so far, which is as good (a heaviest weight of other than 1, rounded
    # too, comes to 1.05, 1.2 and 1.2 of it at the three spreads)
    w = (p / p.amax(-1, keepdim=True))
    same = ((w.bfloat16().double() @ vd) / w.sum(-1, keepdim=True)).bfloat16().double()
    assert float((got - ref).norm()) <= 1.03 * float((same - ref).norm())


@pytest.mark.parametrize("scale", [-0.125, 0.0, 0.3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case", [(2, 4, 2, 100, 163, 64, 65), (1, 2, 1, 64, 600, 128, 512)])  # the latter in splits
def test_any_softmax_scale(case, dtype, scale):
    """The C entry's ``scale`` may be any number, whatever the type: none, or one that turns the order of
    the scores round."""
    import ctypes as C
    from utttcompanion_amd import _native as N
    from utttcompanion_amd import kernels as K
    b, h, hkv, tq, tkv, hd, win = case
    print(f"attention scale {case} {dtype} {scale}", flush=True)
    g = torch.Generator().manual_seed(sum(case))
    q = torch.randn(b, h, tq, hd, generator=g).to(dtype).cuda()
    k, v = (torch.randn(b, hkv, tkv, hd, generator=g).to(dtype).cuda() for _ in range(2))
    out = torch.empty_like(q)
    off = tkv - tq
    lib = N.load_library()
    ws = torch.empty(lib.uttt_swa_prefill_workspace(b, h, tq, tkv, hd, win), dtype=torch.uint8, device="cuda")
    a = K.swa_prefill(q, k, v, win, off, out=out, workspace=ws, build_only=True)
    a.scale = scale
    N.check(lib.uttt_swa_prefill(C.byref(a), torch.cuda.current_stream().cuda_stream), "uttt_swa_prefill")
    kd, vd = (t.double().repeat_interleave(h // hkv, 1) for t in (k, v))
    d = (torch.arange(tq, device="cuda")[:, None] + off) - torch.arange(tkv, device="cuda")
    p = (scale * (q.double() @ kd.transpose(-1, -2))).masked_fill((d < 0) | (d >= win), float("-inf")).softmax(-1)
    ref = p @ vd
    # bf16: half an ulp (2^-8 relative at most) of the output and of each weight; fp32: sums of up to 600 terms
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -14
    assert bool(((out.double() - ref).abs() <= unit * (ref.abs() + 1.1 * (p @ vd.abs()))).all())
