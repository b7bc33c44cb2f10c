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
