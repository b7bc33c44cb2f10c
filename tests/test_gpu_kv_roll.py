"""RoPE, append, history and trimmed cache in one launch against the same steps one by one, bit for
bit: head sizes and lengths at the edges, caches that are views, shared by rows, of another type or
not 16-byte aligned (those take the copies)."""
import pytest
import torch

from oracle import uttt_math as om

pytestmark = pytest.mark.gpu

CASES = [
    # rows, tokens, heads, kv heads, head_dim, history, out_len, kind of history
    (1, 1, 1, 1, 64, 0, 1, "own"),
    (2, 5, 3, 1, 64, 7, 9, "own"),
    (3, 33, 4, 2, 128, 3, 36, "view"),      # everything kept
    (2, 70, 12, 4, 64, 511, 512, "view"),
    (3, 40, 4, 4, 64, 100, 20, "shared"),   # one cache for all rows, only new rows kept
    (2, 9, 2, 2, 32, 5, 6, "own"),          # two pieces a head
    (2, 9, 2, 1, 64, 5, 6, "unaligned"),
    (2, 9, 2, 1, 64, 5, 6, "other type"),
    (2, 9, 2, 1, 24, 5, 6, "own"),          # rows that are not whole pieces
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_roll_equals_the_steps(case, dtype):
    from utttcompanion_amd import kernels as K
    b, t, h, hkv, hd, hist, keep, kind = case
    print(f"kv roll {case} {dtype}", flush=True)
    g = torch.Generator().manual_seed(sum(case[:7]))
    qkv = torch.randn(b, t, h + 2 * hkv, hd, generator=g).to(dtype).cuda()
    n = 1 if kind == "shared" else b
    past = [torch.randn(n, hkv, hist + 6, hd + 8, generator=g) for _ in range(2)]
    past = [p.to(torch.float16 if kind == "other type" else dtype).cuda() for p in past]
    off = {"view": 8, "unaligned": 1}.get(kind, 0)
    past = [p[:, :, 6:, off:off + hd] for p in past]
    if kind not in ("view", "unaligned"):
        past = [p.contiguous() for p in past]
    cos, sin = (x.cuda() for x in om.rope_tables(hd, 600))
    start = hist + 3
    bufs = [torch.full((b, hkv, hist + t, hd), 7.0, dtype=dtype, device="cuda") for _ in range(2)]
    outs = [torch.full((b, hkv, keep, hd), 9.0, dtype=dtype, device="cuda") for _ in range(2)]
    qkv1 = qkv.clone()
    K.rope_kv_append(qkv1[:, :, :h], qkv1[:, :, h:h + hkv], qkv1[:, :, h + hkv:], cos, sin, start, *bufs, hist,
                     history=tuple(past) if hist else None, out=tuple(outs))
    q, k, v = qkv[:, :, :h], qkv[:, :, h:h + hkv], qkv[:, :, h + hkv:]
    rot = lambda x: om.apply_rope(x.transpose(1, 2).cpu(), *(c[start:start + t].cpu() for c in (cos, sin)))
    assert torch.equal(qkv1[:, :, :h].transpose(1, 2).cpu(), rot(q))
    full = [torch.cat((p.expand(b, -1, -1, -1).to(dtype).cpu(), new), 2)
            for p, new in zip(past, (rot(k), v.transpose(1, 2).cpu()))]
    for buf, out, want in zip(bufs, outs, full):
        assert torch.equal(buf.cpu(), want[:, :, -(hist + t):])
        assert torch.equal(out.cpu(), want[:, :, -keep:])
