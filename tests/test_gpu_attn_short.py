"""qe_op_attention's single launch over a short context: every number of passes, positions on both sides
of a pass and of the longest context it takes, one and two q heads per KV head, rows past the context
that hold NaN, and an output that overwrites q, or rows of k or v in use (which takes the runs)."""
import numpy as np
import pytest

import qe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_pos", [1, 7, 63, 64, 65, 128, 129, 191, 255, 256, 257])
@pytest.mark.parametrize("n_heads,n_kv", [(16, 8), (3, 3), (2, 1), (8, 2)])
@pytest.mark.parametrize("in_place", [False, True])
def test_short_context_matches_float64(gpu, n_pos, n_heads, n_kv, in_place):
    import torch
    g = torch.Generator().manual_seed(n_pos * 100 + n_heads)
    q, stride = torch.randn(n_heads, 128, generator=g), n_pos + 3
    k, v = torch.randn(n_kv, stride, 128, generator=g), torch.randn(n_kv, stride, 128, generator=g)
    k[:, n_pos:], v[:, n_pos:] = float("nan"), float("nan")
    qd, kd, vd = q.reshape(-1).cuda(), k.cuda(), v.cuda()
    out = qd if in_place else torch.empty_like(qd)
    work = torch.empty(qe.op_attention_work_bytes(n_heads, n_kv, n_pos), dtype=torch.uint8, device="cuda")
    qe.op_attention(qd, kd, vd, out, n_pos, n_heads, n_kv, work)
    torch.cuda.synchronize()
    qq = q.double().view(n_kv, n_heads // n_kv, 128)
    s = torch.softmax(qq @ k[:, :n_pos].double().transpose(1, 2) / np.sqrt(128.0), -1)
    ref = (s @ v[:, :n_pos].double()).reshape(-1)
    # f32 scores of 128 products (|s| < 8: 2^-19 absolute), weights and sums of n_pos terms
    assert float((out.cpu().double() - ref).abs().max()) < 2e-5


@pytest.mark.parametrize("n_pos", [64, 200, 256])
@pytest.mark.parametrize("over,row", [("k", 0), ("k", -1), ("v", 0), ("v", -1)])
def test_out_over_rows_in_use_equals_out_apart(gpu, n_pos, over, row):
    """out over the first used rows of the cache, or over its end (partly past the used rows): the merge
    writes it after every read of k and v, so the result is the runs' own, bit for bit"""
    import torch
    n_heads, n_kv = 16, 8
    g = torch.Generator().manual_seed(n_pos)
    q, stride = torch.randn(n_heads * 128, generator=g).cuda(), n_pos + 3
    k, v = (torch.randn(n_kv, stride, 128, generator=g).cuda() for _ in range(2))
    work = torch.empty(qe.op_attention_work_bytes(n_heads, n_kv, n_pos), dtype=torch.uint8, device="cuda")
    want = torch.empty_like(q)
    qe.op_attention(q, k, v, want, n_pos, n_heads, n_kv, work, n_splits=(n_pos + 63) // 64)
    flat = {"k": k, "v": v}[over].view(-1)
    out = flat[:n_heads * 128] if row == 0 else flat[-n_heads * 128:]
    qe.op_attention(q, k, v, out, n_pos, n_heads, n_kv, work)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
