"""qe_op_attention's single launch over a short context: every number of passes, positions on both sides
of a pass and of the longest context it takes, one and two q heads per KV head, rows past the context
that hold NaN, and an output that overwrites q (which takes the runs)."""
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
