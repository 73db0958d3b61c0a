"""The GEMMs that load their operands straight into LDS (qe_op_gemm_bf16) at the edges of their
tiles: every k-sliced tile (16 x 16 .. 64 x 128) and every wide one (64 x 128, 64 x 192, 128 x 128,
128 x 192, 128 x 256, and the first two with rings of two slots), both sides of the choice between the two kernels, ragged rows and columns, k of one 32-deep step, an odd number of steps,
fewer 64-deep blocks than waves, and an output whose rows are not 16-byte aligned."""
import numpy as np
import pytest

import qe

pytestmark = pytest.mark.gpu

SHAPES = [
    # k-sliced: 16 x 16, 16 x 32, 32 x 32, 32 x 48, 32 x 64, 48 x 64, 64 x 64, 64 x 128
    (1, 2, 32), (1, 6, 96), (16, 512, 64), (17, 514, 1056), (9, 6144, 1024), (33, 1026, 2048), (130, 1024, 3072),
    (64, 6144, 1024), (333, 1022, 544), (511, 1024, 2048), (130, 4094, 1024), (257, 2048, 480), (200, 4096, 96),
    # k-sliced, up to 8 rows (half an A tile) on 16 x 16, 16 x 32 and 16 x 128, the last on ragged columns
    (8, 1024, 3072), (3, 1022, 96), (7, 6146, 1056), (5, 80002, 288), (8, 65538, 32),
    # k-sliced over many columns: 16 x 128, 32 x 128, 48 x 128, 64 x 128
    (12, 70002, 288), (24, 40002, 96), (40, 40002, 96), (64, 40002, 64),
    # the longest K on a wide tile of one round, the shortest on the k-sliced kernel's 64 x 128
    (512, 4094, 1984), (512, 4094, 2048),
    # wide
    (65, 12290, 64), (449, 4096, 192), (512, 6144, 1024), (513, 6142, 576), (1025, 6146, 640), (2047, 4098, 576),
    # two workgroups a CU over a short k: 64 x 128 and 64 x 192
    (2000, 5110, 64), (1025, 7426, 512), (1500, 6144, 512), (2047, 8194, 64),
    # wide with a half stage at the end (k no multiple of 64), from the only one to one past the ring
    (449, 4096, 32), (449, 4096, 288), (512, 6144, 32), (512, 6144, 416), (513, 6142, 544), (1025, 6146, 1056),
    (2047, 4098, 608), (2000, 5110, 32), (2000, 5110, 96), (1500, 6144, 32), (1500, 6144, 160),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("shift", [0, 1])
def test_gemm_tiles_match_float64(gpu, m, n, k, shift):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n + k)
    a = torch.randn(m, k, generator=g, device="cuda")
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.05).bfloat16()
    buf = torch.full((m * n + 8,), float("nan"), device="cuda")
    c = buf[shift:shift + m * n].view(m, n)  # shift 1: 4-byte aligned only
    qe.op_gemm_bf16(a, w, c)
    torch.cuda.synchronize()
    ref = a.double() @ w.double().T
    # a is split into two bf16 halves (|error| <= 2^-17 |a|); f32 accumulation over k terms
    bound = (2.0 ** -16 + k * 2.0 ** -24) * (a.abs().double() @ w.abs().double().T) + 1e-30
    assert bool(((c.double() - ref).abs() <= bound).all())
    assert bool(torch.isnan(buf[:shift]).all()) and bool(torch.isnan(buf[shift + m * n:]).all())  # nothing past it


@pytest.mark.parametrize("m", [33, 48, 64])
def test_verify_of_many_rows_matches_decode(gpu, tiny_ckpt, m):
    """k tokens in one pass (norm, silu and residual epilogues of the k-sliced GEMM past 32 rows)
    against the same tokens one by one"""
    model = qe.Model.load_model(tiny_ckpt)
    V = model.config().vocab_size
    ids = qe.random_prompt(83, 20 + m, V)
    c1, c2 = qe.KVCache(model, 20 + m), qe.KVCache(model, 20 + m)
    model.prefill(ids[:20], 0, c1, want_logits=False)
    model.prefill(ids[:20], 0, c2, want_logits=False)
    rows = model.verify(ids[20:], 20, c1)
    for i in range(m):
        assert np.max(np.abs(rows[i] - model.forward(int(ids[20 + i]), 20 + i, c2))) < 1e-3, f"row {i}"
