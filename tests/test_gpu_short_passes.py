"""Short verify passes: what they multiply in, and the way of their logits to the host.
Passes of 3 and 4 rows multiply in f32 as a decode step does: what they compute differs from
the same tokens one by one by f32 sums in another order, not by activations held as bf16 halves (gate|up
of 4 rows and the attention of 3 run on the matrix cores, so the checkpoints leave those out of what is
compared)."""
import json

import numpy as np
import pytest

import qe

pytestmark = pytest.mark.gpu

CFG = qe.Config(256, 512, 2, 4, 2, 128, 1000, 1e-6, 1e6, 999)


def load(path, edits):
    """the seeded checkpoint with edits: tensor name -> bf16 bits by a function of them"""
    file = qe.write_random_checkpoint(str(path), 7, CFG)
    raw = np.memmap(file, dtype=np.uint8, mode="r+")
    n = int(raw[:8].view(np.uint64)[0])
    for name, t in json.loads(bytes(raw[8:8 + n])).items():
        for part, f in edits.items():
            if part in name:
                a, b = t["data_offsets"]
                bits = raw[8 + n + a:8 + n + b].view(np.uint16)
                bits[:] = f(bits)
    raw.flush()
    del raw
    return qe.Model.load_model(file)


def times16(bits):  # attention's part of the residual is most of it
    return bits + np.uint16(4 << 7)


def zero(bits):
    return np.uint16(0)


def rel(x, y):
    return float(np.linalg.norm(x - y) / np.linalg.norm(y))


# f32 sums of up to 512 products and f32 softmax in two layers: 2e-7 measured over three seeds;
# activations held in 16 bits (2^-17 each) give 1.4e-6 to 2.8e-6
BOUND = 6e-7


def test_four_rows_project_in_f32(gpu, tmp_path):
    model = load(tmp_path, {"down_proj": zero, "o_proj": times16})
    ids = qe.random_prompt(5, 5, 1000)
    a, b = qe.KVCache(model, 8), qe.KVCache(model, 8)
    rows = model.verify(ids[:4], 0, a)
    for i in range(4):
        assert rel(rows[i], model.forward(int(ids[i]), i, b)) < BOUND, f"row {i}"
    assert rel(model.forward(int(ids[4]), 4, a), model.forward(int(ids[4]), 4, b)) < BOUND


def test_three_rows_project_in_f32(gpu, tmp_path):
    # the second layer's K/V rows come from the first layer's MLP alone
    model = load(tmp_path, {"layers.0.self_attn.o_proj": zero, "layers.1.self_attn.o_proj": times16})
    ids = qe.random_prompt(5, 4, 1000)
    a, b = qe.KVCache(model, 8), qe.KVCache(model, 8)
    model.verify(ids[:3], 0, a)
    for i in range(3):
        model.forward(int(ids[i]), i, b)
    assert rel(model.forward(int(ids[3]), 3, a), model.forward(int(ids[3]), 3, b)) < BOUND


@pytest.mark.parametrize("k", [1, 4, 5, 33, 64])
def test_logits_arrive_whole_in_pageable_and_pinned_memory(gpu, tmp_path, k):
    """40,002 logits a row: one, two, nine and sixteen pieces (the slots taken again) through pinned slots into
    pageable memory; pinned memory is written directly"""
    import ctypes

    import torch
    V = 40002
    model = qe.Model.load_model(qe.write_random_checkpoint(str(tmp_path), 7, qe.Config(256, 512, 1, 2, 2, 128, V, 1e-6,
                                                                                       1e6, 999)))
    ids = np.ascontiguousarray(qe.random_prompt(5, k, V))
    cache = qe.KVCache(model, k)
    pinned = torch.full((k * V + 1,), float("nan"), pin_memory=True)
    paged = np.full(k * V + 1, np.nan, dtype=np.float32)
    for at in (pinned.data_ptr(), paged.ctypes.data):
        qe._check(qe.lib().qe_verify(model._h, ids.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), k, 0, cache._h,
                                     ctypes.cast(at, ctypes.POINTER(ctypes.c_float))))
    np.testing.assert_array_equal(paged, pinned.numpy())
    assert np.isfinite(paged[:-1]).all() and np.isnan(paged[-1])


@pytest.mark.parametrize("hidden", [1024, 1056])
@pytest.mark.parametrize("k", [4, 5, 6, 7])
def test_rows_on_both_sides_of_the_residual_rule(gpu, tmp_path, hidden, k):
    """o_proj and down of 5 and 6 rows: the matvec up to 1024 weight rows, the GEMM past that"""
    model = qe.Model.load_model(qe.write_random_checkpoint(str(tmp_path), 7, qe.Config(hidden, 512, 2, 4, 2, 128, 1000,
                                                                                       1e-6, 1e6, 999)))
    ids = qe.random_prompt(5, 20 + k, 1000)
    a, b = qe.KVCache(model, 20 + k), qe.KVCache(model, 20 + k)
    for c in (a, b):
        model.prefill(ids[:20], 0, c, want_logits=False)
    rows = model.verify(ids[20:], 20, a)
    for i in range(k):  # activations in 16 bits, two layers and the lm_head: some 2^-17 each
        assert rel(rows[i], model.forward(int(ids[20 + i]), 20 + i, b)) < 4e-5, f"row {i}"


def test_single_rows_at_eight_q_heads_per_kv_head(gpu, tmp_path):
    """a verify of one token, and a chunk's last token alone, where its 8 q heads are all rows of a KV head"""
    model = qe.Model.load_model(qe.write_random_checkpoint(str(tmp_path), 7, qe.Config(256, 512, 1, 8, 1, 128, 1000,
                                                                                       1e-6, 1e6, 999)))
    ids = qe.random_prompt(5, 66, 1000)
    a, b = qe.KVCache(model, 66), qe.KVCache(model, 66)
    assert rel(model.prefill_batch(ids[:65], 0, a, chunk=64), model.prefill(ids[:65], 0, b)) < 4e-5
    assert rel(model.verify(ids[65:], 65, a)[0], model.forward(int(ids[65]), 65, b)) < 4e-5
