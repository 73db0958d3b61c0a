"""Causal attention of a pass over cached keys (one tile of 64 positions to many, one run to many)
against the same tokens one by one: passes that normalize, rotate and append their own K/V rows in the
attention launch (up to 64 tokens) at the edges of tiles and token blocks, chunks of one and of two row
blocks per wave, and rows whose scores grow from tile to tile (the deferred rescale)."""
import json

import numpy as np
import pytest

import qe

pytestmark = pytest.mark.gpu

CONFIGS = {
    2: qe.Config(256, 512, 2, 4, 2, 128, 1000, 1e-6, 1e6, 999),
    1: qe.Config(256, 512, 1, 2, 2, 128, 1000, 1e-6, 1e6, 999),
    8: qe.Config(256, 512, 1, 8, 1, 128, 1000, 1e-6, 1e6, 999),
}


@pytest.mark.parametrize("group,n,start,kv", [
    (2, 5, 0, "f32"), (2, 5, 59, "f32"), (2, 6, 60, "bf16"), (2, 33, 31, "f32"), (2, 64, 64, "bf16"),
    (2, 64, 2100, "f32"), (2, 5, 2107, "bf16"), (1, 9, 120, "f32"), (8, 9, 127, "f32"), (8, 64, 1, "bf16"),
    (2, 65, 200, "f32"), (2, 500, 1, "bf16"), (2, 1023, 70, "f32"), (2, 1024, 70, "f32"), (8, 1100, 3, "bf16")])
def test_pass_matches_token_by_token(gpu, tmp_path, group, n, start, kv):
    model = qe.Model.load_model(qe.write_random_checkpoint(str(tmp_path), 11, CONFIGS[group]))
    dtype = qe.QE_KV_BF16 if kv == "bf16" else qe.QE_KV_F32
    ids = qe.random_prompt(5, start + n, 1000)
    a, b = qe.KVCache(model, start + n + 4, dtype), qe.KVCache(model, start + n + 4, dtype)
    if start:
        model.prefill(ids[:start], 0, a, want_logits=False)
        model.prefill(ids[:start], 0, b, want_logits=False)
    # 16-bit mantissas in the products against f32 ones, as the other chunk tests; a bf16 cache's
    # rows next to a rounding boundary fall to either side (2^-8 of a value, averaged over the keys)
    tol = 1e-3 if kv == "f32" else 1e-2
    if n <= 64:
        rows = model.verify(ids[start:], start, a)
        ref = np.stack([model.forward(int(t), start + i, b) for i, t in enumerate(ids[start:])])
        assert np.max(np.abs(rows - ref)) < tol
    else:
        got, ref = model.prefill_batch(ids[start:], start, a, chunk=2048), model.prefill(ids[start:], start, b)
        assert np.max(np.abs(got - ref)) < tol
    for i in range(2):  # the K/V rows of every position are what the next steps attend to
        at = start + n + i
        assert np.max(np.abs(model.forward(int(ids[i]), at, a) - model.forward(int(ids[i]), at, b))) < tol


def test_scores_that_grow_over_the_tiles(gpu, tmp_path):
    """q gains of 8: scores spread over some +-40 in base 2, so that rows pass their running maximum by
    more than 8 in later tiles"""
    path = qe.write_random_checkpoint(str(tmp_path), 11, CONFIGS[2])
    raw = np.memmap(path, dtype=np.uint8, mode="r+")
    n = int(raw[:8].view(np.uint64)[0])
    for name, t in json.loads(bytes(raw[8:8 + n])).items():
        if name.endswith("q_norm.weight"):
            a, b = t["data_offsets"]
            bits = raw[8 + n + a:8 + n + b].view(np.uint16)
            bits[:] = bits + np.uint16(3 << 7)  # bf16 x 8
    raw.flush()
    del raw
    model = qe.Model.load_model(path)
    ids = qe.random_prompt(9, 700, 1000)
    a, b, c = (qe.KVCache(model, 704, qe.QE_KV_F32) for _ in range(3))
    ref = model.prefill(ids, 0, a)
    # a score of 40 carries 2^-16 of itself: 6e-4 of each weight, on logits of order 1
    assert np.max(np.abs(model.prefill_batch(ids, 0, b) - ref)) < 5e-3
    model.prefill(ids[:640], 0, c, want_logits=False)
    rows = [model.verify(ids[640 + i:660 + i], 640 + i, c) for i in (0, 20, 40)]
    assert np.max(np.abs(rows[2][-1] - ref)) < 5e-3


def test_short_chunks_of_widths_that_only_the_matvec_takes(gpu, tmp_path):
    """hidden and intermediate sizes that are no multiple of 32: chunks of up to 3 tokens"""
    model = qe.Model.load_model(qe.write_random_checkpoint(str(tmp_path), 3, qe.Config(264, 520, 2, 4, 2, 128, 1000,
                                                                                      1e-6, 1e6, 999)))
    ids = qe.random_prompt(5, 21, 1000)
    a, b = qe.KVCache(model, 24), qe.KVCache(model, 24)
    assert np.max(np.abs(model.prefill_batch(ids, 0, a, chunk=3) - model.prefill(ids, 0, b))) < 1e-3
