"""Chunks of more than 64 tokens: their GEMMs on split rows (norm, attention and SwiGLU outputs held
as bf16 halves) against the same prompt token by token, at ragged rows, odd numbers of 64-deep
stages, a last column tile that holds one of its two heads, and widths that are no multiple of 64
(the k-sliced GEMMs up to 576 rows of "half_stages", then a half stage at the end of every product).
tests/test_gemm_choice.py holds the cases against the tiles that the products of a chunk run on."""
import numpy as np
import pytest

import qe

pytestmark = pytest.mark.gpu

CONFIGS = {
    "tiny": qe.Config(256, 512, 2, 4, 2, 128, 1000, 1e-6, 1e6, 999),
    "odd_stages": qe.Config(320, 448, 2, 4, 4, 128, 1000, 1e-6, 1e6, 999),
    "half_stage": qe.Config(288, 480, 2, 4, 2, 128, 1000, 1e-6, 1e6, 999),
    "half_stages": qe.Config(288, 2080, 2, 4, 2, 128, 1000, 1e-6, 1e6, 999),
    "93_heads": qe.Config(256, 512, 1, 31, 31, 128, 1000, 1e-6, 1e6, 999),
    # few layers and narrow rows, with the numbers of columns that make each product take its larger tiles
    "k192": qe.Config(192, 1024, 1, 8, 4, 128, 1000, 1e-6, 1e6, 999),
    "k256": qe.Config(256, 1536, 1, 16, 8, 128, 1000, 1e-6, 1e6, 999),
    "wide_mlp": qe.Config(64, 3072, 1, 4, 2, 128, 1000, 1e-6, 1e6, 999),
    "half_mlp": qe.Config(96, 3104, 1, 4, 2, 128, 1000, 1e-6, 1e6, 999),
    "half_mlp_16": qe.Config(96, 3104, 1, 16, 8, 128, 1000, 1e-6, 1e6, 999),
    "half_mlp_2080": qe.Config(96, 2080, 1, 16, 8, 128, 1000, 1e-6, 1e6, 999),
    "half_mlp_4064": qe.Config(96, 4064, 1, 4, 2, 128, 1000, 1e-6, 1e6, 999),
    "half_down": qe.Config(2080, 1056, 1, 4, 2, 128, 1000, 1e-6, 1e6, 999),
}

CASES = [  # (config, tokens in one chunk, cache)
    ("tiny", 65, "f32"), ("tiny", 129, "bf16"), ("tiny", 1025, "f32"), ("odd_stages", 200, "f32"),
    ("half_stage", 150, "f32"), ("half_stages", 576, "f32"), ("half_stages", 577, "f32"),
    ("half_stages", 1100, "bf16"), ("half_stages", 2047, "f32"), ("93_heads", 2001, "f32"),
    ("k192", 1100, "f32"), ("k256", 1100, "f32"), ("wide_mlp", 700, "f32"), ("wide_mlp", 1100, "bf16"),
    ("half_mlp", 400, "f32"), ("half_mlp_16", 513, "f32"), ("half_mlp_2080", 1100, "f32"),
    ("half_mlp_4064", 700, "f32"), ("half_down", 1300, "f32"), ("half_down", 1500, "f32"), ("half_down", 2000, "f32"),
]


@pytest.mark.parametrize("name,n,kv", CASES)
def test_chunk_matches_token_by_token(gpu, tmp_path, name, n, kv):
    model = qe.Model.load_model(qe.write_random_checkpoint(str(tmp_path), 7, CONFIGS[name]))
    dtype = qe.QE_KV_BF16 if kv == "bf16" else qe.QE_KV_F32
    ids = qe.random_prompt(5, n, 1000)
    a, b = qe.KVCache(model, n + 4, dtype), qe.KVCache(model, n + 4, dtype)
    got, ref = model.prefill_batch(ids, 0, a, chunk=2048), model.prefill(ids, 0, b)
    # 16-bit mantissas in the products against f32 ones, as the other chunk tests; a bf16 cache's
    # rows next to a rounding boundary fall to either side (2^-8 of a value, averaged over n keys)
    tol = 1e-3 if kv == "f32" else 1e-2
    assert np.max(np.abs(got - ref)) < tol
    for i in range(2):  # the K/V rows of every position are what the next steps attend to
        d = np.max(np.abs(model.forward(int(ids[i]), n + i, a) - model.forward(int(ids[i]), n + i, b)))
        assert d < tol, f"step {i}: {d}"


# chunks whose attention launch appends their K/V rows (33 and 64 tokens), chunks on the k-sliced GEMMs with
# k_qk_rope (widths that are no multiple of 64), and chunks on split rows with a half stage
@pytest.mark.parametrize("name,n,chunk", [("tiny", 500, 33), ("tiny", 600, 64), ("half_stage", 600, 64),
                                          ("half_stage", 600, 96), ("half_stage", 700, 128), ("half_stages", 2000, 640)])
def test_streams_change_no_result(gpu, tmp_path, monkeypatch, name, n, chunk):
    path = qe.write_random_checkpoint(str(tmp_path), 7, CONFIGS[name])
    ids = qe.random_prompt(5, n, 1000)

    def run(streams):
        monkeypatch.setenv("QE_PREFILL_STREAMS", streams)  # read when the model loads
        model = qe.Model.load_model(path)
        cache = qe.KVCache(model, n + 2)
        return model.prefill_batch(ids, 0, cache, chunk=chunk), model.forward(int(ids[0]), n, cache)

    one = run("1")
    for streams in ("2", "3", "4"):
        for got, want in zip(run(streams), one):
            np.testing.assert_array_equal(got, want, err_msg=f"{streams} streams")
