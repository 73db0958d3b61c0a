"""The engine's measured work: single calls of its device ops and whole calls of the model.

Shapes are those of the Qwen3-0.6B architecture the engine serves (hidden 1024, 16 query heads over
8 KV heads of 128, SwiGLU 3072, vocabulary 151,936, 28 layers) with seeded random-init weights, as
the tests and bench.py use them. The model is loaded once and kept, as a program that serves it
does; every case has its own prompt and its own KV cache.

Kinds (a case's "kind"):
  matvec     one token through one projection (op_matvec_bf16)
  attention  one token's GQA attention over an f32 cache (op_attention)
  gemm       the token rows of a verify pass or a prefill chunk through one projection (op_gemm_bf16)
  verify     k tokens checked in one pass over a cached context (Model.verify)
  prefill    a prompt into an empty cache in chunks (Model.prefill_batch)
  decode     greedy decode over a cached context (Model.decode), then the next token's logits
             (Model.forward)
"""
import importlib
import json
import math
import os
import tempfile

import numpy as np
import torch

qe = importlib.import_module("mac-gpu-compiler_amd.qe")

CFG = qe.QWEN3_0_6B
WEIGHT_SEED = 20260101
D = CFG.head_dim
H, I, V = CFG.hidden_size, CFG.intermediate_size, CFG.vocab_size
NH, NKV, L = CFG.num_attention_heads, CFG.num_key_value_heads, CFG.num_hidden_layers
LAYER_WEIGHTS = H * (NH + 2 * NKV) * D + NH * D * H + 3 * H * I  # elements of one layer's matrices

# (rows, columns) of the projections: q|k|v, o_proj, gate|up, down
PROJECTIONS = [((NH + 2 * NKV) * D, H), (H, NH * D), (2 * I, H), (H, I)]


def listed():
    return [
        # one decode token through o_proj: the smallest weight product of a step
        dict(name="matvec_o_proj", kind="matvec", rows=H, cols=NH * D),
        # one decode token's attention a little past a 130-token prompt, and in a long chat
        dict(name="attention_197", kind="attention", n_pos=197),
        dict(name="attention_4225", kind="attention", n_pos=4225),
        # gate|up of a verify pass with 8 drafts
        dict(name="gemm_verify_9", kind="gemm", m=9, n=2 * I, k=H),
        # down of a 130-token prompt
        dict(name="gemm_prompt_130", kind="gemm", m=130, n=H, k=I),
        # gate|up of a default prefill chunk, and q|k|v of the largest chunk
        dict(name="gemm_chunk_512", kind="gemm", m=512, n=2 * I, k=H),
        dict(name="gemm_chunk_2048", kind="gemm", m=2048, n=(NH + 2 * NKV) * D, k=H),
        # speculative decoding: 3 drafts after a long prompt; lookup's default 4 drafts in a chat
        dict(name="verify_4_at_2048", kind="verify", rows=4, pos=2048, kv="f32"),
        dict(name="verify_5_at_700", kind="verify", rows=5, pos=700, kv="f32"),
        # a prompt of ordinary, odd length into the small cache type
        dict(name="prefill_333_bf16", kind="prefill", n=333, chunk=0, kv="bf16"),
        # a long prompt in default chunks
        dict(name="prefill_2048", kind="prefill", n=2048, chunk=512, kv="f32"),
        # the headline workload: 128 greedy steps after a 130-token prompt
        dict(name="decode_128_at_130", kind="decode", steps=128, pos=130, kv="f32"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["matvec", "attention", "gemm", "gemm", "gemm", "verify", "verify", "prefill", "prefill",
                       "decode"])
    kv = rng.choice(["f32", "f32", "bf16"])
    if kind == "matvec":
        return dict(kind=kind, rows=_log_int(rng, 128, V), cols=8 * _log_int(rng, 32, 384))
    if kind == "attention":
        return dict(kind=kind, n_pos=_log_int(rng, 16, 32768))
    if kind == "gemm":
        m = _log_int(rng, 2, 2048)
        if rng.random() < 0.6:
            n, k = rng.choice(PROJECTIONS)
        else:
            n, k = 2 * _log_int(rng, 128, I), 64 * rng.randint(4, 48)
        return dict(kind=kind, m=m, n=n, k=k)
    if kind == "verify":
        return dict(kind=kind, rows=_log_int(rng, 2, 64), pos=_log_int(rng, 32, 4096), kv=kv)
    if kind == "prefill":
        return dict(kind=kind, n=_log_int(rng, 33, 2048), chunk=rng.choice([0, 0, 128, 256, 1024, 2048]), kv=kv)
    pos = _log_int(rng, 16, 4096)
    return dict(kind=kind, steps=rng.randint(8, 128 if pos <= 1024 else 48), pos=pos, kv=kv)


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
_model = None
_weights = None  # the same checkpoint's matrices for exact()


def _with_checkpoint(use):
    with tempfile.TemporaryDirectory(prefix="qe_cases_") as d:
        return use(qe.write_random_checkpoint(d, WEIGHT_SEED, CFG))


def _the_model():
    global _model
    if _model is None:
        _model = _with_checkpoint(qe.Model.load_model)
    return _model


def _ids(case, seed, n):
    rng = np.random.default_rng([seed, case.get("pos", 0), case.get("n", 0)])
    return rng.integers(0, V, size=n, dtype=np.uint32)


def _op_inputs(case, seed):
    """The op's tensors, made on the host so that they depend on the seed alone."""
    g = torch.Generator().manual_seed((seed * 1000003 + 17) % (1 << 62))

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g) * std

    if case["kind"] == "matvec":  # normalized activations, N(0, 0.02) weights
        return normal(case["cols"]), normal(case["rows"], case["cols"], std=0.02).bfloat16()
    if case["kind"] == "gemm":
        return normal(case["m"], case["k"]), normal(case["n"], case["k"], std=0.02).bfloat16()
    # normalized and rotated q and k; v as a projection of a normalized row; a cache with room left
    stride = case["n_pos"] + 64
    return normal(NH * D), normal(NKV, stride, D), normal(NKV, stride, D, std=0.02 * math.sqrt(H))


def _kv_type(case):
    return qe.QE_KV_BF16 if case["kv"] == "bf16" else qe.QE_KV_F32


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "gemm"):
        x, w = (t.cuda() for t in _op_inputs(case, seed))
        out = torch.empty(*x.shape[:-1], w.shape[0], device="cuda")
        return dict(kind=kind, x=x, w=w, out=out)
    if kind == "attention":
        q, k, v = (t.cuda() for t in _op_inputs(case, seed))
        work = torch.empty(qe.op_attention_work_bytes(NH, NKV, case["n_pos"]), dtype=torch.uint8, device="cuda")
        return dict(kind=kind, q=q, k=k, v=v, out=torch.empty(NH * D, device="cuda"), n_pos=case["n_pos"], work=work)
    m = _the_model()
    st = dict(kind=kind, model=m)
    if kind == "prefill":
        st.update(ids=_ids(case, seed, case["n"]), chunk=case["chunk"], kv=qe.KVCache(m, case["n"] + 64, _kv_type(case)))
        return st
    more = case["rows"] if kind == "verify" else case["steps"] + 1
    ids = _ids(case, seed, case["pos"] + more)
    kv = qe.KVCache(m, case["pos"] + more + 64, _kv_type(case))
    m.prefill_batch(ids[:case["pos"]], 0, kv, want_logits=False)
    st.update(kv=kv, pos=case["pos"])
    if kind == "verify":
        st.update(ids=ids[case["pos"]:])
    else:
        st.update(first=int(ids[case["pos"]]), steps=case["steps"])
    return st


def run(st):
    kind = st["kind"]
    if kind == "matvec":
        qe.op_matvec_bf16(st["w"], st["x"], st["out"])
        return st["out"]
    if kind == "gemm":
        qe.op_gemm_bf16(st["x"], st["w"], st["out"])
        return st["out"]
    if kind == "attention":
        qe.op_attention(st["q"], st["k"], st["v"], st["out"], st["n_pos"], NH, NKV, st["work"])
        return st["out"]
    if kind == "prefill":
        return st["model"].prefill_batch(st["ids"], 0, st["kv"], chunk=st["chunk"])
    if kind == "verify":
        return st["model"].verify(st["ids"], st["pos"], st["kv"])
    toks, _ = st["model"].decode(st["first"], st["pos"], st["steps"], st["kv"])
    logits = st["model"].forward(toks[-1], st["pos"] + st["steps"], st["kv"])
    return dict(tokens=np.asarray(toks, dtype=np.int64), logits=logits)


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "matvec":
        r, c = case["rows"], case["cols"]
        return dict(bytes=2 * r * c + 4 * (r + c), flops=2 * r * c)
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(bytes=4 * m * k + 2 * n * k + 4 * m * n, flops=2 * m * n * k)
    if kind == "attention":
        n = case["n_pos"]
        return dict(bytes=2 * NKV * n * D * 4 + 2 * NH * D * 4, flops=4 * NH * n * D)
    el = 2 if case["kv"] == "bf16" else 4
    row = 2 * L * NKV * D * el  # one position's K and V
    layers, head = 2 * L * LAYER_WEIGHTS, 2 * V * H

    def attend(first, count):  # flops of `count` tokens from position `first`
        return sum(4 * NH * D * (first + i + 1) for i in range(count)) * L

    if kind == "prefill":
        n = case["n"]
        return dict(bytes=layers + head + n * (row + 2 * H) + 4 * V,
                    flops=2 * n * L * LAYER_WEIGHTS + attend(0, n) + 2 * H * V)
    if kind == "verify":
        r, p = case["rows"], case["pos"]
        return dict(bytes=layers + head + (p + r) * row + r * (2 * H + 4 * V),
                    flops=2 * r * (L * LAYER_WEIGHTS + H * V) + attend(p, r))
    s, p = case["steps"] + 1, case["pos"]
    return dict(bytes=s * (layers + head + 2 * H) + row * sum(p + i + 1 for i in range(s)) + 4 * V,
                flops=2 * s * (L * LAYER_WEIGHTS + H * V) + attend(p, s))


def tolerance(case):
    """About four times what each path shows against exact()."""
    if case.get("kv") == "bf16":  # K/V rows next to a rounding boundary fall to either side: 8.6e-4
        return {"rel": 4e-3}
    return {
        "matvec": {"rel": 5e-7},     # f32 sums of up to 3072 products: 1e-7
        "attention": {"rel": 1e-6},  # f32 scores, softmax and sums: 2e-7
        "gemm": {"rel": 1e-5},       # f32 rows as two bf16 halves, f32 sums: 2.5e-6
        "verify": {"rel": 4e-5},     # 28 layers of both, the logits: 1e-5
        "prefill": {"rel": 4e-5},
        "decode": {"rel": 4e-5},
    }[case["kind"]]


# ---------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _read_checkpoint(path):
    """name -> float64 matrix of a safetensors file of bf16 tensors"""
    raw = np.memmap(path, dtype=np.uint8, mode="r")
    n = int(raw[:8].view(np.uint64)[0])
    out = {}
    for name, t in json.loads(bytes(raw[8:8 + n])).items():
        if name == "__metadata__":
            continue
        a, b = t["data_offsets"]
        bits = torch.from_numpy(np.array(raw[8 + n + a:8 + n + b]).view(np.int16)).view(torch.bfloat16)
        out[name] = bits.reshape(t["shape"]).to(_dev())
    return out


def _rms(x, gain):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + CFG.rms_norm_eps) * gain


def _rope(x, pos):
    """x [n, heads, D] at positions pos..: angles are the f32 products of the engine's definition"""
    i = np.arange(D // 2, dtype=np.float64)
    freq = np.power(np.float64(np.float32(CFG.rope_theta)), -2.0 * i / D).astype(np.float32)
    ang = np.arange(pos, pos + x.shape[0], dtype=np.float32)[:, None] * freq[None, :]
    ang = torch.from_numpy(ang.astype(np.float64)).to(x.device)[:, None, :]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


class _Exact:
    """The decoder in float64; the cache holds what its type holds (bf16: rounded rows)."""

    def __init__(self, kv, cap):
        global _weights
        if _weights is None:
            _weights = _with_checkpoint(_read_checkpoint)
        self.w, self.kv = _weights, kv
        self.cache = torch.zeros(2, L, NKV, cap, D, dtype=torch.float64, device=_dev())

    def __call__(self, ids, pos, last):
        """ids at positions pos..; the logits of the last `last` of them"""
        def mat(name):
            return self.w[name].double()

        n = len(ids)
        x = self.w["model.embed_tokens.weight"][torch.from_numpy(np.asarray(ids, np.int64)).to(_dev())].double()
        for l in range(L):
            p = f"model.layers.{l}."
            h = _rms(x, mat(p + "input_layernorm.weight"))
            q = (h @ mat(p + "self_attn.q_proj.weight").T).view(n, NH, D)
            k = (h @ mat(p + "self_attn.k_proj.weight").T).view(n, NKV, D)
            v = (h @ mat(p + "self_attn.v_proj.weight").T).view(n, NKV, D)
            q = _rope(_rms(q, mat(p + "self_attn.q_norm.weight")), pos)
            k = _rope(_rms(k, mat(p + "self_attn.k_norm.weight")), pos)
            if self.kv == "bf16":
                k, v = k.float().bfloat16().double(), v.float().bfloat16().double()
            self.cache[0, l, :, pos:pos + n] = k.transpose(0, 1)
            self.cache[1, l, :, pos:pos + n] = v.transpose(0, 1)
            kk, vv = self.cache[0, l, :, :pos + n], self.cache[1, l, :, :pos + n]
            seen = torch.arange(pos + n, device=x.device)[None, :] <= pos + torch.arange(n, device=x.device)[:, None]
            att = torch.empty(n, NH, D, dtype=torch.float64, device=x.device)
            for j in range(NH):
                s = (q[:, j] @ kk[j * NKV // NH].T) / math.sqrt(D)
                att[:, j] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ vv[j * NKV // NH]
            x = x + att.reshape(n, NH * D) @ mat(p + "self_attn.o_proj.weight").T
            h = _rms(x, mat(p + "post_attention_layernorm.weight"))
            gate = h @ mat(p + "mlp.gate_proj.weight").T
            h = gate * torch.sigmoid(gate) * (h @ mat(p + "mlp.up_proj.weight").T)
            x = x + h @ mat(p + "mlp.down_proj.weight").T
        x = _rms(x[n - last:], mat("model.norm.weight"))
        return (x @ mat("lm_head.weight").T).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "gemm"):
        x, w = (t.to(_dev()).double() for t in _op_inputs(case, seed))
        return x @ w.T
    if kind == "attention":
        q, k, v = (t.to(_dev()).double() for t in _op_inputs(case, seed))
        k, v = k[:, :case["n_pos"]], v[:, :case["n_pos"]]
        s = torch.einsum("gjd,gtd->gjt", q.view(NKV, NH // NKV, D), k) / math.sqrt(D)
        return torch.einsum("gjt,gtd->gjd", torch.softmax(s, -1), v).reshape(NH * D)
    if kind == "prefill":
        return _Exact(case["kv"], case["n"])(_ids(case, seed, case["n"]), 0, 1)[0]
    p = case["pos"]
    more = case["rows"] if kind == "verify" else case["steps"] + 1
    ids = _ids(case, seed, p + more)
    model = _Exact(case["kv"], p + more)
    if kind == "verify":
        return model(ids, 0, more)
    if _dev() == "cpu":
        return None  # 64-bit weights streamed once per step: minutes without a GPU
    model(ids[:p], 0, 1)
    toks, tok = [], int(ids[p])
    for i in range(case["steps"]):
        tok = int(np.argmax(model([tok], p + i, 1)[0]))
        toks.append(tok)
    return dict(tokens=np.asarray(toks, dtype=np.int64), logits=model([tok], p + case["steps"], 1)[0])
