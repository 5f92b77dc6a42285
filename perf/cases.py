"""The work that callers of this library have it do, as cases that can be timed and checked.

A case names an op family, its sizes and its storage types.  `prepare` makes what the
caller's program holds beforehand (activations, weights in the model file's formats, a
paged KV cache and its metadata), `run` makes one pass through the public entry points of
`nano_vllm_cpp_amd.ops`, and `exact` computes the same outputs in 64 bits with plain torch.

Families:
  chain   the per-layer ops around the GEMMs: embedding gather, residual-add + RMSNorm,
          (QK-norm +) RoPE on q and k, SwiGLU
  layer   the embedding and one whole decoder layer of a decode step, Q8_0 weights: norms,
          the four Q8_0 products, bias / QK-norm / RoPE / KV store, paged attention, SwiGLU
  q8      hip_matmul_q8 on activations: row quantizer and Q8_0 product
  matmul  hip_matmul / _u16 / _qk: fp32, fp16, bf16 and K-quant weights
  attn    paged attention of a prefill batch (or a decode batch) over a block table
  moe     routing and expert FFN of a mixture-of-experts layer
"""
from __future__ import annotations

import math

import numpy as np
import torch

from nano_vllm_cpp_amd import ops

DEV = "cuda"
TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
FORMATS = {"f32": ops.W_F32, "f16": ops.W_F16, "bf16": ops.W_BF16, "q4_k": ops.Q4_K, "q5_k": ops.Q5_K,
           "q6_k": ops.Q6_K}
BYTES_PER_WEIGHT = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q4_k": 144 / 256, "q5_k": 176 / 256, "q6_k": 210 / 256}
EPS, THETA, KV_BLOCK = 1e-6, 1e6, 256

# the decoder shapes of the repository's benchmark configurations
MODELS = {
    "qwen2.5-0.5b": dict(vocab=151936, hidden=896, inter=4864, q_heads=14, kv_heads=2, head_dim=64, qk_norm=False),
    "qwen2.5-7b": dict(vocab=152064, hidden=3584, inter=18944, q_heads=28, kv_heads=4, head_dim=128, qk_norm=False),
    "qwen3-8b": dict(vocab=151936, hidden=4096, inter=12288, q_heads=32, kv_heads=8, head_dim=128, qk_norm=True),
}
# Qwen3-30B-A3B's expert layer
EXPERTS = dict(hidden=2048, inter=768, experts=128, top=8)


def listed() -> list[dict]:
    return [
        # a short prompt on the smallest model: launches and latency
        dict(name="chain_64_0.5b", family="chain", model="qwen2.5-0.5b", tokens=64, dtype="f16"),
        # a full prefill chunk through the per-layer ops, with QK-norm
        dict(name="chain_8192_8b", family="chain", model="qwen3-8b", tokens=8192, dtype="bf16"),
        # interactive generation: one sequence, one new token, a long context
        dict(name="layer_decode_1", family="layer", model="qwen2.5-7b", seqs=1, context=4096, dtype="f16"),
        # a serving engine's decode step: 256 sequences of ragged contexts
        dict(name="layer_decode_256", family="layer", model="qwen2.5-7b", seqs=256, context=4096, dtype="f16"),
        # the widest product of a Q8_0 model's prefill, a ragged number of prompt tokens
        dict(name="q8_prefill_gate_up", family="q8", m=3977, n=37888, k=3584, dtype="f16"),
        # the widest product of an unquantized model's prefill
        dict(name="bf16_prefill_gate_up", family="matmul", m=4096, n=24576, k=4096, x="bf16", w="bf16"),
        # the LM head for a small decode batch
        dict(name="bf16_head_24", family="matmul", m=24, n=151936, k=4096, x="bf16", w="bf16"),
        # a Q4_K model's prefill of one odd-sized prompt
        dict(name="q4k_prefill_gate_up", family="matmul", m=1021, n=37888, k=3584, x="f16", w="q4_k"),
        # the same weights for one generated token
        dict(name="q4k_decode_gate_up", family="matmul", m=1, n=37888, k=3584, x="f16", w="q4_k"),
        # attention of a packed prefill of ragged prompts, 16-bit KV cache
        dict(name="attn_prefill_f16", family="attn", lens="4096,3001,2048,777", decode=False, q_heads=28, kv_heads=4,
             head_dim=128, dtype="f16"),
        # the same op on the reference's own dtype
        dict(name="attn_prefill_f32", family="attn", lens="3072,1531,700", decode=False, q_heads=28, kv_heads=4,
             head_dim=128, dtype="f32"),
        # an expert layer for a decode batch of 256 sequences
        dict(name="moe_256", family="moe", rows=256, x="bf16", w="bf16"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _products(rng, heads: bool) -> tuple[int, int]:
    """(n, k) of one of a decoder's weight matrices."""
    c = MODELS[rng.choice(sorted(MODELS))]
    qs, ks = c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    kinds = [(qs + 2 * ks, c["hidden"]), (c["hidden"], qs), (2 * c["inter"], c["hidden"]), (c["hidden"], c["inter"])]
    return rng.choice(kinds + ([(c["vocab"], c["hidden"])] if heads else []))


def draw(rng) -> dict:
    family = rng.choice(["chain", "layer", "q8", "matmul", "matmul", "matmul", "attn", "attn", "moe"])
    if family == "chain":
        return dict(family=family, model=rng.choice(sorted(MODELS)), tokens=_log_int(rng, 1, 6000),
                    dtype=rng.choice(["f32", "f16", "bf16"]))
    if family == "layer":
        return dict(family=family, model=rng.choice(sorted(MODELS)), seqs=_log_int(rng, 1, 256),
                    context=_log_int(rng, 64, 4096), dtype=rng.choice(["f16", "bf16"]))
    if family == "q8":
        n, k = _products(rng, False)
        return dict(family=family, m=_log_int(rng, 1, 3900), n=n, k=k, dtype=rng.choice(["f32", "f16", "bf16"]))
    if family == "matmul":
        x, w = rng.choice([("f16", "f16"), ("bf16", "bf16"), ("f32", "f16"), ("f32", "bf16"), ("f32", "f32"),
                           ("f16", "q4_k"), ("bf16", "q4_k"), ("f32", "q4_k"), ("f16", "q5_k"), ("f16", "q6_k"),
                           ("f32", "q6_k")])
        n, k = _products(rng, True)
        most = 6e11 if x == w and x != "f32" else 1.5e11  # operations: within the largest listed case's time
        return dict(family=family, m=_log_int(rng, 1, max(1, min(4000, int(most / (2.0 * n * k))))), n=n, k=k, x=x, w=w)
    if family == "attn":
        c = MODELS[rng.choice(["qwen2.5-7b", "qwen3-8b"])]
        decode = rng.random() < 0.5
        lens = [_log_int(rng, 64, 3000 if not decode else 4096) for _ in range(_log_int(rng, 1, 3 if not decode else 60))]
        return dict(family=family, lens=",".join(map(str, lens)), decode=decode, q_heads=c["q_heads"],
                    kv_heads=c["kv_heads"], head_dim=c["head_dim"], dtype=rng.choice(["f32", "f16", "bf16"]))
    return dict(family=family, rows=_log_int(rng, 1, 2048), x=rng.choice(["f32", "f16", "bf16"]),
                w=rng.choice(["f16", "bf16"]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype, mean: float = 0.0, std: float = 1.0) -> torch.Tensor:
    out = torch.empty(shape, dtype=dtype, device=DEV)
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 27):  # in pieces: no fp32 copy of a whole weight matrix
        part = flat[i:i + (1 << 27)]
        part.copy_(torch.randn(part.numel(), generator=g, device=DEV).mul_(std).add_(mean))
    return out


def _q8_weights(g, n: int, k: int, lo: float = 2e-4, hi: float = 1e-3) -> tuple[torch.Tensor, torch.Tensor]:
    """Q8_0 split planes: int8 values and one fp16 scale per 32 of them."""
    w8 = torch.randint(-127, 128, (n * k,), generator=g, device=DEV, dtype=torch.int8)
    return w8, torch.empty(n * k // 32, device=DEV).uniform_(lo, hi, generator=g).half().view(torch.int16)


def _fp16_bytes(g, blocks: int, lo: float, hi: float) -> torch.Tensor:
    return torch.empty(blocks, device=DEV).uniform_(lo, hi, generator=g).half().view(torch.uint8).view(blocks, 2)


def _kquant_weights(g, n: int, k: int, fmt: str) -> torch.Tensor:
    """K-quant superblocks of roughly zero-mean weights, as quantized model files hold them:
    w = d sc q - dmin mn with the minimum near the middle of the quants' range."""
    blocks = n * k // 256
    size = {"q4_k": 144, "q5_k": 176, "q6_k": 210}[fmt]
    blk = torch.randint(0, 256, (blocks, size), generator=g, device=DEV, dtype=torch.uint8)
    if fmt == "q6_k":  # [128 low nibbles][64 high bits][16 int8 scales][fp16 d]
        blk[:, 192:208] = torch.randint(-64, 64, (blocks, 16), generator=g, device=DEV, dtype=torch.int8).view(torch.uint8)
        blk[:, 208:210] = _fp16_bytes(g, blocks, 1e-5, 6e-5)
        return blk.view(-1)
    half = 8.0 if fmt == "q4_k" else 16.0
    d = torch.empty(blocks, device=DEV).uniform_(1e-4, 3e-4, generator=g) * (8.0 / half)
    sc = torch.randint(16, 60, (blocks, 8), generator=g, device=DEV, dtype=torch.int32)
    mn = sc + torch.randint(-4, 4, (blocks, 8), generator=g, device=DEV, dtype=torch.int32)
    blk[:, 0:2] = d.half().view(torch.uint8).view(blocks, 2)
    blk[:, 2:4] = (d * half).half().view(torch.uint8).view(blocks, 2)
    blk[:, 4:8] = ((sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
    blk[:, 8:12] = ((mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
    blk[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
    return blk.view(-1)


def _paged(g, seed: int, ctx, q_lens, kv_heads: int, head_dim: int, dtype) -> dict:
    """A paged KV cache of sequences that hold ctx[s] keys, and the metadata of a batch that
    queries the last q_lens[s] positions of each."""
    ctx, q_lens = np.asarray(ctx), np.asarray(q_lens)
    need = -(-ctx // KV_BLOCK)
    perm = np.random.default_rng(seed).permutation(int(need.sum())).astype(np.int32)
    table = np.full((len(ctx), int(need.max())), -1, np.int32)
    at = 0
    for s, nb in enumerate(need):
        table[s, :nb] = perm[at:at + nb]
        at += nb
    seq = np.repeat(np.arange(len(ctx)), q_lens)
    pos = np.concatenate([np.arange(c - n, c) for c, n in zip(ctx, q_lens)])
    slots = table[seq, pos // KV_BLOCK].astype(np.int64) * KV_BLOCK + pos % KV_BLOCK
    rows = int(need.sum()) * KV_BLOCK
    return dict(k_cache=_normal(g, (rows, kv_heads, head_dim), dtype),
                v_cache=_normal(g, (rows, kv_heads, head_dim), dtype),
                query_seq=torch.from_numpy(seq.astype(np.int32)).to(DEV),
                key_len=torch.from_numpy((pos + 1).astype(np.int32)).to(DEV),
                table=torch.from_numpy(table).to(DEV), slots=torch.from_numpy(slots.astype(np.int32)).to(DEV),
                positions=torch.from_numpy(pos.astype(np.int64)).to(DEV),
                cu=np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32), ctx=ctx, host_table=table)


def _contexts(case: dict) -> np.ndarray:
    """The decode batch's key counts: part of the case's shape, not of its inputs."""
    if case["seqs"] == 1:
        return np.array([case["context"]])
    return np.random.default_rng(case["seqs"]).integers(1, case["context"] + 1, case["seqs"])


def prepare(case: dict, seed: int) -> dict:
    g = _generator(seed)
    family = case["family"]
    if family == "chain":
        c, dt, t = MODELS[case["model"]], TYPES[case["dtype"]], case["tokens"]
        hd = c["head_dim"]
        w8, ws = _q8_weights(g, c["vocab"], c["hidden"])
        return dict(case=case, ids=torch.randint(0, c["vocab"], (t,), generator=g, device=DEV), w8=w8, ws=ws,
                    x=_normal(g, (t, c["hidden"]), dt), norm=_normal(g, (c["hidden"],), dt, 1.0, 0.1),
                    q=_normal(g, (t, c["q_heads"] * hd), dt), k=_normal(g, (t, c["kv_heads"] * hd), dt),
                    q_w=_normal(g, (hd,), dt, 1.0, 0.1) if c["qk_norm"] else None,
                    k_w=_normal(g, (hd,), dt, 1.0, 0.1) if c["qk_norm"] else None,
                    positions=torch.arange(t, device=DEV), inv_freq=ops.rope_inv_freq(THETA, hd, DEV),
                    gate_up=_normal(g, (t, 2 * c["inter"]), dt))
    if family == "layer":
        c, dt, t = MODELS[case["model"]], TYPES[case["dtype"]], case["seqs"]
        hd, h, inter = c["head_dim"], c["hidden"], c["inter"]
        qs, ks = c["q_heads"] * hd, c["kv_heads"] * hd
        ctx = _contexts(case)
        s = dict(case=case, ids=torch.randint(0, c["vocab"], (t,), generator=g, device=DEV),
                 emb=_q8_weights(g, c["vocab"], h, 2e-3, 1e-2), qkv=_q8_weights(g, qs + 2 * ks, h),
                 o=_q8_weights(g, h, qs), gate_up=_q8_weights(g, 2 * inter, h), down=_q8_weights(g, h, inter),
                 w_in=_normal(g, (h,), dt, 1.0, 0.1), w_post=_normal(g, (h,), dt, 1.0, 0.1),
                 q_w=_normal(g, (hd,), dt, 1.0, 0.1) if c["qk_norm"] else None,
                 k_w=_normal(g, (hd,), dt, 1.0, 0.1) if c["qk_norm"] else None,
                 bias=None if c["qk_norm"] else _normal(g, (qs + 2 * ks,), torch.float32, 0.0, 0.5),
                 inv_freq=ops.rope_inv_freq(THETA, hd, DEV))
        return dict(s, **_paged(g, seed, ctx, np.ones(t, np.int64), c["kv_heads"], hd, dt))
    if family == "q8":
        w8, ws = _q8_weights(g, case["n"], case["k"])
        return dict(case=case, x=_normal(g, (case["m"], case["k"]), TYPES[case["dtype"]]), w8=w8, ws=ws)
    if family == "matmul":
        n, k, w = case["n"], case["k"], case["w"]
        return dict(case=case, x=_normal(g, (case["m"], k), TYPES[case["x"]]),
                    w=_kquant_weights(g, n, k, w) if w.startswith("q") else _normal(g, (n, k), TYPES[w], 0.0, 0.03))
    if family == "attn":
        lens, dt = [int(v) for v in case["lens"].split(",")], TYPES[case["dtype"]]
        q_lens = [1] * len(lens) if case["decode"] else lens
        p = _paged(g, seed, lens, q_lens, case["kv_heads"], case["head_dim"], dt)
        return dict(p, case=case, q=_normal(g, (int(p["cu"][-1]), case["q_heads"], case["head_dim"]), dt))
    e, dt, wt = EXPERTS, TYPES[case["x"]], TYPES[case["w"]]
    return dict(case=case, x=_normal(g, (case["rows"], e["hidden"]), dt),
                logits=_normal(g, (case["rows"], e["experts"]), torch.float32),
                gu=_normal(g, (e["experts"], 2 * e["inter"], e["hidden"]), wt, 0.0, 0.03),
                dn=_normal(g, (e["experts"], e["hidden"], e["inter"]), wt, 0.0, 0.03),
                slot_of=torch.arange(e["experts"], device=DEV, dtype=torch.int32))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _run_chain(s: dict):
    case = s["case"]
    c, dt = MODELS[case["model"]], TYPES[case["dtype"]]
    residual = ops.embedding_q8_0(s["ids"], s["w8"], s["ws"], c["hidden"], c["vocab"], out_dtype=dt)
    normed = ops.rms_norm_add(s["x"], residual, s["norm"], EPS)
    ops.qk_norm_rope(s["q"], s["k"], s["positions"], s["q_w"], s["k_w"], s["inv_freq"], c["q_heads"], c["kv_heads"],
                     c["head_dim"], EPS)
    return residual, normed, s["q"], s["k"], ops.silu_and_mul(s["gate_up"])


def _run_layer(s: dict):
    case = s["case"]
    c, dt, t = MODELS[case["model"]], TYPES[case["dtype"]], case["seqs"]
    hd, h, inter = c["head_dim"], c["hidden"], c["inter"]
    qs, ks = c["q_heads"] * hd, c["kv_heads"] * hd
    small = t <= 16  # the decode GEMV's fused forms
    residual = ops.embedding_q8_0(s["ids"], *s["emb"], h, c["vocab"], out_dtype=dt)
    if small:
        qkv = ops.matmul_q8_0_rms(residual, s["w_in"], EPS, *s["qkv"], qs + 2 * ks)
    else:
        _, scale, xq = ops.rms_norm_q8(residual, s["w_in"], EPS, want_out=False)
        qkv = ops.matmul_q8_0(xq, scale, *s["qkv"], qs + 2 * ks, dt)
    ops.qk_norm_rope_store_kv(qkv[:, :qs], qkv[:, qs:qs + ks], qkv[:, qs + ks:], s["positions"], s["q_w"], s["k_w"],
                              s["inv_freq"], c["q_heads"], c["kv_heads"], hd, s["k_cache"], s["v_cache"], s["slots"],
                              EPS, qkv_bias=s["bias"])
    att = ops.paged_attention(qkv[:, :qs].view(t, c["q_heads"], hd), s["k_cache"], s["v_cache"], s["query_seq"],
                              s["key_len"], s["table"], KV_BLOCK, hd ** -0.5, max_query_len=1)
    o = ops.matmul_q8_0_act(att.view(t, qs), *s["o"], h) if small else ops.matmul_q8(att.view(t, qs), *s["o"], h)
    _, scale, xq = ops.rms_norm_q8(o, s["w_post"], EPS, residual=residual, want_out=False)
    gate_up = ops.matmul_q8_0(xq, scale, *s["gate_up"], 2 * inter, dt)
    if small:
        down = ops.matmul_q8_0_act(gate_up, *s["down"], h, swiglu=True)
    else:
        _, scale, xq = ops.silu_and_mul_q8(gate_up)
        down = ops.matmul_q8_0(xq, scale, *s["down"], h, dt)
    return qkv, att, residual, down


def run(state: dict):
    case = state["case"]
    family = case["family"]
    if family == "chain":
        return _run_chain(state)
    if family == "layer":
        return _run_layer(state)
    if family == "q8":
        return ops.matmul_q8(state["x"], state["w8"], state["ws"], case["n"])
    if family == "matmul":
        return ops.matmul(state["x"], state["w"], case["n"], FORMATS[case["w"]])
    if family == "attn":
        return ops.paged_attention(state["q"], state["k_cache"], state["v_cache"], state["query_seq"], state["key_len"],
                                   state["table"], KV_BLOCK, case["head_dim"] ** -0.5,
                                   max_query_len=1 if case["decode"] else 0,
                                   cu_seqlens=None if case["decode"] else state["cu"])
    idx, score = ops.moe_route(state["logits"], EXPERTS["top"], True)
    out = ops.moe_ffn(state["x"], idx, score, state["gu"], state["dn"], state["slot_of"], EXPERTS["inter"],
                      EXPERTS["experts"], torch.zeros_like(state["x"]))
    return out, idx, score


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _size(name: str) -> int:
    return 4 if name == "f32" else 2


def work(case: dict) -> dict:
    family = case["family"]
    if family == "chain":
        c, e, t = MODELS[case["model"]], _size(case["dtype"]), case["tokens"]
        h, heads = c["hidden"], (c["q_heads"] + c["kv_heads"]) * c["head_dim"]
        return dict(bytes=t * (h * 34 / 32 + 8 + 3 * h * e + 2 * heads * e + 8 + 3 * c["inter"] * e),
                    flops=t * (6.0 * h + 10.0 * heads + 10.0 * c["inter"]))
    if family == "layer":
        c, e, t = MODELS[case["model"]], _size(case["dtype"]), case["seqs"]
        h, hd = c["hidden"], c["head_dim"]
        qs, ks = c["q_heads"] * hd, c["kv_heads"] * hd
        weights = h * (qs + 2 * ks) + qs * h + 3 * c["inter"] * h
        keys = int(_contexts(case).sum())
        return dict(bytes=weights * 34 / 32 + keys * ks * 2 * e + t * (h * 34 / 32 + (2 * qs + 2 * ks + 2 * h) * e),
                    flops=2.0 * t * weights + 4.0 * keys * qs)
    if family == "q8":
        m, n, k, e = case["m"], case["n"], case["k"], _size(case["dtype"])
        return dict(bytes=m * k * e + n * k * 34 / 32 + m * n * e, flops=2.0 * m * n * k)
    if family == "matmul":
        m, n, k, e = case["m"], case["n"], case["k"], _size(case["x"])
        return dict(bytes=m * k * e + n * k * BYTES_PER_WEIGHT[case["w"]] + m * n * e, flops=2.0 * m * n * k)
    if family == "attn":
        lens, e = [int(v) for v in case["lens"].split(",")], _size(case["dtype"])
        tokens = len(lens) if case["decode"] else sum(lens)
        pairs = sum(lens) if case["decode"] else sum(n * (n + 1) // 2 for n in lens)
        row = case["head_dim"] * e
        return dict(bytes=2.0 * sum(lens) * case["kv_heads"] * row + 2.0 * tokens * case["q_heads"] * row,
                    flops=4.0 * pairs * case["q_heads"] * case["head_dim"])
    c, e, rows = EXPERTS, _size(case["x"]), case["rows"]
    expert = 3 * c["hidden"] * c["inter"]
    used = c["experts"] * (1.0 - (1.0 - c["top"] / c["experts"]) ** rows)  # experts that some row is routed to
    return dict(bytes=used * expert * 2 + rows * (2 * c["hidden"] * e + c["experts"] * 4 + c["top"] * 8),
                flops=2.0 * rows * c["top"] * expert)


def tolerance(case: dict) -> dict:
    family = case["family"]
    kind = case.get("dtype") or case["x"]
    if family == "layer":  # the int8 quantizers truncate: a last-bit change of an input moves some values a whole
        return {"rel": 3e-2}  # step (against 64 bits the down projection's output is 2.2e-2 off)
    if family == "moe":
        return {"rel": {"f32": 1e-5, "f16": 1e-3, "bf16": 8e-3}[kind], "differ": 1e-3}
    return {"rel": {"f32": 1e-5, "f16": 1e-3, "bf16": 8e-3}[kind]}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------
def _stored(x: torch.Tensor, dtype) -> torch.Tensor:
    """A value that the ops keep in the storage type between two calls."""
    return x.to(dtype).double()


def _q8_dequant(w8, ws, n: int, k: int) -> torch.Tensor:
    return (w8.view(-1, 32).double() * ws.view(torch.float16).double()[:, None]).view(n, k)


def _q8_product(x: torch.Tensor, w8, ws, n: int) -> torch.Tensor:
    """The Q8_0 product of x's rows as the path defines it: each row to whole numbers
    (scale 127 / max|x| in fp32, truncated), times the dequantized weights."""
    x = x.float()
    scale = 127.0 / x.abs().amax(1, keepdim=True).clamp_min(1e-8)
    q = (x * scale).clamp(-127.0, 127.0).trunc().double()
    return (q @ _q8_dequant(w8, ws, n, x.shape[1]).T) / scale.double()


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * w.double()


def _silu_mul(gu: torch.Tensor) -> torch.Tensor:
    gate, up = gu.chunk(2, dim=-1)
    return gate * torch.sigmoid(gate) * up


def _rope(x: torch.Tensor, heads: int, hd: int, positions, inv_freq, w) -> torch.Tensor:
    x = x.view(x.shape[0], heads, hd)
    if w is not None:
        x = _rms(x, w)
    angle = (positions.float()[:, None] * inv_freq[None]).double()[:, None]  # the path's angles are fp32
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1).flatten(1)


def _attention(q, k_cache, v_cache, p: dict, q_lens, scale: float) -> torch.Tensor:
    """q [tokens, heads, hd] over the paged caches; sequence s queries its last q_lens[s] keys."""
    heads, kv_heads = q.shape[1], k_cache.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    at = 0
    for s, (ctx, n) in enumerate(zip(p["ctx"], q_lens)):
        j = np.arange(int(ctx))
        rows = torch.from_numpy(p["host_table"][s, j // KV_BLOCK].astype(np.int64) * KV_BLOCK + j % KV_BLOCK).to(DEV)
        keys, values = k_cache[rows].double(), v_cache[rows].double()
        late = torch.arange(int(ctx), device=DEV)[None] > torch.arange(int(ctx) - int(n), int(ctx), device=DEV)[:, None]
        for h in range(heads):
            kv = h // (heads // kv_heads)
            score = (q[at:at + int(n), h].double() @ keys[:, kv].T.contiguous()) * scale
            out[at:at + int(n), h] = score.masked_fill(late, -math.inf).softmax(-1) @ values[:, kv].contiguous()
        at += int(n)
    return out


def _kquant_dequant(blk: torch.Tensor, n: int, k: int, fmt: str) -> torch.Tensor:
    size = {"q4_k": 144, "q5_k": 176, "q6_k": 210}[fmt]
    out = torch.empty(n * k // 256, 256, dtype=torch.float64, device=DEV)
    for i in range(0, out.shape[0], 1 << 18):
        b = blk.view(-1, size)[i:i + (1 << 18)]
        rows = b.shape[0]

        def half(at):
            return b[:, at:at + 2].contiguous().view(torch.float16).double()

        if fmt == "q6_k":
            ql, qh = b[:, :128].int().view(rows, 2, 2, 32), b[:, 128:192].int().view(rows, 2, 32)
            low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
            high = torch.stack([(qh >> (2 * s)) & 3 for s in range(4)], 2)
            q = (low | (high << 4)).double() - 32.0
            sc = b[:, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 1)
            out[i:i + rows] = half(208) * sc * q.reshape(rows, 256)
            continue
        h = b[:, 4:16].int()
        sc = torch.cat([h[:, 0:4] & 63, (h[:, 8:12] & 15) | ((h[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([h[:, 4:8] & 63, (h[:, 8:12] >> 4) | ((h[:, 4:8] >> 6) << 4)], 1).double()
        ql = b[:, size - 128:].int().view(rows, 4, 32)
        q = torch.stack([ql & 15, ql >> 4], 2).view(rows, 8, 32)
        if fmt == "q5_k":
            qh = b[:, 16:48].int()
            q = q | (torch.stack([(qh >> j) & 1 for j in range(8)], 1) << 4)
        out[i:i + rows] = ((half(0) * sc)[..., None] * q.double() - (half(2) * mn)[..., None]).view(rows, 256)
    return out.view(n, k)


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    family = case["family"]
    if family == "chain":
        c, dt = MODELS[case["model"]], TYPES[case["dtype"]]
        h, hd = c["hidden"], c["head_dim"]
        emb = s["w8"].view(c["vocab"], h // 32, 32)[s["ids"]].double()
        emb = (emb * s["ws"].view(torch.float16).view(c["vocab"], h // 32)[s["ids"]].double()[..., None]).view(-1, h)
        residual = _stored(_stored(emb, dt) + s["x"].double(), dt)
        return (residual, _rms(residual, s["norm"]),
                _rope(s["q"].double(), c["q_heads"], hd, s["positions"], s["inv_freq"], s["q_w"]),
                _rope(s["k"].double(), c["kv_heads"], hd, s["positions"], s["inv_freq"], s["k_w"]),
                _silu_mul(s["gate_up"].double()))
    if family == "layer":
        c, dt, t = MODELS[case["model"]], TYPES[case["dtype"]], case["seqs"]
        h, hd, inter = c["hidden"], c["head_dim"], c["inter"]
        qs, ks = c["q_heads"] * hd, c["kv_heads"] * hd
        w8, ws = s["emb"]
        emb = w8.view(c["vocab"], h // 32, 32)[s["ids"]].double()
        emb = (emb * ws.view(torch.float16).view(c["vocab"], h // 32)[s["ids"]].double()[..., None]).view(t, h)
        residual = _stored(emb, dt)
        qkv = _stored(_q8_product(_stored(_rms(residual, s["w_in"]), dt), *s["qkv"], qs + 2 * ks), dt)
        biased = qkv if s["bias"] is None else qkv + s["bias"].double()
        q = _rope(biased[:, :qs], c["q_heads"], hd, s["positions"], s["inv_freq"], s["q_w"])
        k = _rope(biased[:, qs:qs + ks], c["kv_heads"], hd, s["positions"], s["inv_freq"], s["k_w"])
        slots = s["slots"].long()
        s["k_cache"][slots] = k.to(dt).view(t, c["kv_heads"], hd)
        s["v_cache"][slots] = biased[:, qs + ks:].to(dt).view(t, c["kv_heads"], hd)
        att = _attention(_stored(q, dt).view(t, c["q_heads"], hd), s["k_cache"], s["v_cache"], s, np.ones(t, int),
                         hd ** -0.5)
        o = _stored(_q8_product(_stored(att.view(t, qs), dt), *s["o"], h), dt)
        residual = _stored(residual + o, dt)
        gate_up = _stored(_q8_product(_stored(_rms(residual, s["w_post"]), dt), *s["gate_up"], 2 * inter), dt)
        down = _q8_product(_stored(_silu_mul(gate_up), dt), *s["down"], h)
        return torch.cat([q, k, qkv[:, qs + ks:]], 1), att, residual, down
    if family == "q8":
        return _q8_product(s["x"], s["w8"], s["ws"], case["n"])
    if family == "matmul":
        n, k = case["n"], case["k"]
        w = _kquant_dequant(s["w"], n, k, case["w"]) if case["w"].startswith("q") else s["w"].double()
        return s["x"].double() @ w.T
    if family == "attn":
        q_lens = [1] * len(s["ctx"]) if case["decode"] else s["ctx"]
        return _attention(s["q"], s["k_cache"], s["v_cache"], s, q_lens, case["head_dim"] ** -0.5)
    prob = s["logits"].double().softmax(-1)
    score, idx = prob.topk(EXPERTS["top"], dim=-1)
    score = score / score.sum(-1, keepdim=True)
    x, out = s["x"].double(), torch.zeros(s["x"].shape, dtype=torch.float64, device=DEV)
    for e in range(EXPERTS["experts"]):
        row, at = torch.nonzero(idx == e, as_tuple=True)
        if row.numel():
            act = _silu_mul(x[row] @ s["gu"][e].double().T)
            out.index_add_(0, row, (act @ s["dn"][e].double().T) * score[row, at, None])
    return out, None, score
