"""The work that a user of this library has it do, as cases that a measuring program can time and compare.

Seven kinds of call, each through a public entry point:

  forward   flash_attention_forward on dense [B, H, N, D] tensors (inference prefill)
  train     flash_attention and its gradients on dense tensors (a training step's attention)
  packed    flash_attention_varlen and its gradients on packed sequences with grouped heads
  chunks    paged_prefill: new tokens of some sequences against their paged KV cache
  decode    paged_attention_decode: one new token per sequence against the paged KV cache
  mlp       a decoder's MLP block: residual add + norm, gate and up, SwiGLU, down
  step      KVCacheDecoder.step: a whole decode step of the LLaMA-shaped model (logits, caches)
  prompt    KVCacheDecoder.prefill: a whole chunked prefill of it (logits, caches)

listed() names twelve of them; draw() gives others of the same ranges. Sizes are those of the repository's
own workloads (lightserve_amd/workloads.py, model/minimal_llama.py), or generic ones.
"""
import math
import random

import torch

from lightserve_amd.kernels.flash_attention import flash_attention_forward
from lightserve_amd.kernels.flash_attention_backward import flash_attention
from lightserve_amd.kernels.flash_attention_varlen import flash_attention_varlen
from lightserve_amd.kernels.paged_attention import paged_attention_decode, paged_prefill
from lightserve_amd.kernels.tiled_matmul import add_rmsnorm_matmul_shared_input, swiglu_matmul
from lightserve_amd.model.graph_decode import KVCacheDecoder
from lightserve_amd.model.minimal_llama import LayerWeights, LlamaConfig, LlamaWeights

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
VOCAB, LAYERS, EPS = 128256, 4, 1e-5


def listed():
    return [
        # The smallest call: the fp32 attention of a test or of a small fp32 model. Latency.
        dict(name="forward_small_fp32", kind="forward", dtype="fp32", batch=1, heads=4, n=256, dim=64, causal=True,
             heads_inside=False, lse=False),
        # Prefill of a batch of 2048-token prompts at LLaMA-3-8B's layer shape.
        dict(name="forward_prefill_fp16", kind="forward", dtype="fp16", batch=4, heads=32, n=2048, dim=128,
             causal=True, heads_inside=False, lse=False),
        # The repository's headline workload: a training step's attention.
        dict(name="train_bf16", kind="train", dtype="bf16", batch=4, heads=32, n=4096, dim=128, causal=True,
             heads_inside=False, outliers=False),
        # Long context without a mask (encoders, long documents), some keys far larger than the rest.
        dict(name="train_long_bf16", kind="train", dtype="bf16", batch=1, heads=16, n=16384, dim=64, causal=False,
             heads_inside=False, outliers=True),
        # A short, odd-sized training call with a head dim between the tile widths, in the layout in which a
        # projection leaves its heads.
        dict(name="train_short_odd_fp16", kind="train", dtype="fp16", batch=2, heads=12, n=777, dim=80, causal=True,
             heads_inside=True, outliers=False),
        # Training on packed sequences of different lengths with grouped heads.
        dict(name="packed_train_bf16", kind="packed", dtype="bf16", sequences=8, shortest=97, longest=2100, heads=32,
             kv_heads=8, dim=128),
        # A batch of prefill chunks against long cached prefixes (the repository's chunked prefill workload).
        dict(name="chunks_batch_bf16", kind="chunks", dtype="bf16", sequences=8, chunk=512, shortest=1024,
             longest=8192, heads=32, kv_heads=8, dim=128, block=16),
        # One request's prefill chunk, odd-sized, between decode steps of the others.
        dict(name="chunk_single_bf16", kind="chunks", dtype="bf16", sequences=1, chunk=333, shortest=6011,
             longest=6011, heads=32, kv_heads=8, dim=128, block=16),
        # A serving batch's decode attention.
        dict(name="decode_batch_bf16", kind="decode", dtype="bf16", sequences=32, shortest=1024, longest=8192,
             limit=8192, heads=32, kv_heads=8, dim=128, block=16),
        # The MLP of one request's decode step.
        dict(name="mlp_1_row_bf16", kind="mlp", dtype="bf16", rows=1, hidden=4096, inner=14336),
        # A whole decode step of a small batch: logits and the caches it appends to.
        dict(name="step_8_bf16", kind="step", dtype="bf16", sequences=8, shortest=300, longest=1500, limit=2048,
             kv_heads=8, block=16),
        # A whole prompt of odd length, prefilled in chunks.
        dict(name="prompt_bf16", kind="prompt", dtype="bf16", sequences=1, tokens=1001, chunk=512, limit=1024,
             kv_heads=8, block=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes spread over their logarithm, so that most are odd; no dearer than train_long_bf16."""
    kind = rng.choice(["forward", "forward", "train", "train", "packed", "chunks", "chunks", "decode", "decode",
                       "mlp", "mlp", "step", "prompt"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind in ("forward", "train"):
        dtype = rng.choice([half, half, half, "fp32"])
        dim = rng.choice([64, 128, 128, 80, 96, 40])
        n = _log(rng, 128, 2048 if dtype == "fp32" else 8192)
        n = n if rng.random() < 0.7 else -(-n // 128) * 128
        most = {"fp32": 1 << 26}.get(dtype, 1 << 31)  # query-key pairs
        rows = max(1, min(128, most // (n * n)))
        heads = rng.choice([h for h in (4, 8, 12, 16, 32) if h <= rows] or [1])
        case = dict(kind=kind, dtype=dtype, batch=_log(rng, 1, max(1, min(8, rows // heads))), heads=heads, n=n,
                    dim=dim, causal=rng.random() < 0.7, heads_inside=rng.random() < 0.5)
        case.update(dict(lse=rng.random() < 0.3) if kind == "forward" else dict(outliers=rng.random() < 0.2))
        return case
    heads, kv_heads = rng.choice([(32, 8), (32, 8), (32, 32), (16, 2), (28, 4)])
    dim = rng.choice([128, 128, 64])
    if kind == "packed":
        longest = _log(rng, 200, 4000)
        return dict(kind=kind, dtype=half, sequences=_log(rng, 1, 8), shortest=_log(rng, 16, longest), longest=longest,
                    heads=heads, kv_heads=kv_heads, dim=dim)
    if kind == "chunks":
        longest = _log(rng, 64, 16000)
        return dict(kind=kind, dtype=half, sequences=_log(rng, 1, 8), chunk=_log(rng, 16, 1024),
                    shortest=rng.randrange(longest + 1), longest=longest, heads=heads, kv_heads=kv_heads, dim=dim,
                    block=rng.choice([16, 16, 64]))
    if kind == "decode":
        longest = _log(rng, 64, 16000)
        return dict(kind=kind, dtype=half, sequences=_log(rng, 1, 64), shortest=_log(rng, 16, longest),
                    longest=longest, limit=rng.choice([longest, 16384]), heads=heads, kv_heads=kv_heads, dim=dim,
                    block=rng.choice([16, 16, 64]))
    if kind == "mlp":
        hidden = rng.choice([2048, 4096, 4096])
        return dict(kind=kind, dtype=half, rows=_log(rng, 1, 1024), hidden=hidden, inner=hidden * 7 // 2)
    if kind == "step":
        longest = _log(rng, 64, 2000)
        return dict(kind=kind, dtype=half, sequences=_log(rng, 1, 16), shortest=_log(rng, 16, longest),
                    longest=longest, limit=2048, kv_heads=rng.choice([8, 32]), block=rng.choice([16, 64]))
    return dict(kind=kind, dtype=half, sequences=rng.choice([1, 1, 2]), tokens=_log(rng, 50, 400),
                chunk=rng.choice([128, 256, 512]), limit=1024, kv_heads=rng.choice([8, 32]), block=16)


# ------------------------------------------------------------------ inputs
def _lengths(case):
    """The sequences' lengths, from the case alone: shortest .. longest, in no order."""
    n, lo, hi = case["sequences"], case["shortest"], case["longest"]
    order = random.Random(n * 7919 + lo * 31 + hi)
    got = [hi] + [order.randint(lo, hi) for _ in range(n - 1)]
    order.shuffle(got)
    return got


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, shape, dtype, scale=1.0):
    t = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    return t if scale == 1.0 else t.mul_(scale)


def _dense(case, g, scaled_keys=False):
    """q, k, v (and dO) as [B, H, N, D]; with heads_inside as views of [B, N, H, D], as a projection leaves them."""
    b, h, n, d, dtype = case["batch"], case["heads"], case["n"], case["dim"], DTYPES[case["dtype"]]
    got = []
    for _ in range(4 if case["kind"] == "train" else 3):
        t = _randn(g, (b, n, h, d) if case["heads_inside"] else (b, h, n, d), dtype)
        got.append(t.transpose(1, 2) if case["heads_inside"] else t)
    if scaled_keys:  # one key in a hundred is eight times as large
        rows = torch.randperm(n, generator=g, device="cuda")[:max(1, n // 100)]
        got[1][:, :, rows] *= 8.0
    return got


def _offsets(lengths):
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    return torch.tensor(cu, dtype=torch.int32, device="cuda")


def _paged(case, g, lengths, heads):
    """K and V caches [blocks, block, heads, D] with room for `lengths` tokens, and shuffled block tables."""
    block, dtype = case["block"], DTYPES[case["dtype"]]
    need = [-(-n // block) for n in lengths]
    order = torch.randperm(sum(need), generator=g, device="cuda").to(torch.int32)
    tables = torch.zeros(len(lengths), max(need), dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n]
        at += n
    shape = (sum(need), block, heads, case["dim"])
    return _randn(g, shape, dtype), _randn(g, shape, dtype), tables


def _model(case, g):
    """Weights of the 4-layer LLaMA-3-8B-shaped model, N(0, 0.02) as the repository draws them."""
    dtype = DTYPES[case["dtype"]]
    cfg = LlamaConfig(vocab_size=VOCAB, hidden_size=4096, intermediate_size=14336, n_layers=LAYERS, n_heads=32,
                      head_dim=128, max_seq_len=case["limit"], dtype=dtype, n_kv_heads=case["kv_heads"])
    H, I, kv = cfg.hidden_size, cfg.intermediate_size, cfg.kv_heads * cfg.head_dim

    def w(*shape):
        return _randn(g, shape, dtype, 0.02)

    def gain():
        return _randn(g, (H,), dtype, 0.1).add_(1.0)

    layers = [LayerWeights(input_layernorm_weight=gain(), q_proj=w(H, H), k_proj=w(H, kv), v_proj=w(H, kv),
                           o_proj=w(H, H), post_attention_layernorm_weight=gain(), gate_proj=w(H, I), up_proj=w(H, I),
                           down_proj=w(I, H)) for _ in range(LAYERS)]
    return cfg, LlamaWeights(embed_tokens=w(VOCAB, H), layers=layers, norm_weight=gain(), lm_head=w(H, VOCAB))


def prepare(case, seed):
    g, kind, dtype = _gen(seed), case["kind"], DTYPES[case["dtype"]]
    s = dict(case=case)
    if kind == "forward":
        s["q"], s["k"], s["v"] = _dense(case, g)
    elif kind == "train":
        q, k, v, s["do"] = _dense(case, g, case["outliers"])
        s["q"], s["k"], s["v"] = (t.requires_grad_() for t in (q, k, v))
    elif kind == "packed":
        lens = _lengths(case)
        s["cu"], s["longest"] = _offsets(lens), max(lens)
        q, s["do"] = (_randn(g, (sum(lens), case["heads"], case["dim"]), dtype) for _ in range(2))
        k, v = (_randn(g, (sum(lens), case["kv_heads"], case["dim"]), dtype) for _ in range(2))
        s["q"], s["k"], s["v"] = (t.requires_grad_() for t in (q, k, v))
    elif kind == "chunks":
        lens = [n + case["chunk"] for n in _lengths(case)]
        s["k"], s["v"], s["tables"] = _paged(case, g, lens, case["kv_heads"])
        s["q"] = _randn(g, (len(lens) * case["chunk"], case["heads"], case["dim"]), dtype)
        s["cu"] = _offsets([case["chunk"]] * len(lens))
        s["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    elif kind == "decode":
        lens = _lengths(case)
        s["k"], s["v"], s["tables"] = _paged(case, g, lens, case["kv_heads"])
        s["q"] = _randn(g, (len(lens), case["heads"], case["dim"]), dtype)
        s["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    elif kind == "mlp":
        m, h, i = case["rows"], case["hidden"], case["inner"]
        s["x"], s["residual"] = _randn(g, (m, h), dtype, 0.5), _randn(g, (m, h), dtype)
        s["norm"] = _randn(g, (h,), dtype, 0.1).add_(1.0)
        s["gate"], s["up"], s["down"] = (_randn(g, shape, dtype, 0.02) for shape in ((h, i), (h, i), (i, h)))
    else:
        cfg, weights = _model(case, g)
        d = s["decoder"] = KVCacheDecoder(weights, cfg, case["sequences"], block_size=case["block"], seed=seed)
        if kind == "step":
            d.seq_lens.copy_(torch.tensor(_lengths(case), dtype=torch.int32))
            d.tokens.copy_(torch.randint(VOCAB, (case["sequences"],), generator=g, device="cuda"))
            for t in d.k_cache + d.v_cache:  # what was cached before: rows as the projections give them
                t.copy_(_randn(g, t.shape, dtype, 1.28))
        else:
            s["prompt"] = torch.randint(VOCAB, (case["sequences"], case["tokens"]), generator=g, device="cuda")
    return s


# -------------------------------------------------------------------- pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "forward":
        got = flash_attention_forward(s["q"], s["k"], s["v"], case["causal"], return_lse=case["lse"])
        return dict(o=got[0], lse=got[1]) if case["lse"] else dict(o=got)
    if kind == "train":
        o = flash_attention(s["q"], s["k"], s["v"], case["causal"])
        dq, dk, dv = torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])
        return dict(o=o, dq=dq, dk=dk, dv=dv)
    if kind == "packed":
        o = flash_attention_varlen(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["longest"], s["longest"])
        dq, dk, dv = torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])
        return dict(o=o, dq=dq, dk=dk, dv=dv)
    if kind == "chunks":
        return dict(o=paged_prefill(s["q"], s["k"], s["v"], s["tables"], s["cu"], s["lens"],
                                    max_seqlen_q=case["chunk"]))
    if kind == "decode":
        return dict(o=paged_attention_decode(s["q"], s["k"], s["v"], s["tables"], s["lens"],
                                             max_seq_len=case["limit"]))
    if kind == "mlp":
        (gate, up), h = add_rmsnorm_matmul_shared_input(s["x"], s["residual"], s["norm"], EPS, (s["gate"], s["up"]))
        return dict(out=swiglu_matmul(gate, up, s["down"]), residual=h)
    d = s["decoder"]
    if kind == "step":  # the step does not advance the lengths: the next pass writes the same cache rows again
        return dict(logits=d.step(), k=d.k_cache, v=d.v_cache)
    d.seq_lens.zero_()  # a new prompt starts from an empty cache
    return dict(logits=d.prefill(s["prompt"], case["chunk"]), lens=d.seq_lens, k=d.k_cache, v=d.v_cache)


# -------------------------------------------------------------------- work
def _pairs(nq, nk, causal):
    """Visible query-key pairs of one head (the last query sees every key)."""
    return nq * (nk - nq) + nq * (nq + 1) // 2 if causal else nq * nk


def work(case):
    kind, e = case["kind"], 4 if case["dtype"] == "fp32" else 2
    if kind in ("forward", "train"):
        heads = case["batch"] * case["heads"]
        f = 4 * heads * _pairs(case["n"], case["n"], case["causal"]) * case["dim"]
        rows = heads * case["n"] * case["dim"] * e
        # q, k, v in, o out; training adds dO in, dq, dk, dv out, and five products for the forward's two
        if kind == "train":
            return dict(bytes=8 * rows, flops=f * 7 // 2)
        return dict(bytes=4 * rows + (heads * case["n"] * 4 if case["lse"] else 0), flops=f)
    if kind == "packed":
        lens = _lengths(case)
        f = 4 * case["heads"] * case["dim"] * sum(_pairs(n, n, True) for n in lens)
        return dict(bytes=sum(lens) * case["dim"] * 4 * (case["heads"] + case["kv_heads"]) * e, flops=f * 7 // 2)
    if kind == "chunks":
        lens, c = [n + case["chunk"] for n in _lengths(case)], case["chunk"]
        return dict(bytes=2 * case["dim"] * (len(lens) * c * case["heads"] + sum(lens) * case["kv_heads"]) * e,
                    flops=4 * case["heads"] * case["dim"] * sum(_pairs(c, n, True) for n in lens))
    if kind == "decode":
        lens = _lengths(case)
        return dict(bytes=2 * case["dim"] * (len(lens) * case["heads"] + sum(lens) * case["kv_heads"]) * e,
                    flops=4 * case["heads"] * case["dim"] * sum(lens))
    if kind == "mlp":
        m, h, i = case["rows"], case["hidden"], case["inner"]
        return dict(bytes=(3 * h * i + 4 * m * h + h) * e, flops=2 * m * 3 * h * i)
    h, i, kv, b = 4096, 14336, case["kv_heads"] * 128, case["sequences"]
    layer = 2 * h * h + 2 * h * kv + 3 * h * i
    if kind == "step":
        seen = sum(n + 1 for n in _lengths(case))
        return dict(bytes=(LAYERS * (layer + 2 * seen * kv) + h * VOCAB + b * VOCAB) * e,
                    flops=2 * b * (LAYERS * layer + h * VOCAB) + LAYERS * 4 * h * seen)
    n, chunk = case["tokens"], case["chunk"]
    chunks = -(-n // chunk)  # the weights are read for each chunk
    return dict(bytes=(chunks * (LAYERS * layer + h * VOCAB) + LAYERS * 2 * b * n * kv + b * VOCAB) * e,
                flops=2 * b * n * LAYERS * layer + 2 * b * chunks * h * VOCAB + LAYERS * 4 * h * b * _pairs(n, n, True))


# --------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times the distance of the path from exact(): rel 2.1e-3 to 2.5e-3 for attention and its gradients
    in bf16, 2.6e-4 to 3.1e-4 in fp16, 2.4e-7 to 9.2e-7 in fp32, two to three times that in the gradients where some
    scores are eight times as large; 5.2e-3 for the MLP block in bf16. The whole model's logits and cached rows are 1.7e-2 to 2.0e-2 away
    in bf16 after four layers: there 3e-2, the most that still tells a wrong answer from rounding."""
    rel = {"fp32": 4e-6, "fp16": 1.25e-3, "bf16": 1e-2}[case["dtype"]]
    if case["kind"] == "mlp":
        rel *= 2
    elif case["kind"] in ("step", "prompt"):
        rel = {"fp16": 8e-3, "bf16": 3e-2}[case["dtype"]]
    elif case["kind"] == "train" and case["outliers"]:
        rel *= 3 if case["dtype"] == "fp16" else 2
    return {"rel": rel}


# ------------------------------------------------------------------- exact
def _head64(q, k, v, do, causal, scale):
    """One head in 64 bits, in blocks of queries: (o, lse, dq, dk, dv); the last three None without do."""
    q, k, v = q.detach().double(), k.detach().double(), v.detach().double()
    nq, nk = q.shape[0], k.shape[0]
    o, lse = torch.empty_like(q), torch.empty(nq, dtype=torch.float64, device=q.device)
    grads = None
    if do is not None:
        do = do.double()
        grads = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for a in range(0, nq, 2048):
        z = min(nq, a + 2048)
        s = (q[a:z] @ k.T).mul_(scale)
        if causal:
            s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(nk - nq + a + 1), -math.inf)
        lse[a:z] = torch.logsumexp(s, 1)
        p = torch.exp(s.sub_(lse[a:z, None]))
        o[a:z] = p @ v
        if grads is not None:
            grads[2].add_(p.T @ do[a:z])
            ds = p * (do[a:z] @ v.T - (do[a:z] * o[a:z]).sum(1, keepdim=True)) * scale
            grads[0][a:z] = ds @ k
            grads[1].add_(ds.T @ q[a:z])
    return (o, lse) + (grads or (None, None, None))


def _attend64(q, k, v, causal=True):
    """Sequence-major attention in 64 bits: q [n, heads, D], k and v [m, kv heads, D]."""
    group, scale = q.shape[1] // k.shape[1], 1 / math.sqrt(q.shape[2])
    return torch.stack([_head64(q[:, h], k[:, h // group], v[:, h // group], None, causal, scale)[0]
                        for h in range(q.shape[1])], 1)


def _rows(cache, table, n):
    return cache[table.long()].flatten(0, 1)[:n]


def _norm64(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _silu64(x):
    return x / (1 + torch.exp(-x))


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind in ("forward", "train"):
        q, k, v, do = s["q"].detach(), s["k"].detach(), s["v"].detach(), s.get("do")
        o, lse = torch.empty_like(q, dtype=torch.float64), q.new_empty(q.shape[:3], dtype=torch.float64)
        dq, dk, dv = (torch.empty_like(o) if do is not None else None for _ in range(3))
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                got = _head64(q[b, h], k[b, h], v[b, h], None if do is None else do[b, h], case["causal"],
                              1 / math.sqrt(case["dim"]))
                for to, t in zip((o, lse, dq, dk, dv), got):
                    if to is not None:
                        to[b, h] = t
        if kind == "train":
            return dict(o=o, dq=dq, dk=dk, dv=dv)
        return dict(o=o, lse=lse) if case["lse"] else dict(o=o)
    if kind == "packed":
        q, k, v, do = s["q"].detach(), s["k"].detach(), s["v"].detach(), s["do"]
        o, dq = torch.empty_like(q, dtype=torch.float64), torch.empty_like(q, dtype=torch.float64)
        dk, dv = torch.zeros_like(k, dtype=torch.float64), torch.zeros_like(v, dtype=torch.float64)
        group, at = case["heads"] // case["kv_heads"], 0
        for n in _lengths(case):
            r, at = slice(at, at + n), at + n
            for h in range(case["heads"]):
                o[r, h], _, dq[r, h], a, b = _head64(q[r, h], k[r, h // group], v[r, h // group], do[r, h], True,
                                                     1 / math.sqrt(case["dim"]))
                dk[r, h // group] += a
                dv[r, h // group] += b
        return dict(o=o, dq=dq, dk=dk, dv=dv)
    if kind in ("chunks", "decode"):
        c = case["chunk"] if kind == "chunks" else 1
        lens = s["lens"].tolist()
        return dict(o=torch.cat([_attend64(s["q"][i * c:(i + 1) * c], _rows(s["k"], s["tables"][i], n),
                                           _rows(s["v"], s["tables"][i], n)) for i, n in enumerate(lens)]))
    if kind == "mlp":
        h = s["x"].double() + s["residual"].double()
        y = _norm64(h, s["norm"])
        return dict(out=(_silu64(y @ s["gate"].double()) * (y @ s["up"].double())) @ s["down"].double(), residual=h)
    return _model64(s)


def _rope64(x, cos, sin):
    """x [tokens, heads, D] rotated by the rows cos, sin [tokens, D] of the tables."""
    a, b = x.chunk(2, -1)
    return x * cos[:, None] + torch.cat([-b, a], -1) * sin[:, None]


def _model64(s):
    """The model in 64 bits on the tokens of a step or of a prompt, caches and tables as the decoder holds them."""
    case, d = s["case"], s["decoder"]
    new = s["prompt"] if case["kind"] == "prompt" else d.tokens[:, None]
    before = [0] * case["sequences"] if case["kind"] == "prompt" else d.seq_lens.tolist()
    n, heads, kv, block = new.shape[1], 32, case["kv_heads"], case["block"]
    half = torch.arange(0, 64, device="cuda", dtype=torch.float32) / 64
    angle = torch.outer(torch.arange(case["limit"], device="cuda", dtype=torch.float32), 1.0 / (500000.0 ** half))
    cos, sin = (torch.cat([t, t], -1).to(DTYPES[case["dtype"]]).double() for t in (angle.cos(), angle.sin()))
    x = d.w.embed_tokens[new].double()
    caches = [], []
    for i, w in enumerate(d.w.layers):
        kc, vc = d.k_cache[i].double(), d.v_cache[i].double()
        y = _norm64(x, w.input_layernorm_weight)
        q, k, v = (y @ t.double() for t in (w.q_proj, w.k_proj, w.v_proj))
        o = torch.empty_like(q)
        for b, p in enumerate(before):
            at = torch.arange(p, p + n, device="cuda")
            slot = d.block_tables[b].long()[at // block] * block + at % block
            kc.flatten(0, 1)[slot] = _rope64(k[b].view(n, kv, 128), cos[at], sin[at])
            vc.flatten(0, 1)[slot] = v[b].view(n, kv, 128)
            o[b] = _attend64(_rope64(q[b].view(n, heads, 128), cos[at], sin[at]), _rows(kc, d.block_tables[b], p + n),
                             _rows(vc, d.block_tables[b], p + n)).flatten(1)
        caches[0].append(kc)
        caches[1].append(vc)
        x = x + o @ w.o_proj.double()
        y = _norm64(x, w.post_attention_layernorm_weight)
        x = x + (_silu64(y @ w.gate_proj.double()) * (y @ w.up_proj.double())) @ w.down_proj.double()
    logits = _norm64(x[:, -1], d.w.norm_weight) @ d.w.lm_head.double()
    if case["kind"] == "prompt":
        return dict(logits=logits, lens=None, k=caches[0], v=caches[1])
    return dict(logits=logits, k=caches[0], v=caches[1])
