"""The workloads this library is timed on: what a program that uses it calls, from the smallest step to the largest.

Each case is one attention call (forward, or forward and backward) through the public Python entry points, at sizes
of the benchmark's configurations or of the same kind.  ``exact`` is plain torch in float64.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "npu-flex-att_amd"))

import npu_flash_attention as nfa  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"
BLOCK = 128  # block edge of the block-sparse map

# kind: "step" (npu_flash_attention_forward + _backward, as the benchmark's step), "train" (flex_attention under
# autograd), "forward" (prefill and decode).  docs: mean document length of packed sequences (0: one document);
# sparsity: share of the off-diagonal 128 x 128 blocks a block mask removes (0: no block mask).
FIELDS = dict(kind="step", dtype="bf16", B=1, Hq=32, Hkv=8, Sq=4096, Skv=4096, D=128, causal=True, window=0,
              soft_cap=0.0, alibi=False, scale=0.0, spread=1.0, docs=0, sparsity=0.0)


def case(name=None, **kw):
    assert not set(kw) - set(FIELDS), kw
    c = dict(FIELDS, **kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest training step of the latency table: one sequence, two heads; launches and host work count.
        case("step_mha_d64_s128", dtype="fp16", Hq=2, Hkv=2, Sq=128, Skv=128, D=64),
        # The longest of the same table: still far fewer workgroups than the GPU has CUs.
        case("step_mha_d64_s2048", dtype="fp16", Hq=2, Hkv=2, Sq=2048, Skv=2048, D=64),
        # A small model's layer: head dim 32, a local window, ALiBi, a batch of sequences of odd length.
        case("train_d32_window_alibi", kind="train", dtype="bf16", B=4, Hq=8, Hkv=8, Sq=1021, Skv=1021, D=32,
             window=256, alibi=True),
        # Full-precision training or fine-tuning of a grouped-query layer, odd length.
        case("train_fp32_gqa_d128", kind="train", dtype="fp32", B=1, Hq=8, Hkv=2, Sq=1000, Skv=1000, D=128),
        # The benchmark's default workload: a Llama-3-8B-shaped causal grouped-query layer.
        case("step_gqa_d128_s4096", dtype="bf16", B=2, Hq=32, Hkv=8, Sq=4096, Skv=4096, D=128),
        # Gemma2-style layer: head dim 256, sliding window, soft-cap, its own scale.
        case("train_gemma2_d256_s8192", kind="train", dtype="bf16", Hq=16, Hkv=8, Sq=8192, Skv=8192, D=256,
             window=4096, soft_cap=50.0, scale=1.0 / 16, spread=2.0),
        # Every score primitive at once on a long sequence, seven query heads per KV head, Sq != Skv.
        case("step_all_primitives_d64_s16384", dtype="fp16", Hq=28, Hkv=4, Sq=16384, Skv=16383, D=64, window=2048,
             soft_cap=30.0, alibi=True, scale=0.05),
        # Packed pre-training: documents of mixed lengths in one causal sequence.
        case("train_documents_d128_s8192", kind="train", dtype="bf16", Hq=32, Hkv=8, Sq=8192, Skv=8192, D=128,
             docs=700),
        # Block-sparse causal training, half of the off-diagonal blocks removed.
        case("train_block_sparse_d128_s4096", kind="train", dtype="bf16", Hq=32, Hkv=8, Sq=4096, Skv=4096, D=128,
             sparsity=0.5),
        # One prompt's prefill while serving: a few hundred tokens, odd length.
        case("prefill_gqa_d128_s777", kind="forward", dtype="bf16", Sq=777, Skv=777, D=128),
        # Decoding against a long KV cache, a batch of sequences (memory-bound).
        case("decode_gqa_d128_32k", kind="forward", dtype="bf16", B=8, Sq=1, Skv=32768, D=128, causal=False),
        # Decoding of the Gemma2-style layer against a cache of odd length, a small batch.
        case("decode_gemma2_d256_4k", kind="forward", dtype="bf16", B=2, Hq=16, Hkv=8, Sq=1, Skv=4097, D=256,
             causal=False, soft_cap=50.0, scale=1.0 / 16, spread=2.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: sizes spread over their logarithm, odd ones included."""
    family = rng.choice(["small", "d32", "fp32", "gqa", "gemma2", "primitives", "documents", "blocks", "prefill",
                         "decode", "decode"])
    kind = rng.choice(["step", "train"])
    half = rng.choice(["fp16", "bf16"])
    if family == "small":
        s = _log_int(rng, 100, 2048)
        h = rng.choice([1, 2, 4])
        return case(kind=kind, dtype=half, Hq=h, Hkv=h, Sq=s, Skv=s, D=rng.choice([64, 128]))
    if family == "d32":
        s = _log_int(rng, 100, 2000)
        return case(kind=kind, dtype=half, B=rng.randint(1, 8), Hq=8, Hkv=rng.choice([2, 8]), Sq=s, Skv=s, D=32,
                    window=rng.choice([0, 256]), alibi=rng.random() < 0.5)
    if family == "fp32":
        s = _log_int(rng, 128, 2000)
        hkv = rng.choice([1, 2, 8])
        return case(kind=kind, dtype="fp32", B=rng.randint(1, 2), Hq=8, Hkv=hkv, Sq=s, Skv=s,
                    D=rng.choice([64, 128]))
    if family == "gqa":
        s = _log_int(rng, 500, 4096)
        hkv = rng.choice([4, 8, 16])
        return case(kind=kind, dtype=half, B=rng.randint(1, 2), Hq=32, Hkv=hkv, Sq=s, Skv=s, D=rng.choice([64, 128]),
                    causal=rng.random() < 0.7)
    if family == "gemma2":
        s = _log_int(rng, 700, 8192)
        return case(kind=kind, dtype="bf16", Hq=16, Hkv=8, Sq=s, Skv=s, D=256, window=rng.choice([0, 1024, 4096]) if
                    s <= 5000 else 4096, soft_cap=50.0, scale=1.0 / 16, spread=2.0)
    if family == "primitives":
        s = _log_int(rng, 1000, 14000)
        return case(kind=kind, dtype=half, Hq=28, Hkv=4, Sq=s, Skv=s - rng.randint(0, 99), D=64,
                    window=rng.choice([512, 2048]), soft_cap=rng.choice([0.0, 30.0]), alibi=rng.random() < 0.6,
                    scale=0.05)
    if family == "documents":
        s = _log_int(rng, 1000, 8192)
        return case(kind=kind, dtype=half, Hq=32, Hkv=8, Sq=s, Skv=s, D=rng.choice([64, 128]),
                    docs=_log_int(rng, 100, 2000))
    if family == "blocks":
        s = _log_int(rng, 1000, 4096)
        return case(kind=kind, dtype=half, Hq=32, Hkv=8, Sq=s, Skv=s, D=rng.choice([64, 128]),
                    sparsity=rng.uniform(0.3, 0.9))
    if family == "prefill":
        s = _log_int(rng, 64, 4096)
        d = rng.choice([64, 128, 128, 256])
        hq, hkv = (16, 8) if d == 256 else (32, 8)
        return case(kind="forward", dtype=half, Hq=hq, Hkv=hkv, Sq=s, Skv=s, D=d)
    # decoding: one new token, or a few (speculative decoding), against a cache
    d = rng.choice([64, 128, 128, 256])
    hq, hkv = (16, 8) if d == 256 else (32, 8)
    b = _log_int(rng, 1, 16)
    return case(kind="forward", dtype=half, B=b, Hq=hq, Hkv=hkv, Sq=rng.choice([1, 1, 1, 4]),
                Skv=_log_int(rng, 300, min(32768, 262144 // b)), D=d, causal=False,
                soft_cap=50.0 if d == 256 else 0.0)


# ------------------------------------------------------------------ inputs --
def _generator(seed, device):
    return torch.Generator(device=device).manual_seed(seed)


def _document_ids(c, seed):
    """[B, S] ids of packed documents, lengths spread around the mean as in a real mixture (long tail)."""
    g = _generator(seed + 1, "cpu")
    rows = []
    for _ in range(c["B"]):
        n, lengths = 0, []
        while n < c["Sq"]:
            x = int(max(8.0, c["docs"] * math.exp(0.8 * float(torch.randn((), generator=g)) - 0.32)))
            lengths.append(min(x, c["Sq"] - n))
            n += lengths[-1]
        rows.append(torch.repeat_interleave(torch.arange(len(lengths)), torch.tensor(lengths)))
    return torch.stack(rows).to(DEVICE)


def _block_map(c, seed):
    """Dense map [1, 1, nq, nk] of 128 x 128 blocks: the diagonal kept, the share `sparsity` of the others removed."""
    n = -(-c["Sq"] // BLOCK)
    keep = torch.rand(n, n, generator=_generator(seed + 2, "cpu")) >= c["sparsity"]
    keep |= torch.eye(n, dtype=torch.bool)
    return keep.view(1, 1, n, n).to(DEVICE)


def _slopes(c):
    return torch.tensor([2.0 ** (-8.0 * (h + 1) / c["Hq"]) for h in range(c["Hq"])], dtype=torch.float32,
                        device=DEVICE)


def _tensors(c, seed):
    g, t = _generator(seed, DEVICE), DTYPES[c["dtype"]]
    qs, ks = (c["B"], c["Hq"], c["Sq"], c["D"]), (c["B"], c["Hkv"], c["Skv"], c["D"])
    q, k, v, do = (torch.randn(s, generator=g, device=DEVICE, dtype=torch.float32) for s in (qs, ks, ks, qs))
    sp = math.sqrt(c["spread"])  # the scores' spread, shared by Q and K
    return (q * sp).to(t), (k * sp).to(t), v.to(t), do.to(t)


def _options(c, seed):
    o = dict(causal=c["causal"], sliding_window=c["window"], soft_cap=c["soft_cap"])
    if c["scale"]:
        o["scale"] = c["scale"]
    if c["alibi"]:
        o["alibi_slope"] = _slopes(c)
    if c["docs"]:
        o["document_ids"] = _document_ids(c, seed)
    if c["sparsity"]:
        o["block_mask"] = _block_map(c, seed)
    return o


def prepare(case, seed):
    q, k, v, do = _tensors(case, seed)
    s = dict(kind=case["kind"], q=q, k=k, v=v)
    o = _options(case, seed)
    if case["kind"] != "forward":
        s["do"] = do
    if case["kind"] == "train":
        for x in (q, k, v):
            x.requires_grad_(True)
        s["config"] = nfa.AttentionConfig(**o)
    else:
        s["options"] = o
    return s


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    if state["kind"] == "forward":
        return nfa.npu_flash_attention_forward(q, k, v, **state["options"])
    if state["kind"] == "step":
        o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, **state["options"])
        dq, dk, dv = nfa.npu_flash_attention_backward(q, k, v, o, lse, state["do"], **state["options"])
        return o, lse, dq, dk, dv
    o = nfa.flex_attention(q, k, v, config=state["config"])
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
    return o.detach(), dq, dk, dv


# -------------------------------------------------------------------- work --
def _pairs(c):
    """Attended (query row, key) pairs of one head of one sequence, before document and block masks."""
    n = 0
    for i in range(c["Sq"]):
        hi = min(c["Skv"] - 1, i) if c["causal"] else c["Skv"] - 1
        lo = max(0, i - c["window"]) if c["window"] else 0
        n += max(0, hi - lo + 1)
    return n


def work(case):
    c = case
    if c["docs"]:
        # documents of the mean length: what is attended varies with the seed, this is its middle
        pairs = c["Sq"] * min(c["docs"], c["Sq"]) / 2
    elif c["sparsity"]:
        n = -(-c["Sq"] // BLOCK)
        pairs = _pairs(c) * ((1 - c["sparsity"]) * (n - 1) + 1) / n
    else:
        pairs = _pairs(c)
    es = 4 if c["dtype"] == "fp32" else 2
    rows_q, rows_k = c["B"] * c["Hq"] * c["Sq"], c["B"] * c["Hkv"] * c["Skv"]
    if c["kind"] == "forward":
        n_bytes = es * c["D"] * (2 * rows_q + 2 * rows_k)
        flops = 4 * c["D"] * pairs * c["B"] * c["Hq"]
    else:  # q, dO, O, dQ and k, v, dK, dV once each, LSE
        n_bytes = es * c["D"] * (4 * rows_q + 4 * rows_k) + 4 * rows_q
        flops = 14 * c["D"] * pairs * c["B"] * c["Hq"]
    return {"bytes": int(n_bytes), "flops": int(flops)}


# ------------------------------------------------------------------- exact --
def _mask(c, i, j, docs, blocks, b):
    m = torch.ones(len(i), len(j), dtype=torch.bool, device=i.device)
    d = i[:, None] - j[None, :]
    if c["causal"]:
        m &= d >= 0
    if c["window"]:
        m &= d <= c["window"]
    if docs is not None:
        m &= docs[b][i][:, None] == docs[b][j][None, :]
    if blocks is not None:
        m &= blocks[0, 0][(i // BLOCK)[:, None], (j // BLOCK)[None, :]]
    return m


def exact(case, seed):
    c = case
    q, k, v, do = (x.double() for x in _tensors(c, seed))
    o_ = _options(c, seed)
    docs, blocks = o_.get("document_ids"), o_.get("block_mask")
    slopes = o_["alibi_slope"].double() if c["alibi"] else None
    scale, cap, G = c["scale"] or 1.0 / math.sqrt(c["D"]), c["soft_cap"], c["Hq"] // c["Hkv"]
    o = torch.zeros_like(q)
    lse = torch.zeros(q.shape[:3], dtype=torch.float64, device=q.device)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    grads = c["kind"] != "forward"
    j = torch.arange(c["Skv"], device=q.device)
    step = max(128, (1 << 27) // c["Skv"])  # query rows at a time
    for b in range(c["B"]):
        for h in range(c["Hq"]):
            kv = h // G
            K, V = k[b, kv], v[b, kv]
            for r0 in range(0, c["Sq"], step):
                r = slice(r0, min(r0 + step, c["Sq"]))
                i = torch.arange(r.start, r.stop, device=q.device)
                x = (q[b, h, r] @ K.t()).mul_(scale)
                t = None
                if cap > 0:
                    t = torch.tanh(x.div_(cap))
                    x = cap * t
                if slopes is not None:
                    x = x + slopes[h] * (i[:, None] - j[None, :])
                x = x.masked_fill_(~_mask(c, i, j, docs, blocks, b), -math.inf)
                l = torch.logsumexp(x, -1)
                p = torch.exp(x.sub_(torch.where(torch.isinf(l), 0.0, l)[:, None]))
                o[b, h, r] = p @ V
                lse[b, h, r] = l
                if grads:
                    g = do[b, h, r]
                    delta = (o[b, h, r] * g).sum(-1, keepdim=True)
                    dv[b, kv] += p.t() @ g
                    ds = p * ((g @ V.t()) - delta)
                    if t is not None:
                        ds *= 1 - t * t
                    ds *= scale
                    dq[b, h, r] = ds @ K
                    dk[b, kv] += ds.t() @ q[b, h, r]
    if c["kind"] == "forward":
        return o
    if c["kind"] == "step":
        return o, lse, dq, dk, dv
    return o, dq, dk, dv


def tolerance(case):
    # four times the largest error against exact() seen over these ranges (bf16 2.7e-3, fp16 3.4e-4, fp32 1.5e-6)
    return {"rel": {"bf16": 1.1e-2, "fp16": 1.4e-3, "fp32": 6e-6}[case["dtype"]]}
