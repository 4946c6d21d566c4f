"""GPU tests of the kernels that small problems leave for the split ones: the regular forward of every dtype and head dim
(decode_enabled off: flexatt_fwd_regular) and the staged fp32 backward (flexatt_bwd_ws through the C ABI, its workspace
NaN bytes), over the mask primitives, documents, PrefixLM, head groups that are no power of two, and lengths off every
tile grid.  Reference: the float64 oracle at the suite's tolerances.
"""
import pytest
import torch

import flexatt_lib as L
import npu_flash_attention as nfa
from gpu_helpers import alibi_slopes, check, draw
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu

FLAGS = {
    "full_scale_negative": dict(scale=-0.09),
    "causal": dict(causal=True),
    "window_alibi": dict(sliding_window=60, alibi=True),
    "causal_window_alibi_cap": dict(causal=True, sliding_window=70, soft_cap=9.0, alibi=True, scale=0.06),
    "documents": dict(causal=True, docs=True),
    "documents_both_sides_cap": dict(docs=True, soft_cap=20.0),
    "prefix": dict(causal=True, prefix_len=77),
}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
# (Hq, Hkv, Sq, Skv); documents take Sq for both
HEADS = {"g3": (6, 2, 333, 217), "g8": (8, 1, 150, 290), "g1": (2, 2, 130, 129)}


def _case(dtype, d, heads, flags):
    hq, hkv, sq, skv = HEADS[heads]
    kw = dict(FLAGS[flags])
    docs, alibi = kw.pop("docs", False), kw.pop("alibi", False)
    if docs:
        skv = sq
    cpu, dev = draw(hq + d, 2, hq, hkv, sq, skv, d, dtype)
    ref = dict(kw)
    if alibi:
        ref["alibi_slope"] = alibi_slopes(hq)
        kw["alibi_slope"] = ref["alibi_slope"].cuda()
    if docs:
        ref["document_ids"] = (torch.arange(sq) // 45).repeat(2, 1)
        kw["document_ids"] = ref["document_ids"].cuda()
    return cpu, dev, kw, ref


@pytest.mark.parametrize("flags", list(FLAGS))
@pytest.mark.parametrize("heads", list(HEADS))
@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("dtype", list(DTYPES))
def test_regular_forward(gpu_device, monkeypatch, dtype, d, heads, flags):
    dtype = DTYPES[dtype]
    cpu, (q, k, v, _), kw, ref = _case(dtype, d, heads, flags)
    monkeypatch.setattr(nfa, "decode_enabled", False)
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, **kw)
    want, want_lse = orc.forward(*cpu[:3], **ref)
    check("o", o, want, dtype)
    check("lse", lse, want_lse, dtype)


@pytest.mark.parametrize("flags", list(FLAGS))
@pytest.mark.parametrize("heads", list(HEADS))
@pytest.mark.parametrize("d", [32, 64, 128, 256])
def test_staged_fp32_backward(gpu_device, d, heads, flags):
    cpu, (q, k, v, do), kw, ref = _case(torch.float32, d, heads, flags)
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, **kw)
    b, hq, sq, _ = q.shape
    m = nfa._masks(kw.get("causal", False), kw.get("document_ids"), kw.get("prefix_len"), None, b, hq, sq, k.shape[2],
                   q.device)
    p = nfa._problem(q, k, kw.get("scale") or d ** -0.5, kw.get("causal", False), kw.get("sliding_window", 0),
                     kw.get("soft_cap", 0.0), kw.get("alibi_slope"), m)
    lib, T = L.load(), L.tensor
    n = lib.flexatt_bwd_workspace(p)
    ws = torch.full((n,), 0xFF, dtype=torch.uint8, device=q.device)
    got, delta = (torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)), torch.empty_like(lse)
    L.check(lib.flexatt_bwd_ws(p, T(q), T(k), T(v), T(o), T(do), lse.data_ptr(), delta.data_ptr(), *map(T, got),
                               ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream), "flexatt_bwd_ws")
    for name, x, r in zip(("dq", "dk", "dv"), got, orc.backward(*cpu, **ref)):
        check(name, x, r, torch.float32)


# (dtype, D, B, Hq, Hkv, Sq, Skv, causal, window): many row tiles that meet few keys, where the split forward measured
# 1.1 to 1.9 times the regular one's time, and (split) calls either side of the rule
@pytest.mark.parametrize("case, split", [
    (("bf16", 128, 8, 32, 8, 143, 143, True, 0), False), (("fp16", 128, 1, 32, 8, 2286, 72, True, 32), False),
    (("bf16", 64, 4, 128, 16, 144, 144, True, 0), False), (("fp16", 64, 8, 7, 1, 3384, 56, False, 64), False),
    (("fp32", 128, 4, 56, 8, 183, 183, False, 0), False), (("fp32", 128, 4, 64, 8, 118, 2418, False, 64), False), (("bf16", 256, 8, 2, 2, 38, 38, False, 0), False),
    (("bf16", 128, 1, 32, 8, 777, 777, True, 0), True), (("fp16", 64, 1, 2, 2, 128, 128, True, 0), True),
    (("bf16", 128, 1, 8, 2, 143, 143, True, 0), True), (("fp32", 128, 1, 8, 2, 183, 183, True, 0), True),
    (("bf16", 256, 8, 2, 2, 100, 100, False, 0), True),
])
def test_forward_choice_by_size(gpu_device, monkeypatch, case, split):
    # the kernels sum in different orders: the same bits mean the same kernel
    dtype, d, b, hq, hkv, sq, skv, causal, window = case
    _, (q, k, v, _) = draw(1, b, hq, hkv, sq, skv, d, DTYPES[dtype])
    kw = dict(causal=causal, sliding_window=window, return_lse=True)
    chosen = nfa.npu_flash_attention_forward(q, k, v, **kw)
    monkeypatch.setattr(nfa, "decode_enabled", False)
    regular = nfa.npu_flash_attention_forward(q, k, v, **kw)
    assert (not all(torch.equal(x, y) for x, y in zip(chosen, regular))) == split
