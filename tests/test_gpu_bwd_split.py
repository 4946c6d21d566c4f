"""GPU tests of the backward that runs dK/dV and dQ in one launch with the streams split over waves and workgroups
(flexatt_bwd_split), called through the C ABI whatever flexatt_bwd_prefers_split says, and of the kernels it takes small
problems from (the API with ds_staging_enabled off) at the same sizes.

Sizes sit at the edges of the 32-row tiles, of the packed rows (G not a power of two) and of the waves' and splits' shares
(fewer tiles than waves); the reference is the float64 oracle at the suite's tolerances.  The sums' workspace starts as
NaN bytes.
"""
import pytest
import torch

import flexatt_lib as L
import npu_flash_attention as nfa
from gpu_helpers import alibi_slopes, check, draw
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu

FLAGS = {
    "causal": dict(causal=True),
    "full_scale_negative": dict(scale=-0.1),
    "window_alibi": dict(causal=True, sliding_window=40, alibi=True),
    "cap_wide_window": dict(sliding_window=(1 << 31) - 1, soft_cap=15.0),
    "documents": dict(causal=True, docs=True),
}
# (dtype, D, B, Hq, Hkv, Sq, Skv)
SHAPES = [
    (torch.float16, 32, 2, 3, 1, 1, 33),
    (torch.bfloat16, 32, 1, 8, 8, 257, 257),
    (torch.bfloat16, 64, 1, 7, 1, 33, 129),
    (torch.float16, 64, 1, 2, 2, 1025, 1025),  # eight waves
    (torch.bfloat16, 64, 1, 8, 1, 300, 300),   # several workgroups a stream
    (torch.bfloat16, 128, 1, 6, 2, 95, 97),
    (torch.float16, 128, 1, 8, 1, 420, 420),   # several workgroups a stream
    (torch.bfloat16, 128, 2, 1, 1, 32, 1),
    (torch.float32, 32, 1, 3, 1, 70, 70),
    (torch.float32, 64, 2, 2, 2, 1, 33),
    (torch.float32, 128, 1, 6, 2, 95, 97),
    (torch.float32, 128, 1, 8, 1, 260, 260),   # several workgroups a stream
]


def _case(shape, flags):
    dtype, d, b, hq, hkv, sq, skv = shape
    kw = dict(FLAGS[flags])
    cpu, dev = draw(sq + d, b, hq, hkv, sq, skv, d, dtype)
    ref = {}
    if kw.pop("alibi", False):
        kw["alibi_slope"] = alibi_slopes(hq).cuda()
    if kw.pop("docs", False):
        if sq != skv:
            pytest.skip("documents need Sq == Skv")
        ids = (torch.arange(sq) // 45).repeat(b, 1)
        ref["document_ids"], kw["document_ids"] = ids, ids.cuda()
    sl = kw.get("alibi_slope")
    want = orc.backward(*cpu, kw.get("causal", False), kw.get("sliding_window", 0), None if sl is None else sl.cpu(),
                        kw.get("scale"), kw.get("soft_cap", 0.0), **ref)
    return dtype, cpu, dev, kw, want


@pytest.mark.parametrize("flags", list(FLAGS))
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"d{s[1]}_b{s[2]}_h{s[3]}_{s[4]}_{s[5]}x{s[6]}")
def test_split_matches_oracle(gpu_device, shape, flags):
    dtype, _, (q, k, v, do), kw, want = _case(shape, flags)
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, **kw)
    b, hq, sq, d = q.shape
    masks = nfa._masks(kw.get("causal", False), kw.get("document_ids"), None, None, b, hq, sq, k.shape[2], q.device)
    p = nfa._problem(q, k, kw.get("scale") or d ** -0.5, kw.get("causal", False), kw.get("sliding_window", 0),
                     kw.get("soft_cap", 0.0), kw.get("alibi_slope"), masks)
    lib, T = L.load(), L.tensor
    n = lib.flexatt_bwd_split_workspace(p)
    ws = torch.full((max(n, 16),), 0xFF, dtype=torch.uint8, device=q.device)

    def run():
        g = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        delta = torch.empty_like(lse)
        L.check(lib.flexatt_bwd_split(p, T(q), T(k), T(v), T(o), T(do), lse.data_ptr(), delta.data_ptr(), T(g[0]),
                                      T(g[1]), T(g[2]), ws.data_ptr() if n else None, n,
                                      torch.cuda.current_stream().cuda_stream), "flexatt_bwd_split")
        return g

    got = run()
    for name, x, r, y in zip(("dq", "dk", "dv"), got, want, run()):
        check(name, x, r, dtype)
        assert torch.equal(x, y)


@pytest.mark.parametrize("flags", list(FLAGS))
@pytest.mark.parametrize("shape", SHAPES[:6] + SHAPES[8:11],
                         ids=lambda s: f"d{s[1]}_b{s[2]}_h{s[3]}_{s[4]}_{s[5]}x{s[6]}")
def test_other_backward_at_the_same_sizes(gpu_device, monkeypatch, shape, flags):
    monkeypatch.setattr(nfa, "ds_staging_enabled", False)
    dtype, _, (q, k, v, do), kw, want = _case(shape, flags)
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, **kw)
    for name, x, r in zip(("dq", "dk", "dv"), nfa.npu_flash_attention_backward(q, k, v, o, lse, do, **kw), want):
        check(name, x, r, dtype)


@pytest.mark.parametrize("split", [True, False], ids=["split", "other"])
@pytest.mark.parametrize("hq, sq", [(2, 8), (6, 8), (2, 33)])
def test_fp16_d32_rounds_ds_with_the_scale(gpu_device, monkeypatch, hq, sq, split):
    # large (loss-scaled) gradients: dS reaches 8e4 without the scale, past fp16's 65504, and 1.4e4 with it
    cpu, dev = draw(3, 1, hq, 2, sq, 5, 32, torch.float16)
    for q, k, v, do in (cpu, dev):
        q.mul_(0.1), k.mul_(0.1), v.mul_(2), do.mul_(12000)
    ds = orc.score_grad(*cpu).abs().max().item()
    assert 70000 < ds < 65504 * 32 ** 0.5
    monkeypatch.setattr(nfa, "ds_staging_auto", split)
    want = orc.backward(*cpu)
    q, k, v, do = dev
    p = nfa._problem(q, k, 32 ** -0.5, False, 0, 0.0, None)
    assert L.load().flexatt_bwd_prefers_split(p) == 1
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True)
    for name, x, r in zip(("dq", "dk", "dv"), nfa.npu_flash_attention_backward(q, k, v, o, lse, do), want):
        check(name, x, r, torch.float16)
