"""GPU tests of the forward that splits a row tile's keys over the waves of a workgroup, which flexatt_fwd takes where
the query rows fill too few regular workgroups, of flexatt_fwd_split at head_dim 256, and of the regular forward at the
same small lengths (a batch large enough to fill the chip).

Sizes sit at the edges of the 32-row tiles and of the waves' shares (one tile, fewer tiles than waves, one more than a
multiple); the reference is the float64 oracle at the suite's tolerances.
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
    "cap_window_both_sides": dict(sliding_window=65, soft_cap=15.0),
    "documents": dict(causal=True, docs=True),
}
# (dtype, D, B, Hq, Hkv, Sq, Skv)
SHAPES = [
    (torch.float16, 32, 2, 3, 1, 1, 33),
    (torch.bfloat16, 32, 1, 8, 8, 257, 257),
    (torch.float16, 64, 1, 7, 1, 33, 129),
    (torch.bfloat16, 64, 2, 2, 2, 1025, 1025),  # eight waves
    (torch.bfloat16, 128, 1, 6, 2, 95, 97),
    (torch.float16, 128, 1, 2, 1, 2049, 2049),  # eight waves
    (torch.bfloat16, 256, 1, 4, 2, 130, 160),
    (torch.float32, 32, 1, 3, 1, 70, 70),
    (torch.float32, 64, 1, 2, 2, 1, 33),
    (torch.float32, 128, 1, 6, 2, 95, 97),
    # a full grid: the regular forward
    (torch.float32, 32, 48, 16, 8, 100, 100),
    (torch.float32, 128, 48, 16, 8, 60, 60),
    (torch.bfloat16, 64, 64, 32, 8, 150, 150),
    (torch.float16, 128, 24, 16, 8, 150, 150),
]


@pytest.mark.parametrize("flags", list(FLAGS))
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"d{s[1]}_b{s[2]}_h{s[3]}_{s[5]}x{s[6]}")
def test_forward_matches_oracle(gpu_device, shape, flags):
    dtype, d, b, hq, hkv, sq, skv = shape
    kw = dict(FLAGS[flags])
    cpu, (q, k, v, _) = draw(sq + d, b, hq, hkv, sq, skv, d, dtype)
    ref = {}
    if kw.pop("alibi", False):
        kw["alibi_slope"] = alibi_slopes(hq).cuda()
    if kw.pop("docs", False):
        if sq != skv:
            pytest.skip("documents need Sq == Skv")
        ids = (torch.arange(sq) // 45).repeat(b, 1)
        ref["document_ids"], kw["document_ids"] = ids, ids.cuda()
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, **kw)
    sl = kw.get("alibi_slope")
    want, want_lse = orc.forward(*cpu[:3], kw.get("causal", False), kw.get("sliding_window", 0),
                                 None if sl is None else sl.cpu(), kw.get("scale"), kw.get("soft_cap", 0.0), **ref)
    check("o", o, want, dtype)
    check("lse", lse, want_lse, dtype)


@pytest.mark.parametrize("sq, skv, hq, hkv", [(1, 1, 2, 1), (1, 257, 8, 8), (4, 1000, 16, 8), (3, 4097, 10, 1)])
@pytest.mark.parametrize("cap", [0.0, 30.0])
def test_decode_d256_matches_oracle(gpu_device, sq, skv, hq, hkv, cap):
    cpu, (q, k, v, _) = draw(skv, 2, hq, hkv, sq, skv, 256, torch.bfloat16)
    p = nfa._problem(q, k, 1 / 16, False, 0, cap, None)
    lib = L.load()
    assert lib.flexatt_fwd_decode_workspace(p) == 0 and lib.flexatt_fwd_split_workspace(p) > 0
    # strided storage [B, S, H, D] as well
    for x in ((q, k, v), tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))):
        o, lse = nfa.npu_flash_attention_forward(*x, return_lse=True, scale=1 / 16, soft_cap=cap)
        want, want_lse = orc.forward(*cpu[:3], False, 0, None, 1 / 16, cap)
        check("o", o, want, torch.bfloat16)
        check("lse", lse, want_lse, torch.bfloat16)


# (head_dim, partials of a row): 1024 / D partial columns are merged at once, four of each
@pytest.mark.parametrize("d, ns", [(256, 2), (256, 17), (256, 65), (128, 3), (128, 33), (64, 64), (64, 65), (32, 129),
                                   (32, 256)])
def test_merge_of_partials(gpu_device, d, ns):
    skv = 256 * ns - 5
    cpu, (q, k, v, _) = draw(ns, 1, 3, 1, 2, skv + 5, d, torch.bfloat16)
    cpu, (k, v) = (cpu[0], cpu[1][:, :, :skv], cpu[2][:, :, :skv]), (k[:, :, :skv], v[:, :, :skv])
    p = nfa._problem(q, k, 0.1, False, 0, 0.0, None)
    # 3 heads x 2 query rows, D + 1 floats a partial
    assert L.load().flexatt_fwd_split_workspace(p) == 6 * ns * (d + 1) * 4
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, scale=0.1)
    want, want_lse = orc.forward(*cpu, False, 0, None, 0.1, 0.0)
    check("o", o, want, torch.bfloat16)
    check("lse", lse, want_lse, torch.bfloat16)


def _planted(what, d, sq, skv, dtype):
    cpu, dev = draw(d + skv, 1, 4, 2, sq, skv, d, dtype)
    for q, k, v, _ in (cpu, dev):
        t, x = {"nan_query": (q[0, 1, 1], "nan"), "nan_key": (k[0, 1, skv - 5], "nan"), "inf_value": (v[0, 0, skv - 5], "inf")}[what]
        t[3] = float(x)
    return cpu, dev


def _check_planted(cpu, dev, dtype, **kw):
    o, lse = nfa.npu_flash_attention_forward(*dev[:3], return_lse=True, **kw)
    want, want_lse = orc.forward(*cpu[:3])
    assert torch.equal(o.isnan().cpu(), want.isnan()) and torch.equal(lse.isnan().cpu(), want_lse.isnan())
    check("o", o, want, dtype)
    check("lse", lse, want_lse, dtype)


@pytest.mark.parametrize("what", ["nan_query", "nan_key", "inf_value"])
@pytest.mark.parametrize("d, sq, skv", [(64, 2, 40), (64, 2, 3000), (128, 2, 3000), (256, 2, 40), (256, 2, 3000),
                                        (64, 200, 200), (128, 200, 200), (256, 100, 100)])
def test_nan_and_inf_reach_the_row(gpu_device, d, sq, skv, what):
    # one workgroup a row tile (40, 100, 200) and partials merged (3000): a row with a NaN score is not an empty row,
    # and the partials that the merge reads past the last one add nothing
    cpu, dev = _planted(what, d, sq, skv, torch.bfloat16)
    _check_planted(cpu, dev, torch.bfloat16)


@pytest.mark.parametrize("what", ["nan_query", "nan_key", "inf_value"])
@pytest.mark.parametrize("dtype, d", [(torch.bfloat16, 32), (torch.float16, 64), (torch.bfloat16, 128), (torch.bfloat16, 256),
                                      (torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.float32, 256)])
def test_nan_and_inf_reach_the_row_in_the_other_kernels(gpu_device, dtype, d, what):
    # the regular forward (a block map, here of all blocks, keeps a small problem there) and the fp32 kernels
    cpu, dev = _planted(what, d, 200, 150, dtype)
    _check_planted(cpu, dev, dtype, block_mask=torch.ones(1, 1, 2, 2, dtype=torch.bool, device="cuda"))
    _check_planted(cpu, dev, dtype)
