"""GPU tests of the staged dK/dV whose KV blocks' query tiles are shared by several workgroups (flexatt_bwd_ws with
flexatt_bwd_ws_parts_bytes more workspace), against the same call without them, which the staged tests hold to the oracle.

Shares of unequal length, blocks with fewer query tiles than shares (the last causal blocks), block maps whose list is
walked in shares, interval masks, and both passes of head_dim 256.  The workspace starts as NaN bytes.
"""
import pytest
import torch

import flexatt_lib as L
import npu_flash_attention as nfa
from gpu_helpers import alibi_slopes, check, draw

pytestmark = pytest.mark.gpu

# name: (dtype, D, B, Hq, Hkv, Sq, Skv, kwargs)
CASES = {
    "d128_causal": (torch.bfloat16, 128, 1, 4, 1, 700, 700, dict(causal=True)),
    "d128_full_sq_lt_skv": (torch.float16, 128, 1, 3, 1, 270, 900, {}),
    "d128_window_alibi": (torch.bfloat16, 128, 2, 2, 2, 900, 900, dict(causal=True, sliding_window=130, alibi=True)),
    "d128_blocks": (torch.float16, 128, 1, 4, 2, 1000, 1000, dict(causal=True, blocks=True)),
    "d128_documents": (torch.bfloat16, 128, 1, 4, 1, 900, 900, dict(causal=True, docs=True)),
    "d64_cap": (torch.float16, 64, 1, 7, 1, 650, 600, dict(causal=True, soft_cap=20.0)),
    "d64_blocks_documents": (torch.bfloat16, 64, 1, 4, 1, 800, 800, dict(causal=True, blocks=True, docs=True)),
    "d256_causal": (torch.bfloat16, 256, 1, 2, 1, 600, 600, dict(causal=True, soft_cap=30.0)),
    "d256_documents": (torch.float16, 256, 1, 3, 1, 520, 520, dict(docs=True)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_parts_match_whole_streams(gpu_device, case):
    dtype, d, b, hq, hkv, sq, skv, kw = CASES[case]
    kw = dict(kw)
    _, (q, k, v, do) = draw(sq, b, hq, hkv, sq, skv, d, dtype)
    if kw.pop("alibi", False):
        kw["alibi_slope"] = alibi_slopes(hq).cuda()
    ids = blocks = None
    if kw.pop("docs", False):
        ids = kw["document_ids"] = (torch.arange(sq, device="cuda") // 170).repeat(b, 1)
    if kw.pop("blocks", False):
        n = -(-sq // 128)
        g = torch.Generator().manual_seed(1)
        keep = (torch.rand(n, n, generator=g) > 0.5) | torch.eye(n, dtype=torch.bool)
        blocks = kw["block_mask"] = keep.view(1, 1, n, n).cuda()
    o, lse = nfa.npu_flash_attention_forward(q, k, v, return_lse=True, **kw)
    masks = nfa._masks(kw.get("causal", False), ids, None, blocks, b, hq, sq, skv, q.device)
    p = nfa._problem(q, k, d ** -0.5, kw.get("causal", False), kw.get("sliding_window", 0), kw.get("soft_cap", 0.0),
                     kw.get("alibi_slope"), masks)
    lib, T = L.load(), L.tensor
    band, parts = lib.flexatt_bwd_workspace(p), lib.flexatt_bwd_ws_parts_bytes(p)
    assert parts > 0 and parts % (8 * b * hkv * skv * d) == 0 and parts // (8 * b * hkv * skv * d) > 1

    def run(nbytes):
        ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=q.device)
        g = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        delta = torch.empty_like(lse)
        L.check(lib.flexatt_bwd_ws(p, T(q), T(k), T(v), T(o), T(do), lse.data_ptr(), delta.data_ptr(), T(g[0]), T(g[1]),
                                   T(g[2]), ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream), "bwd_ws")
        torch.cuda.synchronize()
        return g

    want, got, again = run(band), run(band + parts), run(band + parts)
    assert torch.equal(got[0], want[0])  # the same staged dS
    for name, x, y, w in zip(("dq", "dk", "dv"), got, again, want):
        assert torch.equal(x, y)
        check(name, x, w, dtype)
