"""GPU tests of the staged backward's walk under interval masks: dK/dV visits (and stages the dS of) only the query
tiles some key of its KV block may meet, and dQ reads exactly those units.

The workspace starts as NaN bytes, so that a unit read without having been written reaches dQ.  The reference is
eager float64 autograd over the same mask; tolerances are the suite's.
"""
import pytest
import torch

import flexatt_lib as L
import npu_flash_attention as nfa
from gpu_helpers import check, draw

pytestmark = pytest.mark.gpu


def _documents(lengths):
    edges = torch.tensor([0] + lengths).cumsum(0)
    lo = torch.repeat_interleave(edges[:-1], torch.tensor(lengths))
    hi = torch.repeat_interleave(edges[1:], torch.tensor(lengths))
    b = torch.stack((lo, hi), -1)
    return b, b


def _transpose(rows, skv):
    """The query rows each key meets, for non-decreasing row bounds."""
    j = torch.arange(skv)
    lo = (rows[:, 1].view(-1, 1) <= j).sum(0)
    hi = (rows[:, 0].view(-1, 1) <= j).sum(0)
    return rows, torch.stack((lo, hi), -1)


def _steps(sq, skv):
    """Row bounds that jump: key blocks no row meets, and rows that meet no key."""
    i = torch.arange(sq)
    lo = torch.where(i < 37, 0, torch.where(i < 38, 20, torch.where(i < 200, 300, 640)))
    hi = torch.where(i < 37, 10, torch.where(i < 200, 330, 900)).clamp(max=skv)
    return _transpose(torch.stack((torch.minimum(lo, hi), hi), -1), skv)


# name: (dtype, D, Hq, Hkv, Sq, Skv, causal, window, bounds)
CASES = {
    "edges_of_blocks_d128": (torch.bfloat16, 128, 4, 1, 700, 700, True, 0, lambda: _documents([128, 127, 1, 129, 255, 60])),
    "edges_of_tiles_d64": (torch.float16, 64, 2, 2, 650, 650, True, 0, lambda: _documents([32, 31, 33, 1, 159, 256, 138])),
    "not_causal_d256": (torch.bfloat16, 256, 2, 1, 520, 520, False, 0, lambda: _documents([5, 250, 1, 264])),
    "window_d128": (torch.float16, 128, 6, 2, 900, 900, True, 150, lambda: _documents([200, 500, 200])),
    "one_row_documents_d128": (torch.bfloat16, 128, 8, 8, 385, 385, False, 0, lambda: _documents([1] * 385)),
    "jumps_d128": (torch.bfloat16, 128, 4, 2, 333, 1000, False, 0, lambda: _steps(333, 1000)),
    "jumps_d64": (torch.float16, 64, 3, 1, 333, 777, False, 0, lambda: _steps(333, 777)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_walk_covers_what_dq_reads(gpu_device, case):
    dtype, d, hq, hkv, sq, skv, causal, window, bounds = CASES[case]
    rows, cols = bounds()
    (qc, kc, vc, doc), (q, k, v, do) = draw(7, 1, hq, hkv, sq, skv, d, dtype)
    i, j = torch.arange(sq).view(-1, 1), torch.arange(skv).view(1, -1)
    ok = (j >= rows[:, :1]) & (j < rows[:, 1:])
    assert torch.equal(ok, (i >= cols[:, 0]) & (i < cols[:, 1]))  # one mask, described twice
    ok = ok & ((j <= i) if causal else True) & ((i - j <= window) if window else True)

    x = [t.double().requires_grad_(True) for t in (qc, kc, vc)]
    ke, ve = (t.repeat_interleave(hq // hkv, 1) for t in x[1:])
    s = (x[0] @ ke.transpose(-1, -2)) / d ** 0.5
    e = torch.where(ok, torch.exp(s - s.detach().amax(-1, keepdim=True)), 0.0)
    ref_o = (e / e.sum(-1, keepdim=True).clamp(min=1e-300)) @ ve
    ref = torch.autograd.grad(ref_o, x, doc.double())

    dev = [t.to(torch.int32).unsqueeze(0).contiguous().cuda() for t in (rows, cols)]
    masks = nfa._Masks(causal, *dev)
    o, lse = torch.empty_like(q), torch.empty(1, hq, sq, device=q.device)
    nfa._forward_into(q, k, v, o, lse, causal=causal, sliding_window=window, alibi=None, scale=d ** -0.5, soft_cap=0.0,
                      masks=masks)
    p = nfa._problem(q, k, d ** -0.5, causal, window, 0.0, None, masks)
    lib, T = L.load(), L.tensor
    n = lib.flexatt_bwd_workspace(p)
    ws = torch.full((n,), 0xFF, dtype=torch.uint8, device=q.device)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    delta = torch.empty_like(lse)
    L.check(lib.flexatt_bwd_ws(p, T(q), T(k), T(v), T(o), T(do), lse.data_ptr(), delta.data_ptr(), T(dq), T(dk), T(dv),
                               ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream), "bwd_ws")
    torch.cuda.synchronize()
    check("o", o, ref_o, dtype)
    for name, a, r in zip(("dq", "dk", "dv"), (dq, dk, dv), ref):
        check(name, a, r, dtype)
