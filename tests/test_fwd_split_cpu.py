"""flexatt_fwd_split's range and argument checks (no kernel is launched)."""
import pytest

import flexatt_lib as L
from test_capi_cpu import FAKE, problem, tens


@pytest.mark.parametrize("kw, inside", [
    (dict(head_dim=256, seqlen_q=1), True), (dict(head_dim=128, seqlen_q=16), True), (dict(head_dim=64, seqlen_q=17), False),
    (dict(head_dim=256, seqlen_q=1, dtype=L.F32), False), (dict(seqlen_q=1, block_map=FAKE, block_heads=1), False),
    (dict(seqlen_q=1, seqlen_kv=1, doc_bounds=FAKE), False), (dict(head_dim=96, seqlen_q=1), False),
])
def test_split_workspace_range(kw, inside):
    lib, p = L.load(), problem(**kw)
    n = lib.flexatt_fwd_split_workspace(p)
    assert (n > 0) == inside
    if inside and kw["head_dim"] <= 128:
        assert n == lib.flexatt_fwd_decode_workspace(p)


def test_split_rejections():
    lib, p = L.load(), problem(head_dim=256, seqlen_q=1)
    t = tens(stride_s=256, stride_h=64 * 256, stride_b=4 * 64 * 256)
    need = lib.flexatt_fwd_split_workspace(p)
    assert lib.flexatt_fwd_split(problem(head_dim=256, seqlen_q=64), t, t, t, t, FAKE, FAKE, need, None) == -6
    assert lib.flexatt_fwd_split(p, t, t, t, t, FAKE, FAKE, need - 1, None) == -1
    assert lib.flexatt_fwd_split(p, t, t, t, t, FAKE, None, need, None) == -1
    assert lib.flexatt_fwd_split(p, t, t, t, t, None, FAKE, need, None) == -1
    assert lib.flexatt_fwd_split(p, t, t, t, t, FAKE, FAKE + 8, need, None) == -5


@pytest.mark.parametrize("kw, code", [
    (dict(head_dim=256), -6), (dict(dtype=L.F32, head_dim=256), -6), (dict(block_map=FAKE, block_heads=1), -6), (dict(head_dim=48), -3),
])
def test_bwd_split_range(kw, code):
    lib, p = L.load(), problem(**kw)
    t = tens(stride_s=p.head_dim, stride_h=64 * p.head_dim, stride_b=4 * 64 * p.head_dim)
    assert lib.flexatt_bwd_prefers_split(p) == 0 and lib.flexatt_bwd_split_workspace(p) == 0
    assert lib.flexatt_bwd_split(p, t, t, t, t, t, FAKE, FAKE, t, t, t, None, 0, None) == code


def test_bwd_split_workspace_checks():
    lib, p, t = L.load(), problem(heads_q=16, heads_kv=1, seqlen_q=640, seqlen_kv=640), tens(stride_h=640 * 64,
                                                                                             stride_b=16 * 640 * 64)
    need = lib.flexatt_bwd_split_workspace(p)
    assert lib.flexatt_bwd_prefers_split(p) == 1 and need > 0  # the sums of two or more splits
    args = (p, t, t, t, t, t, FAKE, FAKE, t, t, t)
    assert lib.flexatt_bwd_split(*args, None, need, None) == -1
    assert lib.flexatt_bwd_split(*args, FAKE, need - 1, None) == -1
    assert lib.flexatt_bwd_split(*args, FAKE + 8, need, None) == -5
