"""flexatt_document_bounds: the kernel that turns document ids into interval bounds, against the tensor-operation form
of the same bounds (``_doc_bounds`` without ``native``), at the edges of its 8192-position chunks."""
import pytest
import torch

import flexatt_lib as L
import npu_flash_attention as nfa

FAKE = 1 << 20  # an aligned non-null address that is never dereferenced


@pytest.mark.parametrize("args, status", [
    ((None, 4, 1, 8, FAKE), -1), ((FAKE, 4, 1, 8, None), -1), ((FAKE, 3, 1, 8, FAKE), -1), ((FAKE, 4, 0, 8, FAKE), -1),
    ((FAKE, 4, 1, 0, FAKE), -1), ((FAKE, 4, 1 << 16, 1 << 15, FAKE), -4), ((FAKE + 4, 8, 1, 8, FAKE), -5),
])
def test_rejections(args, status):
    assert L.load().flexatt_document_bounds(*args, None) == status


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.int16, torch.uint8])
@pytest.mark.parametrize("b, s, mean", [(1, 1, 1), (3, 7, 2), (2, 8192, 50), (1, 8191, 9000), (2, 8193, 1),
                                        (1, 20000, 6000), (2, 16384, 16384)])
def test_bounds_match_tensor_operations(gpu_device, b, s, mean, dtype):
    g = torch.Generator().manual_seed(s + mean)
    starts = torch.rand(b, s, generator=g) < 1.0 / mean
    ids = (starts.cumsum(1) % 3).to(dtype)  # neighbours differ, values repeat
    wide = torch.stack((ids, ids + 1), -1).cuda()[..., 0]  # not contiguous
    want = nfa._doc_bounds(ids, b, s, s, "cpu")
    for x in (ids.cuda(), wide):
        got = nfa._doc_bounds(x, b, s, s, "cuda", native=True)
        assert got.dtype == torch.int32 and torch.equal(got.cpu(), want)


@pytest.mark.gpu
def test_wide_ids_take_tensor_operations(gpu_device):
    ids = torch.tensor([[1, 1, 2, 2, 2, 1]]).to(torch.complex128)
    want = nfa._doc_bounds(ids, 1, 6, 6, "cpu")
    assert torch.equal(nfa._doc_bounds(ids.cuda(), 1, 6, 6, "cuda", native=True).cpu(), want)
