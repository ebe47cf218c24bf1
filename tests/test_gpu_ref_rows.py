"""The row-staging partial scores and the compacted candidate scores at the edges of their tiles and at any
alignment, and the int32 list ids, against the oracle."""

import numpy as np
import pytest
import torch

from kv_cache_amd import _lib
from kv_cache_amd import qabs_cuda_kernels as Q
from oracle import ref_semantics as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("keys", [1, 63, 64, 65, 129, 1025, 2050])
@pytest.mark.parametrize("pad", [0, 1, 8])   # elements before each row: unaligned rows for 1
def test_scores_at_tile_edges(dtype, keys, pad):
    g = torch.Generator().manual_seed(keys + pad)
    b, h, d, dims = 2, 3, 128, 13
    buf = torch.randn((b, h, keys, d + pad), generator=g).to(dtype).to(DEV)
    k = buf[..., pad:]
    q = (torch.randint(-9, 10, (b, h, d), generator=g) * 0.25).to(dtype).to(DEV)
    qn, kn = q.float().cpu().numpy(), k.float().cpu().numpy()
    assert np.array_equal(Q.partial_scores(q, k, dims).cpu().numpy(), R.partial_scores(qn, kn, dims))
    masks = [torch.rand((b, h, keys), generator=g) < p for p in (0.1, 0.3, 0.02)]
    for prev, fin, sink, recent in ((None, None, 0, 0), (masks[1], masks[2], 4, 16), (None, masks[2], keys + 5, 0),
                                    (masks[1], None, 1, keys + 5)):
        got = Q.candidate_full_scores(q, k, masks[0].to(DEV), None if prev is None else prev.to(DEV),
                                      None if fin is None else fin.to(DEV), sink, recent, 0.3).cpu().numpy()
        want = R.candidate_full_scores(qn, kn, masks[0].numpy(), None if prev is None else prev.numpy(),
                                       None if fin is None else fin.numpy(), sink, recent, 0.3)
        assert np.array_equal(got, want)


# both sides of the lines between whole rows and single dims: 61 and 203 MB of fp32, 406 MB of bf16
@pytest.mark.parametrize("dtype,keys,dims", [(torch.float32, 3900, 4), (torch.float32, 3900, 5), (torch.float32, 13000, 5),
                                             (torch.float32, 13000, 6), (torch.bfloat16, 52000, 1),
                                             (torch.bfloat16, 52000, 2)])
def test_few_dims_of_a_large_history(dtype, keys, dims):
    g = torch.Generator(device=DEV).manual_seed(keys + dims)
    k = torch.randn((1, 32, keys, 128), generator=g, device=DEV).to(dtype)
    q = torch.randn((1, 32, 128), generator=g, device=DEV).to(dtype)
    got = Q.partial_scores(q, k, dims)
    for h in (0, 17, 31):
        want = R.partial_scores(q[:, h : h + 1].float().cpu().numpy(), k[:, h : h + 1].float().cpu().numpy(), dims)
        assert np.array_equal(got[:, h : h + 1].cpu().numpy(), want)


def test_token_ids():
    idx = torch.tensor([0, 5, 6, -1, 2 ** 40, -2 ** 40, 3, 2 ** 32 + 1], device=DEV)
    valid = torch.tensor([1, 1, 1, 1, 1, 1, 0, 1], dtype=torch.uint8, device=DEV)
    ids = torch.empty(8, dtype=torch.int32, device=DEV)
    lib = _lib.load()
    _lib.check(lib.qkv_token_ids(idx.data_ptr(), valid.data_ptr(), 8, 6, ids.data_ptr(), _lib.stream_of(idx)))
    assert ids.tolist() == [0, 5, -1, -1, -1, -1, -1, -1]
    assert lib.qkv_token_ids(idx.data_ptr(), valid.data_ptr(), -1, 6, ids.data_ptr(), _lib.stream_of(idx)) == -1
