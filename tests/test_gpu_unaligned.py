"""Dim-major copies whose rows start at any element (odd capacities, odd offsets): the partial scores and
the one-launch candidates equal the oracle's, as they do on aligned copies."""

import numpy as np
import pytest
import torch

from kv_cache_amd import _lib
from kv_cache_amd import reuse as RU
from oracle import ref_semantics as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def copy_at(k, offset, pad):
    """K [B, H, T, D] as a dim-major view [B, H, D, T] whose rows start `offset` elements into rows of T + pad."""
    b, h, t, d = k.shape
    buf = torch.zeros((b, h, d, t + pad), dtype=k.dtype, device=DEV)
    view = buf[..., offset:offset + t]
    view.copy_(k.transpose(2, 3))
    return view


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("offset,pad", [(0, 0), (1, 1), (3, 4), (7, 8)])
@pytest.mark.parametrize("batch,hist", [(1, 1), (1, 7), (1, 8), (1, 9), (1, 2049), (1, 2055),
                                        (32, 1003)])   # (32 x 4 rows: the one-launch candidates)
def test_partial_scores_at_any_alignment(dtype, offset, pad, batch, hist):
    g = torch.Generator().manual_seed(hist + offset)
    hq, hkv, d, dims = 4, 2, 128, 12
    k = torch.randn((batch, hkv, hist, d), generator=g).to(dtype).to(DEV)
    q = torch.randint(-3, 4, (batch, hq, d), generator=g).to(dtype).to(DEV)   # |q| ties: the lower dim first
    kdm = copy_at(k, offset, pad)
    want = R.partial_scores(q.float().cpu().numpy(), np.repeat(k.float().cpu().numpy(), hq // hkv, axis=1), dims)
    got = RU.reuse_partial_scores(q, kdm, hist, dims).cpu().numpy().reshape(batch, hq, hist)
    assert np.array_equal(got, want)
    lib = _lib.load()
    rows, keep = batch * hq, max(1, hist // 20)
    need = lib.qkv_reuse_candidates_workspace_bytes(rows, hist, keep)
    ws = torch.zeros((need + 3) // 4, dtype=torch.float32, device=DEV)
    partial = torch.empty((rows, hist), dtype=torch.float32, device=DEV)
    bits = torch.zeros((rows, -(-hist // 64)), dtype=torch.int64, device=DEV)
    _lib.check(lib.qkv_reuse_candidates(
        q.data_ptr(), kdm.data_ptr(), _lib.strides(*kdm.stride()), _lib.DTYPE_CODES[dtype], batch, hq, hkv, hist, d,
        dims, keep, partial.data_ptr(), hist, None, 0, bits.data_ptr(), bits.stride(0), None, ws.data_ptr(),
        ws.numel() * 4, _lib.stream_of(q)))
    assert np.array_equal(partial.cpu().numpy().reshape(batch, hq, hist), want)
    flat = want.reshape(rows, hist)
    kth = np.sort(flat, axis=1)[:, hist - keep][:, None]
    assert np.array_equal(RU.expand_bits(bits, hist).cpu().numpy(), flat >= kth)
