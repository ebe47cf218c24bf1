"""The one-workgroup-per-row selections at the edges of their keys-per-thread classes: rows of equal,
few-valued and normal scores, against a stable sort."""

import numpy as np
import pytest
import torch

from kv_cache_amd import _lib
from kv_cache_amd import reuse as RU

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("step", [4, 8, 12, 16, 20, 24, 28, 32, 40])   # keys per thread
@pytest.mark.parametrize("edge", [0, 1])
def test_selection_and_mask_at_class_edges(step, edge):
    n = 1024 * step + edge if step < 40 else 1024 * 40 - edge
    g = torch.Generator().manual_seed(n)
    rows = torch.stack([torch.randn(n, generator=g), torch.randint(0, 5, (n,), generator=g).float(),
                        torch.zeros(n), torch.randn(n, generator=g)])
    rows[3, ::3] = -float("inf")
    frac = 0.07
    keep = int(np.ceil(frac * n))
    idx, valid, _, mask = RU.qabs_candidate_select(rows.to(DEV), n + 1, frac, 0, 0, False)
    order = np.argsort(-rows.numpy(), axis=1, kind="stable")[:, :keep]
    want = np.sort(order, axis=1)
    assert np.array_equal(idx[:, :keep].cpu().numpy(), want)
    hit = np.zeros(rows.shape, dtype=bool)
    np.put_along_axis(hit, want, True, axis=1)
    assert np.array_equal(mask.cpu().numpy(), hit) and bool(valid.all())
    kth = np.sort(rows.numpy(), axis=1)[:, n - keep][:, None]
    got = torch.zeros((4, n), dtype=torch.uint8, device=DEV)
    need = _lib.load().qkv_threshold_mask_workspace_bytes(4, n, keep)
    ws = torch.empty(max(1, need // 4 + 1), dtype=torch.float32, device=DEV)
    RU.threshold_mask(rows.to(DEV), n, keep, got, ws)
    assert np.array_equal(got.cpu().numpy().astype(bool), rows.numpy() >= kth)
