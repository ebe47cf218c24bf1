"""Prefill block scores where the two-blocks-ahead loads of a key chunk begin
and end: chunks of 1 to 4 and of 15 to 16 visible blocks, ending in unmasked
and in masked blocks of either parity, with 1, 2 and 4 waves per workgroup."""

import numpy as np
import pytest
import torch

from kv_cache_amd import int4 as K
from kv_cache_amd import prefill as P
from oracle import qkv_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 15, 16, 17, 18, 19, 20])
@pytest.mark.parametrize("hidden", [0, 70, 200])
def test_block_scores_at_chunk_edges_match_oracle(group, blocks, hidden):
    # The queries stand at the end (hidden = 0: the walk's last blocks need no
    # mask but for the ragged one) or `hidden` tokens before it (its last
    # blocks are masked, or seen by no query).
    t = 64 * blocks - 5
    nq = min(3, t)
    q_pos0 = max(t - nq - hidden, 0)
    g = torch.Generator().manual_seed(100 * blocks + hidden + group)
    q = torch.randn((1, 2 * group, nq, 128), generator=g).to(torch.bfloat16)
    k = torch.randn((1, 2, t, 128), generator=g).to(torch.bfloat16)
    packed, scales = K.int4_pack_k(k.to(DEV), 128)
    q8, _ = P.quantize_query(q.to(DEV))
    got = P.block_scores(q8, packed, scales, t, q_pos0).cpu().numpy()
    want_q8, _ = O.quantize_query_rows(q.float().numpy())
    kp, ks = O.int4_pack_k(k.float().numpy(), 128)
    want = O.prefill_block_scores(want_q8, kp, ks[..., 0], 64, q_pos0)
    # whole numbers scaled by one rounding each: bit-equal
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
