"""Top-k of long rows by row histogram and slices: every tie pattern, boundary bins that hold few keys,
most of them or all, lists in registers and in memory, and the decode call that counts as it scores;
and the calls that take one workgroup per row or the chunk lists instead."""

import numpy as np
import pytest
import torch

from kv_cache_amd import _lib
from kv_cache_amd import int4 as K

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rows_of(n, seed):
    g = torch.Generator().manual_seed(seed)
    few = torch.randint(-3, 4, (n,), generator=g).float()
    inf = torch.randn(n, generator=g)
    inf[torch.rand(n, generator=g) < 0.4] = -float("inf")
    return torch.stack([
        torch.randn(n, generator=g),                  # some 2% of the keys in the boundary bin
        few,                                          # large groups of equal keys
        torch.zeros(n),                               # every key equal: the lists overflow
        100.0 + torch.rand(n, generator=g),           # one bin: the lists overflow
        100.0 + 40.0 * torch.rand(n, generator=g),    # a tenth of the keys in a bin
        inf,
    ])


def want(vals, k):
    order = np.argsort(-vals.numpy(), axis=1, kind="stable")[:, :k]
    return np.sort(order, axis=1)


@pytest.mark.parametrize("n", [4097, 8192, 20003, 65536, 131072, 196608])
@pytest.mark.parametrize("share", [0.0, 0.1, 0.5, 1.0])
@pytest.mark.parametrize("copies", [1, 20])   # 6 or 120 rows: other keys per thread
def test_large_k_equals_stable_sort(n, share, copies):
    k = max(1025, min(n, int(share * n)))
    vals = rows_of(n, n + copies)
    assert _lib.load().qkv_topk_workspace_bytes(6, n, k) > 0
    ws = K.topk_workspace(6 * copies, n, k, DEV)
    ws.fill_(float("nan"))   # contents irrelevant
    dev = vals.repeat(copies, 1).to(DEV)
    for _ in range(2):
        got = K.block_topk(dev, k, workspace=ws).cpu().numpy().reshape(copies, 6, k)
        assert np.array_equal(got[0], want(vals, k))
        assert (got == got[:1]).all()


@pytest.mark.parametrize("n", [4097, 9001, 20003, 131072, 196608])
@pytest.mark.parametrize("k", [1, 300, 513, 1024])
@pytest.mark.parametrize("copies", [1, 20])
def test_boundary_bins_of_many_keys(n, k, copies):
    """Slices that hold more keys of the boundary bin than are wanted of it list only their first ones."""
    few = torch.full((2, n), -float("inf"))    # k past the finite keys: the rest is -inf, lowest index first
    few[0, 5::(n // 40)] = 1.0
    few[1, : min(n, 900)] = torch.randn(min(n, 900), generator=torch.Generator().manual_seed(k))
    narrow = 100.0 + 0.5 * torch.randn((2, n), generator=torch.Generator().manual_seed(n))
    narrow[1, n // 2 :] = 100.25               # equal keys behind distinct ones of the same bin
    vals = torch.cat([rows_of(n, n + k), few, narrow])
    rows = vals.size(0)
    ws = K.topk_workspace(rows * copies, n, k, DEV)
    got = K.block_topk(vals.repeat(copies, 1).to(DEV), k, workspace=ws).cpu().numpy().reshape(copies, rows, k)
    assert np.array_equal(got[0], want(vals, k))
    assert (got == got[:1]).all()


@pytest.mark.parametrize("rows,n,k", [(257, 4097, 700), (300, 20003, 64), (257, 33000, 1000), (512, 135169, 1000), (257, 135169, 1000),
                                      (513, 8193, 1100), (257, 12289, 1100)])
def test_more_rows_than_workgroups_at_once(rows, n, k):
    g = torch.Generator(device=DEV).manual_seed(rows)
    vals = torch.randn((rows, n), generator=g, device=DEV)
    vals[rows // 2] = 3.0
    got = K.block_topk(vals, k)
    some = [0, 1, rows // 2, 255, 256, rows - 1]
    assert np.array_equal(got[some].cpu().numpy(), want(vals[some].cpu(), k))
    order = torch.sort(vals, dim=1, descending=True, stable=True).indices[:, :k]
    assert torch.equal(got, order.sort(dim=1).values.int())


@pytest.mark.parametrize("batch,tokens,k", [(33, 33000, 700), (33, 4200, 64), (17, 9000, 1100), (4, 12288, 1500),
                                            (4, 12289, 6000), (1, 8192, 1025)])
def test_decode_topk_by_rows_and_k(batch, tokens, k):
    """Both sides of the lines between the row histogram, the chunk lists and one workgroup per row, with
    and without a kept state, which stays zero whichever is taken."""
    g = torch.Generator(device=DEV).manual_seed(tokens)
    key = torch.randn((batch, 8, tokens, 128), generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn((batch, 16, 128), generator=g, device=DEV).to(torch.bfloat16)
    cache = K.Int4KCache.from_prefill(key, 32, 16)
    scores = K.decode_scores(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, 1)
    order = torch.sort(scores.view(-1, tokens), dim=1, descending=True, stable=True).indices[:, :k]
    state = K.topk_state(batch * 8, tokens, k, DEV)
    for st in (None, state, state):
        got = K.decode_topk(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, k, state=st)
        assert torch.equal(got.view(-1, k), order.sort(dim=1).values.int())
    assert not state.any()


def test_calls_without_the_larger_workspace_still_run():
    lib = _lib.load()
    vals = rows_of(9000, 4).to(DEV)
    out = torch.empty((6, 2000), dtype=torch.int32, device=DEV)
    _lib.check(lib.qkv_topk_ws(vals.data_ptr(), 6, 9000, 9000, 2000, out.data_ptr(), None, 0, _lib.stream_of(vals)))
    assert np.array_equal(out.cpu().numpy(), want(vals.cpu(), 2000))


@pytest.mark.parametrize("tokens,k,selected", [(5000, 1024, 16), (5000, 1200, 16), (20011, 2002, 32), (70001, 7001, 64), (8192, 8192, 128)])
def test_decode_topk_counts_as_it_scores(tokens, k, selected):
    g = torch.Generator().manual_seed(tokens)
    key = torch.randn((2, 3, tokens, 128), generator=g).to(torch.bfloat16).to(DEV)
    q = torch.randn((2, 12, 128), generator=g).to(torch.bfloat16).to(DEV)
    cache = K.Int4KCache.from_prefill(key, 32, selected)
    scores = torch.empty((2, 3, tokens), device=DEV)
    got = K.decode_topk(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, k, scores=scores)
    bmax = K.decode_scores(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, 1)
    assert torch.equal(scores, bmax)
    assert np.array_equal(got.cpu().numpy().reshape(6, k), want(bmax.cpu().view(6, tokens), k))


def test_large_k_in_a_graph():
    vals = rows_of(30000, 8).to(DEV)
    ws = K.topk_workspace(6, 30000, 3000, DEV)
    out = torch.empty((6, 3000), dtype=torch.int32, device=DEV)
    K.block_topk(vals, 3000, out=out, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        K.block_topk(vals, 3000, out=out, workspace=ws)
    for seed in range(3):
        vals.copy_(rows_of(30000, 50 + seed))
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want(vals.cpu(), 3000))


@pytest.mark.parametrize("tokens,k", [(4097, 1), (9001, 300), (40000, 1024), (131072, 4000)])
def test_kept_state_returns_to_zero(tokens, k):
    g = torch.Generator().manual_seed(k)
    key = torch.randn((1, 4, tokens, 128), generator=g).to(torch.bfloat16).to(DEV)
    cache = K.Int4KCache.from_prefill(key, 32, 32)
    state = K.topk_state(4, tokens, k, DEV)
    ws = K.topk_workspace(4, tokens, k, DEV)
    for seed in range(3):
        q = torch.randn((1, 8, 128), generator=g).to(torch.bfloat16).to(DEV)
        scores = torch.empty((1, 4, tokens), device=DEV)
        got = K.decode_topk(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, k, scores=scores, workspace=ws,
                            state=state)
        assert np.array_equal(got.cpu().numpy().reshape(4, k), want(scores.cpu().view(4, tokens), k))
        assert int(state.abs().sum()) == 0
    with pytest.raises(RuntimeError, match="state needs"):
        K.decode_topk(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, k, workspace=ws, state=state[:64])


@pytest.mark.parametrize("tokens,k", [(5000, 300), (40000, 1024), (131072, 4000)])
def test_state_left_with_counts(tokens, k):
    """Counts left in a state (here k keys of the highest bin, which the row does not hold): no index
    is stale, and the call leaves the state zero, so that the next one is exact."""
    g = torch.Generator().manual_seed(k)
    key = torch.randn((1, 4, tokens, 128), generator=g).to(torch.bfloat16).to(DEV)
    cache = K.Int4KCache.from_prefill(key, 32, 32)
    q = torch.randn((1, 8, 128), generator=g).to(torch.bfloat16).to(DEV)
    state = K.topk_state(4, tokens, k, DEV)
    stride = 4096 + 64 + 8
    state[4095 : 4 * stride : stride] = k
    scores = torch.empty((1, 4, tokens), device=DEV)
    out = torch.full((1, 4, k), 7, dtype=torch.int32, device=DEV)
    K.decode_topk(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, k, scores=scores, out=out, state=state)
    assert bool((out == -1).all()) and int(state.abs().sum()) == 0
    K.decode_topk(q, cache.chan_idx, cache.slab, cache.slab_scales, tokens, k, scores=scores, out=out, state=state)
    assert np.array_equal(out.cpu().numpy().reshape(4, k), want(scores.cpu().view(4, tokens), k))


def test_state_arguments():
    key = torch.randn((1, 2, 5000, 128), generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(DEV)
    cache = K.Int4KCache.from_prefill(key, 32, 32)
    q = torch.randn((1, 4, 128), generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(DEV)
    words = K.topk_state(2, 5000, 64, DEV).numel()

    def call(state):
        return K.decode_topk(q, cache.chan_idx, cache.slab, cache.slab_scales, 5000, 64, state=state)

    with pytest.raises(RuntimeError, match="contiguous"):
        call(torch.zeros(1, dtype=torch.int32, device=DEV).expand(words))
    with pytest.raises(RuntimeError, match="device"):
        call(torch.zeros(words, dtype=torch.int32))
    with pytest.raises(RuntimeError, match="state needs"):   # bytes, not elements
        call(torch.zeros(words, dtype=torch.uint8, device=DEV))
    assert torch.equal(call(torch.zeros(words, device=DEV)), call(None))


@pytest.mark.parametrize("n,k", [(5000, 64), (9000, 1000), (131072, 1024), (196609, 500)])
def test_smaller_workspaces_take_the_chunk_lists(n, k):
    """Workspaces sized for the chunk lists (their size does not depend on the row histogram) are still accepted."""
    vals = rows_of(n, k).to(DEV)
    chunks = -(-n // 4096)
    ws = torch.empty(6 * chunks * (66 + 2 * k + 1), dtype=torch.float32, device=DEV)
    out = torch.empty((6, k), dtype=torch.int32, device=DEV)
    lib = _lib.load()
    _lib.check(lib.qkv_topk_ws(vals.data_ptr(), 6, n, n, k, out.data_ptr(), ws.data_ptr(), ws.numel() * 4,
                               _lib.stream_of(vals)))
    assert np.array_equal(out.cpu().numpy(), want(vals.cpu(), k))
