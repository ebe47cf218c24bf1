"""A workspace sized once, for the longest row or the capacity, is never too small for a shorter one (host only)."""

import math

import pytest

from kv_cache_amd import _lib

lib = _lib.load()
# both sides of every length at which a selection changes its path: 4096-key chunks, one workgroup's
# 40960 positions, the row histogram's 196608, 64 chunks
LENGTHS = sorted({n + d for n in (1, 4096, 8192, 20000, 34133, 40960, 65536, 100000, 131072, 163840, 196608, 200000,
                                  204800, 262144, 300000) for d in (-1, 0, 1) if n + d > 0})


def budget(n, fraction):
    return min(n, max(1, math.ceil(fraction * n)))


@pytest.mark.parametrize("rows", [1, 8, 32, 300])
@pytest.mark.parametrize("k", [1, 64, 513, 1000, 1024])
def test_topk_size_grows_with_the_row(rows, k):
    sizes = [lib.qkv_topk_workspace_bytes(rows, n, k) for n in LENGTHS if n >= k]
    assert sizes == sorted(sizes)


@pytest.mark.parametrize("rows", [1, 8, 32, 300])
@pytest.mark.parametrize("fraction", [0.0, 0.0004, 0.005, 0.02, 0.03, 0.1, 1.0])
def test_sizes_at_the_capacity_cover_shorter_histories(rows, fraction):
    sizes = {
        "qabs_candidates": lambda n: lib.qkv_qabs_candidates_workspace_bytes(rows, n, fraction),
        "qabs_candidate_select": lambda n: lib.qkv_qabs_candidate_select_workspace_bytes(rows, n, fraction),
        "reuse_select": lambda n: lib.qkv_reuse_select_workspace_bytes(rows, n, fraction),
        "reuse_candidates": lambda n: lib.qkv_reuse_candidates_workspace_bytes(rows, n, budget(n, fraction)),
        "threshold_mask": lambda n: lib.qkv_threshold_mask_workspace_bytes(rows, n, budget(n, fraction)),
    }
    for name, size in sizes.items():
        got = [size(n) for n in LENGTHS]
        assert got[0] >= 0 and got == sorted(got), name


@pytest.mark.parametrize("rows,fraction,capacity,history", [
    (32, 0.03, 262144, 65536), (32, 0.03, 262144, 131072), (32, 0.03, 262144, 196608), (32, 0.03, 262144, 30000),
    (8, 0.01, 196610, 196608), (8, 0.01, 300000, 4097)])
def test_candidate_attention_step_sizes(rows, fraction, capacity, history):
    """QabsCandidateAttentionStep sizes its workspace once, at capacity - 1 history tokens."""
    assert lib.qkv_qabs_candidates_workspace_bytes(rows, capacity - 1, fraction) >= \
        lib.qkv_qabs_candidates_workspace_bytes(rows, history, fraction)
