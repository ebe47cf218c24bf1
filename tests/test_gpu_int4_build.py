"""Pack, channel statistic and slab at the edges of their tiles, against the oracle."""

import numpy as np
import pytest
import torch

from kv_cache_amd import _lib
from kv_cache_amd import int4 as K
from oracle import qkv_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def f32(t):
    return t.float().cpu().numpy()


def make(b, h, t, d, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    k = torch.randn((b, h, t, d), generator=g) * scale
    k[..., 5] *= 8.0
    k[:, :, ::7] *= torch.rand((b, h, (t + 6) // 7, 1), generator=g)
    return k.to(dtype).to(DEV)


# one token, a tile of the pack (64 tokens at D = 128) and of the slab (64), a chunk of the statistic (128), +- 1
@pytest.mark.parametrize("tokens", [1, 63, 64, 65, 127, 128, 129, 1000])
@pytest.mark.parametrize("d,group,count", [(64, 32, 16), (64, 64, 64), (128, 32, 32), (128, 128, 64), (128, 64, 128),
                                           (256, 128, 128), (256, 32, 16)])
def test_build_edges(tokens, d, group, count):
    dtype = torch.float16 if (tokens + d) % 2 else torch.bfloat16
    key = make(2, 3, tokens, d, dtype, tokens + d)
    packed, scales = K.int4_pack_k(key, group)
    want_p, want_s = O.int4_pack_k(f32(key), group)
    assert np.array_equal(packed[:, :, :tokens].cpu().numpy(), want_p)
    assert np.array_equal(scales[:, :, :tokens].view(torch.int16).cpu().numpy().view(np.uint16), want_s)
    chan, stats = K.select_channels(packed, scales, tokens, group, count)
    want = O.channel_stats(want_p, want_s, group)
    assert np.array_equal(stats.cpu().numpy().view(np.uint64).reshape(6, d), want.reshape(6, d))
    assert np.array_equal(chan.cpu().numpy().reshape(6, count), O.select_channels(want.reshape(6, d), count))
    slabs = []
    for kk in (key, unaligned(key)):   # 16-byte rows, and the path for any alignment
        slab = torch.zeros((2, 3, K.round_capacity(tokens), count // 2), dtype=torch.uint8, device=DEV)
        ss = torch.zeros(slab.shape[:3], dtype=torch.float16, device=DEV)
        K.build_slab(kk, chan, slab=slab, slab_scales=ss)
        slabs.append((slab.cpu().numpy(), ss.view(torch.int16).cpu().numpy().view(np.uint16)))
    want_slab, want_ss = O.build_slab(f32(key).reshape(6, tokens, d), chan.cpu().numpy().reshape(6, count))
    want_stored = O.swizzle_slab(want_slab, K.round_capacity(tokens))
    for slab, ss in slabs:
        assert np.array_equal(slab.reshape(6, -1), want_stored)
        assert np.array_equal(ss.reshape(6, -1)[:, :tokens], want_ss)


def unaligned(key):
    b, h, t, d = key.shape
    buf = torch.zeros((b, h, t, d + 2), dtype=key.dtype, device=DEV)
    buf[..., 1:d + 1] = key
    return buf[..., 1:d + 1]


@pytest.mark.parametrize("dtype,scale", [(torch.float16, 2.0e4), (torch.bfloat16, 1.0e6), (torch.float16, 1.0e-6)])
def test_scales_at_the_ends_of_fp16(dtype, scale):
    """Scales of 256 and more (the statistic's high words), saturated ones, subnormal and zero ones."""
    key = make(1, 2, 300, 128, dtype, 3, scale).clamp(-6.0e4, 6.0e4) if dtype is torch.float16 else \
        make(1, 2, 300, 128, dtype, 3, scale)
    packed, scales = K.int4_pack_k(key, 64)
    want_p, want_s = O.int4_pack_k(f32(key), 64)
    assert np.array_equal(packed[:, :, :300].cpu().numpy(), want_p)
    chan, stats = K.select_channels(packed, scales, 300, 64, 32)
    want = O.channel_stats(want_p, want_s, 64)
    assert np.array_equal(stats.cpu().numpy().view(np.uint64).reshape(2, 128), want.reshape(2, 128))


def test_nan_and_infinity():
    """A NaN is left out of its group's scale; its code is -8, and 0 where the scale is 0 (a group of NaN
    and zeros).  An infinity saturates the scale and takes the outermost code."""
    key = torch.zeros((1, 1, 64, 128), dtype=torch.bfloat16, device=DEV)
    key[0, 0, :, 3] = float("nan")       # group 0: NaN and zeros
    key[0, 0, :, 40] = float("nan")      # group 1: NaN among ordinary values
    key[0, 0, :, 41:48] = 7.0
    key[0, 0, :, 70] = float("inf")      # group 2
    key[0, 0, :, 71] = -float("inf")
    packed, scales = K.int4_pack_k(key, 32)
    codes = torch.stack([packed[0, 0, :64] & 15, packed[0, 0, :64] >> 4], dim=-1).view(64, 128).cpu()
    codes = torch.where(codes > 7, codes.int() - 16, codes.int())
    want = torch.zeros(128, dtype=torch.int32)
    want[40], want[41:48], want[70], want[71] = -8, 7, 7, -8
    assert torch.equal(codes, want.expand(64, 128))
    assert scales[0, 0, 0].tolist() == [0.0, 1.0, 65504.0, 0.0]
    chan = torch.arange(16, dtype=torch.int32, device=DEV).view(1, 1, 16)   # the first group's channels only
    for kk in (key, unaligned(key)):
        slab = torch.full((1, 1, K.round_capacity(64), 8), 7, dtype=torch.uint8, device=DEV)
        ss = torch.zeros(slab.shape[:3], dtype=torch.float16, device=DEV)
        K.build_slab(kk, chan, slab=slab, slab_scales=ss)
        stored = O.swizzle_slab(np.zeros((1, 64, 8), np.uint8), K.round_capacity(64)).reshape(-1)
        mask = O.swizzle_slab(np.full((1, 64, 8), 255, np.uint8), K.round_capacity(64)).reshape(-1) != 0
        assert np.array_equal(slab.cpu().numpy().reshape(-1)[mask], stored[mask])


def test_statistic_without_workspace():
    key = make(2, 4, 3000, 128, torch.bfloat16, 9)
    packed, scales = K.int4_pack_k(key, 32)
    chan, stats = K.select_channels(packed, scales, 2999, 32, 32)
    chan2, stats2 = torch.empty_like(chan), torch.empty_like(stats)
    lib = _lib.load()
    _lib.check(lib.qkv_int4_select_channels(packed.data_ptr(), scales.data_ptr(), 8, 2999, packed.size(2), 128, 32, 32,
                                            stats2.data_ptr(), chan2.data_ptr(), _lib.stream_of(packed)))
    assert torch.equal(stats, stats2) and torch.equal(chan, chan2)
    # a workspace that is too small is refused
    assert lib.qkv_int4_select_channels_ws(packed.data_ptr(), scales.data_ptr(), 8, 2999, packed.size(2), 128, 32, 32,
                                           stats2.data_ptr(), chan2.data_ptr(), stats.data_ptr(), 64,
                                           _lib.stream_of(packed)) == -1
