"""Scratch of latent attention: what a caller sized for its longest sequences serves every shorter step, at latents of every form that the attention kernels have."""
import ctypes

import pytest

from ming_univision_amd import _lib

LENS = [1, 63, 64, 65, 127, 128, 129, 255, 256, 257] + list(range(320, 4353, 64)) + [8191, 8192, 8193, 16384, 32768, 65536]


@pytest.mark.parametrize("r", [40, 64, 128, 256, 264, 384, 512, 576, 1024])
def test_splits_grow_with_the_length_and_fall_with_the_runs(r):
    L = _lib.lib()
    last = None
    for blk in list(range(1, 130)) + [255, 256, 257, 511, 512, 513, 1000, 5000]:
        ks = [L.mn_latent_attn_splits(blk, n, r) for n in LENS]
        assert ks == sorted(ks) and ks[0] == 1 and ks[-1] <= 64, (r, blk)
        assert last is None or all(a >= b for a, b in zip(last, ks)), (r, blk)
        last = ks


@pytest.mark.parametrize("arith", [0, 1])
@pytest.mark.parametrize("r", [40, 128, 256, 384, 512])
def test_scratch_of_a_step_grows_with_its_lengths(r, arith):
    L = _lib.lib()
    layer = (_lib.SeqLayer * 2)()
    for ly in layer:
        ly.kind, ly.heads, ly.dim, ly.vdim, ly.kv_rank, ly.q_rank, ly.ff, ly.writes_arena = 0, 16, 128, 128, r, 384, 2048, 1
    m = _lib.SeqModel(width=1024, n_layers=2, taps=2, arith=arith, eps=1e-5)
    m.layers = ctypes.cast(layer, ctypes.POINTER(_lib.SeqLayer))
    for M in (1, 2, 8, 28, 29, 32, 61, 64, 65, 121, 128, 300, 1500):
        size = [L.mn_seq_workspace_bytes(ctypes.byref(m), M, n) for n in LENS]
        assert size[0] > 0 and size == sorted(size), (r, M)
