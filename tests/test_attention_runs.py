"""Tiled attention whose tiles leave CUs idle: key steps cut into runs over
several blocks, merged by the split-merge kernel (flash_attention_tiled.hip,
pairTiles 3): the rule on the CPU, and outputs against the oracle on the GPU."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

FAKE = 1 << 20


def _kernel(pa, t, B, Nq, Nkv, Sq, Sk, cap, Hd, mask, q=None, k=None, v=None, out=None):
    def fake(*shape):
        return pa.Tensor(FAKE, shape, t)

    q, out = q or fake(B, Nq, Sq, Hd), out or fake(B, Nq, Sq, Hd)
    k, v = k or fake(B, Nkv, cap, Hd), v or fake(B, Nkv, cap, Hd)
    return pa.Kernels.FlashAttention(q, k, v, out=out, scale=Hd ** -0.5, mask=pa.AttentionMask(*mask), batch=B,
                                     query_heads=Nq, kv_heads=Nkv, query_len=Sq, key_len=Sk, head_dim=Hd,
                                     key_capacity=cap)


def test_runs_rule():
    import popcorn_amd as pa

    def runs(Nq, Sq, Sk, Hd=256, t="bf16", mask=(0, -1)):
        return len(_kernel(pa, t, 1, Nq, Nq, Sq, Sk, Sk, Hd, mask).function_names) == 2

    assert runs(8, 500, 8692) and runs(8, 1000, 1000) and runs(32, 300, 3000, 128) and runs(8, 100, 5000, 64)
    assert runs(8, 200, 2500, mask=(2, -1))
    assert not runs(2, 640, 640)              # under 768 keys: one launch
    assert not runs(24, 768, 768, 64) and not runs(16, 900, 900, 128)  # pairs are faster
    assert not runs(16, 2048, 2048)           # a tile per CU
    assert not runs(8, 500, 8692, 512) and not runs(8, 500, 8692, t="f32")  # whole tiles only
    assert not runs(16, 1000, 4000, mask=(1, 64))  # a window of 7 steps: nothing to cut


@pytest.mark.gpu
@pytest.mark.parametrize("t", ["f16", "bf16"])
@pytest.mark.parametrize("B,Nq,Nkv,Sq,Sk,cap,Hd,mask", [
    (1, 2, 1, 33, 800, 800, 256, (0, -1)),     # a tile of 33 rows, a short last step
    (1, 4, 2, 300, 1201, 1300, 256, (0, -1)),  # ragged tiles behind a cache, rows past the keys
    (2, 2, 2, 130, 2050, 2050, 128, (2, -1)),  # every key, two sequences
    (1, 4, 1, 200, 1500, 1501, 128, (1, 700)),  # a window that cuts the first steps
    (1, 2, 1, 128, 3000, 3000, 64, (0, -1)),   # the 32-row kernel
    (1, 2, 1, 40, 900, 900, 200, (0, -1)),     # a head dim padded to 256
    (1, 2, 2, 900, 900, 900, 256, (0, -1)),    # a prompt: some tiles of one run, some of several
])
def test_runs_vs_oracle(t, B, Nq, Nkv, Sq, Sk, cap, Hd, mask):
    import oracle as O
    from conftest import assert_out
    from gpu_util import EPS, download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    q = rounded(O.normal(Sq, (B, Nq, Sq, Hd)), t)
    k, v = (rounded(O.normal(Sk + i, (B, Nkv, cap, Hd)), t) for i in (1, 2))
    out = upload(pa, np.full((B, Nq, Sq, Hd), np.nan, np.float32), t)
    kern = _kernel(pa, t, B, Nq, Nkv, Sq, Sk, cap, Hd, mask, upload(pa, q, t), upload(pa, k, t), upload(pa, v, t), out)
    assert len(kern.function_names) == 2 and kern.function_names[1].startswith("flash_attention_split_merge_")
    ref = O.attention_naive(q, k, v, Hd ** -0.5, key_len=Sk, mask_kind=mask[0], window=mask[1])
    enc.encode(kern)
    stream.synchronize()
    got = download(out, stream)
    assert_out(got, ref, EPS[t], t, "runs")

    # no scratch to be had: the whole tiles give the same rows
    class Empty(pa.KernelScratchAllocator):
        def borrow(self, length):
            raise MemoryError

    out.copy_from(np.full((B, Nq, Sq, Hd), 0x7FFF, np.uint16), stream)
    pa.KernelCommandEncoder(lib, stream, Empty()).encode(kern)
    stream.synchronize()
    assert_out(download(out, stream), ref, EPS[t], t, "whole tiles")


@pytest.mark.gpu
@pytest.mark.parametrize("Hd", [64, 128, 256])
def test_infinite_value_stays_infinite(Hd):
    # an infinity in V at the last key, which every row sees, in the last run
    # of each tile: the dims it reaches are infinite, no dim is a NaN. Queries
    # of 0 weigh every key alike, so the rest are the keys' mean.
    import oracle as O
    from gpu_util import download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    B, Nq, Nkv, Sq, Sk = 1, 4, 2, 40, 2000
    k, v = (rounded(O.normal(Sk + i, (B, Nkv, Sk, Hd)), "f16") for i in (1, 2))
    v[..., Sk - 1, 3], v[..., Sk - 1, Hd - 1] = np.inf, -np.inf
    q = np.zeros((B, Nq, Sq, Hd), np.float32)
    out = upload(pa, q, "f16")
    kern = _kernel(pa, "f16", B, Nq, Nkv, Sq, Sk, Sk, Hd, (2, -1), upload(pa, q, "f16"), upload(pa, k, "f16"), upload(pa, v, "f16"), out)
    assert len(kern.function_names) == 2 and kern.function_names[1].startswith("flash_attention_split_merge_")
    enc.encode(kern)
    stream.synchronize()
    got = download(out, stream)
    want = np.repeat(v.astype(np.float64).mean(2), Nq // Nkv, 1)[:, :, None].repeat(Sq, 2)
    assert np.isposinf(got[..., 3]).all() and np.isneginf(got[..., Hd - 1]).all()
    ok = np.isfinite(want)
    # means of 2000 values under 5: f32 sums and one rounding to f16, of a unit of 2^-11 at 0.15 at most
    assert ok.sum() == want.size // Hd * (Hd - 2) and np.abs(got[ok] - want[ok]).max() < 2e-4
