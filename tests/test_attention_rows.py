"""Attention of 2 to 31 query rows on the matrix cores (flash_attention_rows_*):
the rule that takes a call there on the CPU, outputs against the oracle on the
GPU at the edges of row tiles, key steps, partitions and head dims."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

FAKE = 1 << 20


def _kernel(pa, t, B, Nq, Nkv, Sq, Sk, cap, Hd, mask=(0, -1), scale=None, q=None, k=None, v=None, out=None, ot=None, **kw):
    def fake(*shape):
        return pa.Tensor(FAKE, shape, t)

    q, out = q or fake(B, Nq, Sq, Hd), out or pa.Tensor(FAKE, (B, Nq, Sq, Hd), ot or t)
    k, v = k or fake(B, Nkv, cap, Hd), v or fake(B, Nkv, cap, Hd)
    return pa.Kernels.FlashAttention(q, k, v, out=out, scale=Hd ** -0.5 if scale is None else scale,
                                     mask=pa.AttentionMask(*mask), batch=B, query_heads=Nq, kv_heads=Nkv, query_len=Sq,
                                     key_len=Sk, head_dim=Hd, key_capacity=cap, **kw)


def test_rows_rule():
    import popcorn_amd as pa

    def name(Nq, Nkv, Sq, Sk, Hd=256, t="bf16", **kw):
        return _kernel(pa, t, 1, Nq, Nkv, Sq, Sk, Sk, Hd, **kw).function_names

    assert name(8, 4, 8, 4104) == ["flash_attention_rows_bf16_bf16_d256_r1", "flash_decoding_reduce_bf16_ext"]
    assert name(8, 4, 31, 200) == ["flash_attention_rows_bf16_bf16_d256_r1"]  # up to 12 steps: one partition
    assert name(32, 8, 31, 30000, 128)[0] == "flash_attention_rows_bf16_bf16_d128_r4"
    assert name(8, 8, 2, 200, 72, ot="f32") == ["flash_attention_rows_bf16_f32_d128_r1"]
    old = "flash_decoding_partial_"
    assert name(8, 4, 1, 4104)[0].startswith(old)
    assert name(8, 4, 8, 4104, t="f32")[0].startswith(old)
    assert name(8, 4, 8, 4104, 252)[0].startswith(old)        # rows not in 16-byte chunks
    assert name(8, 4, 8, 4104, scale=-1.0)[0].startswith(old)  # maxima are taken on unscaled scores
    pos = pa.Tensor(FAKE, (1,), "i32")
    assert name(8, 4, 8, 4104, position=pos)[0].startswith(old)
    q = pa.Tensor(FAKE + 2, (1, 8, 8, 256), "bf16")
    assert name(8, 4, 8, 4104, q=q)[0].startswith(old)
    assert name(8, 4, 8, 4104, ot="f16")[0].startswith(old)
    # measured both ways at Hd 256 and 512: a longer chain of key steps per wave
    # than the one-row kernels', until these read K and V too often
    for case, rows in {(8, 4, 2, 700): False, (8, 4, 8, 384): False, (8, 4, 8, 1500): True, (16, 16, 2, 300): False,
                       (8, 1, 2, 300): True, (8, 4, 2, 64): True, (8, 4, 31, 300, 512): False, (8, 4, 31, 5000, 512): True,
                       (16, 16, 2, 2000, 512): False, (16, 16, 2, 500, 128): False, (8, 2, 6, 500, 320): True}.items():
        assert name(*case)[0].startswith("flash_attention_rows_" if rows else old), case


@pytest.mark.gpu
@pytest.mark.parametrize("t,ot", [("f16", "f16"), ("f16", "f32"), ("bf16", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("B,Nq,Nkv,Sq,Sk,cap,Hd,mask,form", [
    (1, 2, 2, 2, 2, 2, 64, (0, -1), "d64_r1"),             # fewer keys than a step, rows of one head
    (1, 4, 2, 8, 33, 40, 256, (0, -1), "d256_r1"),         # 16 rows exactly; a second step of one key
    (2, 6, 2, 11, 500, 512, 128, (0, -1), "d128_r1"),      # 33 rows: a third tile of one row; 16 steps: partitions
    (1, 8, 1, 31, 1100, 1100, 256, (0, -1), "d256_r1"),    # 248 rows of one KV head
    (1, 16, 2, 24, 700, 701, 512, (0, -1), "d512_r1"),
    (1, 2, 1, 5, 700, 701, 400, (0, -1), "d512_r1"),       # padded to 512
    (1, 4, 4, 3, 450, 450, 200, (2, -1), "d256_r1"),       # padded head dim, every key
    (1, 4, 2, 9, 900, 1000, 72, (1, 100), "d128_r1"),      # a window: most partitions of the keys unseen
    (1, 4, 1, 20, 600, 600, 128, (1, 3), "d128_r1"),
    (8, 32, 8, 8, 1030, 1031, 64, (0, -1), "d64_r2"),      # 2 and 4 row tiles per block
    (8, 32, 8, 16, 2050, 2050, 64, (0, -1), "d64_r4"),
    (8, 32, 8, 8, 1030, 1030, 128, (0, -1), "d128_r2"),
    (8, 32, 8, 16, 1030, 1030, 128, (0, -1), "d128_r4"),
    (8, 16, 8, 16, 1100, 1100, 256, (0, -1), "d256_r2"),
])
def test_rows_vs_oracle(t, ot, B, Nq, Nkv, Sq, Sk, cap, Hd, mask, form):
    import oracle as O
    from conftest import assert_out
    from gpu_util import EPS, download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    q = rounded(O.normal(Sq, (B, Nq, Sq, Hd)), t)
    k, v = (rounded(O.normal(Sk + i, (B, Nkv, cap, Hd)), t) for i in (1, 2))
    k[:, :, Sk:] = v[:, :, Sk:] = np.nan  # rows past the keys
    guard = 64
    buf = upload(pa, np.full(q.size + guard, 7.0, np.float32), ot)
    kern = _kernel(pa, t, B, Nq, Nkv, Sq, Sk, cap, Hd, mask, None, upload(pa, q, t), upload(pa, k, t), upload(pa, v, t),
                   buf.view([B, Nq, Sq, Hd]))
    assert kern.function_names[0] == f"flash_attention_rows_{t}_{ot}_{form}"
    ref = O.attention_naive(q, k, v, Hd ** -0.5, key_len=Sk, mask_kind=mask[0], window=mask[1])

    class Empty(pa.KernelScratchAllocator):
        def borrow(self, length):
            raise MemoryError

    # with the plan's partitions, and with no scratch for them: one partition
    for e in (enc, pa.KernelCommandEncoder(lib, stream, Empty())):
        buf.copy_from(np.full(q.size + guard, 7.0, np.float32) if ot == "f32" else
                      O.to_bits(np.full(q.size + guard, 7.0, np.float32), {"f16": O.F16, "bf16": O.BF16}[ot]), stream)
        e.encode(kern)
        stream.synchronize()
        got = download(buf, stream)
        assert (got[q.size:] == 7.0).all(), "wrote past the output"
        assert_out(got[:q.size].reshape(q.shape), ref, EPS[t], ot, f"rows {kern.function_names}")


@pytest.mark.gpu
@pytest.mark.parametrize("t", ["f16", "bf16"])
def test_rows_wide_score_range(t):
    # scores over hundreds of natural-log units: the reference max moves on
    # most steps, in waves and partitions of their own
    import oracle as O
    from conftest import assert_out
    from gpu_util import EPS, download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    q, k = (rounded(3.0 * O.normal(s, sh), t) for s, sh in ((1, (1, 4, 31, 256)), (2, (1, 2, 640, 256))))
    v = rounded(O.normal(3, (1, 2, 640, 256)), t)
    out = pa.Tensor.empty([1, 4, 31, 256], t)
    kern = _kernel(pa, t, 1, 4, 2, 31, 640, 640, 256, (0, -1), 1.0, upload(pa, q, t), upload(pa, k, t), upload(pa, v, t), out)
    assert kern.function_names[0].startswith("flash_attention_rows_")
    enc.encode(kern)
    stream.synchronize()
    assert_out(download(out, stream), O.attention_naive(q, k, v, 1.0), EPS[t], t, "wide range")


def _own_keys(q, k, v, scale, mask=(0, -1)):
    """Attention in 64 bits, each row over the keys it sees and no others."""
    B, Nq, Sq, Hd = q.shape
    Nkv, Sk = k.shape[1:3]
    out = np.zeros(q.shape)
    with np.errstate(all="ignore"):  # the tests put infinities and NaN in K and V
        for b, h, i in np.ndindex(B, Nq, Sq):
            pos = Sk - Sq + i
            lo = max(0, pos - mask[1] + 1) if mask[0] == 1 else 0
            kk, vv = (x[b, h // (Nq // Nkv), lo:pos + 1].astype(np.float64) for x in (k, v))
            s = kk @ q[b, h, i].astype(np.float64) * scale
            w = np.exp(s - s.max())
            out[b, h, i] = w @ vv / w.sum()
    return out


# every kernel of the rule, by a call that takes it
FORMS = [(1, 4, 2, 4, 300, 64, "d64_r1"), (8, 32, 8, 8, 1030, 64, "d64_r2"), (8, 32, 8, 16, 1030, 64, "d64_r4"),
         (1, 8, 4, 8, 1500, 128, "d128_r1"), (8, 32, 8, 8, 1030, 128, "d128_r2"), (8, 32, 8, 16, 1030, 128, "d128_r4"),
         (1, 8, 4, 8, 1500, 256, "d256_r1"), (8, 16, 8, 16, 1030, 256, "d256_r2"), (1, 8, 2, 24, 1500, 512, "d512_r1")]


@pytest.mark.gpu
@pytest.mark.parametrize("t", ["f16", "bf16"])
@pytest.mark.parametrize("B,Nq,Nkv,Sq,Sk,Hd,form", FORMS)
def test_rows_hold_f32_precision(t, B, Nq, Nkv, Sq, Sk, Hd, form):
    # An f32 output against 64 bits. With the weights and every sum in f32 its
    # error is a handful of roundings of 2^-24 per term (a score, its exponent,
    # the weight, two products and sums), the terms' own averaged over the
    # keys: 6e-7 is ten. Weights of one f16 give 1.4e-4, of two bf16 1.7e-6.
    import oracle as O
    from gpu_util import download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    q = rounded(O.normal(Sq, (B, Nq, Sq, Hd)), t)
    k, v = (rounded(O.normal(Sk + i, (B, Nkv, Sk, Hd)), t) for i in (1, 2))
    out = upload(pa, np.zeros(q.shape, np.float32), "f32")
    kern = _kernel(pa, t, B, Nq, Nkv, Sq, Sk, Sk, Hd, (0, -1), None, upload(pa, q, t), upload(pa, k, t), upload(pa, v, t), out)
    assert kern.function_names[0] == f"flash_attention_rows_{t}_f32_{form}"
    enc.encode(kern)
    stream.synchronize()
    want = _own_keys(q[:2], k[:2], v[:2], Hd ** -0.5)
    err = download(out, stream)[:2].astype(np.float64) - want
    assert np.linalg.norm(err) / np.linalg.norm(want) < 6e-7


@pytest.mark.gpu
@pytest.mark.parametrize("t", ["f16", "bf16"])
@pytest.mark.parametrize("B,Nq,Nkv,Sq,Sk,Hd,form", FORMS)
def test_rows_non_finite_values(t, B, Nq, Nkv, Sq, Sk, Hd, form):
    # infinities and NaN in the K and V of single keys change only the rows
    # that see them: K of NaN at the last key (only the last query sees it), V of
    # NaN at the one before, and an infinity of V in the middle of the cache,
    # which every row sees; with a window, those before it change no row
    import oracle as O
    from conftest import assert_out
    from gpu_util import EPS, download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    q = rounded(O.normal(Sq, (B, Nq, Sq, Hd)), t)
    k, v = (rounded(O.normal(Sk + i, (B, Nkv, Sk, Hd)), t) for i in (1, 2))
    first, win = Sk - Sq, 1000 if Hd == 512 else 70  # the first query's own key; a window that takes these kernels
    for mask in ((0, -1), (1, win)):
        kk, vv = k.copy(), v.copy()
        kk[:, :, Sk - 1], vv[:, :, Sk - 2] = np.nan, np.nan
        if mask[0] == 0:
            vv[:, :, 40, Hd - 3] = np.inf
        else:
            vv[:, :, first - win], kk[:, :, first - win - 1], vv[:, :, first - win - 5] = -np.inf, np.nan, np.nan
            vv[:, :, first - 5, 1] = -np.inf  # inside every window
        out = upload(pa, np.zeros(q.shape, np.float32), t)
        kern = _kernel(pa, t, B, Nq, Nkv, Sq, Sk, Sk, Hd, mask, None, upload(pa, q, t), upload(pa, kk, t), upload(pa, vv, t), out)
        name = kern.function_names[0]
        assert name.startswith(f"flash_attention_rows_{t}_{t}_d{Hd}_") and (mask[0] or name.endswith(form))
        enc.encode(kern)
        stream.synchronize()
        got, ref = download(out, stream)[:2, :, :-1], _own_keys(q[:2], kk[:2], vv[:2], Hd ** -0.5, mask)[:, :, :-1]
        assert np.isfinite(ref[:, :, 0, 2]).all() and np.isnan(ref[:, :, -1]).all() and np.isinf(ref[:, :, 0]).any()
        ok = np.isfinite(ref)
        np.testing.assert_array_equal(np.isfinite(got), ok, err_msg=f"{name} {mask}")
        if len(kern.function_names) == 1:  # (the combine of partitions may make a NaN of an infinity)
            np.testing.assert_array_equal(got == np.inf, ref == np.inf, err_msg=f"{name} {mask}")
            np.testing.assert_array_equal(got == -np.inf, ref == -np.inf, err_msg=f"{name} {mask}")
        assert_out(got[ok], ref[ok], EPS[t], t, f"{name} {mask}")


@pytest.mark.gpu
@pytest.mark.parametrize("t", ["f16", "bf16"])
@pytest.mark.parametrize("B,Nq,Nkv,Sq,Sk,Hd,form", FORMS)
def test_rows_nan_in_the_first_key(t, B, Nq, Nkv, Sq, Sk, Hd, form):
    # a row whose first score is NaN gives what the one-row kernels give for it,
    # not the attention over its other keys
    import oracle as O
    from gpu_util import download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    q = rounded(O.normal(Sq, (B, Nq, Sq, Hd)), t)
    k, v = (rounded(O.normal(Sk + i, (B, Nkv, Sk, Hd)), t) for i in (1, 2))
    k[:, :, 0] = np.nan
    kt, vt = upload(pa, k, t), upload(pa, v, t)
    out = upload(pa, np.full(q.shape, 7.0, np.float32), t)
    kern = _kernel(pa, t, B, Nq, Nkv, Sq, Sk, Sk, Hd, (0, -1), None, upload(pa, q, t), kt, vt, out)
    assert kern.function_names[0].endswith(form)
    enc.encode(kern)
    for i in (0, Sq - 1):
        one = upload(pa, np.full((B, Nq, 1, Hd), 7.0, np.float32), t)
        enc.encode(_kernel(pa, t, B, Nq, Nkv, 1, Sk - Sq + i + 1, Sk, Hd, (0, -1), None, upload(pa, q[:, :, i:i + 1], t), kt, vt, one))
        stream.synchronize()
        np.testing.assert_array_equal(download(out, stream)[:, :, i], download(one, stream)[:, :, 0], err_msg=form)
