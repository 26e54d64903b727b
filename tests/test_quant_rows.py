"""4-bit Matmul of a few bf16 rows on the matrix cores (aq_rows.hip): the rule
that takes a call there on the CPU, and on the GPU exact integer products and
the oracle at the edges of row tiles, chunks, units, phases and tiles."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

FAKE = 1 << 20
PREFIX = "aq_matvec_simd4_bf16_bf16_bf16_b4_g64_m"


def _names(M, N, K, ot="bf16", x_ptr=FAKE, xt="bf16"):
    import popcorn_amd as pa

    w = pa.AffineQuantizedTensor(pa.Tensor(FAKE, [N, K // 8], "u32"), pa.Tensor(FAKE, [N, K // 64], "bf16"),
                                 pa.Tensor(FAKE, [N, K // 64], "bf16"), [N, K])
    return pa.Kernels.Matmul(pa.Tensor(x_ptr, [M, K], xt), w, pa.Tensor(FAKE, [M, N], ot)).function_names


def test_rows_rule():
    assert _names(8, 9216, 2304) == [PREFIX + "1_s2"]
    assert _names(15, 2304, 9216) == [PREFIX + "1_s8"]
    assert _names(5, 24576, 3072) == [PREFIX + "1_s1"]
    assert _names(32, 9216, 2304) == [PREFIX + "2_s2"] and _names(48, 9216, 2304) == [PREFIX + "4_s2"]
    assert _names(40, 5000, 1024) == [PREFIX + "4_s4"]  # under 2^27 weight bytes: not the prompt GEMM's
    old = ("aq_matvec_simd4_bf16_bf16_bf16_b4_g64_l", "aq_matvec_simd4_bf16_bf16_f32_b4_g64_l")
    assert _names(2, 9216, 2304)[0].startswith(old)        # two rows: from 2^26 multiply-adds
    assert _names(4, 1024, 1024)[0].startswith(old)        # small matrices
    assert _names(8, 500, 8192)[0].startswith(old)         # few rows of W
    assert _names(8, 9216, 2304, "f32")[0].startswith(old)
    assert not _names(8, 9216, 2304 + 64)[0].startswith(PREFIX)  # not whole chunks of 128
    assert not _names(8, 9216, 2304, x_ptr=FAKE + 2)[0].startswith(PREFIX)
    assert _names(16, 16448, 1024)[0] == "aq_gemm_prep_bf16" and _names(64, 9216, 2304)[0] == "aq_gemm_prep_bf16"
    assert _names(32, 2304, 9216)[0] == "aq_gemm_prep_bf16"


def _matrix(env, packed, s, b, N, K):
    from gpu_util import upload

    pa = env[0]
    return pa.AffineQuantizedTensor(pa.Tensor.from_numpy(packed.view(np.uint32), "u32"), upload(pa, s, "bf16"),
                                    upload(pa, b, "bf16") if b is not None else None, [N, K])


def _run(env, x, w, N):
    from gpu_util import download, upload

    pa, lib, stream, enc = env
    M, guard = x.shape[0], 64
    buf = upload(pa, np.full(M * N + guard, np.nan, np.float32), "bf16")
    k = pa.Kernels.Matmul(upload(pa, x, "bf16"), w, buf.view([M, N]))
    assert k.function_names[0].startswith(PREFIX)
    enc.encode(k)
    stream.synchronize()
    out = download(buf, stream)
    assert np.isnan(out[M * N:]).all(), "wrote past C"
    return out[:M * N].reshape(M, N)


@pytest.fixture(scope="module")
def env():
    from gpu_util import gpu_env

    return gpu_env()


SHAPES = [(3, 9216, 1024),     # two units, two waves per tile
          (15, 2300, 1408),    # 11 chunks: a unit of three; rows of W past N in the last tile
          (16, 1030, 2304),    # every row of a tile; eight waves per tile, 18 chunks
          (17, 4100, 640),     # a second row tile of one row; a unit of one chunk
          (33, 1100, 1152), (48, 1024, 2048),
          (13, 1040, 8192),    # x in two phases
          (9, 33000, 128)]     # one chunk; one wave per tile


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_rows_integer_exact(env, M, N, K):
    # One x of 1 or -1 in each group of a row, at a value that the rows and the
    # passes walk through, so that every value of K meets every row of W. The
    # scales differ by powers of two and the biases are whole: every sum is a
    # whole number under 2^24, exact in f32 whatever the order, and the output is
    # its one rounding to bf16. A wrong nibble, x, scale, bias or index moves
    # whole rows or columns by whole units.
    import oracle as O
    from q4util import pack_q4

    rng = np.random.default_rng(M + N + K)
    q = rng.integers(0, 16, (N, K)).astype(np.uint32)
    s = 2.0 ** rng.integers(0, 4, (N, K // 64)).astype(np.float32)
    b = rng.integers(-8, 8, (N, K // 64)).astype(np.float32)
    dense = (q * np.repeat(s, 64, 1) + np.repeat(b, 64, 1)).astype(np.float32)
    w, seen = _matrix(env, pack_q4(q), s, b, N, K), np.zeros(K, bool)
    for p in range(0, 64, M):
        x = np.zeros((M, K // 64, 64), np.float32)
        for r in range(M):
            x[r, :, (p + r) % 64] = rng.choice([-1.0, 1.0], K // 64)
        x = x.reshape(M, K)
        seen |= (x != 0).any(0)
        np.testing.assert_array_equal(_run(env, x, w, N), O.round_to(x @ dense.T, O.BF16))
    assert seen.all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("bias", [True, False])
def test_rows_vs_oracle(env, M, N, K, bias):
    import oracle as O
    from conftest import assert_out
    from gpu_util import EPS, rounded
    from q4util import quantize_q4

    rng = np.random.default_rng(M * 7 + N + K)
    packed, s, b, _ = quantize_q4(0.05 * rng.standard_normal((N, K)).astype(np.float32), bias=bias)
    x = rounded(rng.standard_normal((M, K)).astype(np.float32), "bf16")
    assert_out(_run(env, x, _matrix(env, packed, s, b, N, K), N), O.aq_matmul(x, packed, s, b, N, K), EPS["bf16"], "bf16", f"{M}x{N}x{K} bias={bias}")


def test_prompt_wave_forms_rule():
    # waves of 64 x 64 in one round of blocks with more than 36 groups each
    name = "aq_gemm_mfma_bf16_bf16_"
    assert _names(129, 1031, 2432)[1] == name + "bf16_b4_g64_w64" and _names(129, 1031, 2304)[1] == name + "bf16_b4_g64"
    assert _names(1100, 2900, 4864)[1] == name + "splitk_b4_g64_w64" and _names(1100, 2900, 4608)[1] == name + "splitk_b4_g64"
    assert _names(777, 9216, 3072)[1] == name + "bf16_b4_g64_w64"   # 504 blocks
    assert _names(1000, 9216, 3072)[1] == name + "bf16_b4_g64"      # 576


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(129, 1031, 2432), (1100, 2900, 4864)])  # whole K, and split
def test_prompt_wave_form_integer_exact(env, M, N, K):
    # small integers: every product and sum is an exact f32 integer in any order
    from gpu_util import download, upload
    from q4util import pack_q4

    pa, lib, stream, enc = env
    rng = np.random.default_rng(M + N + K)
    q = rng.integers(0, 16, (N, K)).astype(np.uint32)
    s = 2.0 ** rng.integers(0, 2, (N, K // 64)).astype(np.float32)
    b = rng.integers(-8, 8, (N, K // 64)).astype(np.float32)
    x = rng.integers(-3, 4, (M, K)).astype(np.float32)
    w = _matrix(env, pack_q4(q), s, b, N, K)
    guard = 64
    buf = upload(pa, np.full(M * N + guard, np.nan, np.float32), "f32")
    k = pa.Kernels.Matmul(upload(pa, x, "bf16"), w, buf.view([M, N]))
    assert k.function_names[1].endswith("_w64")
    enc.encode(k)
    stream.synchronize()
    out = download(buf, stream)
    assert np.isnan(out[M * N:]).all(), "wrote past C"
    dense = q.astype(np.float64) * np.repeat(s, 64, 1) + np.repeat(b, 64, 1)
    np.testing.assert_array_equal(out[:M * N].reshape(M, N), (x.astype(np.float64) @ dense.T).astype(np.float32))
