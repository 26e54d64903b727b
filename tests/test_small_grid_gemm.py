"""The 16-bit Matmul on grids of few tiles: the four-stage whole-line tiles
(f64x64, f128x64, f128x128), K not a multiple of a stage, K split unevenly
over blocks and its reduction where M N is odd, against exact integer
products; and the rule that picks tile and splits, on the CPU."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

FAKE = 1 << 20


def _names(M, K, N, dtype="bf16", out_ptr=FAKE):
    import popcorn_amd as pa

    def t(shape, ptr=FAKE):
        return pa.Tensor(ptr, shape, dtype)

    return pa.Kernels.Matmul(t([M, K]), t([N, K]), t([M, N], out_ptr), True).function_names


def test_small_grid_plan():
    # few 128 x 128 tiles: a smaller tile, or K split over blocks
    assert _names(137, 9216, 2304)[1] == "matmul_splitk_reduce_bf16"
    assert _names(1000, 2304, 1024) == ["matmul_mfma_bf16_bf16_bf16_f64x64"]
    # between one and two 128 x 128 tiles per CU: split only for a clear gain
    assert _names(389, 4096, 14336) == ["matmul_mfma_bf16_bf16_bf16_e128x128"] and len(_names(1156, 4096, 4096)) == 1
    assert len(_names(1153, 24576, 3072)) == 2 and len(_names(403, 4896, 10227)) == 2
    # C off 16-byte alignment: the reduction's vector stores are out, one pass
    assert len(_names(137, 9216, 2304, out_ptr=FAKE + 2)) == 1
    # under 2^29 multiply-adds: one 128 x 128 pass
    assert _names(100, 2304, 2304) == ["matmul_mfma_bf16_bf16_bf16_e128x128"]
    # more than two tiles per CU: the score over the large tiles
    assert _names(1000, 2304, 9216) == ["matmul_mfma_bf16_bf16_bf16_e256x192"]
    assert _names(512, 2304, 9216 * 2) == ["matmul_mfma_bf16_bf16_bf16_e128x192"]
    assert _names(700, 3072, 24576) == ["matmul_mfma_bf16_bf16_bf16_e192x384"]
    assert _names(4601, 9216, 4096) == ["matmul_mfma_bf16_bf16_bf16_e256x320"]
    assert _names(2964, 3072, 4096) == ["matmul_mfma_bf16_bf16_bf16_e192x256"]
    # K of whole 16-byte chunks but not whole stages takes the same tiles
    assert _names(190, 2136, 9088)[0].split("_")[-1][0] in "ef"
    # rows too long for a tile's 32-bit offsets, not in whole 64-byte runs
    assert _names(65, (1 << 23) + 8, 2)[0].startswith("matmul_tiled")


def _run(env, a, b, at, ot, guard=64):
    from gpu_util import download, upload

    pa, lib, stream, enc = env
    M, N = a.shape[0], b.shape[0]
    buf = upload(pa, np.full(M * N + guard, np.nan, np.float32), ot)
    k = pa.Kernels.Matmul(upload(pa, a, at), upload(pa, b, at), buf.view([M, N]), True)
    enc.encode(k)
    stream.synchronize()
    out = download(buf, stream)
    assert np.isnan(out[M * N:]).all(), "wrote past C"
    return out[:M * N].reshape(M, N), k.function_names


def _ints(seed, M, K, N):
    rng = np.random.default_rng(seed)
    a, b = (rng.integers(-4, 5, s).astype(np.float32) for s in ((M, K), (N, K)))
    return a, b, (a.astype(np.float64) @ b.T.astype(np.float64)).astype(np.float32)  # |sums| < 2^24: exact


@pytest.fixture(scope="module")
def env():
    from gpu_util import gpu_env

    return gpu_env()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", ["f64x64", "f128x64", "f128x128", "e128x128", "e256x256", "e256x288", "e256x320",
                                  "e192x384", "e256x192", "e192x256"])
def test_tiles_any_k_integer_exact(env, monkeypatch, tile):
    # 1 to 6 stages (fewer and more than are in flight), the last one whole,
    # or of 1, 2 or 7 chunks; M and N ragged
    monkeypatch.setenv("POPCORN_GEMM_TILE", tile)
    for at in ("f16", "bf16"):
        for M, K, N in [(70, 64, 131), (130, 8, 90), (65, 200, 64), (300, 272, 67), (129, 312, 200), (200, 384, 129)]:
            a, b, want = _ints(M + K, M, K, N)
            got, names = _run(env, a, b, at, "f32")
            assert names == [f"matmul_mfma_{at}_{at}_f32_{tile}"]
            np.testing.assert_array_equal(got, want, err_msg=f"{tile} {at} {M}x{K}x{N}")


@pytest.mark.gpu
@pytest.mark.parametrize("at", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N", [(137, 9216, 2304),   # the plan's own split, even
                                   (131, 9000, 2003),   # M N odd: the reduction element by element; K ragged
                                   (66, 16384, 500), (300, 8200, 260), (257, 4104, 2308)])
def test_split_plans_integer_exact(env, at, M, K, N):
    a, b, want = _ints(M + K, M, K, N)
    got, names = _run(env, a, b, at, "f32")
    assert names == _names(M, K, N, at)[:1] + ["matmul_splitk_reduce_f32"] and "_splitk_" in names[0]
    np.testing.assert_array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("at,ot", [("f16", "f16"), ("bf16", "bf16"), ("bf16", "f32")])
def test_split_plan_rounds_once(env, at, ot):
    import oracle as O
    from conftest import assert_out
    from gpu_util import EPS, rounded

    M, K, N = 131, 9000, 2003
    a = rounded(O.normal(1, (M, K)), at)
    b = rounded(O.normal(2, (N, K), std=0.02), at)
    got, _ = _run(env, a, b, at, ot)
    rows = [0, 63, 64, 127, 128, M - 1]
    ref = O.matmul(a[rows], b, len(rows), K, N, True).reshape(len(rows), N)
    if ot == "f32":  # f32 sums of K terms in another order: 1e-5 of the terms' magnitudes
        mag = np.abs(a[rows]).astype(np.float64) @ np.abs(b).T.astype(np.float64)
        assert (np.abs(got[rows] - ref) <= 1e-5 * mag).all()
    else:
        assert_out(got[rows], ref, EPS[at], ot, f"split {at}->{ot}")


@pytest.mark.gpu
def test_split_without_scratch_runs_whole(env):
    # an allocator with nothing to give: the product still runs, unsplit
    pa, lib, stream, enc = env

    class Empty(pa.KernelScratchAllocator):
        def borrow(self, length):
            raise MemoryError

    a, b, want = _ints(3, 137, 9216, 1000)
    got, names = _run((pa, lib, stream, pa.KernelCommandEncoder(lib, stream, Empty())), a, b, "bf16", "f32")
    assert len(names) == 2  # the plan splits it
    np.testing.assert_array_equal(got, want)
