"""RMSNorm of many rows on a few lanes each (rmsnorm_rows_*): the rule on the
CPU, and on the GPU the oracle at the edges of lanes, vectors and blocks."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

FAKE = 1 << 20


def test_rows_rule():
    import popcorn_amd as pa

    def name(rows, H, t="bf16", x_ptr=FAKE, w_ptr=FAKE):
        return pa.Kernels.RMSNorm(pa.Tensor(x_ptr, [rows, H], t), pa.Tensor(w_ptr, [H], "f32"),
                                  pa.Tensor(FAKE, [rows, H], t), eps=1e-6).describe()

    assert name(8, 2304) == "rmsnorm_rows_bf16_l64_v8" and name(8000, 256) == "rmsnorm_rows_bf16_l32_v1"
    assert name(100, 128, "f16") == "rmsnorm_rows_f16_l16_v1" and name(600, 4096, "f32") == "rmsnorm_rows_f32_l64_v16"
    # long f32 rows: a block per row while they are few
    assert name(9, 4096, "f32") == "rmsnorm" and name(400, 4096, "f32") == "rmsnorm" and name(255, 1536, "f32") == "rmsnorm"
    assert name(256, 1536, "f32") == "rmsnorm_rows_f32_l64_v8" and name(9, 1528, "f32") == "rmsnorm_rows_f32_l64_v8"
    assert name(7, 2304) == "rmsnorm_bf16" and name(100, 2300) == "rmsnorm_bf16" and name(100, 8200) == "rmsnorm_bf16"
    assert name(100, 256, x_ptr=FAKE + 2) == "rmsnorm_bf16" and name(100, 256, w_ptr=FAKE + 4) == "rmsnorm_bf16"


@pytest.mark.gpu
@pytest.mark.parametrize("t", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,H", [(8, 8), (33, 128), (9, 136), (1000, 256), (17, 264), (8, 512), (8, 520), (65, 2048),
                                    (10, 2304), (2100, 256), (9, 4096), (3000, 64)])
@pytest.mark.parametrize("weight,add_one", [(True, False), (True, True), (False, False)])
def test_rows_vs_oracle(t, rows, H, weight, add_one):
    import oracle as O
    from conftest import assert_out
    from gpu_util import EPS, download, gpu_env, rounded, upload

    pa, lib, stream, enc = gpu_env()
    if t == "f32" and H >= 1536:
        rows += 512  # fewer long f32 rows take a block each
    x = rounded(O.normal(rows + H, (rows, H)), t)
    x[rows // 2] = 0.0  # a row of zeros: its scale is 1 / sqrt(eps)
    w = O.normal(H, (H,), mean=1.0, std=0.1) if weight else None
    guard = 64
    buf = upload(pa, np.full(rows * H + guard, 7.0, np.float32), t)
    k = pa.Kernels.RMSNorm(upload(pa, x, t), upload(pa, w, "f32") if weight else None, buf.view([rows, H]), eps=1e-6,
                           add_one_to_weight=add_one)
    assert k.describe().startswith(f"rmsnorm_rows_{t}_")
    enc.encode(k)
    stream.synchronize()
    got = download(buf, stream)
    assert (got[rows * H:] == 7.0).all(), "wrote past the output"
    assert_out(got[:rows * H].reshape(rows, H), O.rmsnorm(x, w, 1e-6, add_one), EPS[t], t, f"rmsnorm {t} {rows}x{H}")
