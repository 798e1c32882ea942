"""One and two rows against q8_0 weights at every number of columns a team of waves takes (two to sixteen, by the columns a CU gets): either side of each, against 64-bit
products."""
import numpy as np
import pytest

from gpu_common import Dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = Dev()
    yield d
    d.ctx.close()


# K 64: eight teams of a wave a workgroup, 2048 columns a step on 256 CUs; K 4160: teams of four waves, 512
@pytest.mark.parametrize("rows,K,step,k", [(1, 64, 2048, 1), (2, 64, 2048, 2), (1, 64, 2048, 6), (2, 64, 2048, 14), (1, 64, 2048, 16), (1, 4160, 512, 3), (2, 4160, 512, 8)])
def test_columns_per_team(dev, rows, K, step, k):
    rng = np.random.default_rng(K + k)
    N = step * k + 3
    blob = np.empty((N, K // 32, 34), dtype=np.uint8)
    d = rng.uniform(0.001, 0.01, size=(N, K // 32)).astype(np.float16)
    q = rng.integers(-127, 128, size=(N, K // 32, 32)).astype(np.int8)
    blob[:, :, :2], blob[:, :, 2:] = d.view(np.uint8).reshape(N, K // 32, 2), q.view(np.uint8)
    w = (d.astype(np.float64)[:, :, None] * q).reshape(N, K)
    a = rng.standard_normal((rows, K)).astype(np.float32)
    for n in (N - 4, N - 3, N):
        da, dw, dc = dev.up(a), dev.up(blob[:n]), dev.zeros(rows * n * 4)
        dev.call("m40llm_ext_gemm_f32xq80_gguf_f32", da.ptr, dw.ptr, dc.ptr, rows, n, K)
        dev.sync()
        want = a.astype(np.float64) @ w[:n].T
        bound = np.abs(a).astype(np.float64) @ np.abs(w[:n]).T * 2.0 ** -20          # 32 products a chain, a sum of at most 64 of those by halves
        assert np.all(np.abs(dc.download(np.float32, (rows, n)) - want) <= bound)
