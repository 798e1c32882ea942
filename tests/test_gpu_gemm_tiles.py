"""The many-row product f32 [M][K] x f16 [N][K]^T over the tiles and K splits that row, column and K counts choose, at their edges."""
import numpy as np
import pytest

from tests.gpu_common import Dev, f16bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return Dev()


# 64 x 64 (one part, several parts), 64 x 128, 128 x 128 and 128 x 256 tiles; rows, columns and k that fill no tile, an odd number of steps of
# 32, one step, fewer steps than buffers, columns that no float4 divides, more than one round of tiles
@pytest.mark.parametrize("M,N,K", [(33, 16, 32), (33, 17, 64), (64, 64, 2048), (65, 130, 2112), (127, 1030, 5632), (129, 2048, 320), (200, 2560, 2080), (257, 2048, 5632),
                                   (257, 2049, 2048), (385, 2044, 1984), (522, 2048, 2048), (522, 2560, 2048), (522, 2050, 5600), (640, 2048, 2016), (1030, 2048, 2048),
                                   (1030, 5640, 96), (1301, 3001, 352), (2049, 2300, 160)])
def test_many_rows_tiles_vs_float64(dev, M, N, K):
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    A[::5] *= 1e-4
    A[M - 1] *= 1e4
    B = f16bits(rng.standard_normal((N, K)) * 0.05)
    got = dev.gemm_gguf(A, B, M, N, K).astype(np.float64)
    B64 = B.view(np.float16).astype(np.float64)
    # against the sum of the products' magnitudes: K additions in float32 in some order err by 2^-24 each at random signs (4 sqrt(K) of them
    # covers the largest of all elements), the two f16 parts of an activation by 2^-22 of the row's largest; elements share one bound
    mag = np.abs(A.astype(np.float64)) @ np.abs(B64).T
    row_max = np.abs(A).max(axis=1, keepdims=True).astype(np.float64) * np.abs(B64).sum(axis=1)
    bound = mag * 4.0 * np.sqrt(K) * 2.0 ** -24 + row_max * 2.0 ** -22
    err = np.abs(got - A.astype(np.float64) @ B64.T)
    i = int(np.argmax(err / bound))
    assert (err <= bound).all(), (i // N, i % N, float(err.flat[i]), float(bound.flat[i]))
