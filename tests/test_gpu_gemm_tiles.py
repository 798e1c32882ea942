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
                                   (1030, 5640, 96), (1301, 3001, 352), (2049, 2300, 160), (1030, 5640, 864), (2065, 2300, 800)])
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


# where the tile of thousands of rows changes over: the same bits as the rows of a call that takes 128 x 128 tiles, and as those of one row of tiles more or less
@pytest.mark.parametrize("M,N,K", [(2048, 2560, 320), (2049, 2560, 320), (3333, 2560, 288), (3500, 2304, 64)])
def test_rows_of_the_large_tiles_are_the_same(dev, M, N, K):
    rng = np.random.default_rng(M)
    A, B = rng.standard_normal((M, K)).astype(np.float32), f16bits(rng.standard_normal((N, K)) * 0.05)
    got = dev.gemm_gguf(A, B, M, N, K).view(np.uint32)
    for first, rows in ((0, 1100), (M - 1100, 1100), (0, M - 128), (1, M - 1)):
        assert np.array_equal(dev.gemm_gguf(np.ascontiguousarray(A[first:first + rows]), B, rows, N, K).view(np.uint32), got[first:first + rows]), (first, rows)


@pytest.mark.parametrize("norm_dtype", [0, 1])
@pytest.mark.parametrize("M,F,K", [(33, 16, 64), (65, 48, 128), (100, 5632, 2048), (129, 1024, 320), (300, 5632, 256), (522, 272, 2048), (1030, 2816, 96), (2049, 1040, 160)])
def test_gate_up_swiglu_equals_separate_calls(dev, M, F, K, norm_dtype):
    rng = np.random.default_rng(M + F + K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[2] *= 1e-4
    w = (1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    dw, dx = dev.up(w if norm_dtype else f16bits(w)), dev.up(x)
    gate, up = (f16bits(rng.standard_normal((F, K)) * 0.05) for _ in range(2))
    dg, du = dev.up(gate), dev.up(up)
    g, u, want, got = (dev.zeros(M * F * 4) for _ in range(4))
    dev.call("m40llm_ext_prefill_gemm_fused_async", 1, dx.ptr, None, dw.ptr, norm_dtype, 1e-5, M, K, 2, dg.ptr, F, g.ptr, None, du.ptr, F, u.ptr, None, 0, None, 0)
    dev.sync()
    dev.call("m40llm_swiglu_f32_async", g.ptr, u.ptr, want.ptr, M * F)
    dev.sync()
    dev.call("m40llm_ext_prefill_norm_gate_up_swiglu_async", dx.ptr, dw.ptr, norm_dtype, 1e-5, M, K, dg.ptr, du.ptr, F, got.ptr, 0)
    dev.sync()
    want, got = want.download(np.float32, (M, F)), got.download(np.float32, (M, F))
    if (M + 127) // 128 * ((F + 127) // 128) * 2 > 128:        # larger grids are cut nowhere: the same sums
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    # otherwise the two may add k in other blocks: two products of about sqrt(K) roundings each, relative to their own size
    assert (np.abs(got - want) <= 2.0 ** -22 * np.sqrt(K) * (np.abs(want) + np.abs(want).max())).all()


def test_gate_up_swiglu_declines_and_checks(dev):
    M, K, F = 64, 64, 48
    x, w, b, o = dev.zeros(M * K * 4), dev.zeros(K * 4), dev.zeros(F * K * 2), dev.zeros(M * F * 4)
    name = "m40llm_ext_prefill_norm_gate_up_swiglu_async"
    dev.call(name, x.ptr, w.ptr, 1, 1e-5, 32, K, b.ptr, b.ptr, F, o.ptr, 0, expect=1)           # few rows
    dev.call(name, x.ptr, w.ptr, 1, 1e-5, M, K, b.ptr, b.ptr, 40, o.ptr, 0, expect=1)           # columns in no groups of 16
    dev.call(name, x.ptr, w.ptr, 1, 1e-5, M, 32, b.ptr, b.ptr, F, o.ptr, 0, expect=1)           # a small grid, an odd number of steps
    dev.call(name, x.ptr, None, 1, 1e-5, M, K, b.ptr, b.ptr, F, o.ptr, 0, expect=-1)
    dev.call(name, x.ptr, w.ptr, 2, 1e-5, M, K, b.ptr, b.ptr, F, o.ptr, 0, expect=-2)


# the first product whole, in two and in more parts of K; fewer k than columns (the parts would lie under the next product's rows); as gate and up and as Q/K/V
@pytest.mark.parametrize("M,K0,D,Ns,gated", [(33, 2048, 2048, (1024, 1024), 1), (101, 2048, 2048, (5632, 5632), 1), (101, 5632, 2048, (2048, 256, 256), 0), (250, 11008, 2048, (2048, 256, 256), 0),
                                             (522, 5632, 2048, (2048, 256, 256), 0), (522, 512, 2048, (272, 272), 1), (1030, 2048, 2048, (2816, 2816), 1), (65, 96, 160, (50,), 0),
                                             (300, 1024, 64, (48, 33), 0), (40, 4096, 260, (16,), 0)])
def test_project_norm_project_equals_separate_calls(dev, M, K0, D, Ns, gated):
    rng = np.random.default_rng(M + K0 + D)
    x, r = rng.standard_normal((M, K0)).astype(np.float32), rng.standard_normal((M, D)).astype(np.float32)
    w = (1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    dx, dr, dw, dB0 = dev.up(x), dev.up(r), dev.up(w), dev.up(f16bits(rng.standard_normal((D, K0)) * 0.05))
    dB = [dev.up(f16bits(rng.standard_normal((n, D)) * 0.05)) for n in Ns]
    none = [None, 0, None]
    supported = K0 % 32 == 0 and D % 32 == 0
    name = "m40llm_ext_prefill_project_norm_project_async"
    c0, got = dev.zeros(M * D * 4), [dev.zeros(M * n * 4) for n in Ns]
    args = sum([[b.ptr, n, o.ptr] for b, n, o in zip(dB, Ns, got)], []) + none * (3 - len(Ns))
    dev.call(name, dx.ptr, M, K0, dB0.ptr, D, dr.ptr, c0.ptr, dw.ptr, 1, 1e-5, gated, len(Ns), *args, 0, expect=0 if supported else 1)
    dev.sync()
    if not supported:
        return
    want0, want = dev.zeros(M * D * 4), [dev.zeros(M * n * 4) for n in Ns]
    fused = "m40llm_ext_prefill_gemm_fused_async"
    dev.call(fused, 0, dx.ptr, None, None, 0, 1e-5, M, K0, 1, dB0.ptr, D, want0.ptr, dr.ptr, None, 0, None, None, 0, None, 0)
    if gated:
        dev.call("m40llm_ext_prefill_norm_gate_up_swiglu_async", want0.ptr, dw.ptr, 1, 1e-5, M, D, dB[0].ptr, dB[1].ptr, Ns[0], want[0].ptr, 0)
    else:
        a = sum([[b.ptr, n, o.ptr] + ([None] if i == 0 else []) for i, (b, n, o) in enumerate(zip(dB, Ns, want))], []) + none * (3 - len(Ns))
        dev.call(fused, 1, want0.ptr, None, dw.ptr, 1, 1e-5, M, D, len(Ns), *a, 0)
    dev.sync()
    for n, g, o in [(D, c0, want0)] + list(zip(Ns, got, want)):
        assert np.array_equal(g.download(np.uint32, (M, n)), o.download(np.uint32, (M, n))), n
    dev.call(name, dx.ptr, M, K0, dB0.ptr, D, None, c0.ptr, dw.ptr, 1, 1e-5, gated, len(Ns), *args, 0, expect=-1)
    dev.call(name, dx.ptr, M, K0, dB0.ptr, D, dr.ptr, c0.ptr, dw.ptr, 1, 1e-5, gated, 0, *args, 0, expect=-2)
