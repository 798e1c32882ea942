"""Projections of a decode step for up to 32 rows (m40llm_ext_batched_wide_*): every row count at the edges of its tiles of sixteen, K that gives
the eight waves unequal numbers of blocks of 64, columns that end in the middle of a tile, every number of column tiles per workgroup, against 64-bit products."""
import numpy as np
import pytest

from gpu_common import Dev, close, f16bits, m40

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = Dev()
    yield d
    d.ctx.close()


def _rows(rng, rows, K):
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[rows // 2] *= 3e3                       # rows of very different magnitude
    x[rows - 1] *= 1e-3
    x[0, :K // 2] *= 1e-4                     # and chunks
    return x


def _f64(w):
    return w.view(np.float16).astype(np.float64)


def _normed(x, nw, eps):
    x = x.astype(np.float64)
    return x / np.sqrt((x * x).mean(axis=1, keepdims=True) + eps) * nw


def _same(got, want):
    # f32 sums of at most 5632 products of operands exact to 2^-22: a few 1e-7 of the row's largest value
    sc = np.abs(want).max(axis=1, keepdims=True)
    close(got / sc, want / sc, 1e-5, 2e-6)


# column tiles of sixteen: 1 and 129 (one a workgroup, halves of K or not), 300, 700, 1000, 1500 (two, three, four and six a workgroup)
@pytest.mark.parametrize("rows,N,K", [(9, 7, 256), (16, 2048, 5632), (17, 2063, 768), (32, 2048, 1024), (31, 4800, 512), (12, 11195, 256), (32, 16000, 768),
                                      (25, 24000, 256), (1, 2048, 2816), (24, 4100, 1280)])
def test_residual_onto_zero(dev, rows, N, K):
    rng = np.random.default_rng(rows * 7 + N)
    a, w = _rows(rng, rows, K), f16bits(rng.standard_normal((N, K)) * 0.03)
    res = rng.standard_normal((rows, N)).astype(np.float32)
    da, dw, dres, out = dev.up(a), dev.up(w), dev.up(res), dev.zeros(rows * N * 4)
    want = a.astype(np.float64) @ _f64(w).T
    dev.call("m40llm_ext_batched_wide_gemm_residual_onto_zero_async", da.ptr, dw.ptr, dres.ptr, out.ptr, rows, N, K)
    dev.sync()
    got = out.download(np.float32, (rows, N))
    _same(got, want + res)
    again = dev.zeros(rows * N * 4)
    dev.call("m40llm_ext_batched_wide_gemm_residual_onto_zero_async", da.ptr, dw.ptr, dres.ptr, again.ptr, rows, N, K)
    dev.sync()
    assert np.array_equal(again.download(np.float32, (rows, N)), got)          # the same bits whichever half of K arrives first
    dev.call("m40llm_ext_batched_wide_gemm_residual_onto_zero_async", da.ptr, dw.ptr, dres.ptr, dres.ptr, rows, N, K)      # in place: overwritten
    dev.sync()
    _same(dres.download(np.float32, (rows, N)), want + res)
    dev.call("m40llm_ext_batched_wide_gemm_residual_onto_zero_async", da.ptr, dw.ptr, dres.ptr, out.ptr, 33, N, K, expect=-6)
    dev.call("m40llm_ext_batched_wide_gemm_residual_onto_zero_async", da.ptr, dw.ptr, dres.ptr, out.ptr, rows, N, K - 64, expect=-6)


@pytest.mark.parametrize("rows,F,K,norm_dtype", [(9, 1004, 256, 1), (16, 5632, 2048, 0), (17, 2049, 768, 1), (32, 11003, 512, 0)])
def test_norm_gate_up_and_norm_product(dev, rows, F, K, norm_dtype):
    rng = np.random.default_rng(rows + F)
    x = _rows(rng, rows, K)
    nw = (1 + 0.1 * rng.standard_normal(K)).astype(np.float16).astype(np.float32)
    wg, wu = (f16bits(rng.standard_normal((F, K)) * 0.05) for _ in range(2))
    dx, dnw, dwg, dwu = dev.up(x), dev.up(f16bits(nw) if norm_dtype == 0 else nw), dev.up(wg), dev.up(wu)
    hid, out, clear = dev.zeros(rows * F * 4), dev.zeros(rows * F * 4), dev.up(np.full(rows * 1000 + 3, 5.0, dtype=np.float32))
    dev.call("m40llm_ext_batched_wide_norm_gate_up_swiglu_async", dx.ptr, dnw.ptr, norm_dtype, 1e-5, dwg.ptr, dwu.ptr, hid.ptr, rows, F, K, clear.ptr, rows * 1000)
    dev.call("m40llm_ext_batched_wide_norm_gemm_async", dx.ptr, dnw.ptr, norm_dtype, 1e-5, dwg.ptr, out.ptr, rows, F, K)
    dev.sync()
    xn = _normed(x, nw, 1e-5)
    g, u = xn @ _f64(wg).T, xn @ _f64(wu).T
    _same(out.download(np.float32, (rows, F)), g)
    _same(hid.download(np.float32, (rows, F)), g / (1 + np.exp(-g)) * u)
    assert np.array_equal(clear.download(np.float32, (rows * 1000 + 3,)), [0.0] * (rows * 1000) + [5.0] * 3)


@pytest.mark.parametrize("rows,qh,kvh,hd,K,layout,bias", [(9, 32, 4, 64, 2048, 0, False), (32, 16, 2, 128, 2048, 1, True), (17, 5, 5, 16, 768, 1, True),
                                                          (30, 3, 1, 32, 256, 0, True)])
def test_norm_qkv_rope_append(dev, rows, qh, kvh, hd, K, layout, bias):
    rng = np.random.default_rng(rows * 3 + hd)
    x, nw = _rows(rng, rows, K), (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    w = [f16bits(rng.standard_normal((n * hd, K)) * 0.03) for n in (qh, kvh, kvh)]
    b = [rng.standard_normal(n * hd).astype(np.float32) for n in (qh, kvh, kvh)]
    slots, lens = rng.permutation(rows + 3)[:rows].astype(np.uint32), rng.integers(0, 60, rows).astype(np.uint32)
    kv = m40.KVCache(dev.ctx, 64, rows + 3, kvh, hd)
    dx, dnw, dw, db = dev.up(x), dev.up(nw), [dev.up(t) for t in w], [dev.up(t) for t in b]
    ds, dl, q, clear = dev.up(slots), dev.up(lens), dev.zeros(rows * qh * hd * 4), dev.up(np.full(77, 5.0, dtype=np.float32))
    dev.call("m40llm_ext_batched_wide_norm_qkv_rope_append_async", kv.h, ds.ptr, dl.ptr, rows, dx.ptr, dnw.ptr, 1, 1e-5, *(t.ptr for t in dw),
             *(t.ptr if bias else None for t in db), K, qh, 1e4, 1.0, layout, q.ptr, clear.ptr, 76)
    dev.sync()
    xn = _normed(x, nw, 1e-5)
    y = [xn @ _f64(t).T + (c if bias else 0.0) for t, c in zip(w, b)]

    def rotated(t):
        t = t.reshape(rows, -1, hd).copy()
        a = lens[:, None, None] * 1e4 ** (-np.arange(0, hd, 2) / hd)
        i, j = (slice(0, hd // 2), slice(hd // 2, hd)) if layout else (slice(0, hd, 2), slice(1, hd, 2))
        u, v = t[..., i].copy(), t[..., j].copy()
        t[..., i], t[..., j] = u * np.cos(a) - v * np.sin(a), v * np.cos(a) + u * np.sin(a)
        return t.reshape(rows, -1)
    want_q, want_k = rotated(y[0]), rotated(y[1])
    got = q.download(np.float32, (rows, qh * hd))
    close(got / np.abs(want_q).max(axis=1, keepdims=True), want_q / np.abs(want_q).max(axis=1, keepdims=True), 1e-5, 2e-5)      # 2^-24 of an angle of 60 in f32
    for r in range(rows):
        k16, v16 = kv.read_token(int(slots[r]), int(lens[r]))
        for bits, want in ((k16, want_k[r]), (v16, y[2][r])):
            close(bits.view(np.float16) / np.abs(want).max(), want / np.abs(want).max(), 1e-3, 1e-4)
    assert np.array_equal(clear.download(np.float32, (77,)), [0.0] * 76 + [5.0])
    kv.destroy()


def test_results_that_overlap_the_rows(dev):
    """One launch reads all rows in every workgroup: results (and what is cleared) in them are refused, a result that is its own residual is not.  The calls for
    up to 16 rows take a result in place of the rows as before, in two launches."""
    rng, rows, K, D = np.random.default_rng(4), 12, 1024, 1024
    a, w = _rows(rng, rows, K), f16bits(rng.standard_normal((D, K)) * 0.03)
    res, ones = rng.standard_normal((rows, D)).astype(np.float32), np.ones(K, np.float32)
    da, dw, dn, dres, out = dev.up(a), dev.up(w), dev.up(ones), dev.up(np.concatenate([res.ravel(), np.zeros(4, np.float32)])), dev.zeros(rows * D * 4 + 64)
    last = da.ptr + rows * K * 4 - 16                  # the rows' last 16 bytes
    onto, wide = "m40llm_ext_batched_wide_gemm_residual_onto_zero_async", "m40llm_ext_batched_wide_norm_gate_up_swiglu_async"
    for to in (da.ptr, last, da.ptr - rows * D * 4 + 16):
        dev.call(onto, da.ptr, dw.ptr, dres.ptr, to, rows, D, K, expect=-6)
        dev.call("m40llm_ext_batched_wide_norm_gemm_async", da.ptr, dn.ptr, 1, 1e-5, dw.ptr, to, rows, D, K, expect=-6)
        dev.call(wide, da.ptr, dn.ptr, 1, 1e-5, dw.ptr, dw.ptr, to, rows, D, K, None, 0, expect=-6)
    dev.call(onto, da.ptr, dw.ptr, dres.ptr, dres.ptr + 16, rows, D, K, expect=-6)          # a residual half under the result
    dev.call(wide, da.ptr, dn.ptr, 1, 1e-5, dw.ptr, dw.ptr, out.ptr, rows, D, K, last, 4, expect=-6)
    dev.call(wide, da.ptr, dn.ptr, 1, 1e-5, dw.ptr, dw.ptr, out.ptr, rows, D, K, out.ptr + rows * D * 4 - 16, 8, expect=-6)
    kv = m40.KVCache(dev.ctx, 64, rows, 2, 64)
    ids, lens = dev.up(np.arange(rows, dtype=np.uint32)), dev.zeros(rows * 4)
    dev.call("m40llm_ext_batched_wide_norm_qkv_rope_append_async", kv.h, ids.ptr, lens.ptr, rows, da.ptr, dn.ptr, 1, 1e-5, dw.ptr, dw.ptr, dw.ptr, None, None, None, K, 8, 1e4, 1.0, 0,
             last, None, 0, expect=-6)
    dev.sync()
    assert np.array_equal(da.download(np.float32, (rows, K)), a)                            # nothing was enqueued
    want = a.astype(np.float64) @ _f64(w).T + res
    for name in ("m40llm_ext_batched_gemm_residual_f32xf16_async", "m40llm_ext_batched_gemm_residual_onto_zero_f32xf16_async"):
        dev.call(name, da.ptr, dw.ptr, dres.ptr, da.ptr, rows, D, K)
        dev.sync()
        _same(da.download(np.float32, (rows, D)), want)
        da = dev.up(a)
    kv.destroy()


@pytest.mark.parametrize("rows,N,K", [(9, 2048, 1024), (16, 512, 5632), (16, 4097, 2048)])
def test_results_of_nine_and_more_rows_are_overwritten(dev, rows, N, K):
    """Only up to eight rows are added onto zeros by the call for up to 16: whatever the result holds before, more rows overwrite it."""
    rng = np.random.default_rng(rows + N)
    a, w, res = _rows(rng, rows, K), f16bits(rng.standard_normal((N, K)) * 0.03), rng.standard_normal((rows, N)).astype(np.float32)
    da, dw, dres, out = dev.up(a), dev.up(w), dev.up(res), dev.up(np.full((rows, N), 7.0, np.float32))
    want = a.astype(np.float64) @ _f64(w).T + res
    for _ in range(2):
        dev.call("m40llm_ext_batched_gemm_residual_onto_zero_f32xf16_async", da.ptr, dw.ptr, dres.ptr, out.ptr, rows, N, K)
        dev.sync()
        _same(out.download(np.float32, (rows, N)), want)


@pytest.mark.parametrize("rows,N,K", [(9, 2048, 2048), (32, 2048, 5632), (17, 333, 1024), (32, 16000, 768)])
def test_residual_is_rounded_once(dev, rows, N, K):
    """The product is finished before a residual of a hundred times its size is added: half a unit in the last place of the result, and the product's own
    error, at most a third of that here."""
    rng = np.random.default_rng(rows + K)
    a, w = rng.standard_normal((rows, K)).astype(np.float32), f16bits(rng.standard_normal((N, K)) / np.sqrt(K))
    res = (100.0 + 27.0 * rng.random((rows, N))).astype(np.float32) * rng.choice([-1.0, 1.0], (rows, N)).astype(np.float32)
    a[0] = 0.0                                        # a product of zeros: the residual itself
    da, dw, dres = dev.up(a), dev.up(w), dev.up(res)
    want = a.astype(np.float64) @ _f64(w).T + res
    for _ in range(3):
        out = dev.zeros(rows * N * 4)
        dev.call("m40llm_ext_batched_wide_gemm_residual_onto_zero_async", da.ptr, dw.ptr, dres.ptr, out.ptr, rows, N, K)
        dev.sync()
        got = out.download(np.float32, (rows, N))
        assert np.array_equal(got[0], res[0])
        ulp = np.spacing(np.abs(got)).astype(np.float64)
        assert (np.abs(got - want) <= 0.5 * ulp + 5.0 * 2.0 ** -22).all()           # products of up to five, their error 1e-7 of that
    out = dev.zeros(rows * N * 4)
    dev.call("m40llm_ext_batched_wide_gemm_residual_onto_zero_async", da.ptr, dw.ptr, None, out.ptr, rows, N, K)
    dev.sync()
    got = out.download(np.float32, (rows, N))
    assert not got[0].any()
    _same(got[1:], (want - res)[1:])
