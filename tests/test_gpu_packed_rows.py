"""O and down projection of rows that the launch before left as matrix operands (m40llm_ext_batched_packed_*, ..._packed_async): every padded row count, K that gives
the waves unequal numbers of blocks, columns that end in the middle of a tile, K whole and in halves, units of zeros, against 64-bit products of the rows that the
f32 form of the same call makes."""
import numpy as np
import pytest

from gpu_common import Dev, close, f16bits, m40

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = Dev()
    yield d
    d.ctx.close()


def _bytes(rows, K):
    pad = 8 if rows <= 8 else (16 if rows <= 16 else 32)
    return pad * K * 4 + pad * K // 8 * 4


def _f64(w):
    return w.view(np.float16).astype(np.float64)


def _project(dev, packed, rows64, w, res, rows, N, K):
    """Residual, no residual and the same bits twice, onto zeros; `rows64`: the rows the buffer holds."""
    dw, dres = dev.up(w), dev.up(res)
    want = rows64 @ _f64(w).T
    # operands exact to 2^-22 of themselves and 2^-31 of the largest of their eight; f32 sums of K products: a few 2^-24 of
    # the row's largest sum of magnitudes a wave's share
    bound = np.abs(rows64) @ np.abs(_f64(w)).T * 2.0 ** -21
    got = []
    for r in (res, None, res):
        out = dev.zeros(rows * N * 4)
        dev.call("m40llm_ext_batched_packed_gemm_residual_onto_zero_async", packed.ptr, dw.ptr, None if r is None else dres.ptr, out.ptr, rows, N, K)
        dev.sync()
        got.append(out.download(np.float32, (rows, N)))
        full = want + (0.0 if r is None else r)
        assert np.all(np.abs(got[-1] - full) <= bound + np.abs(full) * 2.0 ** -23)
    assert np.array_equal(got[0], got[2])           # the same bits whichever half of K arrives first
    dev.call("m40llm_ext_batched_packed_gemm_residual_onto_zero_async", packed.ptr, dw.ptr, dres.ptr, dres.ptr, rows, N, K, expect=-6)
    dev.call("m40llm_ext_batched_packed_gemm_residual_onto_zero_async", packed.ptr, dw.ptr, dres.ptr, out.ptr, 33, N, K, expect=-6)
    dev.call("m40llm_ext_batched_packed_gemm_residual_onto_zero_async", packed.ptr, dw.ptr, dres.ptr, out.ptr, rows, N, K - 64, expect=-6)


@pytest.mark.parametrize("rows,F,D,N", [(1, 256, 2048, 7), (3, 5632, 2048, 2048), (8, 11008, 2048, 2048), (9, 768, 256, 2063), (16, 5632, 512, 2048), (17, 1024, 256, 4100),
                                        (32, 2816, 2048, 2048), (25, 4864, 256, 900)])
def test_feed_forward(dev, rows, F, D, N):
    rng = np.random.default_rng(rows * 5 + F)
    x = rng.standard_normal((rows, D)).astype(np.float32)
    x[rows // 2] *= 3e3
    x[rows - 1] *= 1e-3
    nw = np.abs(1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    wg, wu = (rng.standard_normal((F, D)) * 0.08 for _ in range(2))
    wu[8:16] = 0.0                                  # a unit of zeros
    wu[16:24] *= 1e-4                               # units of very different magnitude that meet in one instruction
    dx, dnw, dwg, dwu = dev.up(x), dev.up(nw), dev.up(f16bits(wg)), dev.up(f16bits(wu))
    hid, clear = dev.zeros(rows * F * 4), dev.up(np.full(rows * 99 + 3, 5.0, dtype=np.float32))
    packed = dev.up(np.full(_bytes(rows, F), 0xFF, dtype=np.uint8))     # rows that are not there: NaN
    plain = "m40llm_ext_batched_norm_gate_up_swiglu_clear_async" if rows <= 8 else "m40llm_ext_batched_wide_norm_gate_up_swiglu_async"
    dev.call(plain, dx.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, hid.ptr, rows, F, D, None, 0)
    dev.call("m40llm_ext_batched_norm_gate_up_swiglu_packed_async", dx.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, packed.ptr, rows, F, D, clear.ptr, rows * 99)
    dev.sync()
    assert np.array_equal(clear.download(np.float32, (rows * 99 + 3,)), [0.0] * (rows * 99) + [5.0] * 3)
    w = f16bits(rng.standard_normal((N, F)) * 0.03)
    _project(dev, packed, hid.download(np.float32, (rows, F)).astype(np.float64), w, rng.standard_normal((rows, N)).astype(np.float32), rows, N, F)
    dev.call("m40llm_ext_batched_norm_gate_up_swiglu_packed_async", dx.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, packed.ptr, rows, F - 64, D, None, 0, expect=-6)
    dev.call("m40llm_ext_batched_norm_gate_up_swiglu_packed_async", dx.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, dx.ptr, rows, F, D, None, 0, expect=-6)


# one chunk and several, the kernel for short rows and the one on matrix instructions
@pytest.mark.parametrize("rows,qh,kvh,hd,longest", [(2, 4, 2, 64, 60), (8, 16, 2, 128, 700), (5, 32, 4, 64, 400), (9, 8, 8, 64, 530), (17, 4, 4, 128, 40), (32, 32, 4, 64, 1000)])
def test_attention(dev, rows, qh, kvh, hd, longest):
    rng = np.random.default_rng(rows + longest)
    kv = m40.KVCache(dev.ctx, 1024, rows, kvh, hd)
    lens = rng.integers(1, longest + 1, rows).astype(np.uint32)
    lens[0] = longest
    for r in range(rows):
        k, v = (f16bits(rng.standard_normal((int(lens[r]), kvh, hd))) for _ in range(2))
        dev.fill_dense(kv, r, k, v)
    K, N = qh * hd, 2048 if qh * hd > 512 else 130
    q = rng.standard_normal((rows, K)).astype(np.float32)
    dq, out, ids, dlens = dev.up(q), dev.zeros(q.nbytes), dev.up(np.arange(rows, dtype=np.uint32)), dev.up(lens)
    packed = dev.up(np.full(_bytes(rows, K), 0xFF, dtype=np.uint8))
    dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_async", kv.h, ids.ptr, dlens.ptr, 0, rows, longest, dq.ptr, qh, out.ptr)
    dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_packed_async", kv.h, ids.ptr, dlens.ptr, 0, rows, longest, dq.ptr, qh, packed.ptr)
    dev.sync()
    w = f16bits(rng.standard_normal((N, K)) * 0.03)
    _project(dev, packed, out.download(np.float32, (rows, K)).astype(np.float64), w, rng.standard_normal((rows, N)).astype(np.float32), rows, N, K)
    kv.destroy()


@pytest.mark.parametrize("rows,qh,kvh,hd", [(2, 14, 2, 64), (9, 1, 1, 64), (32, 5, 5, 64), (4, 1, 1, 128), (33, 4, 4, 64)])
def test_refused_attention(dev, rows, qh, kvh, hd):
    """Rows that the buffer has no form for (q heads x head size no multiple of 256, more than 32): its size is 0, the call refuses, and nothing is written."""
    K = qh * hd
    kv = m40.KVCache(dev.ctx, 16, rows, kvh, hd)
    ids, lens, q = dev.up(np.arange(rows, dtype=np.uint32)), dev.up(np.full(rows, 3, dtype=np.uint32)), dev.zeros(rows * K * 4)
    packed = dev.up(np.full(64, 0xFF, dtype=np.uint8))
    assert dev.lib.m40llm_ext_packed_rows_bytes(rows, K) == 0
    dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_packed_async", kv.h, ids.ptr, lens.ptr, 0, rows, 16, q.ptr, qh, packed.ptr, expect=-6)
    dev.sync()
    assert (packed.download(np.uint8, (64,)) == 0xFF).all()
    kv.destroy()


def test_refused_buffers(dev):
    """A buffer, or q, that is not aligned, and one that lies over q; the size is that of the rows' padded number."""
    rows, qh, hd = 9, 4, 64
    K = qh * hd
    kv = m40.KVCache(dev.ctx, 16, rows, qh, hd)
    ids, lens, q = dev.up(np.arange(rows, dtype=np.uint32)), dev.up(np.full(rows, 3, dtype=np.uint32)), dev.zeros(rows * K * 4 + 16)
    for r in (1, 8, 9, 16, 17, 32): assert dev.lib.m40llm_ext_packed_rows_bytes(r, K) == _bytes(r, K)
    packed = dev.zeros(_bytes(rows, K) + 16)
    call = lambda qp, pp, expect: dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_packed_async", kv.h, ids.ptr, lens.ptr, 0, rows, 16, qp, qh, pp, expect=expect)
    call(q.ptr, packed.ptr + 4, -6)
    call(q.ptr + 4, packed.ptr, -6)
    call(packed.ptr, packed.ptr, -6)
    call(packed.ptr + _bytes(rows, K) - 16, packed.ptr, -6)
    call(None, packed.ptr, -1)
    call(q.ptr, None, -1)
    call(q.ptr, packed.ptr, 0)
    dev.sync()
    kv.destroy()


# one launch on matrix cores (width 2048, up to eight rows), nine rows and more, the vector-ALU form, product and epilogue
@pytest.mark.parametrize("rows,qh,kvh,hd,D", [(1, 32, 4, 64, 2048), (8, 16, 2, 128, 2048), (5, 4, 2, 64, 256), (12, 8, 8, 64, 512), (16, 4, 1, 128, 2048), (3, 8, 2, 64, 4096)])
@pytest.mark.parametrize("floats", [1, 1000])
def test_clear_beside_qkv(dev, rows, qh, kvh, hd, D, floats):
    """Q, K and V with a range cleared on the side: the bits of the call without one, zeros in the range and nothing behind it; a range that lies over the rows or q is refused."""
    rng = np.random.default_rng(rows * 7 + D)
    x, nw = rng.standard_normal((rows, D)).astype(np.float32), (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    dx, dnw = dev.up(x), dev.up(nw)
    w = [dev.up(f16bits(rng.standard_normal((n * hd, D)) * 0.05)) for n in (qh, kvh, kvh)]
    ids, lens = dev.up(np.arange(rows, dtype=np.uint32)), dev.up(rng.integers(0, 8, rows).astype(np.uint32))
    got = []
    for name, clear in (("m40llm_ext_batched_norm_qkv_rope_append_async", False), ("m40llm_ext_batched_norm_qkv_rope_append_clear_async", True)):
        kv, q = m40.KVCache(dev.ctx, 16, rows, kvh, hd), dev.zeros(rows * qh * hd * 4)
        zone = dev.up(np.full(floats + 3, 5.0, dtype=np.float32))
        args = lambda *tail: (kv.h, ids.ptr, lens.ptr, rows, dx.ptr, dnw.ptr, 1, 1e-5, *(t.ptr for t in w), None, None, None, D, qh, 1e4, 1.0, 0, q.ptr, *tail)
        if clear:
            for at in (dx.ptr, dx.ptr + rows * D * 4 - 4, q.ptr, q.ptr + rows * qh * hd * 4 - 4): dev.call(name, *args(at, floats), expect=-6)
            dev.sync()
            assert np.array_equal(dx.download(np.float32, (rows, D)), x) and not q.download(np.uint32, (rows * qh * hd,)).any()
        dev.call(name, *args(*((zone.ptr, floats) if clear else ())))
        dev.sync()
        assert np.array_equal(zone.download(np.float32, (floats + 3,)), ([0.0] if clear else [5.0]) * floats + [5.0] * 3)
        got.append([q.download(np.uint32, (rows * qh * hd,))] + [t for r in range(rows) for p in range(8) for t in kv.read_token(r, p)])
        kv.destroy()
    assert all(np.array_equal(a, b) for a, b in zip(*got))


# `far`: log2 between the units that meet in an instruction, either side of where each is multiplied on its own
@pytest.mark.parametrize("rows,F,D,N", [(2, 512, 2048, 40), (8, 2816, 2048, 2048), (13, 1024, 256, 70), (32, 2816, 256, 2048)])
@pytest.mark.parametrize("far", [4, 8, 12, 20, 25, 30, 39])
def test_outliers(dev, rows, F, D, N, far):
    """A unit far above its neighbours, whose columns have no weight: nothing of the small ones is lost beside it."""
    rng = np.random.default_rng(far + F)
    x, nw = rng.standard_normal((rows, D)).astype(np.float32), np.ones(D, np.float32)
    wg, wu = (rng.standard_normal((F, D)) * 0.02 for _ in range(2))
    unit = np.arange(F) // 8
    large, low = unit % 8 == unit // 8 % 8, min(far, 24)
    wu[~large] *= 2.0 ** -(low // 2)
    wg[~large] *= 2.0 ** -(low - low // 2)
    wu[large] *= 2.0 ** (far - low)
    dx, dnw, dwg, dwu = dev.up(x), dev.up(nw), dev.up(f16bits(wg)), dev.up(f16bits(wu))
    hid, packed = dev.zeros(rows * F * 4), dev.up(np.full(_bytes(rows, F), 0xFF, dtype=np.uint8))
    plain = "m40llm_ext_batched_norm_gate_up_swiglu_clear_async" if rows <= 8 else "m40llm_ext_batched_wide_norm_gate_up_swiglu_async"
    dev.call(plain, dx.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, hid.ptr, rows, F, D, None, 0)
    dev.call("m40llm_ext_batched_norm_gate_up_swiglu_packed_async", dx.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, packed.ptr, rows, F, D, None, 0)
    dev.sync()
    a = hid.download(np.float32, (rows, F)).astype(np.float64)
    w = rng.standard_normal((N, F)) * 0.03
    w[:, large] = 0.0
    w = f16bits(w)
    dw, out = dev.up(w), dev.zeros(rows * N * 4)
    dev.call("m40llm_ext_batched_packed_gemm_residual_onto_zero_async", packed.ptr, dw.ptr, None, out.ptr, rows, N, F)
    dev.sync()
    most = np.repeat(np.abs(a).reshape(rows, F // 8, 8).max(axis=2), 8, axis=1)
    # a value is exact to 2^-22 of itself and 2^-31 of its unit's largest; f32 sums of K products (2^-22 of the sum of magnitudes)
    bound = (np.abs(a) * 2.0 ** -21 + most * 2.0 ** -30) @ np.abs(_f64(w)).T
    err = np.abs(out.download(np.float32, (rows, N)) - a @ _f64(w).T)
    assert np.all(err <= bound), (err / bound).max()


@pytest.mark.parametrize("rows,qh,kvh,hd,length", [(3, 4, 2, 64, 40), (8, 32, 4, 64, 128), (9, 4, 4, 64, 70), (32, 16, 2, 128, 256)])
def test_infinities(dev, rows, qh, kvh, hd, length):
    """A row with one infinity gives infinities, of each weight's sign; rows of very large and very small values beside it keep theirs."""
    rng = np.random.default_rng(rows + length)
    K, N = qh * hd, 130
    kv = m40.KVCache(dev.ctx, length, rows, kvh, hd)
    for r in range(rows):
        k, v = (rng.standard_normal((length, kvh, hd)).astype(np.float16) for _ in range(2))
        v *= np.float16(2.0 ** (13 if r % 3 == 1 else -10))          # |v| < 2^3: within f16
        if r % 3 == 0: v[r % length, r % kvh, 5] = np.inf
        dev.fill_dense(kv, r, f16bits(0.1 * k), v.view(np.uint16))
    q = rng.standard_normal((rows, K)).astype(np.float32)
    dq, out, ids, dlens = dev.up(q), dev.zeros(q.nbytes), dev.up(np.arange(rows, dtype=np.uint32)), dev.up(np.full(rows, length, dtype=np.uint32))
    packed, y = dev.up(np.full(_bytes(rows, K), 0xFF, dtype=np.uint8)), dev.zeros(rows * N * 4)
    dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_async", kv.h, ids.ptr, dlens.ptr, 0, rows, length, dq.ptr, qh, out.ptr)
    dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_packed_async", kv.h, ids.ptr, dlens.ptr, 0, rows, length, dq.ptr, qh, packed.ptr)
    w = rng.standard_normal((N, K)) * 0.03
    w = f16bits(np.where(np.abs(w) < 1e-3, 1e-3, w))
    # one head of the infinite kv head alone keeps its weight's sign: the heads that share it would add infinities of both
    group = qh // kvh
    w64 = _f64(w).reshape(N, kvh, group, hd)
    w64[:, :, 1:, 5] = np.abs(w64[:, :, :1, 5]) * np.sign(w64[:, :, :1, 5])
    w = f16bits(w64.reshape(N, K))
    dw = dev.up(w)
    dev.call("m40llm_ext_batched_packed_gemm_residual_onto_zero_async", packed.ptr, dw.ptr, None, y.ptr, rows, N, K)
    dev.sync()
    a, got = out.download(np.float32, (rows, K)).astype(np.float64), y.download(np.float32, (rows, N))
    want, fine = a @ _f64(w).T, np.arange(rows) % 3 != 0
    assert np.isinf(want[~fine]).all() and np.array_equal(got[~fine], want[~fine])
    assert np.all(np.abs(got[fine] - want[fine]) <= np.abs(a[fine]) @ np.abs(_f64(w)).T * 2.0 ** -21)
    kv.destroy()
