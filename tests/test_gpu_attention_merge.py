"""Merge of chunk partials: one, some and more than 64 chunks a row, rows of one batch with very different numbers of them, and partials of an earlier, longer call
(infinities) left in the buffer, against 64-bit attention."""
import numpy as np
import pytest

from gpu_common import Dev, close, f16bits, m40

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = Dev()
    yield d
    d.ctx.close()


@pytest.mark.parametrize("qh,kvh,hd,lens,hint", [(4, 2, 64, [8192], 8192), (4, 2, 128, [8193], 8704), (2, 1, 128, [16500, 1, 700], 16512), (16, 2, 64, [129, 128, 1000, 3], 1024),
                                                 (8, 8, 128, [640], 640)])
def test_merge_of_chunks(dev, qh, kvh, hd, lens, hint):
    rng = np.random.default_rng(hd + len(lens))
    B, L = len(lens), max(lens)
    kv = m40.KVCache(dev.ctx, hint, B + 1, kvh, hd)
    Kc, Vc = (rng.standard_normal((B, L, kvh, hd)).astype(np.float16) for _ in range(2))
    for b, n in enumerate(lens): dev.fill_dense(kv, b, Kc[b, :n].view(np.uint16), Vc[b, :n].view(np.uint16))
    dev.fill_dense(kv, B, f16bits(np.zeros((hint, kvh, hd))), f16bits(np.full((hint, kvh, hd), np.inf)))
    q = (2.0 * rng.standard_normal((B, qh * hd))).astype(np.float32)
    dq, out = dev.up(q), dev.zeros(q.nbytes)
    call = "m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_async"
    stale = dev.up(np.full(B, B, dtype=np.uint32)), dev.up(np.full(B, hint, dtype=np.uint32))
    ids, dlens = dev.up(np.arange(B, dtype=np.uint32)), dev.up(np.asarray(lens, dtype=np.uint32))
    dev.call(call, kv.h, stale[0].ptr, stale[1].ptr, 0, B, hint, dq.ptr, qh, out.ptr)
    dev.call(call, kv.h, ids.ptr, dlens.ptr, 0, B, hint, dq.ptr, qh, out.ptr)
    dev.sync()
    got = out.download(np.float32, (B, qh, hd)).astype(np.float64)
    for b, n in enumerate(lens):
        k, v = (np.repeat(t[b, :n].astype(np.float64), qh // kvh, axis=1) for t in (Kc, Vc))
        s = np.einsum("hd,thd->ht", q[b].reshape(qh, hd).astype(np.float64), k) / np.sqrt(hd)
        w = np.exp(s - s.max(axis=1, keepdims=True))
        want = np.einsum("ht,thd->hd", w / w.sum(axis=1, keepdims=True), v)
        # q exact to 2^-22 and sums of f32: scores of up to 40 off by a few 2^-20, the weights by as much
        close(got[b], want, 1e-5, 2e-5)
    kv.destroy()


# 16, 17, 32 and 33 chunks of 128 tokens: what a merge asks for at once, and one more
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("hint", [2048, 2049, 4096, 4097])
def test_merge_at_the_edges_of_a_request(dev, hd, hint):
    test_merge_of_chunks(dev, 4, 2, hd, [hint, 129], hint)


# short rows in batches of few and many q heads: one chunk and several, rows of a token, uneven rows
@pytest.mark.parametrize("qh,kvh,hd,rows,hint", [(32, 4, 64, 15, 128), (32, 4, 64, 16, 128), (32, 4, 64, 63, 256), (32, 4, 64, 64, 256), (32, 4, 64, 15, 512), (32, 4, 64, 16, 512),
                                                 (8, 8, 64, 64, 130), (64, 4, 128, 15, 256), (64, 4, 128, 16, 256), (16, 2, 128, 15, 400), (16, 2, 128, 16, 400), (64, 4, 128, 4, 257)])
def test_short_rows_of_a_batch(dev, qh, kvh, hd, rows, hint):
    rng = np.random.default_rng(qh + rows)
    lens = rng.integers(1, hint + 1, rows)
    lens[0], lens[-1] = hint, 1
    test_merge_of_chunks(dev, qh, kvh, hd, [int(n) for n in lens], hint)


@pytest.mark.parametrize("qh,kvh,hd,rows,hint", [(32, 4, 64, 4, 128), (32, 4, 64, 16, 128), (32, 4, 64, 32, 500), (16, 2, 128, 32, 120), (16, 2, 128, 16, 400), (32, 8, 128, 32, 256)])
def test_short_rows_of_a_batch_keep_infinities(dev, qh, kvh, hd, rows, hint):
    """An infinite value of a short row stays an infinity however many rows a call has, and no other element sees it; the error of the finite ones, q four times as
    large, stays that of f32 sums (a few 2^-24 of scores of up to 40)."""
    rng = np.random.default_rng(rows + hint)
    lens = rng.integers(2, hint + 1, rows)
    kv = m40.KVCache(dev.ctx, hint, rows, kvh, hd)
    Kc, Vc = (rng.standard_normal((rows, hint, kvh, hd)).astype(np.float16) for _ in range(2))
    Kc *= np.float16(0.25)
    for b, n in enumerate(lens):
        Vc[b, b % n, b % kvh, 3] = np.inf * (-1) ** b
        dev.fill_dense(kv, b, Kc[b].view(np.uint16), Vc[b].view(np.uint16))
    q = (4.0 * rng.standard_normal((rows, qh * hd))).astype(np.float32)
    dq, out, ids, dlens = dev.up(q), dev.zeros(q.nbytes), dev.up(np.arange(rows, dtype=np.uint32)), dev.up(lens.astype(np.uint32))
    dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_async", kv.h, ids.ptr, dlens.ptr, 0, rows, hint, dq.ptr, qh, out.ptr)
    dev.sync()
    got = out.download(np.float32, (rows, qh, hd)).astype(np.float64)
    for b, n in enumerate(lens):
        k, v = (np.repeat(t[b, :n].astype(np.float64), qh // kvh, axis=1) for t in (Kc, Vc))
        s = np.einsum("hd,thd->ht", q[b].reshape(qh, hd).astype(np.float64), k) / np.sqrt(hd)
        w = np.exp(s - s.max(axis=1, keepdims=True))
        want = np.einsum("ht,thd->hd", w / w.sum(axis=1, keepdims=True), v)
        assert np.array_equal(np.isinf(want), np.isinf(got[b])) and np.array_equal(want[np.isinf(want)], got[b][np.isinf(want)])
        fine = np.isfinite(want)
        close(got[b][fine], want[fine], 2e-6, 4e-6)
    kv.destroy()

# more rows and kv heads than two workgroups a CU: rows of one chunk, and long rows that then have one as well
@pytest.mark.parametrize("qh,kvh,hd,rows,hint", [(8, 8, 64, 65, 100), (4, 4, 128, 129, 128), (8, 4, 64, 129, 520), (8, 8, 128, 65, 2100)])
def test_more_rows_than_the_chip_takes_at_once(dev, qh, kvh, hd, rows, hint):
    rng = np.random.default_rng(rows + hint)
    lens = rng.integers(1, min(hint, 600) + 1, rows)
    lens[0], lens[-1] = hint, 1
    test_merge_of_chunks(dev, qh, kvh, hd, [int(n) for n in lens], hint)

@pytest.mark.parametrize("qh,kvh,hd,hint", [(32, 4, 64, 512), (6, 2, 64, 256), (5, 5, 64, 100), (16, 2, 128, 256), (12, 3, 128, 128), (40, 8, 128, 480)])
def test_short_row_in_a_launch_for_more(dev, qh, kvh, hd, hint):
    """Lengths at the edges of the steps of a pass, in a launch sized for `hint` tokens and in one of the row's own size: the same bits; rows behind the end hold NaN, and
    an infinity in the last one stays an infinity."""
    rng = np.random.default_rng(hint + hd)
    L, step = hint + 1, 8 * 512 // hd
    kv = m40.KVCache(dev.ctx, L, 1, kvh, hd)
    for n in sorted({1, step - 1, step, step + 1, 2 * step, 2 * step + 1, 4 * step, 4 * step + 1, hint - 1, hint}):
        if n > hint: continue
        Kc, Vc = (rng.standard_normal((L, kvh, hd)).astype(np.float16) for _ in range(2))
        Kc[n:], Vc[n:] = np.nan, np.nan
        Vc[n - 1, 0, 3] = np.inf
        dev.fill_dense(kv, 0, Kc.view(np.uint16), Vc.view(np.uint16))
        q = (2.0 * rng.standard_normal((qh, hd))).astype(np.float32)
        dq, out, own, pos = dev.up(q), dev.zeros(q.nbytes), dev.zeros(q.nbytes), dev.up(np.array([n - 1], dtype=np.uint32))
        dev.call("m40llm_ext_attention_last_token_f32_gqa_position_dev_async", kv.h, 0, dq.ptr, qh, pos.ptr, hint, out.ptr)
        dev.call("m40llm_attention_last_token_f32_gqa_async", kv.h, 0, dq.ptr, qh, n, own.ptr)
        dev.sync()
        got = out.download(np.float32, (qh, hd))
        if hint <= 8 * step: assert np.array_equal(got.view(np.uint32), own.download(np.uint32, (qh, hd)))
        k, v = (np.repeat(t[:n].astype(np.float64), qh // kvh, axis=1) for t in (Kc, Vc))
        s = np.einsum("hd,thd->ht", q.astype(np.float64), k) / np.sqrt(hd)
        w = np.exp(s - s.max(axis=1, keepdims=True))
        want = np.einsum("ht,thd->hd", w / w.sum(axis=1, keepdims=True), v)
        # scores of up to 2 hd terms in f32 and sums of n: (hd + n) 2^-24 of values of a few units, with room for exp
        assert np.array_equal(np.isinf(got), np.isinf(want))
        keep = np.isfinite(want)
        assert np.abs(got[keep] - want[keep]).max() <= 4 * (hd + n) * 2.0 ** -24 * np.abs(want[keep]).max() + 1e-6


# a row of every number of steps (64 tokens each, 32 with heads of 128), full and with one token more; one and four q heads a workgroup; an infinity in the last
# token's values, whose rows past the end repeat it
@pytest.mark.parametrize("qh,kvh,hd", [(4, 2, 64), (4, 2, 128), (32, 8, 64), (32, 8, 128)])
def test_every_number_of_steps(dev, qh, kvh, hd):
    step = 64 if hd == 64 else 32
    lens = [k * step + o for k in range(1, 8) for o in (0, 1)] + [1, 8 * step]
    test_merge_of_chunks(dev, qh, kvh, hd, lens, 8 * step)
    rng, rows, hint = np.random.default_rng(hd), len(lens), 8 * step
    kv = m40.KVCache(dev.ctx, hint, rows, kvh, hd)
    K, V = (rng.standard_normal((rows, hint, kvh, hd)).astype(np.float16) for _ in range(2))
    for b, n in enumerate(lens):
        V[b, n - 1, :, 5] = np.inf
        dev.fill_dense(kv, b, K[b].view(np.uint16), V[b].view(np.uint16))
    q = rng.standard_normal((rows, qh * hd)).astype(np.float32)
    dq, out, ids, dlens = dev.up(q), dev.zeros(q.nbytes), dev.up(np.arange(rows, dtype=np.uint32)), dev.up(np.asarray(lens, dtype=np.uint32))
    dev.call("m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_async", kv.h, ids.ptr, dlens.ptr, 0, rows, hint, dq.ptr, qh, out.ptr)
    dev.sync()
    got = out.download(np.float32, (rows, qh, hd))
    assert np.all(got[:, :, 5] == np.inf) and np.all(np.isfinite(np.delete(got, 5, axis=2)))
    kv.destroy()


# rows of a step that are 2^32 bytes and more from its address (64 rows of 64 columns, 32 of 128), and as many kv heads as have 32-bit offsets
@pytest.mark.parametrize("kvh,hd,n", [(540_672, 64, 64), (540_672, 64, 70), (541_300, 128, 32), (1 << 18, 64, 70)])
def test_rows_far_apart(dev, kvh, hd, n):
    """A key that takes nearly all weight in the last token, none in the others; a value there that says whose head it is."""
    kv = m40.KVCache(dev.ctx, n, 1, kvh, hd)
    value = np.repeat((np.arange(kvh) % 7 + 1).astype(np.float32), hd)
    zero, ones, dvalue, out = dev.zeros(value.nbytes), dev.up(np.ones(kvh * hd, np.float32)), dev.up(value), dev.zeros(value.nbytes)
    for t in range(n): dev.call("m40llm_kvcache_append_token_f32_async", kv.h, 0, (ones if t == n - 1 else zero).ptr, (dvalue if t == n - 1 else zero).ptr)
    dev.call("m40llm_attention_last_token_f32_gqa_async", kv.h, 0, ones.ptr, kvh, n, out.ptr)
    dev.sync()
    weight = np.exp(np.sqrt(hd)) / (np.exp(np.sqrt(hd)) + n - 1)
    # scores exact, a weight and a division in f32: a few 2^-24
    assert np.abs(out.download(np.float32, value.shape) / value - weight).max() <= 2e-6
    kv.destroy()
