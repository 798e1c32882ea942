"""Prompts from Q, K and V to the feed-forward's hidden rows in one call (m40llm_ext_prefill_attention_project_gate_up_async): the attention leaves its result as the O
projection's operands.  Against the two calls that write it as f32 in between, and the projection against 64 bits of those f32 rows: ragged lengths that start inside tiles
of sixteen rows, both head sizes, one and two query blocks a wave, K whole and in parts, values of one sequence fifty times another's and, within one,
a hundred times the first tokens', values that are not finite."""
import importlib

import numpy as np
import pytest

from gpu_common import Dev, f16bits, m40

pytestmark = pytest.mark.gpu
syn = importlib.import_module("m40-llm_amd.synthetic")
u32 = lambda a: np.asarray(a, dtype=np.uint32)


@pytest.fixture(scope="module")
def dev():
    d = Dev()
    yield d
    d.ctx.close()


@pytest.mark.parametrize("hd,qh,kvh,D,F,lens,layout,bias", [(64, 4, 1, 256, 512, [1, 63, 64, 65], 0, False), (64, 32, 4, 2048, 512, [23, 187, 90, 61, 161], 0, False),
                                                            (128, 16, 2, 2048, 256, [130, 700], 1, True), (64, 32, 4, 256, 256, [4096], 0, False), (128, 2, 2, 64, 64, [33], 1, True)])
def test_attention_project_gate_up(dev, hd, qh, kvh, D, F, lens, layout, bias):
    rng = np.random.default_rng(sum(lens) + hd)
    rows, K, n = sum(lens), qh * hd, len(lens)
    q, k, v = (rng.standard_normal((rows, w)).astype(np.float32) for w in (K, kvh * hd, kvh * hd))
    offs = u32(np.concatenate([[0], np.cumsum(lens)[:-1]]))
    v[offs[-1]:] *= 50.0
    v[offs[-1] + lens[-1] // 2:] *= 1e2
    if n > 1: v[offs[1] + lens[1] // 2, 0] = np.inf
    dq, dk, dv = (dev.up(t) for t in (q, k, v))
    biases = [dev.up(0.1 * rng.standard_normal(w).astype(np.float32)) for w in (K, kvh * hd, kvh * hd)]
    b = [t.ptr if bias else None for t in biases]
    wo, wg, wu = (f16bits(0.05 * rng.standard_normal(s)) for s in ((D, K), (F, D), (F, D)))
    res, nw = rng.standard_normal((rows, D)).astype(np.float32), np.ones(D, np.float32)
    dwo, dwg, dwu, dres, dnw = (dev.up(t) for t in (wo, wg, wu, res, nw))
    h_lens, slots = u32(lens), u32(range(n))
    d_offs, d_lens, angles = dev.up(offs), dev.up(h_lens), dev.zeros(rows * hd // 2 * 8)
    dev.call("m40llm_ext_prefill_angles_async", n, h_lens.ctypes.data, hd, 1e4, 1.0, angles.ptr, 0)
    att, got = dev.zeros(rows * K * 4), []
    for whole in (False, True):
        kv = m40.KVCache(dev.ctx, max(lens) + 1, n, kvh, hd)
        x, hid = dev.zeros(rows * D * 4), dev.zeros(rows * F * 4)
        head = [kv.h, dq.ptr, dk.ptr, dv.ptr, d_offs.ptr, d_lens.ptr, n, slots.ctypes.data, offs.ctypes.data, h_lens.ctypes.data, qh, layout, angles.ptr, *b]
        if whole:
            tail = [dwo.ptr, D, dres.ptr, x.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, F, hid.ptr]
            call = "m40llm_ext_prefill_attention_project_gate_up_async"
            dev.call(call, *head, rows, *tail)
            dev.call(call, *head, rows - 1, *tail, expect=1)
            same = u32([0] * n)
            if n > 1: dev.call(call, *(head[:7] + [same.ctypes.data] + head[8:]), rows, *tail, expect=-8)
        else:
            dev.call("m40llm_ext_prefill_attention_rope_append_async", *head, att.ptr)
            dev.call("m40llm_ext_prefill_project_norm_project_async", att.ptr, rows, K, dwo.ptr, D, dres.ptr, x.ptr, dnw.ptr, 1, 1e-5, 1, 2, dwg.ptr, F, hid.ptr, dwu.ptr, F, None,
                     None, 0, None, 0)
        dev.sync()
        got.append((x.download(np.float32, (rows, D)), hid.download(np.float32, (rows, F)), [kv.read_token(s, lens[s] - 1) for s in range(n)]))
        kv.destroy()
    a = att.download(np.float32, (rows, K)).astype(np.float64)
    fine = np.isfinite(a).all(axis=1)
    assert fine.all() == (n == 1)
    w64 = wo.view(np.float16).astype(np.float64)
    want, bound = a[fine] @ w64.T + res[fine], np.abs(a[fine]) @ np.abs(w64).T * 2.0 ** -20
    for x, _, _ in got:
        # operands exact to 2^-22 each, f32 sums of K products in chains of at most K / 32 steps
        assert np.all(np.abs(x[fine] - want) <= bound + np.abs(want) * 2.0 ** -23)
    rms = [np.sqrt(np.mean(((x[fine] - want) / np.sqrt(np.mean(want ** 2, axis=1, keepdims=True))) ** 2)) for x, _, _ in got]
    assert rms[1] <= 1.05 * rms[0], rms
    assert not np.isfinite(got[1][0][~fine]).any()
    sc = np.abs(got[0][1][fine]).max(axis=1, keepdims=True)
    assert np.all(np.abs(got[1][1][fine] - got[0][1][fine]) <= 1e-5 * sc)
    for s in range(n):
        for i in range(2): assert np.array_equal(got[0][2][s][i], got[1][2][s][i])


@pytest.mark.parametrize("lens", [[1], [5, 3], [31, 1], [32], [33], [20, 14]])
def test_few_rows_of_prompts(dev, lens):
    """Prompts of fewer rows than the many-row products take go through them with rows behind theirs: the same bits whatever an earlier, longer call left in the buffers,
    and the hidden rows of the tokens one by one (whose keys and values pass through f16)."""
    cfg = dict(n_layers=2, d_model=256, q_heads=4, kv_heads=2, head_dim=64, ffn=512, vocab=500, rms_eps=1e-5, rope_base=1e4, rope_scale=1.0, rope_layout=0, qkv_bias=False)
    W = syn.make_weights(cfg, seed=4, std=0.08, emb_std=1.0)
    rng = np.random.default_rng(sum(lens))
    prompts, long = [rng.integers(0, 500, n) for n in lens], [rng.integers(0, 500, 200)]
    got = []
    for before in (False, True):
        dm = syn.DeviceModel(dev.ctx, cfg, W, max_seq_len=256, max_sequences=3)
        dm.set_mode(2)
        if before: dm.forward_prefill([2], long)
        got.append(dm.forward_prefill(range(len(lens)), prompts))
        for s, p in enumerate(prompts):
            for t, tok in enumerate(p): h, l = dm.forward_token(2, t, int(tok))
            for a, b in zip((got[-1][0][s], got[-1][1][s]), (h, l)):
                assert np.abs(a - b).max() <= 2e-3 * np.abs(b).max()
        dm.close()
    assert all(np.array_equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("hd,qh,kvh,D,lens,at", [(64, 4, 1, 256, [300, 65], [77, 1]), (64, 32, 4, 2048, [23, 187, 90, 61, 161], [5, 130, 64, 60, 100]), (128, 16, 2, 256, [130, 700], [129, 33]),
                                                 (128, 5, 5, 320, [97], [40]), (64, 32, 4, 256, [4096], [2100])])
def test_rows_do_not_see_what_comes_behind_them(dev, hd, qh, kvh, D, lens, at):
    """Values a million times larger from a token on: the rows ahead of it have the bits that they have without, and the error against 64 bits that f32 rows have."""
    rng = np.random.default_rng(sum(lens) + hd)
    rows, K, n, F = sum(lens), qh * hd, len(lens), 64
    q, k, v = (rng.standard_normal((rows, w)).astype(np.float32) for w in (K, kvh * hd, kvh * hd))
    v *= 0.01
    offs = u32(np.concatenate([[0], np.cumsum(lens)[:-1]]))
    large, ahead = v.copy(), np.zeros(rows, bool)
    for o, m, t in zip(offs, lens, at):
        large[o + t:o + m] *= np.float32(2.0 ** 20)
        ahead[o:o + t] = True
    dq, dk = dev.up(q), dev.up(k)
    wo, wg, wu = (f16bits(0.05 * rng.standard_normal(s)) for s in ((D, K), (F, D), (F, D)))
    dwo, dwg, dwu, dres, dnw = (dev.up(t) for t in (wo, wg, wu, np.zeros((rows, D), np.float32), np.ones(D, np.float32)))
    h_lens, slots = u32(lens), u32(range(n))
    d_offs, d_lens, angles = dev.up(offs), dev.up(h_lens), dev.zeros(rows * hd // 2 * 8)
    dev.call("m40llm_ext_prefill_angles_async", n, h_lens.ctypes.data, hd, 1e4, 1.0, angles.ptr, 0)
    kv, att, got = m40.KVCache(dev.ctx, max(lens), n, kvh, hd), dev.zeros(rows * K * 4), []
    for values in (v, large):
        dv, x, hid = dev.up(values), dev.zeros(rows * D * 4), dev.zeros(rows * F * 4)
        head = [kv.h, dq.ptr, dk.ptr, dv.ptr, d_offs.ptr, d_lens.ptr, n, slots.ctypes.data, offs.ctypes.data, h_lens.ctypes.data, qh, 0, angles.ptr, None, None, None]
        dev.call("m40llm_ext_prefill_attention_project_gate_up_async", *head, rows, dwo.ptr, D, dres.ptr, x.ptr, dnw.ptr, 1, 1e-5, dwg.ptr, dwu.ptr, F, hid.ptr)
        dev.call("m40llm_ext_prefill_attention_rope_append_async", *head, att.ptr)
        dev.sync()
        got.append(x.download(np.float32, (rows, D)))
    assert np.array_equal(got[0][ahead].view(np.uint32), got[1][ahead].view(np.uint32))
    a, w64 = att.download(np.float32, (rows, K)).astype(np.float64), wo.view(np.float16).astype(np.float64)
    # operands exact to 2^-22 each, f32 sums of K products in chains of at most K / 32 steps
    assert np.all(np.abs(got[1] - a @ w64.T) <= np.abs(a) @ np.abs(w64).T * 2.0 ** -20)
    kv.destroy()
