"""Batched greedy runs on either side of the length from which their steps are recorded as a graph, and across a change of the attention's size: the picks and gaps
of the run whose steps go out one by one (mode 1)."""
import importlib

import numpy as np
import pytest

from gpu_common import m40

pytestmark = pytest.mark.gpu
syn = importlib.import_module("m40-llm_amd.synthetic")


@pytest.mark.parametrize("rows,steps,longest", [(2, 48, 20), (2, 49, 20), (9, 70, 20), (3, 60, 500)])
def test_recorded_steps(rows, steps, longest):
    ctx = m40.Context(0)
    cfg = dict(n_layers=2, d_model=256, q_heads=4, kv_heads=2, head_dim=64, ffn=512, vocab=500, rms_eps=1e-5, rope_base=10000.0, rope_scale=1.0, rope_layout=0,
               qkv_bias=False)
    dm = syn.DeviceModel(ctx, cfg, syn.make_weights(cfg, seed=3, std=0.08, emb_std=1.0), max_seq_len=longest + steps + 2, max_sequences=rows)
    rng = np.random.default_rng(rows)
    lens = np.full(rows, longest, dtype=np.uint32)
    k16, v16 = (ctx.to_device(rng.standard_normal((longest, 2, 64)).astype(np.float16).view(np.uint16)) for _ in range(2))
    for r in range(rows):
        for l in range(2):
            m40.check(ctx.lib.m40llm_ext_kvcache_bulk_fill_f16(ctx.h, dm.kv_handle(), dm.H.m40host_model_kv_slot(dm.h, r, l), k16.ptr, v16.ptr, longest))
    got = {}
    for mode in (1, 2, 2):
        dm.set_mode(mode)
        ids, gaps = dm.decode_batch_greedy(np.arange(rows), lens, np.arange(rows, dtype=np.uint32), steps)
        if mode in got:
            assert np.array_equal(ids, got[mode][0]) and np.array_equal(gaps, got[mode][1])
        got[mode] = ids.copy(), gaps.copy()
    assert np.array_equal(got[1][0], got[2][0]) and np.array_equal(got[1][1], got[2][1])
    dm.close()
    ctx.close()
