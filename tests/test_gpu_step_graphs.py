"""Steps of single tokens that a layered decoder replays from a graph: every step's logits are the bits of the launches one by one, with prompts, other
forms of step, released sequences and replaced buffers in between."""
import ctypes as C
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from gpu_common import m40  # noqa: E402

layered = importlib.import_module("m40-llm_amd.layered")
bench = importlib.import_module("m40-llm_amd.layered_bench")


def config(design):
    s = dict(bench.SHAPES["2k"], layers=4)
    cfg = bench.pimosun_config(s) if design == "pimosun" else getattr(bench, design + "_config")("2k")
    cfg["layers"] = cfg["layers"][:4]
    return dict(cfg, vocab=1000)


@pytest.fixture(scope="module")
def ctx():
    yield m40.Context(0)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("design", ["pimosun", "gulidra", "natatar", "fomunex"])
def test_replayed_steps_equal_launched_steps(ctx, design, dtype):
    models = [layered.LayeredModel.random(ctx, config(design), seed=3, std=0.05, dtype=dtype, max_tokens=2048, max_sequences=4, max_rows=256) for _ in range(2)]
    models[1].set_mode(0)
    rng = np.random.default_rng(1)

    def step(entries):
        entries = [(s, rng.integers(0, 1000, n), want) for s, n, want in entries]
        a, b = (m.step(entries) for m in models)
        assert a.shape == b.shape and np.array_equal(a.view(np.uint32), b.view(np.uint32)), (design, entries)
        assert np.isfinite(a).all()

    def singles(n, seqs, want=lambda s: [0]):
        for _ in range(n):
            step([(s, 1, want(s)) for s in seqs])

    def counts(since=(0, 0, 0)):
        assert models[1].step_counts() == (0, 0, 0)
        return tuple(a - b for a, b in zip(models[0].step_counts(), since))
    step([(0, 5, [4]), (1, 58, [0, 57]), (2, 130, [129])])
    singles(12, (0, 1, 2))                                   # one sequence grows past its first page
    replayed, recorded, _ = counts()
    assert replayed >= 3 and 1 <= recorded <= 3              # four steps at least before and behind what the launches are split for anew
    singles(6, (2, 0), lambda s: [0] if s else [])           # another form, one place wanted
    before = counts()
    step([(3, 700, [699]), (0, 1, [0])])                     # a prompt beside a token, whose tables are larger than any before
    assert counts(before)[0] == 0 and models[0].step_counts()[1] == models[0].step_counts()[2]      # every graph went
    singles(5, (0, 1, 2))
    singles(5, (3, 1, 0, 2))
    for m in models:
        m.release(1)
    singles(4, (0, 2, 3), lambda s: [])                      # no logits at all
    step([(1, 1, [0])])
    singles(5, (1, 0, 2))
    before = counts()
    models[0].set_mode(2)
    assert counts(before)[2] >= 1
    singles(5, (1, 0, 2))
    assert counts(before)[:2] == (2, 1)
    for n in range(10):                                      # more forms than are kept, and back to the first
        singles(4, [(0, 1, 2, 3)[i] for i in range(4) if n + 1 >> i & 1])
    singles(4, (1, 0, 2))
    ids = [m.decode_batch_timed([0, 2], [m.length(0), m.length(2)], [5, 6], 2, 4)[0] for m in models]
    assert np.array_equal(*ids)
    singles(5, (0, 2))


@pytest.mark.parametrize("design", ["pimosun", "gulidra", "natatar", "fomunex"])
def test_more_logits_than_one_head_takes(ctx, design):
    """Single tokens whose places are wanted 300 times (the head takes 256 rows at once), with a prompt of another row count in between."""
    models = [layered.LayeredModel.random(ctx, config(design), seed=3, std=0.05, max_tokens=2048, max_sequences=4, max_rows=256) for _ in range(2)]
    models[1].set_mode(0)
    rng = np.random.default_rng(2)

    def step(entries):
        entries = [(s, rng.integers(0, 1000, n), want) for s, n, want in entries]
        a, b = (m.step(entries) for m in models)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (design, entries)
    step([(1, 70, [69])])
    for _ in range(5):
        step([(0, 1, [0] * 300)])
    step([(2, 70, [69])])
    for _ in range(2):
        step([(0, 1, [0] * 300), (1, 1, [0])])
        step([(0, 1, [0] * 300)])


def test_a_recording_leaves_the_contexts_stream_alone(ctx):
    """Between a recorder's begin and end the context's stream runs what it is given; the graph holds what the recorder was given, replay after replay."""
    lib = ctx.lib
    rec = C.c_void_p(lib.m40llm_ext_create_recorder(ctx.h))
    assert rec.value and not lib.m40llm_ext_create_recorder(rec) and not lib.m40llm_ext_create_recorder(None)
    src, mine, theirs = ctx.to_device(np.arange(64, dtype=np.uint32)), ctx.to_device(np.zeros(64, np.uint32)), ctx.to_device(np.zeros(64, np.uint32))
    for _ in range(2):                                       # a recorder records more than once
        m40.check(lib.m40llm_cuda_graph_begin_capture(rec, 1), "begin")
        m40.check(lib.m40llm_ext_copy_words_async(rec, mine.ptr, src.ptr, 64, 1), "recorded")
        m40.check(lib.m40llm_ext_copy_words_async(ctx.h, theirs.ptr, src.ptr, 64, 1), "launched")
        ctx.sync(1)
        graph = C.c_void_p()
        m40.check(lib.m40llm_cuda_graph_end_capture(rec, 1, C.byref(graph)), "end")
        assert np.array_equal(theirs.download(np.uint32, (64,)), np.arange(64)) and not mine.download(np.uint32, (64,)).any()
        for _ in range(3):
            m40.check(lib.m40llm_ext_clear_u32_async(ctx.h, mine.ptr, 64, 1), "clear")
            m40.check(lib.m40llm_ext_clear_u32_async(ctx.h, theirs.ptr, 64, 1), "clear")
            m40.check(lib.m40llm_cuda_graph_launch(ctx.h, graph, 1), "replay")
            ctx.sync(1)
            assert np.array_equal(mine.download(np.uint32, (64,)), np.arange(64)) and not theirs.download(np.uint32, (64,)).any()
        m40.check(lib.m40llm_ext_clear_u32_async(ctx.h, mine.ptr, 64, 1), "clear")
        ctx.sync(1)
        lib.m40llm_cuda_graph_destroy(graph)
    lib.m40llm_destroy_context(rec)
    m40.check(lib.m40llm_ext_copy_words_async(ctx.h, theirs.ptr, src.ptr, 64, 1), "after the recorder is gone")
    ctx.sync(1)


NARROW = bench.pimosun_config(dict(bench.SHAPES["2k"], width=256, heads=2, kv_rank=64, q_rank=64, ff=704, layers=2))


@pytest.mark.parametrize("cfg,vocab", [(config("gulidra"), 1000), (config("pimosun"), 1001), (config("pimosun"), 40_000), (NARROW, 30_000), (NARROW, 40_000), (NARROW, 1001)],
                         ids=["gulidra", "pimosun", "pimosun wide vocabulary", "narrow", "narrow wide vocabulary", "narrow few words"])
def test_rows_of_logits_that_the_head_stores_itself_and_one_more(ctx, cfg, vocab):
    """Up to four rows of logits (of narrow models up to 128 k words) are written to the host's memory by the head, more go there by a copy: the same bits, launched and replayed."""
    models = [layered.LayeredModel.random(ctx, dict(cfg, vocab=vocab), seed=3, std=0.05, max_tokens=2048, max_sequences=5, max_rows=256) for _ in range(4)]
    models[3].set_mode(0)
    rng = np.random.default_rng(4)
    for n in [7] + 9 * [1]:
        tokens = rng.integers(0, vocab, (5, n))
        five, four, three, launched = (m.step([(s, tokens[s], [n - 1] if s < k else []) for s in range(5)]) for m, k in zip(models, (5, 4, 3, 5)))
        assert five.shape == (5, vocab) and np.isfinite(five).all()
        for other in (four, three, launched):
            assert np.array_equal(five[:len(other)].view(np.uint32), other.view(np.uint32)), (n, len(other))
    assert all(m.step_counts()[0] >= 4 for m in models[:3])
