"""Products of many packed bf16 rows over the tile sizes that row, column and k counts choose, at their edges."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pimosun_common import c_struct, close_to, from_act, ld, m40, pack_tiles, unpack_tiles, up32  # noqa: E402
from test_gpu_layer_kernels import ACT, ADD, KEYS, PROJECT, STORE, STORE_ACT, VALUES, bf16w, call, gemm, rounded  # noqa: E402

Gemm = c_struct("M40llmPackedGemm")


@pytest.fixture(scope="module")
def ctx():
    yield m40.Context(0)


# 64 x 64 tiles alone on their CU (65 .. 500 rows of few columns) and two to a CU, 64 x 128 (odd number of k tiles, or rows between), 128 x 128, 128 x 256
# (whole rounds of them); k of one tile, of fewer stages than buffers, of one stage more than a period; rows and columns that fill no tile
@pytest.mark.parametrize("rows,n,k", [(65, 144, 32), (65, 150, 64), (127, 2048, 384), (200, 500, 352), (300, 1040, 2112), (500, 2048, 256), (700, 2050, 320), (700, 2048, 992),
                                      (1300, 1504, 96), (1300, 2050, 160), (1700, 2310, 2112), (2049, 3000, 352), (4096, 2048, 192), (4000, 2040, 224)])
def test_tiles_store_and_add(ctx, rows, n, k):
    rng = np.random.default_rng(rows + n + k)
    A, W = rng.standard_normal((rows, k)), bf16w(rng, n, k)
    want = rounded(A, "bfloat16") @ W.T.astype(np.float64)
    for ld_out in (n, (n + 3) // 4 * 4 + 4):
        old = rng.standard_normal((rows, ld_out)).astype(np.float32)
        got = gemm(ctx, "bfloat16", STORE, A, W, out_f32=old, ld_out=ld_out, cols=n)["out_f32"]
        close_to(got[:, :n], want, "float32", factor=2)
        assert np.array_equal(got[:, n:], old[:, n:])
        added = gemm(ctx, "bfloat16", ADD, A, W, out_f32=old, ld_out=ld_out, cols=n)["out_f32"]
        assert np.array_equal(added[:, :n], old[:, :n] + got[:, :n])       # one addition, whichever way the results are written
        assert np.array_equal(added[:, n:], old[:, n:])


# few rows: 16, 8 and 4 waves a tile and pairs of tiles (an odd last one); k tiles that no wave count divides, fewer than a wave's batch, more than one
@pytest.mark.parametrize("rows,n,k", [(1, 4096, 544), (3, 4100, 512), (5, 8200, 2080), (16, 16390, 512), (16, 16400, 1408), (17, 4000, 2048), (30, 4112, 608), (32, 8230, 992),
                                      (33, 4097, 3000), (64, 8210, 1100), (2, 2048, 5632), (1, 12304, 768)])
def test_few_rows_waves_and_pairs(ctx, rows, n, k):
    rng = np.random.default_rng(rows + n + k)
    A, W = rng.standard_normal((rows, k)), bf16w(rng, n, k)
    want = rounded(A, "bfloat16") @ W.T.astype(np.float64)
    ld_out = (n + 3) // 4 * 4 + 4
    old = rng.standard_normal((rows, ld_out)).astype(np.float32)
    got = gemm(ctx, "bfloat16", STORE, A, W, out_f32=old, ld_out=ld_out, cols=n)["out_f32"]
    close_to(got[:, :n], want, "float32", factor=2)
    assert np.array_equal(got[:, n:], old[:, n:])


# up to 4, 8 and 16 sums of k tiles (fewer than 16, fewer than 64, more), each kept by one wave, or by 8 or 4 waves that keep two or four of them
@pytest.mark.parametrize("k", [480, 512, 2016, 2048, 2080])
@pytest.mark.parametrize("rows", [1, 16, 20, 64])
def test_waves_and_pairs_change_no_bit(ctx, rows, k):
    rng = np.random.default_rng(rows + k)
    tiles = [4, 400, 600]                              # times up to one tile of rows: up to a CU each, up to two, more
    A, W = rng.standard_normal((rows, k)), bf16w(rng, 16 * tiles[-1], k)
    got = [gemm(ctx, "bfloat16", STORE, A, W[:16 * t], out_f32=np.zeros((rows, 16 * t), np.float32), ld_out=16 * t, cols=16 * t)["out_f32"] for t in tiles]
    assert np.abs(got[0]).max(axis=1).min() > 0
    for g in got[1:]:
        assert np.array_equal(g[:, :64].view(np.uint32), got[0].view(np.uint32))
    assert np.array_equal(got[1].view(np.uint32), got[2][:, :16 * tiles[1]].view(np.uint32))
    last = 16 * tiles[-1] - 64                         # and the wide product's last columns by a narrow one
    tail = gemm(ctx, "bfloat16", STORE, A, W[last:], out_f32=np.zeros((rows, 64), np.float32), ld_out=64, cols=64)["out_f32"]
    assert np.array_equal(got[2][:, last:].view(np.uint32), tail.view(np.uint32))


# up to 16 rows: one tile a workgroup and (more than eight rows of more than four tiles a CU) two, gate and up over 8 and (more than one pair a CU, at most
# two) 4 waves; rows that are not there hold no numbers
@pytest.mark.parametrize("rows,k", [(1, 2048), (8, 2080), (9, 2048), (15, 2368), (16, 3000), (3, 1000), (9, 96)])
def test_forms_of_few_rows_change_no_bit(ctx, rows, k):
    rng, K = np.random.default_rng(rows + k), up32(k)
    A, W = rng.standard_normal((rows, k)), bf16w(rng, 16 * 1100, k)
    full = np.full((16, K), np.nan)
    full[:rows, :k], full[:rows, k:] = A, 0.0
    want, bufs = rounded(A, "bfloat16") @ W.T.astype(np.float64), [ctx.to_device(pack_tiles(b)) for b in (ld.f32_to_bf16(full), ld.f32_to_bf16(W))]

    def product(tiles, kind):
        n = 16 * tiles if kind == STORE else 8 * tiles
        out = ctx.to_device(np.zeros((rows, n), np.float32) if kind == STORE else np.zeros((16, n), np.uint16))
        g = Gemm(act_dtype=ACT["bfloat16"], epilogue=kind, a=bufs[0].ptr, lda=K, w=bufs[1].ptr, n_tiles=tiles, k_tiles=K // 32, rows=rows, batches=1, activation=1)
        if kind == STORE:
            g.out_f32, g.ld_out, g.cols = out.ptr, n, n
        else:
            g.out_act, g.ld_act = out.ptr, n
        call(ctx, "m40llm_ext_packed_gemm_async", C.byref(g), 1)
        return out.download(np.float32, (rows, n)) if kind == STORE else unpack_tiles(out.download(np.uint16, (16 * n,)), rows, n)
    wide = product(1100, STORE)
    close_to(wide, want, "float32", factor=2)
    assert np.array_equal(wide[:, :64].view(np.uint32), product(4, STORE).view(np.uint32))
    act = product(1100, PROJECT)                       # 550 pairs, 300, 4
    gate, up = want.reshape(rows, 550, 2, 16).transpose(2, 0, 1, 3).reshape(2, rows, -1)
    close_to(from_act(act, "bfloat16"), gate / (1.0 + np.exp(-gate)) * up, "bfloat16", factor=2)
    for tiles in (600, 8):
        assert np.array_equal(act[:, :64], product(tiles, PROJECT)[:, :64])


# 64 x 64 tiles (two k tiles a stage), 64 x 128, 128 x 128 (one and two a stage), 128 x 256 (long sums)
@pytest.mark.parametrize("k", [992, 2048, 2112])
def test_tile_shapes_change_no_bit(ctx, k):
    rng, n = np.random.default_rng(k), 2048
    A, W = rng.standard_normal((4096, k)), bf16w(rng, n, k)
    product = lambda first, rows: gemm(ctx, "bfloat16", STORE, A[first:first + rows], W, out_f32=np.zeros((rows, n), np.float32), ld_out=n, cols=n)["out_f32"].view(np.uint32)
    whole = product(0, 4096)
    for first, rows in ((0, 65), (4000, 77), (100, 300), (2048, 700), (1000, 1300), (16, 2500)):
        assert np.array_equal(product(first, rows), whole[first:first + rows]), (first, rows)


@pytest.mark.parametrize("rows,ff,k", [(1, 4112, 512), (20, 4200, 352), (65, 64, 64), (129, 1024, 352), (300, 72, 128), (700, 1024, 96), (1300, 1504, 160), (4096, 1024, 64)])
def test_tiles_gated_pairs(ctx, rows, ff, k):
    """The first 32 columns plain, then pairs of tiles of gate and up."""
    rng = np.random.default_rng(rows + ff)
    tiles = (ff + 15) // 16
    gate, up, plain = (bf16w(rng, m, k, 2.0) for m in (tiles * 16, tiles * 16, 32))
    W = np.concatenate([plain] + [np.concatenate([gate[i * 16:i * 16 + 16], up[i * 16:i * 16 + 16]]) for i in range(tiles)])
    A = rng.standard_normal((rows, k))
    a = rounded(A, "bfloat16")
    want = ld.gelu_tanh(a @ gate.T.astype(np.float64)) * (a @ up.T.astype(np.float64))
    ld_act = up32(tiles * 16)
    out = gemm(ctx, "bfloat16", PROJECT, A, W, out_f32=np.zeros((rows, 32), np.float32), ld_out=32, out_act=np.zeros((rows + 15) // 16 * 16 * ld_act, np.uint16), ld_act=ld_act,
               plain_tiles=2, cols=W.shape[0])
    close_to(out["out_f32"], a @ plain.T.astype(np.float64), "float32", factor=2)
    got = (unpack_tiles(out["out_act"], rows, ld_act).astype(np.uint32) << 16).view(np.float32)[:, :tiles * 16]
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 1e-5 * np.abs(want).max()).all()      # one rounding to 8 bits, and f32 sums


@pytest.mark.parametrize("k", [2048, 2080])
@pytest.mark.parametrize("n", [304, 1280])
def test_expert_jobs_of_short_and_long_sums(ctx, n, k):
    """Jobs of up to 128 rows take 128-column tiles up to 64 k tiles and 256-column ones beyond; an unused expert, ragged rows, a ragged last tile."""
    counts, rng, keep = [130, 0, 17, 128], np.random.default_rng(n + k), []
    W, jobs, slots = [bf16w(rng, n, k) for _ in counts], [], 0
    for e, m in enumerate(counts):
        jobs += [(e, slots + j, min(128, m - j), 0) for j in range(0, m, 128)]
        slots += (m + 15) // 16 * 16
    A = rng.standard_normal((slots, k))
    dev = lambda a: keep.append(ctx.to_device(np.ascontiguousarray(a))) or keep[-1].ptr
    out = ctx.to_device(np.full(slots * n, 0x4b4b, np.uint16))
    g = Gemm(act_dtype=ACT["bfloat16"], epilogue=STORE_ACT, lda=k, a=dev(pack_tiles(ld.f32_to_bf16(A))), w=dev(np.concatenate([pack_tiles(ld.f32_to_bf16(w)).reshape(-1) for w in W])),
             n_tiles=n // 16, k_tiles=k // 32, w_batch=n // 16 * (k // 32) * 512, rows=slots, batches=1, out_act=out.ptr, ld_act=n, cols=n,
             jobs=dev(np.concatenate([[len(jobs), slots, 0, 0], np.array(jobs).reshape(-1)]).astype(np.uint32)), max_jobs=len(jobs) + 2, job_rows=128)
    call(ctx, "m40llm_ext_packed_gemm_async", C.byref(g), 1)
    got = from_act(out.download(np.uint16, (slots, n)), "bfloat16")
    for e, first, m, _ in jobs:
        close_to(got[first:first + m], rounded(A[first:first + m], "bfloat16") @ W[e].T.astype(np.float64), "bfloat16")


# 128 x 256 and 256 x 256 tiles of eight waves: one round of the CUs and a part of a next one, rows and columns that fill no tile, an even and an odd number of k tiles, the fewest that
# they take and one less; every part of the result against a narrower tile's
@pytest.mark.parametrize("rows,n,k", [(4090, 2040, 1536), (500, 12600, 1568), (4090, 3990, 1536), (4000, 4000, 1568), (700, 16400, 1568), (4090, 2040, 1504), (2050, 11010, 2048)])
def test_large_tiles_change_no_bit(ctx, rows, n, k):
    rng = np.random.default_rng(rows + n + k)
    A, W = rng.standard_normal((rows, k)), bf16w(rng, n, k)
    old = rng.standard_normal((rows, n)).astype(np.float32)
    store = lambda first, m: gemm(ctx, "bfloat16", STORE, A[first:first + m], W, out_f32=np.zeros((m, n), np.float32), ld_out=n, cols=n)["out_f32"]
    whole = store(0, rows)
    some = np.array([0, 15, 127, 128, 255, 256, rows - 1])
    close_to(whole[some], rounded(A[some], "bfloat16") @ W.T.astype(np.float64), "float32", factor=2)
    for first in (0, 120, 256, rows // 2, rows - 77):
        assert np.array_equal(store(first, 77).view(np.uint32), whole[first:first + 77].view(np.uint32)), first
    added = gemm(ctx, "bfloat16", ADD, A, W, out_f32=old, ld_out=n, cols=n)["out_f32"]
    assert np.array_equal(added, old + whole)
    act = gemm(ctx, "bfloat16", STORE_ACT, A, W, out_act=np.zeros((rows, up32(n)), np.uint16), ld_act=up32(n), cols=n)["out_act"]
    assert np.array_equal(act[:, :n], ld.f32_to_bf16(whole))


@pytest.mark.parametrize("rows,tiles,k", [(4090, 128, 1536), (700, 1026, 1568), (500, 790, 1536)])
def test_large_tiles_gated_pairs(ctx, rows, tiles, k):
    """Two plain tiles and pairs of gate and up behind it; rows of the result against a launch of few rows."""
    rng = np.random.default_rng(tiles)
    A, W, width = rng.standard_normal((rows, k)), bf16w(rng, tiles * 16, k), up32((tiles - 2) * 8)
    def project(first, m):
        out = gemm(ctx, "bfloat16", PROJECT, A[first:first + m], W, out_f32=np.zeros((m, 32), np.float32), ld_out=32, plain_tiles=2, cols=W.shape[0],
                   out_act=np.zeros((m + 15) // 16 * 16 * width, np.uint16), ld_act=width)
        return out["out_f32"].view(np.uint32), unpack_tiles(out["out_act"], m, width)[:, :(tiles - 2) * 8]
    whole = project(0, rows)
    for first, m in ((0, 65), (112, 70), (240, 77), (rows - 70, 70)):
        for a, b in zip(project(first, m), whole):
            assert np.array_equal(a, b[first:first + m]), first


@pytest.mark.parametrize("kind", [KEYS, VALUES])
@pytest.mark.parametrize("tiles", [128, 256])
def test_large_tiles_over_pages(ctx, kind, tiles):
    """Scattered pages of 50 k tiles, of which the product takes 48; the results of a page are one piece."""
    rng, pages = np.random.default_rng(tiles), 63
    cache, W = rng.standard_normal((pages + 2, 64, 1600)), bf16w(rng, tiles * 16, 1536)
    order = rng.permutation(pages + 2)[:pages].astype(np.uint32)
    dc, dw = ctx.to_device(np.concatenate([pack_tiles(ld.f32_to_bf16(p)).reshape(-1) for p in cache])), ctx.to_device(pack_tiles(ld.f32_to_bf16(W)))
    def product(first, n):
        out, dl = ctx.to_device(np.zeros((n, 64 * tiles * 16), np.uint16)), ctx.to_device(order[first:first + n])
        g = Gemm(act_dtype=ACT["bfloat16"], epilogue=kind, a=dc.ptr, w=dw.ptr, n_tiles=tiles, k_tiles=48, rows=64 * n, batches=1, out_act=out.ptr, pages=dl.ptr, page_k_tiles=50)
        call(ctx, "m40llm_ext_packed_gemm_async", C.byref(g), 1)
        return out.download(np.uint16, (n, 64 * tiles * 16))
    whole = product(0, pages)
    for first, n in ((0, 1), (3, 3), (30, 5), (61, 2)):
        assert np.array_equal(product(first, n), whole[first:first + n])
    want = rounded(cache[order[5]][:, :1536], "bfloat16") @ W.T.astype(np.float64)
    close_to(np.sort(from_act(whole[5], "bfloat16")), np.sort(want.reshape(-1)), "bfloat16", factor=2)
