"""The norm before a routed feed-forward with the router's product and the choice of experts in its launch, and the experts' first product with the list of rows by expert in its,
beside the launches one by one: the same bits everywhere."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pimosun_common import c_struct, close_to, from_act, ld, m40, pack_tiles, unpack_tiles, up32  # noqa: E402
from test_gpu_layer_kernels import PROJECT, bf16w, call, rounded  # noqa: E402

NormAdd, Update, Route, Gemm = (c_struct("M40llm" + n) for n in ("NormAdd", "StreamUpdate", "Route", "PackedGemm"))


@pytest.fixture(scope="module")
def ctx():
    yield m40.Context(0)


def run(ctx, fused, rows, width, streams, experts, identity, top, groups, sigmoid, weighted, source, odd=False, times=3):
    rng, keep = np.random.default_rng(rows * width + experts), []
    f32 = lambda *s: rng.standard_normal(s).astype(np.float32)          # noqa: E731

    def put(a):
        keep.append(ctx.to_device(np.ascontiguousarray(a)))
        return keep[-1]
    all_, ldh, tiles = experts + identity, up32(width), (experts + identity + 15) // 16
    W = np.zeros((tiles * 16, ldh), np.float32)
    W[:all_, :width] = 3 * f32(all_, width) / np.sqrt(width)
    router = put(pack_tiles(ld.f32_to_bf16(W)))
    correction = put(0.1 * f32(all_))
    planes = f32(3, rows, width)
    if odd:
        planes[0, 0, 5] = np.nan
        planes[1, -1, 7] = np.inf
    sub = dict(act_dtype=0, rows=rows, width=width, eps=1e-5, mult=0.7, ld_h=ldh, w=put(1 + 0.2 * f32(width)).ptr)
    if source == "planes":
        sub.update(planes=put(planes).ptr, n_planes=3, plane_stride=rows * width)
    else:
        place = rng.permutation(rows * 3).astype(np.uint32).reshape(rows, 3)
        if not streams:
            place[0, 1] = 0xffffffff
        sub.update(expert_out=put(ld.f32_to_bf16(f32(rows * 3, width))).ptr, ld_expert=width, place=put(place).ptr, weight=put(np.abs(f32(rows, 3))).ptr, top=3)
    if streams:
        x, stride = put(f32(streams, rows, width)), rows * width
        sub.update(streams=streams, streams_x=x.ptr, stream_stride=stride, mix=put(f32(streams, streams)).ptr, share=put(f32(streams)).ptr, take=put(f32(streams)).ptr)
    else:
        x = put(f32(rows, width))
        sub.update(x=x.ptr)
    slots = ctx.lib.m40llm_ext_expert_slots(rows, experts, top)
    jobs_n = 4 + 4 * ctx.lib.m40llm_ext_expert_max_jobs(rows, experts, top, 16)
    gate_up = put(ld.f32_to_bf16(f32(experts * 96 * ldh) / np.sqrt(width)))      # any numbers in the order of the tiles: six column tiles an expert
    out = dict(act=put(np.zeros((slots, 64), np.uint16)), h=put(np.zeros(16 * ldh, np.uint16)), h_rows=put(np.zeros((rows, ldh), np.uint16)), ids=put(np.full(rows * top, 77, np.uint32)), weight=put(f32(rows * top)),
               place=put(np.zeros(rows * top, np.uint32)), jobs=put(np.zeros(jobs_n, np.uint32)), x=x)
    rows_of, slot_weight = put(np.full(slots, 99, np.uint32)), put(np.zeros(slots, np.float32))
    logits = put(np.zeros((rows, tiles * 16), np.float32))
    q = Route(rows=rows, experts=experts, identity=identity, top=top, job_rows=16, groups=groups, keep=max(1, groups // 2), score=int(sigmoid), scale=1.5, logits=logits.ptr, ld_logits=tiles * 16,
              correction=correction.ptr, ids=out["ids"].ptr, weight=out["weight"].ptr, rows_of=rows_of.ptr, place=out["place"].ptr, jobs=out["jobs"].ptr,
              slot_weight=slot_weight.ptr if weighted else None)
    sub.update(h=out["h"].ptr, h_rows=out["h_rows"].ptr)
    name, struct = ("m40llm_ext_stream_update_async", Update) if streams else ("m40llm_ext_norm_add_rows_async", NormAdd)
    got = []
    for _ in range(times):       # the rows and streams go on from time to time, over the list of the time before
        if fused:
            call(ctx, name, C.byref(struct(**sub, route=C.addressof(q), router=router.ptr, router_tiles=tiles)), 1)
        else:
            call(ctx, name, C.byref(struct(**sub)), 1)
            g = Gemm(act_dtype=0, epilogue=0, a=out["h"].ptr, lda=ldh, w=router.ptr, n_tiles=tiles, k_tiles=ldh // 32, rows=rows, batches=1, out_f32=logits.ptr, ld_out=tiles * 16, cols=tiles * 16)
            call(ctx, "m40llm_ext_packed_gemm_async", C.byref(g), 1)
            call(ctx, "m40llm_ext_route_rows_async", C.byref(q), 1)
        g = Gemm(act_dtype=0, epilogue=PROJECT, a=out["h_rows"].ptr, lda=ldh, w=gate_up.ptr, n_tiles=6, k_tiles=ldh // 32, rows=rows, batches=1, w_batch=96 * ldh, out_act=out["act"].ptr, ld_act=64, activation=1)
        if fused:
            g.route = C.addressof(q)
        else:
            g.jobs, g.gather, g.max_jobs, g.job_rows, g.row_scale = out["jobs"].ptr, rows_of.ptr, (jobs_n - 4) // 4, 16, slot_weight.ptr if weighted else None
        call(ctx, "m40llm_ext_packed_gemm_async", C.byref(g), 1)
        ctx.sync(1)
        got.append({n: b.download(np.uint8, (b.nbytes,)) for n, b in out.items()})
    return got


@pytest.mark.parametrize("rows,width,streams,experts,identity,top,groups,sigmoid,weighted,source", [
    (1, 2048, 0, 32, 2, 4, 0, False, False, "planes"), (8, 2048, 0, 32, 2, 4, 0, False, False, "experts"), (10, 4096, 0, 62, 2, 6, 0, True, True, "planes"),
    (1, 2048, 1, 32, 0, 4, 0, True, True, "planes"), (5, 2072, 1, 20, 0, 2, 0, False, True, "experts"), (1, 2048, 1, 48, 0, 48, 0, True, False, "planes"),
    (1, 2048, 4, 32, 0, 4, 8, False, False, "planes"), (3, 4064, 4, 64, 0, 4, 8, False, False, "experts"), (16, 2048, 4, 8, 0, 1, 0, True, True, "planes"), (16, 2048, 0, 33, 31, 4, 0, False, False, "planes"),
    (2, 2080, 0, 1, 0, 1, 0, False, False, "planes")])
@pytest.mark.parametrize("odd", [False, True])
def test_norm_with_the_router_behind_it(ctx, odd, rows, width, streams, experts, identity, top, groups, sigmoid, weighted, source):
    want, got = (run(ctx, fused, rows, width, streams, experts, identity, top, groups, sigmoid, weighted, source, odd) for fused in (False, True))
    for i, (a, b) in enumerate(zip(want, got)):
        for n in a:
            assert np.array_equal(a[n], b[n]), (i, n)


def test_what_the_launch_has_no_form_for_is_refused(ctx):
    x = ctx.to_device(np.zeros(4096 * 32, np.float32))
    p = x.ptr

    def rc(rows=2, width=2048, streams=0, tiles=2, experts=32, job_rows=16, top=4, router=p, dtype=0, ids=p, ld=None):
        q = Route(rows=rows, experts=experts, top=top, job_rows=job_rows, ids=ids, weight=p, rows_of=p, place=p, jobs=p)
        both = dict(act_dtype=dtype, rows=rows, width=width, ld_h=ld or up32(width), planes=p, n_planes=1, plane_stride=width, w=p, h=p, route=C.addressof(q), router=router, router_tiles=tiles)
        if streams:
            return ctx.lib.m40llm_ext_stream_update_async(ctx.h, C.byref(Update(streams=streams, streams_x=p, stream_stride=width, mix=p, share=p, take=p, **both)), 1)
        return ctx.lib.m40llm_ext_norm_add_rows_async(ctx.h, C.byref(NormAdd(x=p, **both)), 1)
    for streams in (0, 1):
        assert rc(streams=streams, ids=None) == -1
        for bad in (dict(rows=17), dict(width=2016), dict(width=4128), dict(width=2044), dict(tiles=0), dict(tiles=5), dict(tiles=1), dict(router=None), dict(router=p + 4), dict(dtype=1),
                    dict(top=33)):
            assert rc(streams=streams, **bad) == -3, bad
    assert rc(streams=2) == rc(streams=16) == -3
    route = dict(experts=32, job_rows=16, top=4, ids=p, weight=p, rows_of=p, place=p, jobs=p)
    gemm = dict(act_dtype=0, epilogue=PROJECT, a=p, lda=2048, w=p, n_tiles=2, k_tiles=64, batches=1, out_act=p, ld_act=32)

    def product(more={}, **kw):
        q = Route(**dict(dict(route, rows=2), **kw))
        return ctx.lib.m40llm_ext_packed_gemm_async(ctx.h, C.byref(Gemm(**dict(gemm, rows=2, route=C.addressof(q), **more))), 1)
    assert product(dict(jobs=p)) == product(dict(gather=p)) == product(dict(row_scale=p)) == product(dict(plain_tiles=2, out_f32=p)) == -3
    assert [product(**dict(dict(route, rows=2), **bad)) for bad in (dict(rows=17), dict(job_rows=32), dict(top=33), dict(experts=65), dict(rows=16, top=5), dict(rows=0))] == [-3] * 6
    assert product(**dict(route, ids=None)) == -1
    for rows, of_route in ((1, 2), (2, 3), (15, 16)):          # fewer rows than the route has choices of: none past the end of a is read
        q = Route(**dict(route, rows=of_route))
        assert ctx.lib.m40llm_ext_packed_gemm_async(ctx.h, C.byref(Gemm(**dict(gemm, rows=rows, route=C.addressof(q)))), 1) == -3


@pytest.mark.parametrize("rows,top,expert", [(16, 4, 5), (5, 4, 0), (16, 4, None)])
def test_repeated_ids_stay_in_their_experts_slots(ctx, rows, top, expert):
    """Ids that a caller wrote: one expert for all pairs (64 and 20), or the same two in every row; the list names slots of the expert's own job alone, and the first 16 pairs'
    products are those of the rows."""
    rng, ldh, experts = np.random.default_rng(rows), 2048, 8
    ids = np.full((rows, top), expert) if expert is not None else np.tile([3, 6, 3, 6], (rows, 1))
    A, W = rng.standard_normal((rows, ldh)), bf16w(rng, experts * 32, ldh)           # 16 rows of gate, 16 of up an expert
    x, w = ld.f32_to_bf16(A.astype(np.float32)), pack_tiles(ld.f32_to_bf16(W))
    slots, n_jobs = ctx.lib.m40llm_ext_expert_slots(rows, experts, top), ctx.lib.m40llm_ext_expert_max_jobs(rows, experts, top, 16)
    bufs = [ctx.to_device(a) for a in (ids.astype(np.uint32), np.ones((rows, top), np.float32), np.full(rows * top, 9999, np.uint32), np.zeros(4 + 4 * n_jobs, np.uint32), x, w)]
    dids, weight, place, jobs, dx, dw = bufs
    act = ctx.to_device(np.full((slots, 32), 0x4242, np.uint16))
    q = Route(rows=rows, experts=experts, top=top, job_rows=16, ids=dids.ptr, weight=weight.ptr, rows_of=place.ptr, place=place.ptr, jobs=jobs.ptr)
    g = Gemm(act_dtype=0, epilogue=PROJECT, a=dx.ptr, lda=ldh, w=dw.ptr, n_tiles=2, k_tiles=ldh // 32, rows=rows, batches=1, w_batch=32 * ldh, out_act=act.ptr, ld_act=32, activation=1)
    g.route = C.addressof(q)
    call(ctx, "m40llm_ext_packed_gemm_async", C.byref(g), 1)
    ctx.sync(1)
    used = sorted(set(ids.ravel().tolist()))
    want = np.zeros(rows * top, np.uint32)
    for job, e in enumerate(used):
        mine = np.flatnonzero(ids.ravel() == e)
        want[mine] = 16 * job + np.minimum(np.arange(len(mine)), 15)
    assert np.array_equal(place.download(np.uint32, (rows * top,)), want)
    j = jobs.download(np.uint32, (4 + 4 * n_jobs,))
    assert j[0] == len(used) and j[4:4 + 4 * len(used)].reshape(-1, 4).tolist() == [[e, 16 * i, 16, 0] for i, e in enumerate(used)]
    got = act.download(np.uint16, (slots * 32,))
    assert np.all(got[512 * len(used):] == 0x4242)
    y = (rounded(A, "bfloat16") @ W.T.astype(np.float64)).reshape(rows, experts, 2, 16)
    gate, up = y[:, :, 0], y[:, :, 1]
    y, first = gate / (1.0 + np.exp(-gate)) * up, [np.flatnonzero(want == s)[0] for s in range(16 * len(used))]
    close_to(from_act(unpack_tiles(got, 16 * len(used), 32)[:, :16], "bfloat16"), np.stack([y[p // top, ids.ravel()[p]] for p in first]), "bfloat16", factor=2)
