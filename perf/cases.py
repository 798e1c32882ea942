"""The work by which this framework's speed is judged: calls that a user's program makes through the public entry points, over the
sizes that the framework is used with.

Every kind of case stands for one use:

  attention     last-token attention of one sequence over its f16 cache (m40llm_attention_last_token_f32_gqa_async), the smallest call
                that a decode loop built on the C interface makes; 16 to 32768 tokens of context
  block_select  attention over compressed long-context caches of one to eight sequences, one call for all of them
  ffn_q80       one q8_0 feed-forward (gate, up, SwiGLU, down) of a decode step, one to sixteen rows
  decode        greedy generation by a dense f16 model from filled caches: one sequence, a server's batch, a batch of 32; afterwards the
                logits behind the last token of the first sequence, as a program that goes on sampling by itself takes them
  prefill       the prompts of a dense f16 model as one packed batch, then the first token behind the first prompt (which reads the cache
                that the prompts left)
  layered       a model opened from its folder serves prompts and then single tokens through the step call, all logits of the
                generated places returned; sequences given back at the end.  One design each with what is typical for serving: a long
                prompt, a batch that generates, ragged prompts, one conversation

Weights are random with the shapes of the repository's own configurations (two dense models of synthetic.py; the four designs at width
2048 of layered_bench.py, the first four layers).  Dense models hold f16 weights N(0, 0.02); caches hold N(0, 1).
"""
import importlib
import json
import math
import os
import random
import tempfile
import zlib

import numpy as np
import torch

m40 = importlib.import_module("m40-llm_amd")
syn = importlib.import_module("m40-llm_amd.synthetic")
layered = importlib.import_module("m40-llm_amd.layered")
layered_bench = importlib.import_module("m40-llm_amd.layered_bench")

DENSE = dict(tinyllama=syn.TINYLLAMA_1B, qwen=syn.QWEN25_3B)
DESIGNS = ("pimosun", "gulidra", "natatar", "fomunex")
HEADS = ((32, 4, 64), (16, 2, 128), (32, 8, 128))          # query heads, kv heads, head size of the attention benchmarks
FFN = ((4096, 14336), (2048, 5632), (2048, 11008))
SELECT = dict(q_heads=32, kv_heads=8, head_dim=128, window=512, block=64, top=64)


# ---- the cases ----------------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # the reference configuration of single-token attention: latency of one small launch
        dict(name="attention 512", kind="attention", q_heads=32, kv_heads=4, head_dim=64, context=512),
        # a long-context decode step of four sequences over compressed caches, V in groups of 32
        dict(name="block select 4x32k", kind="block_select", sequences=4, context=32768, backing=3),
        # a small batch through a q8_0 feed-forward of an 8B-sized model
        dict(name="ffn q8_0 4 rows", kind="ffn_q80", rows=4, d_model=4096, ffn=14336),
        # one user: 32 tokens behind a context of a few hundred
        dict(name="decode tinyllama 1", kind="decode", model="tinyllama", rows=1, shortest=301, longest=301, steps=32),
        # a server's batch of eight with ragged contexts
        dict(name="decode qwen 8", kind="decode", model="qwen", rows=8, shortest=256, longest=4093, steps=16),
        # a throughput batch of 32
        dict(name="decode tinyllama 32", kind="decode", model="tinyllama", rows=32, shortest=128, longest=1021, steps=4),
        # a long prompt
        dict(name="prefill tinyllama 4096", kind="prefill", model="tinyllama", prompts=1, shortest=4096, longest=4096),
        # several short prompts that arrive together
        dict(name="prefill tinyllama 5 short", kind="prefill", model="tinyllama", prompts=5, shortest=23, longest=187),
        dict(name="pimosun prompt 4096", kind="layered", design="pimosun", sequences=1, shortest=4096, longest=4096, steps=0),
        dict(name="gulidra 8 generate", kind="layered", design="gulidra", sequences=8, shortest=61, longest=327, steps=16),
        dict(name="natatar 3 prompts", kind="layered", design="natatar", sequences=3, shortest=301, longest=1501, steps=2),
        dict(name="fomunex 1 chat", kind="layered", design="fomunex", sequences=1, shortest=77, longest=77, steps=24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    case = known[0]
    while case in known:
        case = _drawn(rng)
    return case


def _drawn(rng):
    kind = rng.choice(("attention", "block_select", "ffn_q80", "decode", "decode", "prefill", "prefill", "layered", "layered", "layered"))
    if kind == "attention":
        q, kv, hd = rng.choice(HEADS)
        return dict(kind=kind, q_heads=q, kv_heads=kv, head_dim=hd, context=_log_int(rng, 16, 32768))
    if kind == "block_select":
        return dict(kind=kind, sequences=rng.randint(1, 4), context=_log_int(rng, 1500, 32768), backing=rng.choice((2, 3)))
    if kind == "ffn_q80":
        d, f = rng.choice(FFN)
        return dict(kind=kind, rows=_log_int(rng, 1, 16), d_model=d, ffn=f)
    if kind == "decode":
        model = rng.choice(("tinyllama", "tinyllama", "qwen"))
        rows = _log_int(rng, 1, 32 if model == "tinyllama" else 8)
        longest = _log_int(rng, 32, 1000 if rows > 16 else 2000)
        shortest = longest if rows == 1 else rng.randint(longest // 4, longest)
        return dict(kind=kind, model=model, rows=rows, shortest=shortest, longest=longest, steps=4 if rows > 16 else rng.randint(8, 15))
    if kind == "prefill":
        model = rng.choice(("tinyllama", "tinyllama", "qwen"))
        prompts = _log_int(rng, 1, 8)
        longest = _log_int(rng, 16, 4000 // prompts if model == "tinyllama" else 1300 // prompts)
        return dict(kind=kind, model=model, prompts=prompts, shortest=longest if prompts == 1 else rng.randint(max(1, longest // 8), longest), longest=longest)
    sequences = _log_int(rng, 1, 8)
    longest = _log_int(rng, 17, 2400 // sequences)
    return dict(kind=kind, design=rng.choice(DESIGNS), sequences=sequences, shortest=longest if sequences == 1 else rng.randint(max(1, longest // 4), longest),
                longest=longest, steps=rng.choice((0, 2, 8, 16)))


def _lengths(case, n):
    """n lengths between shortest and longest, fixed by the case."""
    if n == 1:
        return [case["longest"]]
    r = random.Random(zlib.crc32(json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True).encode()))
    a, b = case["shortest"], case["longest"]
    return [a, b] + [r.randint(a, b) for _ in range(n - 2)]


# ---- inputs --------------------------------------------------------------------------------------------------------------------------
_ctx = None


def _context():
    """The program's one device context."""
    global _ctx
    if _ctx is None:
        _ctx = m40.Context(0)
    return _ctx


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, dtype=torch.float16, std=1.0, mean=0.0):
    return torch.empty(shape, device="cuda", dtype=dtype).normal_(mean, std, generator=g)


def _ids(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, size=n).astype(np.uint32)


def _dense_weights(cfg, g):
    D, F, KV = cfg["d_model"], cfg["ffn"], cfg["kv_heads"] * cfg["head_dim"]
    layers = []
    for _ in range(cfg["n_layers"]):
        w = {n: _normal(g, r, k, std=0.02) for n, r, k in (("wq", D, D), ("wk", KV, D), ("wv", KV, D), ("wo", D, D), ("wgate", F, D), ("wup", F, D), ("wdown", D, F))}
        for n, r in (("bq", D), ("bk", KV), ("bv", KV)) if cfg["qkv_bias"] else ():
            w[n] = _normal(g, r, dtype=torch.float32, std=0.02)
        w["attn_norm"], w["ffn_norm"] = (_normal(g, D, dtype=torch.float32, std=0.1, mean=1.0) for _ in range(2))
        layers.append(w)
    return dict(layers=layers, out_norm=_normal(g, D, dtype=torch.float32, std=0.1, mean=1.0), lm_head=_normal(g, cfg["vocab"], D, std=0.02),
                tok_emb=_normal(g, cfg["vocab"], D, std=0.02))


class _Dense(syn.DeviceModel):
    """A dense model over weights that are on the device already."""

    def __init__(self, ctx, cfg, weights, max_seq_len, max_sequences):
        self.ctx, self.cfg, self.weights, self.bufs, self.H = ctx, cfg, weights, [], m40.host()
        self.layers = (syn.HostLayerWeights * cfg["n_layers"])()
        for l, w in zip(self.layers, weights["layers"]):
            for name, t in w.items():
                setattr(l, name, t.data_ptr())
        hc = syn.HostModelConfig(*(cfg[k] for k in ("n_layers", "d_model", "q_heads", "kv_heads", "head_dim", "ffn", "vocab", "rms_eps", "rope_base", "rope_scale",
                                                    "rope_layout")), 1 if cfg["qkv_bias"] else 0, 1, max_seq_len, max_sequences)
        torch.cuda.synchronize()
        self.h = self.H.m40host_model_create(ctx.h, syn.C.byref(hc), self.layers, *(weights[k].data_ptr() for k in ("out_norm", "lm_head", "tok_emb")), None)
        if not self.h:
            raise RuntimeError(self.H.m40host_last_error().decode())
        self.set_mode(2)


def _caches(case, cfg, g):
    """Keys and values of every sequence, f16 [rows][longest][kv heads][head size]; all layers hold the same."""
    return [_normal(g, case["rows"], case["longest"], cfg["kv_heads"], cfg["head_dim"]) for _ in range(2)]


def _design_config(design):
    s = dict(layered_bench.SHAPES["2k"], layers=4)
    if design == "pimosun":
        return layered_bench.pimosun_config(s)
    cfg = getattr(layered_bench, design + "_config")("2k")
    cfg["layers"] = cfg["layers"][:4]
    return cfg


def _design_weights(design, cfg, g):
    """bf16 tensors of a model folder, by name."""
    T, D = {}, cfg["width"]

    def mat(name, n, k, gain=1.0):
        T[name] = _normal(g, n, k, dtype=torch.bfloat16, std=gain / math.sqrt(k))

    def vec(name, n, mean=1.0, std=0.2):
        T[name] = _normal(g, n, dtype=torch.bfloat16, std=std, mean=mean)

    def spread(name, n, lo, hi):
        T[name] = torch.empty(n, device="cuda").uniform_(lo, hi, generator=g).bfloat16()

    def conv(name, n, taps, gain=1.0):
        T[name] = _normal(g, n, taps, dtype=torch.bfloat16, std=gain / math.sqrt(taps))

    def gated(p, ff, gain=1.0, down=1.0):
        mat(p + "gate", ff, D, gain), mat(p + "up", ff, D, gain), mat(p + "down", D, ff, down)
    T["embed"] = _normal(g, cfg["vocab"], D, dtype=torch.bfloat16, std=3.0 if design == "fomunex" else 1.0)
    if design == "pimosun":
        T["bigram"] = _normal(g, cfg["embedding"]["bigram"]["buckets"] + 1, D, dtype=torch.bfloat16)
    if "max_positions" in cfg:
        T["pos"] = _normal(g, cfg["max_positions"], D, dtype=torch.bfloat16, std=1.0 if design == "fomunex" else 0.5)
    for i, layer in enumerate(cfg["layers"]):
        p, x, m, kind, mlp = f"l{i}.", f"l{i}.mix.", layer["mixer"], layer["type"], layer["mlp"]
        for q in "1" if design == "pimosun" else "12":
            if design == "fomunex":
                T[p + "norm" + q] = torch.tensor(1.1 if q == "1" else 0.9, device="cuda").bfloat16()
            else:
                vec(p + "norm" + q, D, *((0.0, 0.3) if design == "natatar" else (1.0, 0.2)))
            if design == "natatar":
                s = cfg["streams"]
                vec(f"{p}hc{q}.in", s, 1.0 / s, 0.3), vec(f"{p}hc{q}.out", s, 1.0, 0.3)
                T[f"{p}hc{q}.mix"] = (torch.eye(s, device="cuda") * 0.8 + 0.2 / s + _normal(g, s, s, dtype=torch.float32, std=0.15)).bfloat16()
        if kind == "latent_attention":
            H = m["heads"]
            mat(x + "dq", m["q_rank"], D), vec(x + "dq.norm", m["q_rank"]), mat(x + "uq", H * (m["dim"] + m["rot_dim"]), m["q_rank"], 1.6)
            if "kv_from" not in m:
                mat(x + "dkv", m["kv_rank"] + m["rot_dim"], D), vec(x + "dkv.norm", m["kv_rank"])
            mat(x + "uk", H * m["dim"], m["kv_rank"], 1.6), mat(x + "uv", H * m["vdim"], m["kv_rank"])
            vec(x + "sink", H, 0.5, 1.5), mat(x + "g", H, D), mat(x + "o", D, H * m["vdim"])
        elif design == "gulidra" and kind == "attention":
            for c, n in (("q", 2 * m["heads"] * m["dim"]), ("k", 2 * m["kv_heads"] * m["dim"]), ("v", m["kv_heads"] * m["vdim"])):
                if c == "q" or "kv_from" not in m:
                    mat(x + c, n, D), conv(x + c + ".conv", n, m["conv"])
                    if c != "v":
                        vec(x + c + ".norm", m["dim"], 1.2)
            for c in ("lq1", "lk1", "lq2", "lk2"):
                vec(x + c, m["dim"], 0.0, 0.8 * m["dim"] ** -0.5)
            mat(x + "g", m["heads"], D), mat(x + "o", D, m["heads"] * m["vdim"])
        elif kind == "lightning":
            for c, n in (("q", m["dim"]), ("k", m["dim"]), ("v", m["vdim"]), ("g", m["vdim"])):
                mat(x + c, m["heads"] * n, D, 1.5)
            vec(x + "norm", m["heads"] * m["vdim"]), mat(x + "o", D, m["heads"] * m["vdim"])
        elif kind in ("attention", "parallel"):
            y, n = (x + "left.", m["left"]) if kind == "parallel" else (x, m)
            for c, r in (("q", n["heads"] * n["dim"]), ("k", n["kv_heads"] * n["dim"]), ("v", n["kv_heads"] * n["vdim"])):
                mat(y + c, r, D)
                if design == "natatar" and kind == "attention":
                    vec(y + c + ".b", r, 0.0, 0.5)
                    if c != "v":
                        vec(y + c + ".norm", r, 1.2)
            mat(y + "o", D, n["heads"] * n["vdim"])
            if design == "fomunex":
                vec(x + "sink", m["heads"], 1.0, 1.5)
            elif kind == "attention":
                T[x + "vmix"] = torch.tensor(0.4 + 0.1 * i, device="cuda").bfloat16()
            else:
                mat(y + "g", n["heads"] * n["vdim"], D)
                y, n = x + "right.", m["right"]
                H, v = n["heads"], n["heads"] * n["vdim"]
                for c, r in (("q", H * n["dim"]), ("k", H * n["dim"]), ("v", v), ("g", v), ("i", H), ("f", H)):
                    mat(y + c, r, D, 2.0 if c in "if" else 1.0)
                mat(y + "o", D, v), vec(y + "norm", v), vec(y + "i.b", H, 0.0, 1.5), vec(y + "f.b", H, 3.0, 2.0)
        elif kind == "channel_delta":
            H, G = m["heads"], m["kv_heads"]
            for c, r in (("q", G * m["dim"]), ("k", G * m["dim"]), ("v", H * m["vdim"])):
                mat(x + c, r, D), conv(x + c + ".conv", r, m["conv"])
            mat(x + "b", H, D, 2.0), spread(x + "A_log", H, -2.0, 1.5), vec(x + "dt_bias", H * m["dim"], -2.5, 1.5), vec(x + "norm", m["vdim"])
            mat(x + "a1", 64, D), mat(x + "a2", H * m["dim"], 64), mat(x + "g1", 64, D), mat(x + "g2", H * m["vdim"], 64), mat(x + "o", D, H * m["vdim"])
        elif kind == "wkv":
            n = m["heads"] * m["dim"]
            for c in "rkvgw":
                spread(x + "mu." + c, D, -0.2, 1.2)
            for c in "rkvg":
                mat(x + c, n, D)
            mat(x + "w1", 64, D), mat(x + "w2", n, 64), spread(x + "w0", n, -5.0, 1.0), vec(x + "norm", n), mat(x + "o", D, n)
            T[x + "u"] = _normal(g, m["heads"], m["dim"], dtype=torch.bfloat16)
        else:
            H, inner = m["heads"], m["heads"] * m["vdim"]
            cols = inner + 2 * m["groups"] * m["state"]
            mat(x + "in", inner + cols + H, D), conv(x + "conv", cols, m["conv"], 1.5), vec(x + "conv.b", cols, 0.1, 0.4)
            spread(x + "dt_bias", H, -3.0, 0.5), spread(x + "A_log", H, -2.5, 1.5), vec(x + "D", H, 0.8, 0.5), vec(x + "norm", inner), mat(x + "o", D, inner)
        if mlp["kind"] == "moe":
            r = mlp["router"]
            n = r["experts"] + r.get("identity", 0)
            for e in range(r["experts"]):      # few experts carry the weight: a close call among the last moves little
                gated(f"{p}mlp.e{e}.", mlp["expert"]["ff"], *((1.5, 0.1) if design == "fomunex" else ()))
            mat(p + "mlp.router", n, D, 3.0)
            if design == "gulidra":
                vec(p + "mlp.correction", n, 0.0, 0.1)
        elif design == "fomunex":
            mat(p + "mlp.up", mlp["ff"], D), mat(p + "mlp.down", D, mlp["ff"])
            T[p + "mlp.act"] = (torch.tensor([0.8, -0.5, 0.3, 0.2], device="cuda") + _normal(g, 4, dtype=torch.float32, std=0.2)).bfloat16()
        else:
            gated(p + "mlp.", mlp["ff"])
    if design == "fomunex":
        T["final.norm"] = torch.tensor(1.2, device="cuda").bfloat16()
    else:
        vec("final.norm", D, *((0.0, 0.3) if design == "natatar" else (1.0, 0.2)))
    if design != "natatar":
        mat("head", cfg["vocab"], D, 3.0 if design == "fomunex" else 1.0)
    return T


def _write_folder(path, cfg, T):
    head, at = {}, 0
    for name, t in T.items():
        head[name] = dict(dtype="BF16", shape=list(t.shape), data_offsets=[at, at + 2 * t.numel()])
        at += 2 * t.numel()
    text = json.dumps(head).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg, f)
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(len(text).to_bytes(8, "little") + text)
        for t in T.values():
            t.reshape(-1).view(torch.int16).cpu().numpy().tofile(f)


def _select_inputs(case, g):
    s, n = SELECT, case["sequences"]
    lens = [case["context"] - 37 * i for i in range(n)]
    kv = [[_normal(g, l, s["kv_heads"], s["head_dim"]) for _ in range(2)] for l in lens]
    return lens, kv, _normal(g, n, s["q_heads"], s["head_dim"], dtype=torch.float32)


def _q80(g, n, k):
    """n columns of k weights in blocks of 32: an f16 scale and 32 signed bytes."""
    w = torch.empty(n, k // 32, 34, device="cuda", dtype=torch.uint8)
    w[:, :, :2] = torch.empty(n, k // 32, 1, device="cuda").uniform_(0.001, 0.01, generator=g).half().view(torch.uint8)
    w[:, :, 2:] = torch.randint(-127, 128, (n, k // 32, 32), device="cuda", dtype=torch.int8, generator=g).view(torch.uint8)
    return w


def _ffn_inputs(case, g):
    d, f = case["d_model"], case["ffn"]
    return _normal(g, case["rows"], d, dtype=torch.float32), _q80(g, f, d), _q80(g, f, d), _q80(g, d, f)


def _attention_inputs(case, g):
    k, v = (_normal(g, case["context"], case["kv_heads"], case["head_dim"]) for _ in range(2))
    return k, v, _normal(g, case["q_heads"], case["head_dim"], dtype=torch.float32)


def _prompts(case, n, seed, vocab):
    """Token ids of n prompts, each followed by the tokens of the generated places."""
    return [_ids((seed, i), l + case.get("steps", 0), vocab) for i, l in enumerate(_lengths(case, n))]


def prepare(case, seed):
    ctx, g, kind = _context(), _generator(seed), case["kind"]
    if kind == "attention":
        k, v, q = _attention_inputs(case, g)
        cache = m40.KVCache(ctx, case["context"], 1, case["kv_heads"], case["head_dim"])
        torch.cuda.synchronize()
        m40.check(ctx.lib.m40llm_ext_kvcache_bulk_fill_f16(ctx.h, cache.h, 0, k.data_ptr(), v.data_ptr(), case["context"]), "bulk fill")
        ctx.sync()
        return dict(case=case, cache=cache, q=q, out=torch.zeros_like(q))
    if kind == "block_select":
        s, (lens, kv, q) = SELECT, _select_inputs(case, g)
        cache = m40.KVCache(ctx, case["context"], len(lens), s["kv_heads"], s["head_dim"],
                            compressed=dict(recent_window=s["window"], block_size=s["block"], top_blocks=s["top"], exact_old_backing=case["backing"]))
        torch.cuda.synchronize()
        for i, (k, v) in enumerate(kv):
            m40.check(ctx.lib.m40llm_ext_kvcache_bulk_fill_f16(ctx.h, cache.h, i, k.data_ptr(), v.data_ptr(), lens[i]), "bulk fill")
        ctx.sync()
        return dict(case=case, cache=cache, q=q, out=torch.zeros_like(q), ids=np.arange(len(lens), dtype=np.uint32), lens=np.array(lens, dtype=np.uint32))
    if kind == "ffn_q80":
        x, gate, up, down = _ffn_inputs(case, g)
        return dict(case=case, x=x, gate=gate, up=up, down=down, scratch=torch.empty(2, case["rows"], case["ffn"], device="cuda"), out=torch.zeros_like(x))
    if kind == "decode":
        cfg, rows = DENSE[case["model"]], case["rows"]
        lens = _lengths(case, rows)
        weights = _dense_weights(cfg, g)
        model = _Dense(ctx, cfg, weights, case["longest"] + case["steps"] + 2, rows)
        k, v = _caches(case, cfg, g)
        torch.cuda.synchronize()
        for r in range(rows):
            for l in range(cfg["n_layers"]):
                slot = model.H.m40host_model_kv_slot(model.h, r, l)
                m40.check(ctx.lib.m40llm_ext_kvcache_bulk_fill_f16(ctx.h, model.kv_handle(), slot, k[r].data_ptr(), v[r].data_ptr(), lens[r]), "bulk fill")
        ctx.sync()
        return dict(case=case, model=model, lens=np.array(lens, dtype=np.uint32), rows=np.arange(rows), first=_ids(seed, rows, cfg["vocab"]))
    if kind == "prefill":
        cfg, n = DENSE[case["model"]], case["prompts"]
        model = _Dense(ctx, cfg, _dense_weights(cfg, g), case["longest"] + 2, n)
        return dict(case=case, model=model, rows=np.arange(n), prompts=_prompts(case, n, seed, cfg["vocab"]))
    cfg, n = _design_config(case["design"]), case["sequences"]
    tokens = _prompts(case, n, seed, cfg["vocab"])
    with tempfile.TemporaryDirectory(dir="/dev/shm" if os.path.isdir("/dev/shm") else None) as d:
        _write_folder(d, cfg, _design_weights(case["design"], cfg, g))
        model = layered.LayeredModel.open(ctx, d, max_tokens=sum((len(t) + 63) // 64 * 64 for t in tokens), max_sequences=n, max_rows=4096)
    torch.cuda.empty_cache()
    return dict(case=case, model=model, tokens=tokens, lens=_lengths(case, n))


# ---- one pass ------------------------------------------------------------------------------------------------------------------------
def run(s):
    case, ctx = s["case"], _context()
    kind = case["kind"]
    if kind == "attention":
        m40.check(ctx.lib.m40llm_attention_last_token_f32_gqa_async(ctx.h, s["cache"].h, 0, s["q"].data_ptr(), case["q_heads"], case["context"], s["out"].data_ptr()))
        return s["out"]
    if kind == "block_select":
        c = SELECT
        m40.check(ctx.lib.m40llm_ext_attention_block_select_fp16_k_q4_v_multi_async(
            ctx.h, s["cache"].h, len(s["ids"]), s["ids"].ctypes.data, s["lens"].ctypes.data, s["q"].data_ptr(), c["q_heads"], c["window"], c["block"], c["top"],
            s["out"].data_ptr()))
        return s["out"]
    if kind == "ffn_q80":
        m40.check(ctx.lib.m40llm_ext_ffn_swiglu_q80_f32_async(ctx.h, s["x"].data_ptr(), s["gate"].data_ptr(), s["up"].data_ptr(), s["down"].data_ptr(),
                                                              s["scratch"].data_ptr(), s["out"].data_ptr(), case["rows"], case["d_model"], case["ffn"]))
        return s["out"]
    if kind == "decode":
        model, n = s["model"], case["steps"]
        if case["rows"] == 1:
            ids, gaps = model.decode_greedy(0, s["first"], n, start_pos=int(s["lens"][0]))
            ids, gaps = ids[None, 1:], gaps[None]
        else:
            ids, gaps = model.decode_batch_greedy(s["rows"], s["lens"], s["first"], n)
        hidden, logits = model.forward_token(0, int(s["lens"][0]) + n, ids[0, -1])
        return dict(ids=ids, gaps=gaps, hidden=hidden, logits=logits)
    if kind == "prefill":
        hidden, logits = s["model"].forward_prefill(s["rows"], s["prompts"])
        next_hidden, next_logits = s["model"].forward_token(0, len(s["prompts"][0]), int(np.argmax(logits[0])))
        return dict(hidden=hidden, logits=logits, next_hidden=next_hidden, next_logits=next_logits)
    model, lens = s["model"], s["lens"]
    out = [model.step([(i, t[:n], [n - 1]) for i, (t, n) in enumerate(zip(s["tokens"], lens))])]
    for k in range(case["steps"]):
        out.append(model.step([(i, t[n + k:n + k + 1], [0]) for i, (t, n) in enumerate(zip(s["tokens"], lens))]))
    for i in range(len(lens)):
        model.release(i)
    return np.stack(out)


# ---- what a pass cannot do without -------------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "attention":
        q, kv, hd, n = case["q_heads"], case["kv_heads"], case["head_dim"], case["context"]
        return dict(bytes=4 * n * kv * hd + 8 * q * hd, flops=4 * n * q * hd)
    if kind == "block_select":
        s, b, f = SELECT, 0, 0
        hd, vbytes = s["head_dim"], s["head_dim"] // 2 + (4 if case["backing"] == 2 else s["head_dim"] // 8)
        for i in range(case["sequences"]):
            old = max(0, case["context"] - 37 * i - s["window"])
            taken = min(old, s["top"] * s["block"])
            b += old * s["kv_heads"] * hd * 2 + min(s["kv_heads"] * old, s["q_heads"] * taken) * vbytes + 4 * s["kv_heads"] * s["window"] * hd + 8 * s["q_heads"] * hd
            f += 2 * old * s["kv_heads"] * hd + 4 * (taken + s["window"]) * s["q_heads"] * hd
        return dict(bytes=b, flops=f)
    if kind == "ffn_q80":
        n = 3 * case["d_model"] * case["ffn"]
        return dict(bytes=n * 34 // 32 + 8 * case["rows"] * case["d_model"], flops=2 * n * case["rows"])
    if kind in ("decode", "prefill"):
        cfg = DENSE[case["model"]]
        D, kv, L, V = cfg["d_model"], cfg["kv_heads"] * cfg["head_dim"], cfg["n_layers"], cfg["vocab"]
        layers, head = L * (2 * D * D + 2 * kv * D + 3 * D * cfg["ffn"]), V * D
        if kind == "decode":
            lens, n = _lengths(case, case["rows"]), case["steps"]
            seen = sum((l + n / 2) for l in lens) * L
            one = lens[0] * L
            return dict(bytes=(n + 1) * 2 * (layers + head) + 4 * kv * (n * seen + one), flops=(n * len(lens) + 1) * 2 * (layers + head) + 4 * D * (n * seen + one))
        lens = _lengths(case, case["prompts"])
        rows, pairs = sum(lens), sum(l * (l + 1) / 2 for l in lens)
        return dict(bytes=2 * 2 * (layers + head) + rows * L * kv * 4, flops=2 * (rows + 1) * layers + 2 * (len(lens) + 1) * head + 4 * L * D * (pairs + lens[0]))
    cfg, lens, steps = _design_config(case["design"]), _lengths(case, case["sequences"]), case["steps"]
    D, rows, pairs = cfg["width"], sum(lens), sum(l * (l + 1) / 2 for l in lens)
    read = lambda share, n: 1.0 - (1.0 - share) ** n          # noqa: E731  the part of the experts that n rows choose from
    b = (steps + 1) * 2 * cfg["vocab"] * D
    f = 2 * len(lens) * (steps + 1) * cfg["vocab"] * D
    for layer in cfg["layers"]:
        m, mlp, tokens = layer["mixer"], layer["mlp"], rows + steps * len(lens)
        if layer["type"] == "latent_attention":
            w = D * (m["q_rank"] + m["heads"]) + m["q_rank"] * m["heads"] * (m["dim"] + m["rot_dim"]) + m["heads"] * (m["dim"] + m["vdim"]) * m["kv_rank"] + m["heads"] * m["vdim"] * D
            w += 0 if "kv_from" in m else D * (m["kv_rank"] + m["rot_dim"])
            per_key, per_pair = 2 * (m["kv_rank"] + m["rot_dim"]), 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
        elif layer["type"] in ("attention", "parallel"):
            n = m.get("left", m)
            maps = 2 if case["design"] == "gulidra" else 1
            w = D * (maps * n["heads"] * n["dim"] + n["kv_heads"] * (maps * n["dim"] + n["vdim"]) + n["heads"] * n["vdim"])
            if layer["type"] == "parallel":
                r = m["right"]
                w += D * n["heads"] * n["vdim"] + D * r["heads"] * (2 * r["dim"] + 3 * r["vdim"])
            per_key, per_pair = 2 * n["kv_heads"] * (maps * n["dim"] + n["vdim"]), 2 * n["heads"] * maps * (n["dim"] + n["vdim"])
        else:
            per_key = per_pair = 0
            w = {"lightning": lambda: D * m["heads"] * (2 * m["dim"] + 3 * m["vdim"]), "channel_delta": lambda: D * (2 * m["kv_heads"] * m["dim"] + 2 * m["heads"] * m["vdim"]) + 256 * D,
                 "wkv": lambda: 5 * D * m["heads"] * m["dim"] + 128 * D, "mamba2": lambda: D * (3 * m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"])}[layer["type"]]()
        b += (steps + 1) * 2 * w + per_key * (tokens + steps * rows)
        f += 2 * tokens * w + per_pair * (pairs + steps * rows)
        if mlp["kind"] == "moe":
            r, e = mlp["router"], 3 * D * mlp["expert"]["ff"]
            n = r["experts"] + r.get("identity", 0)
            b += 2 * r["experts"] * e * (read(r["top"] / n, rows) + steps * read(r["top"] / n, len(lens)))
            f += 2 * tokens * r["top"] * e * r["experts"] / n
        else:
            e = D * mlp["ff"] * (2 if case["design"] == "fomunex" else 3)
            b += (steps + 1) * 2 * e
            f += 2 * tokens * e
    return dict(bytes=b, flops=f)


def tolerance(case):
    """About four times what the paths differ by from 64-bit results."""
    if case["kind"] == "layered":      # bf16 activations, and experts that are chosen by them
        return {"rel": 0.03, "max": 0.9}
    if case["kind"] == "decode":       # a new key or value that f16 rounds the other way; gaps are small differences of logits
        return {"rel": 1.5e-3, "max": 0.05}
    if case["kind"] == "prefill":
        return {"rel": 4e-4, "max": 0.02}
    return {"rel": 1e-5, "max": 4e-4}


# ---- 64-bit results ------------------------------------------------------------------------------------------------------------------
def _softmax_values(scores, v):
    return torch.softmax(scores, dim=-1) @ v


def _rms(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _attention_exact(q, k, v, heads_of):
    """q [heads][dim], k / v [tokens][kv heads][dim]: one token's attention."""
    k, v = (t.double().repeat_interleave(heads_of, dim=1).transpose(0, 1) for t in (k, v))
    return _softmax_values(q[:, None] @ k.transpose(1, 2) / math.sqrt(q.shape[-1]), v)[:, 0]


def _select_exact(case, g):
    s, (lens, kv, q) = SELECT, _select_inputs(case, g)
    out = torch.empty(q.shape, device="cuda", dtype=torch.float64)
    groups, hd = s["q_heads"] // s["kv_heads"], s["head_dim"]
    seven, fifteen = (torch.full((1,), n, device="cuda") for n in (7.0, 15.0))      # on the device: a plain number would be multiplied by its inverse
    for i, (k16, v16) in enumerate(kv):
        old = max(0, lens[i] - s["window"])
        k, v = k16.double(), v16.double()
        if old and case["backing"] == 3:      # groups of 32 under an f16 scale and an f16 minimum
            x = v16[:old].float().reshape(old, s["kv_heads"], hd // 32, 32)
            low, high = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
            d, m = ((high - low) / fifteen).half().float(), low.half().float()
            n = torch.where(d > 0, ((x - m) / d).round().clamp(0, 15), torch.zeros_like(x))
            v[:old] = (n.double() * d + m).reshape(old, s["kv_heads"], hd)
        elif old:                             # one f32 scale a row
            x = v16[:old].float()
            d = x.abs().amax(-1, keepdim=True) / seven
            n = torch.where(d > 0, (x / d).round().clamp(-7, 7), torch.zeros_like(x))
            v[:old] = (n * d).half().double()
        blocks = -(-old // s["block"])
        for h in range(s["q_heads"]):
            kh, vh, qh = k[:, h // groups], v[:, h // groups], q[i, h].double()
            seen = torch.ones(lens[i], device="cuda", dtype=torch.bool)
            scores = kh @ qh / math.sqrt(hd)
            if blocks > s["top"]:
                total = torch.zeros(blocks, device="cuda", dtype=torch.float64).index_add_(0, torch.arange(old, device="cuda") // s["block"], scores[:old])
                size = torch.full((blocks,), s["block"], device="cuda", dtype=torch.float64)
                size[-1] = old - (blocks - 1) * s["block"]
                taken = torch.zeros(blocks, device="cuda", dtype=torch.bool)
                taken[torch.topk(total / size, s["top"]).indices] = True
                seen[:old] = taken.repeat_interleave(s["block"])[:old]
            out[i, h] = _softmax_values(scores.masked_fill(~seen, -math.inf)[None], vh)[0]
    return out


def _q80_double(w):
    n, blocks, _ = w.shape
    return (w[:, :, 2:].contiguous().view(torch.int8).double() * w[:, :, :2].contiguous().view(torch.float16).double()).reshape(n, blocks * 32)


def _rope(x, pos, cfg):
    """x [tokens][heads][dim] at positions pos."""
    hd = x.shape[-1]
    a = pos.double()[:, None] * cfg["rope_base"] ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    c, s = a.cos()[:, None], a.sin()[:, None]
    if cfg["rope_layout"]:
        u, v = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([u * c - v * s, v * c + u * s], dim=-1)
    u, v = x[..., ::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], dim=-1).flatten(-2)


class _DenseExact:
    def __init__(self, cfg, weights):
        self.cfg, self.w = cfg, weights
        self.layers = [{n: t.double() for n, t in l.items()} for l in weights["layers"]]

    def layer(self, l, x, pos, attend):
        c, w, n = self.cfg, self.layers[l], len(x)
        h = _rms(x, c["rms_eps"]) * w["attn_norm"]
        q, k, v = ((h @ w["w" + t].T + (w["b" + t] if c["qkv_bias"] else 0.0)).reshape(n, -1, c["head_dim"]) for t in "qkv")
        x = x + attend(l, _rope(q, pos, c), _rope(k, pos, c), v).reshape(n, -1) @ w["wo"].T
        h = _rms(x, c["rms_eps"]) * w["ffn_norm"]
        return x + (torch.nn.functional.silu(h @ w["wgate"].T) * (h @ w["wup"].T)) @ w["wdown"].T

    def logits(self, x):
        return (_rms(x, self.cfg["rms_eps"]) * self.w["out_norm"].double()) @ self.w["lm_head"].double().T

    def tokens(self, ids, pos, k, v):
        """One token of each sequence: k / v [layer][sequence] are lists of f16 rows, which grow by the token's."""
        x, heads_of = self.w["tok_emb"][torch.as_tensor(np.asarray(ids, dtype=np.int64), device="cuda")].double(), self.cfg["q_heads"] // self.cfg["kv_heads"]
        at = torch.as_tensor(np.asarray(pos, dtype=np.int64), device="cuda")

        def attend(l, q, kn, vn):
            for r in range(len(ids)):
                k[l][r], v[l][r] = torch.cat([k[l][r], kn[r:r + 1].half()]), torch.cat([v[l][r], vn[r:r + 1].half()])
            return torch.stack([_attention_exact(q[r], k[l][r], v[l][r], heads_of) for r in range(len(ids))])
        for l in range(self.cfg["n_layers"]):
            x = self.layer(l, x, at, attend)
        return x


def _decode_exact(case, seed, g):
    cfg, rows, n = DENSE[case["model"]], case["rows"], case["steps"]
    lens = _lengths(case, rows)
    model = _DenseExact(cfg, _dense_weights(cfg, g))
    k16, v16 = _caches(case, cfg, g)
    k, v = ([[t[r, :lens[r]] for r in range(rows)] for _ in range(cfg["n_layers"])] for t in (k16, v16))
    ids, pos, picked, gaps = _ids(seed, rows, cfg["vocab"]), np.array(lens), [], []
    for _ in range(n):
        x = model.tokens(ids, pos, k, v)
        top = model.logits(x).topk(2, dim=-1)
        ids, pos = top.indices[:, 0].cpu().numpy(), pos + 1
        picked.append(ids)
        gaps.append((top.values[:, 0] - top.values[:, 1]).cpu().numpy())
    x = model.tokens(ids[:1], pos[:1], [[t[0]] for t in k], [[t[0]] for t in v])
    return dict(ids=np.stack(picked, 1).astype(np.uint32), gaps=np.stack(gaps, 1), hidden=x[0], logits=model.logits(x)[0])


def _prefill_exact(case, seed, g):
    cfg, n = DENSE[case["model"]], case["prompts"]
    model, heads_of = _DenseExact(cfg, _dense_weights(cfg, g)), cfg["q_heads"] // cfg["kv_heads"]
    hidden = []
    for i, tokens in enumerate(_prompts(case, n, seed, cfg["vocab"])):
        ids = torch.as_tensor(tokens.astype(np.int64), device="cuda")
        x, pos = model.w["tok_emb"][ids].double(), torch.arange(len(ids), device="cuda")
        past = torch.ones(len(ids), len(ids), device="cuda", dtype=torch.bool).tril()
        kept = [[], []]

        def attend(l, q, k, v):
            if i == 0:
                kept[0].append([k.half()]), kept[1].append([v.half()])
            return torch.stack([_softmax_values((q[:, h] @ k[:, h // heads_of].T / math.sqrt(cfg["head_dim"])).masked_fill(~past, -math.inf), v[:, h // heads_of])
                                for h in range(cfg["q_heads"])], dim=1)
        for l in range(cfg["n_layers"]):
            x = model.layer(l, x, pos, attend)
        hidden.append(x[-1])
        if i == 0:
            first = kept, len(ids)
    hidden = torch.stack(hidden)
    logits = model.logits(hidden)
    x = model.tokens([int(logits[0].argmax())], [first[1]], *first[0])
    return dict(hidden=hidden, logits=logits, next_hidden=x[0], next_logits=model.logits(x)[0])


class _DesignExact:
    """All tokens of one sequence through a layered design, from its equations."""

    def __init__(self, design, cfg, T):
        self.design, self.cfg, self.eps = design, cfg, cfg["norm"]["eps"]
        self.T = T

    def t(self, name):
        return self.T[name].double()

    def lin(self, x, name):
        return x @ self.t(name).T

    def conv(self, u, w):
        w, taps, n = w.double(), w.shape[1], len(u)
        u = torch.cat([torch.zeros(taps - 1, u.shape[1], device="cuda", dtype=torch.float64), u])
        return sum(w[:, j] * u[j:j + n] for j in range(taps))

    def rotate(self, x, rot):
        n, s = rot["dims"], rot["scaling"]
        i = torch.arange(n // 2, device="cuda", dtype=torch.float64)
        f = rot["base"] ** (-2.0 * i / n)
        where = lambda turns: n * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))          # noqa: E731
        lo, hi = max(math.floor(where(s["fast"])), 0), min(math.ceil(where(s["slow"])), n - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        a = torch.arange(len(x), device="cuda", dtype=torch.float64)[:, None] * (f / s["factor"] * ramp + f * (1.0 - ramp))
        mag = 0.1 * math.log(s["factor"]) + 1.0
        c, sn = a.cos() * mag, a.sin() * mag
        if x.dim() == 3:
            c, sn = c[:, None], sn[:, None]
        u, v = x[..., 0:n:2], x[..., 1:n:2]
        return torch.cat([torch.stack([u * c - v * sn, v * c + u * sn], dim=-1).flatten(-2), x[..., n:]], dim=-1)

    def causal(self, q, k, v, scale, sink=None, cap=None, falloff=0.0, window=None):
        """One head's attention."""
        n = len(q)
        i = torch.arange(n, device="cuda")
        away = i[:, None] - i[None, :]
        s = q @ k.T * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        s = (s - falloff * away).masked_fill((away < 0) | (away >= (window or n)), -math.inf)
        if sink is None:
            return _softmax_values(s, v)
        return torch.softmax(torch.cat([s, sink.expand(n, 1)], dim=1), dim=1)[:, :n] @ v

    # mixers: output before the last projection
    def latent_attention(self, h, p, m, i):
        H, dim, n = m["heads"], m["dim"], len(h)
        q = self.lin(_rms(self.lin(h, p + "dq"), self.eps) * self.t(p + "dq.norm"), p + "uq").reshape(n, H, -1)
        q = torch.cat([q[..., :dim], self.rotate(q[..., dim:], m["rot"])], dim=-1)
        if "kv_from" not in m:
            both = self.lin(h, p + "dkv")
            self.kept[i] = (_rms(both[:, :m["kv_rank"]], self.eps) * self.t(p + "dkv.norm"), self.rotate(both[:, m["kv_rank"]:], m["rot"]))
        c, r = self.kept[m.get("kv_from", i)]
        k, v = self.lin(c, p + "uk").reshape(n, H, -1), self.lin(c, p + "uv").reshape(n, H, -1)
        gate, sink = torch.sigmoid(self.lin(h, p + "g")), self.t(p + "sink")
        return torch.cat([self.causal(q[:, a], torch.cat([k[:, a], r], dim=1), v[:, a], m["scale"], sink[a]) * gate[:, a:a + 1] for a in range(H)], dim=1)

    def differential(self, h, p, m, i):
        H, G, dim, n = m["heads"], m["kv_heads"], m["dim"], len(h)
        proj = lambda c: self.conv(self.lin(h, p + c), self.T[p + c + ".conv"])          # noqa: E731
        q = (_rms(proj("q").reshape(n, 2 * H, dim), self.eps) * self.t(p + "q.norm")).reshape(n, H, 2, dim)
        if "kv_from" not in m:
            self.kept[i] = ((_rms(proj("k").reshape(n, 2 * G, dim), self.eps) * self.t(p + "k.norm")).reshape(n, G, 2, dim), proj("v").reshape(n, G, -1))
        k, v = self.kept[m.get("kv_from", i)]
        lam = torch.exp((self.t(p + "lq1") * self.t(p + "lk1")).sum()) - torch.exp((self.t(p + "lq2") * self.t(p + "lk2")).sum()) + m["diff"]
        gate, out = torch.sigmoid(self.lin(h, p + "g")), []
        for a in range(H):
            one, two = (self.causal(q[:, a, j], k[:, a * G // H, j], v[:, a * G // H], m["scale"]) for j in (0, 1))
            out.append(_rms(one - lam * two, self.eps) * (1.0 - m["diff"]) * gate[:, a:a + 1])
        return torch.cat(out, dim=1)

    def walk(self, n, S, step):
        """Outputs of a recurrence, token after token."""
        out = []
        for t in range(n):
            S, o = step(t, S)
            out.append(o)
        return torch.stack(out)

    def zeros(self, *shape):
        return torch.zeros(shape, device="cuda", dtype=torch.float64)

    def lightning(self, h, p, m):
        n, H = len(h), m["heads"]
        q, k, v = (torch.nn.functional.silu(self.lin(h, p + c)).reshape(n, H, -1) for c in "qkv")
        decay = torch.tensor(m["decay"], device="cuda", dtype=torch.float64)[:, None, None]

        def step(t, S):
            S = decay * S + k[t][:, :, None] * v[t][:, None, :]
            return S, (q[t][:, None] @ S)[:, 0]
        o = self.walk(n, self.zeros(H, m["dim"], m["vdim"]), step).reshape(n, -1)
        return _rms(o, self.eps) * self.t(p + "norm") * torch.sigmoid(self.lin(h, p + "g"))

    def memory(self, h, p, m):
        n, H = len(h), m["heads"]
        q, k, v = (self.lin(h, p + c).reshape(n, H, -1) for c in "qkv")
        q, cap = q * m["dim"] ** -0.5, lambda z: m["gate_cap"] * torch.tanh(z / m["gate_cap"])
        i, f = cap(self.lin(h, p + "i") + self.t(p + "i.b")), torch.nn.functional.logsigmoid(cap(self.lin(h, p + "f") + self.t(p + "f.b")))
        v = torch.cat([v, torch.ones_like(v[..., :1])], dim=-1)          # the normalizer as one more column

        def step(t, state):
            S, top0 = state
            top = torch.maximum(f[t] + top0, i[t])
            S = torch.exp(f[t] + top0 - top)[:, None, None] * S + (torch.exp(i[t] - top)[:, None] * k[t])[:, :, None] * v[t][:, None, :]
            o = (q[t][:, None] @ S)[:, 0]
            return (S, top), o[:, :-1] / (torch.maximum(o[:, -1:].abs(), torch.exp(-top)[:, None]) + 1e-6)
        o = self.walk(n, (self.zeros(H, m["dim"], m["vdim"] + 1), self.zeros(H)), step)
        return _rms(o, self.eps).reshape(n, -1) * self.t(p + "norm") * torch.sigmoid(self.lin(h, p + "g"))

    def delta(self, h, p, m):
        n, H, G, dim = len(h), m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (torch.nn.functional.silu(self.conv(self.lin(h, p + c), self.T[p + c + ".conv"])) for c in "qkv")
        q, k = ((x / torch.sqrt(x.square().sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, dim=1) for x in (q.reshape(n, G, dim), k.reshape(n, G, dim)))
        q, v, beta = q * dim ** -0.5, v.reshape(n, H, -1), torch.sigmoid(self.lin(h, p + "b"))
        a = self.lin(self.lin(h, p + "a1"), p + "a2").reshape(n, H, dim)
        g = torch.exp(-torch.exp(self.t(p + "A_log"))[:, None] * torch.nn.functional.softplus(a + self.t(p + "dt_bias").reshape(H, dim), threshold=60.0))

        def step(t, S):
            S = g[t][:, :, None] * S
            u = beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0])
            S = S + k[t][:, :, None] * u[:, None, :]
            return S, (q[t][:, None] @ S)[:, 0]
        o = self.walk(n, self.zeros(H, dim, m["vdim"]), step)
        return (_rms(o, self.eps) * self.t(p + "norm")).reshape(n, -1) * torch.sigmoid(self.lin(self.lin(h, p + "g1"), p + "g2"))

    def normed_attention(self, h, p, m):
        n, H, G = len(h), m["heads"], m["kv_heads"]
        q, k, v = (self.lin(h, p + c) + self.t(p + c + ".b") for c in "qkv")
        q, k = _rms(q, self.eps) * self.t(p + "q.norm"), _rms(k, self.eps) * self.t(p + "k.norm")
        if self.first is None:
            self.first = v
        else:
            lam = self.t(p + "vmix")
            v = (1.0 - lam) * v + lam * self.first
        return self.heads(q.reshape(n, H, -1), k.reshape(n, G, -1), v.reshape(n, G, -1), m["scale"])

    def heads(self, q, k, v, scale):
        per = q.shape[1] // k.shape[1]
        return torch.cat([self.causal(q[:, a], k[:, a // per], v[:, a // per], scale) for a in range(q.shape[1])], dim=1)

    def parallel(self, h, p, m):
        n, l = len(h), m["left"]
        q, k, v = (self.lin(h, p + "left." + c).reshape(n, r, -1) for c, r in (("q", l["heads"]), ("k", l["kv_heads"]), ("v", l["kv_heads"])))
        left = self.heads(self.rotate(q, l["rot"]), self.rotate(k, l["rot"]), v, l["scale"]) * torch.sigmoid(self.lin(h, p + "left.g"))
        return m["left_scale"] * self.lin(left, p + "left.o") + m["right_scale"] * self.lin(self.memory(h, p + "right.", m["right"]), p + "right.o")

    def windowed(self, h, p, m):
        n, H, G = len(h), m["heads"], m["kv_heads"]
        q, k, v = (self.lin(h, p + c).reshape(n, r, -1) for c, r in (("q", H), ("k", G), ("v", G)))
        q, k, sink = _rms(q, self.eps), _rms(k, self.eps), self.t(p + "sink")
        return torch.cat([self.causal(q[:, a], k[:, a * G // H], v[:, a * G // H], m["scale"], sink[a], m["softcap"], 2.0 ** (-8.0 * (a + 1) / H), m["mask"]["size"])
                          for a in range(H)], dim=1)

    def time_mixing(self, h, p, m):
        n, H, d = len(h), m["heads"], m["dim"]
        before = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
        mix = {c: h + (before - h) * self.t(p + "mu." + c) for c in "rkvgw"}
        r, k, v = (self.lin(mix[c], p + c).reshape(n, H, d) for c in "rkv")
        w = torch.exp(-torch.exp(self.lin(torch.tanh(self.lin(mix["w"], p + "w1")), p + "w2") + self.t(p + "w0"))).reshape(n, H, d)
        u = self.t(p + "u")[:, :, None]

        def step(t, S):
            kv = k[t][:, :, None] * v[t][:, None, :]
            return w[t][:, :, None] * S + kv, (r[t][:, None] @ (S + u * kv))[:, 0]
        o = self.walk(n, self.zeros(H, d, d), step)
        return _rms(o, self.eps).reshape(n, -1) * self.t(p + "norm") * torch.nn.functional.silu(self.lin(mix["g"], p + "g"))

    def state_space(self, h, p, m):
        n, H, e, N, G = len(h), m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * e
        z, xbc, dt = torch.split(self.lin(h, p + "in"), [inner, inner + 2 * G * N, H], dim=1)
        x, B, C = torch.split(torch.nn.functional.silu(self.conv(xbc, self.T[p + "conv"]) + self.t(p + "conv.b")), [inner, G * N, G * N], dim=1)
        x, (B, C) = x.reshape(n, H, e), (y.reshape(n, G, N).repeat_interleave(H // G, dim=1) for y in (B, C))
        dt = torch.nn.functional.softplus(dt + self.t(p + "dt_bias"), threshold=60.0)
        keep = torch.exp(-torch.exp(self.t(p + "A_log")) * dt)

        def step(t, S):
            S = keep[t][:, None, None] * S + (dt[t][:, None] * B[t])[:, :, None] * x[t][:, None, :]
            return S, (C[t][:, None] @ S)[:, 0]
        y = (self.walk(n, self.zeros(H, N, e), step) + self.t(p + "D")[:, None] * x).reshape(n, inner) * torch.nn.functional.silu(z)
        return _rms(y.reshape(n, m["norm_groups"], -1), self.eps).reshape(n, inner) * self.t(p + "norm")

    # feed-forwards
    def experts(self, h, p, mlp):
        r, z = mlp["router"], self.lin(h, p + "router")
        s = torch.sigmoid(z) if self.design == "fomunex" else torch.softmax(z, dim=1)
        c = s + self.t(p + "correction") if self.design == "gulidra" else s
        if r.get("groups"):
            best = c.reshape(len(h), r["groups"]["count"], -1).amax(-1)
            ok = torch.zeros_like(best, dtype=torch.bool).scatter_(1, best.topk(r["groups"]["keep"], dim=1).indices, True)
            c = c.masked_fill(~ok.repeat_interleave(c.shape[1] // r["groups"]["count"], dim=1), -math.inf)
        chosen = c.topk(r["top"], dim=1).indices
        weight, out = s.gather(1, chosen) * r.get("scale", 1.0), torch.zeros_like(h)
        for e in range(s.shape[1]):
            t, j = torch.nonzero(chosen == e, as_tuple=True)
            if len(t) == 0:
                continue
            w, x, q = weight[t, j][:, None], h[t], f"{p}e{e}."
            if self.design == "fomunex":
                a, limit = self.lin(w * x, q + "gate").clamp(max=mlp["expert"]["limit"]), mlp["expert"]["limit"]
                out[t] += self.lin(a * torch.sigmoid(1.702 * a) * (self.lin(w * x, q + "up").clamp(-limit, limit) + 1.0), q + "down")
            else:
                out[t] += w * (x if e >= r["experts"] else self.gated(x, q, torch.nn.functional.silu))
        return out

    def gated(self, h, p, act):
        return self.lin(act(self.lin(h, p + "gate")) * self.lin(h, p + "up"), p + "down")

    def polynomial(self, h, p):
        z, a = self.lin(h, p + "up"), self.t(p + "act")
        return self.lin(sum(a[i] * _rms(z ** (i + 1), self.eps) for i in range(3)) + a[3], p + "down")

    def __call__(self, tokens, places):
        """Logits of the places."""
        cfg, design, ids = self.cfg, self.design, torch.as_tensor(tokens.astype(np.int64), device="cuda")
        self.kept, self.first = {}, None
        x = self.T["embed"][ids].double() * cfg.get("embedding", {}).get("scale", 1.0)
        if design == "pimosun":
            b = cfg["embedding"]["bigram"]
            row = torch.cat([torch.tensor([b["buckets"]], device="cuda"), (ids[:-1] * b["mul_prev"] + ids[1:] * b["mul_cur"]) % b["buckets"]])
            x = x + self.T["bigram"][row].double()
        if "pos" in self.T:
            x = x + self.T["pos"][:len(ids)].double()
        streams = torch.stack([x] * cfg.get("streams", 1))
        mult, ln = cfg.get("residual_mult", 1.0), lambda y: torch.nn.functional.layer_norm(y, y.shape[-1:], eps=self.eps)          # noqa: E731
        gelu = lambda y: torch.nn.functional.gelu(y, approximate="tanh")          # noqa: E731
        for i, layer in enumerate(cfg["layers"]):
            p, q, m, kind, mlp = f"l{i}.", f"l{i}.mix.", layer["mixer"], layer["type"], layer["mlp"]
            mixers = dict(latent_attention=lambda h: self.lin(self.latent_attention(h, q, m, i), q + "o"), lightning=lambda h: self.lin(self.lightning(h, q, m), q + "o"),
                          parallel=lambda h: self.parallel(h, q, m), channel_delta=lambda h: self.lin(self.delta(h, q, m), q + "o"),
                          wkv=lambda h: self.lin(self.time_mixing(h, q, m), q + "o"), mamba2=lambda h: self.lin(self.state_space(h, q, m), q + "o"),
                          attention=lambda h: self.lin(dict(gulidra=lambda: self.differential(h, q, m, i), natatar=lambda: self.normed_attention(h, q, m),
                                                            fomunex=lambda: self.windowed(h, q, m))[design](), q + "o"))
            dense = dict(pimosun=lambda h: self.gated(h, p + "mlp.", gelu), fomunex=lambda h: self.polynomial(h, p + "mlp."))
            feed = (lambda h: self.experts(h, p + "mlp.", mlp)) if mlp["kind"] == "moe" else dense.get(design, lambda h: self.gated(h, p + "mlp.", torch.nn.functional.silu))
            if design == "pimosun":
                h = ln(x) * self.t(p + "norm1")
                x = x + mixers[kind](h) + feed(h)
            for k, f in enumerate((mixers[kind], feed) if design != "pimosun" else ()):
                norm = self.t(f"{p}norm{k + 1}")
                if design == "gulidra":
                    x = x + mult * _rms(f(x), self.eps) * norm
                elif design == "fomunex":
                    x = x + f(_rms(x, self.eps) * norm)
                else:
                    hc = f"{p}hc{k + 1}."
                    y = f(_rms(torch.einsum("s,snd->nd", self.t(hc + "in"), streams), self.eps) * (1.0 + norm))
                    streams = torch.einsum("st,snd->tnd", self.t(hc + "mix"), streams) + mult * self.t(hc + "out")[:, None, None] * y
        x = (streams.sum(0) if design == "natatar" else x)[places]
        x = ln(x) * self.t("final.norm") if design == "pimosun" else _rms(x, self.eps) * (self.t("final.norm") + (1.0 if design == "natatar" else 0.0))
        logits = self.lin(x, "embed" if design == "natatar" else "head") * cfg.get("logit_scale", 1.0)
        return cfg["logit_softcap"] * torch.tanh(logits / cfg["logit_softcap"]) if "logit_softcap" in cfg else logits


def exact(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind == "attention":
        k, v, q = _attention_inputs(case, g)
        return _attention_exact(q.double(), k, v, case["q_heads"] // case["kv_heads"])
    if kind == "block_select":
        return _select_exact(case, g)
    if kind == "ffn_q80":
        x, gate, up, down = _ffn_inputs(case, g)
        x = x.double()
        return (torch.nn.functional.silu(x @ _q80_double(gate).T) * (x @ _q80_double(up).T)) @ _q80_double(down).T
    if kind == "decode":
        return _decode_exact(case, seed, g)
    if kind == "prefill":
        return _prefill_exact(case, seed, g)
    cfg = _design_config(case["design"])
    model = _DesignExact(case["design"], cfg, _design_weights(case["design"], cfg, g))
    out = [model(t, list(range(n - 1, n + case["steps"]))) for t, n in zip(_prompts(case, case["sequences"], seed, cfg["vocab"]), _lengths(case, case["sequences"]))]
    return torch.stack(out, dim=1)
