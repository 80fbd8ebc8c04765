"""The work a program has this library do, as cases that can be timed and compared.

A case is a dict of plain values. ``prepare`` makes what a caller has in hand before the call
(pools, tables, weights, workspaces, a captured graph where an engine replays one), ``run``
makes one pass through the public entry points (``crucible_amd.gpu.Gpu``,
``crucible_amd.gpu_model.GpuModel``) and returns everything it computed, ``exact`` gives the
same outputs in 64-bit arithmetic from plain torch.

Operations (``case["op"]``):

* ``decode``  - the attention of one batched decode step: per layer the fused append +
  attention launch (from separate q, k, v or from the fused q/k/v rows with RoPE), or the
  attention alone. The layers of a step replay from one graph, as the engine's step does.
* ``prefill`` - causal attention of whole prompts whose keys are in the pool.
* ``chunk``   - chunks of prompts continued on a cached history: the K and the V append of
  every layer and the tiled attention, called eagerly (chunk sizes differ from call to call).
* ``proj``    - the projections of one decoder layer over some rows: q/k/v with its norm, o
  with the residual, gate/up with norm and SwiGLU, down with the residual.
* ``step``    - a whole batched greedy decode step of the decoder, replayed from a graph.
* ``model``   - ``GpuModel.prefill_logits``: packed prompts to last-row logits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from crucible_amd.gpu import Gpu, pool_elems
from crucible_amd.gpu_model import GpuModel, ModelConfig, rope_tables, weight_names, weight_shape
from crucible_amd.paged import segments_from_cu_seqlens

PAGE = 16
VOCAB = 50257
_DTYPE = {"f16": torch.float16, "f32": torch.float32}


# ------------------------------------------------------------------------------- the cases

def listed():
    return [
        # One user, one step: the smallest decode call, 12 short launches (config 2's shape),
        # fed from the fused q/k/v rows as the engine's step feeds it.
        _decode("decode_b1", batch=1, n_head=12, n_kv=3, head_dim=64, layers=12, capacity=1024,
                lo=1024, hi=1024, entry="qkv"),
        # Continuous batching at batch 16, contexts 64..2048 (config 3, the headline).
        _decode("decode_b16", batch=16, n_head=12, n_kv=3, head_dim=64, layers=12, capacity=2048,
                lo=64, hi=2048, entry="append", q="f16"),
        # A loaded server: a large batch, where bandwidth counts.
        _decode("decode_b128", batch=128, n_head=12, n_kv=3, head_dim=64, layers=4, capacity=2048,
                lo=64, hi=2048, entry="append", q="f16"),
        # A head dimension other than the presets' 64, which the entry points take as well.
        _decode("decode_hd128", batch=16, n_head=12, n_kv=3, head_dim=128, layers=4, capacity=2048,
                lo=64, hi=2048, entry="append", q="f16"),
        # One 512-token prompt (config 1), all layers.
        _prefill("prefill_512", lens="512", n_head=12, n_kv=12, head_dim=64, layers=12, q="f16"),
        # Eight ragged prompts packed (config 4: 16/4 heads, 32..512 tokens), f32 queries as
        # the projections leave them.
        _prefill("prefill_packed", lens="137,420,46,311,98,275,402,190", n_head=16, n_kv=4,
                 head_dim=64, layers=12, q="f32"),
        # A long prompt.
        _prefill("prefill_8192", lens="8192", n_head=12, n_kv=12, head_dim=64, layers=1, q="f16"),
        # Prompts at another head dimension.
        _prefill("prefill_hd128", lens="1000,333,777,64", n_head=12, n_kv=3, head_dim=128,
                 layers=1, q="f16"),
        # Chunked prefill on cached history: the engine's heterogeneous batch (starts
        # 0/63/255/512, lengths 17/64/129/257), appends included.
        _chunk("chunk_append", starts="0,63,255,512", lens="17,64,129,257", n_head=12, n_kv=3,
               head_dim=64, layers=12),
        # One layer's projections over a medium prompt batch.
        _proj("proj_1003", rows=1003, n_embd=768, hidden=2048, n_head=12, n_kv=3),
        # A whole decode step of the 120m decoder at batch 16, logits out.
        _step("step_b16", batch=16, capacity=1024, lo=64, hi=767, layers=12),
        # Sixteen prompts of 64..512 tokens to logits through the whole 120m decoder.
        _model("model_prompts", prompts=16, lo=64, hi=512, layers=12),
    ]


def _decode(name=None, **kw):
    return _case(name, dict(op="decode", q="f32", out="f32", **{k: v for k, v in kw.items()
                                                                 if k not in ("q", "out")})
                 | {k: kw[k] for k in ("q", "out") if k in kw})


def _prefill(name=None, form="tiled", **kw):
    return _case(name, dict(op="prefill", form=form, **kw))


def _chunk(name=None, **kw):
    return _case(name, dict(op="chunk", **kw))


def _proj(name=None, **kw):
    return _case(name, dict(op="proj", **kw))


def _step(name=None, **kw):
    return _case(name, dict(op="step", **kw))


def _model(name=None, **kw):
    return _case(name, dict(op="model", **kw))


def _case(name, d):
    return d if name is None else dict(d, name=name)


_HEADS = [(12, 3), (12, 12), (16, 4)]  # the presets' GQA shapes and the MHA one


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))))))


def draw(rng):
    """One more case of the ranges above."""
    u = rng.random()
    if u < 0.36:
        n_head, n_kv = rng.choice(_HEADS)
        hd = 64 if rng.random() < 0.75 else rng.choice([32, 96, 128])
        capacity = 16 * _log_int(rng, 8, 192)
        batch = _log_int(rng, 1, 128)
        per_layer = batch * capacity * n_kv * hd * 2
        layers = max(1, min(12, int(250e6 // per_layer)))
        hi = rng.randint(max(1, capacity // 3), capacity)
        lo = rng.randint(1, hi)
        entry = rng.choice(["append", "qkv", "decode"])
        return _decode(batch=batch, n_head=n_head, n_kv=n_kv, head_dim=hd, layers=layers,
                       capacity=capacity, lo=lo, hi=hi, entry=entry,
                       q="f32" if entry == "qkv" else rng.choice(["f16", "f32"]),
                       out=rng.choice(["f32", "f32", "f16"]))
    if u < 0.66:
        n_head, n_kv = rng.choice(_HEADS)
        hd = 64 if rng.random() < 0.75 else rng.choice([32, 96, 128])
        form = rng.choice(["tiled", "tiled", "packed", "paged"])
        n = 1 if form == "paged" else _log_int(rng, 1, 16)
        longest = 6000 if hd == 64 else 1200
        lens = [_log_int(rng, 8, longest) for _ in range(n)]
        limit = 20e6 if hd == 64 else 1e6  # visible pairs
        while sum(x * (x + 1) // 2 for x in lens) > limit:
            lens = [max(1, x * 3 // 4) for x in lens]
        small = sum(lens) <= 2048
        return _prefill(lens=",".join(map(str, lens)), n_head=n_head, n_kv=n_kv, head_dim=hd,
                        layers=rng.choice([4, 12]) if small and hd == 64 else 1,
                        q=rng.choice(["f16", "f32"]), form=form)
    if u < 0.78:
        n_head, n_kv = rng.choice(_HEADS)
        n = _log_int(rng, 1, 12)
        return _chunk(starts=",".join(str(rng.choice([0, _log_int(rng, 1, 1500)])) for _ in range(n)),
                      lens=",".join(str(_log_int(rng, 1, 400)) for _ in range(n)),
                      n_head=n_head, n_kv=n_kv, head_dim=64, layers=12)
    if u < 0.93:
        n_embd, hidden, n_head, n_kv = rng.choice([(768, 2048, 12, 3), (1024, 2752, 16, 4)])
        return _proj(rows=_log_int(rng, 1, 5000), n_embd=n_embd, hidden=hidden, n_head=n_head,
                     n_kv=n_kv)
    if u < 0.97:
        hi = rng.randint(100, 1000)
        return _step(batch=_log_int(rng, 1, 32), capacity=1024, lo=rng.randint(1, hi), hi=hi,
                     layers=12)
    hi = rng.randint(40, 500)
    return _model(prompts=_log_int(rng, 1, 16), lo=rng.randint(8, hi), hi=hi, layers=12)


# ------------------------------------------------------------------------------- inputs

class _Seeded:
    """Values on the device and whole numbers on the host, from one seed."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", 0)
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(int(seed))
        self.host = np.random.default_rng(int(seed))

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        x = torch.empty(shape, dtype=dtype, device=self.dev)
        return x.normal_(0.0, std, generator=self.g)

    def to(self, a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(self.dev)


def _tables(host, lens, stride, longest=None):
    """Disjoint page tables over a shuffled pool with room for `longest` tokens (by default
    the lengths themselves) a request."""
    need = [-(-int(n) // PAGE) for n in lens]
    n_pages = 8 + (sum(need) if longest is None else len(need) * -(-longest // PAGE))
    perm = host.permutation(n_pages).astype(np.int32)
    tables = np.zeros((len(lens), stride), np.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[at:at + n]
        at += n
    return tables, n_pages


def _graph(step):
    """A graph of one pass: warm-up on a side stream, then capture."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    return g


def _decode_lens(case, host):
    """Visible lengths, the appended token included."""
    lens = host.integers(case["lo"], case["hi"] + 1, size=case["batch"]).astype(np.int32)
    return np.minimum(lens, case["capacity"])


def _prepare_decode(case, seed, graph=True):
    r, gpu = _Seeded(seed), Gpu(0)
    b, hd, layers = case["batch"], case["head_dim"], case["layers"]
    kv = case["n_kv"] * hd
    lens = _decode_lens(case, r.host)
    stride = case["capacity"] // PAGE
    tables, n_pages = _tables(r.host, lens, stride, min(case["hi"], case["capacity"]))
    s = {
        "case": case, "gpu": gpu, "seq_lens": lens, "n_pages": n_pages,
        "k_pool": r.normal(pool_elems(n_pages, layers, kv), dtype=torch.float16),
        "v_pool": r.normal(pool_elems(n_pages, layers, kv), dtype=torch.float16),
        "tables": r.to(tables), "lens": r.to(lens), "positions": r.to(lens - 1),
        "out": torch.zeros((layers, b, case["n_head"] * hd), dtype=_DTYPE[case["out"]],
                           device=r.dev),
        "ws": gpu.workspace(b, case["n_head"], case["capacity"]),
    }
    if case["entry"] == "qkv":
        s["qkv"] = r.normal(layers, b, case["n_head"] * hd + 2 * kv)
        cos, sin = rope_tables(hd, case["capacity"], 10000.0)
        s["cos"], s["sin"] = r.to(cos), r.to(sin)
    else:
        s["q"] = r.normal(layers, b, case["n_head"] * hd, dtype=_DTYPE[case["q"]])
        if case["entry"] == "append":
            s["k_new"] = r.normal(layers, b, kv)
            s["v_new"] = r.normal(layers, b, kv)

    def step():
        shape = (b, case["n_head"], case["n_kv"], hd, stride, layers)
        for i in range(layers):
            tail = (s["out"][i], s["tables"])
            if case["entry"] == "qkv":
                gpu.attention_decode_qkv_paged_append(
                    s["qkv"][i], s["cos"], s["sin"], s["k_pool"], s["v_pool"], *tail,
                    s["positions"], s["lens"], *shape, i, kv, case["capacity"],
                    workspace=s["ws"])
            elif case["entry"] == "append":
                gpu.attention_decode_paged_append(
                    s["q"][i], s["k_new"][i], s["v_new"][i], s["k_pool"], s["v_pool"], *tail,
                    s["positions"], s["lens"], *shape, i, kv, case["capacity"],
                    workspace=s["ws"])
            else:
                gpu.attention_decode_paged(
                    s["q"][i], s["k_pool"], s["v_pool"], *tail, s["lens"], *shape, i, kv,
                    case["capacity"], workspace=s["ws"])

    if graph:
        s["graph"] = _graph(step)
    return s


def _run_decode(s):
    s["graph"].replay()
    if s["case"]["entry"] == "decode":
        return {"out": s["out"]}
    return {"out": s["out"], "k_pool": s["k_pool"], "v_pool": s["v_pool"]}


def _ints(text):
    return np.array([int(x) for x in text.split(",")], np.int32)


def _prepare_prefill(case, seed, graph=True):
    r, gpu = _Seeded(seed), Gpu(0)
    lens, hd, layers = _ints(case["lens"]), case["head_dim"], case["layers"]
    kv, rows = case["n_kv"] * hd, int(lens.sum())
    stride = -(-int(lens.max()) // PAGE)
    tables, n_pages = _tables(r.host, lens, stride)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    seg, max_chunk = segments_from_cu_seqlens(cu)
    params = np.zeros(8, np.int32)
    s = {
        "case": case, "gpu": gpu, "seq_lens": lens, "n_pages": n_pages,
        "k_pool": r.normal(pool_elems(n_pages, layers, kv), dtype=torch.float16),
        "v_pool": r.normal(pool_elems(n_pages, layers, kv), dtype=torch.float16),
        "q": r.normal(layers, rows, case["n_head"] * hd, dtype=_DTYPE[case["q"]]),
        "out": torch.zeros((layers, rows, case["n_head"] * hd), dtype=torch.float32,
                           device=r.dev),
        "tables": r.to(tables), "segments": r.to(seg), "params": r.to(params),
        "owners": r.to(np.repeat(np.arange(len(lens), dtype=np.int32), lens)),
        "positions": r.to(np.concatenate([np.arange(n, dtype=np.int32) for n in lens])),
    }

    def step():
        heads = (case["n_head"], case["n_kv"], hd, layers)
        for i in range(layers):
            q, out = s["q"][i], s["out"][i]
            if case["form"] == "tiled":
                gpu.attention_prefill_tiled(q, s["k_pool"], s["v_pool"], None, None, out,
                                            s["tables"], s["segments"], len(lens), max_chunk,
                                            stride, *heads, i, kv)
            elif case["form"] == "packed":
                gpu.attention_prefill_packed(q, s["k_pool"], s["v_pool"], out, s["tables"],
                                             s["owners"], s["positions"], rows, stride, *heads,
                                             i, kv, stride * PAGE)
            else:
                gpu.attention_prefill_paged(q, s["k_pool"], s["v_pool"], out, s["tables"], rows,
                                            *heads, i, kv, stride * PAGE, s["params"])

    s["step"] = step
    # Several layers of short prompts replay from a graph (a launch takes less time than the
    # call that makes it); a single long layer is called as it is.
    if graph and layers > 1:
        s["graph"] = _graph(step)
    return s


def _run_prefill(s):
    if "graph" in s:
        s["graph"].replay()
    else:
        s["step"]()
    return {"out": s["out"]}


def _prepare_chunk(case, seed, graph=True):
    r, gpu = _Seeded(seed), Gpu(0)
    starts, lens, hd, layers = _ints(case["starts"]), _ints(case["lens"]), 64, case["layers"]
    kv, rows = case["n_kv"] * hd, int(lens.sum())
    stride = -(-int((starts + lens).max()) // PAGE)
    tables, n_pages = _tables(r.host, starts + lens, stride)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    seg, max_chunk = segments_from_cu_seqlens(cu, starts)
    return {
        "case": case, "gpu": gpu, "starts": starts, "seq_lens": lens, "n_pages": n_pages,
        "rows": rows, "stride": stride, "max_chunk": max_chunk,
        "k_pool": r.normal(pool_elems(n_pages, layers, kv), dtype=torch.float16),
        "v_pool": r.normal(pool_elems(n_pages, layers, kv), dtype=torch.float16),
        "q": r.normal(layers, rows, case["n_head"] * hd),
        "k": r.normal(layers, rows, kv), "v": r.normal(layers, rows, kv),
        "out": torch.zeros((layers, rows, case["n_head"] * hd), dtype=torch.float32,
                           device=r.dev),
        "tables": r.to(tables), "segments": r.to(seg),
        "owners": r.to(np.repeat(np.arange(len(lens), dtype=np.int32), lens)),
        "positions": r.to(np.concatenate([a + np.arange(n, dtype=np.int32)
                                          for a, n in zip(starts, lens)]).astype(np.int32)),
    }


def _run_chunk(s):
    case, gpu = s["case"], s["gpu"]
    kv, layers = case["n_kv"] * 64, case["layers"]
    for i in range(layers):
        for kind in ("k", "v"):
            gpu.cache_store_packed_paged(s[kind][i], s[kind + "_pool"], s["tables"], s["owners"],
                                         s["positions"], s["rows"], kv, s["stride"], layers, i,
                                         kind=kind)
        gpu.attention_prefill_tiled(s["q"][i], s["k_pool"], s["v_pool"], None, None, s["out"][i],
                                    s["tables"], s["segments"], len(s["seq_lens"]),
                                    s["max_chunk"], s["stride"], case["n_head"], case["n_kv"], 64,
                                    layers, i, kv)
    return {"out": s["out"], "k_pool": s["k_pool"], "v_pool": s["v_pool"]}


def _hidden_rows(r, rows, n):
    """Hidden-state rows: channels of different scales, as a trained decoder's are."""
    return r.normal(rows, n) * torch.exp(0.5 * r.normal(n))


def _prepare_proj(case, seed, graph=True):
    r, gpu = _Seeded(seed), Gpu(0)
    rows, d, hid = case["rows"], case["n_embd"], case["hidden"]
    width = d + 2 * case["n_kv"] * (d // case["n_head"])
    f = dict(dtype=torch.float32, device=r.dev)
    s = {
        "case": case, "gpu": gpu, "x": _hidden_rows(r, rows, d), "attn": r.normal(rows, d, std=0.5),
        "norm1": 1.0 + 0.1 * r.normal(d), "norm2": 1.0 + 0.1 * r.normal(d),
        "wqkv": r.normal(width, d, dtype=torch.float16, std=0.02),
        "wo": r.normal(d, d, dtype=torch.float16, std=0.02),
        "wg": r.normal(hid, d, dtype=torch.float16, std=0.02),
        "wu": r.normal(hid, d, dtype=torch.float16, std=0.02),
        "wd": r.normal(d, hid, dtype=torch.float16, std=0.02),
        "qkv": torch.empty((rows, width), **f), "h": torch.empty((rows, d), **f),
        "act": torch.empty((rows, hid), **f), "y": torch.empty((rows, d), **f),
    }

    def step():
        gpu.linear_f64acc(s["x"], s["wqkv"], s["qkv"], norm_w=s["norm1"])
        gpu.linear_f64acc(s["attn"], s["wo"], s["h"], resid=s["x"])
        gpu.linear_swiglu_f64acc(s["h"], s["wg"], s["wu"], s["act"], norm_w=s["norm2"])
        gpu.linear_f64acc(s["act"], s["wd"], s["y"], resid=s["h"])

    s["step"] = step
    if graph and rows <= 64:  # a decode batch: part of a captured step
        s["graph"] = _graph(step)
    return s


def _run_proj(s):
    if "graph" in s:
        s["graph"].replay()
    else:
        s["step"]()
    return {k: s[k] for k in ("qkv", "h", "act", "y")}


def _config(case):
    return ModelConfig(n_layer=case["layers"])  # the 120m preset


def _weights(cfg, r):
    """fp16 weights of the decoder on the device: matrices N(0, 0.02), norms about 1."""
    w = {}
    for name in weight_names(cfg):
        shape = weight_shape(cfg, name)
        if name.endswith("norm.weight"):
            w[name] = (1.0 + 0.1 * r.normal(*shape)).half()
        else:
            w[name] = r.normal(*shape, dtype=torch.float16, std=0.02)
    return w


def _prepare_step(case, seed, graph=True):
    r, gpu, cfg = _Seeded(seed), Gpu(0), _config(case)
    b, d, kv, hid, n = case["batch"], cfg.n_embd, cfg.kv_dim, cfg.hidden, cfg.n_layer
    w = _weights(cfg, r)
    layers = []
    for i in range(n):
        p = f"blocks.{i}."
        layers.append({
            "attn_norm": w[p + "attn_norm.weight"].float(),
            "mlp_norm": w[p + "mlp_norm.weight"].float(),
            "wqkv": torch.cat([w[p + f"attn.{x}_proj.weight"] for x in "qkv"]),
            "wo": w[p + "attn.o_proj.weight"],
            "wgu": torch.cat([w[p + "mlp.gate_proj.weight"], w[p + "mlp.up_proj.weight"]]),
            "wd": w[p + "mlp.down_proj.weight"],
        })
    lens = _decode_lens(case, r.host)
    stride = case["capacity"] // PAGE
    tables, n_pages = _tables(r.host, lens, stride, min(case["hi"], case["capacity"]))
    cos, sin = rope_tables(64, case["capacity"], cfg.rope_theta)
    f = dict(dtype=torch.float32, device=r.dev)
    s = {
        "case": case, "gpu": gpu, "cfg": cfg, "layers": layers, "seq_lens": lens,
        "n_pages": n_pages,
        "emb": w["tok_emb.weight"].float(), "head": w["tok_emb.weight"],
        "final_norm": w["final_norm.weight"].float(),
        "tokens_in": r.to(r.host.integers(0, VOCAB, size=b)),
        "k_pool": r.normal(pool_elems(n_pages, n, kv), dtype=torch.float16),
        "v_pool": r.normal(pool_elems(n_pages, n, kv), dtype=torch.float16),
        "tables": r.to(tables), "lens": r.to(lens), "positions": r.to(lens - 1),
        "cos": r.to(cos), "sin": r.to(sin),
        "ws": gpu.workspace(b, cfg.n_head, case["capacity"]),
        "x": torch.empty((b, d), **f), "qkv": torch.empty((b, d + 2 * kv), **f),
        "attn": torch.empty((b, d), **f), "act": torch.empty((b, hid), **f),
        "logits": torch.empty((b, VOCAB), **f),
        "tokens": torch.empty(b, dtype=torch.int32, device=r.dev),
    }

    def step():
        eps = float(np.float32(cfg.norm_eps))
        torch.index_select(s["emb"], 0, s["tokens_in"], out=s["x"])
        x = s["x"]
        for i, layer in enumerate(layers):
            nxt = layers[i + 1]["wqkv"] if i + 1 < n else None
            gpu.linear_f64acc(x, layer["wqkv"], s["qkv"], norm_w=layer["attn_norm"], eps=eps,
                              prefetch=layer["wo"])
            gpu.attention_decode_qkv_paged_append(
                s["qkv"], s["cos"], s["sin"], s["k_pool"], s["v_pool"], s["attn"], s["tables"],
                s["positions"], s["lens"], b, cfg.n_head, cfg.n_kv_head, 64, stride, n, i, kv,
                case["capacity"], workspace=s["ws"])
            gpu.linear_f64acc(s["attn"], layer["wo"], x, resid=x, prefetch=layer["wgu"])
            gpu.linear_swiglu_f64acc(x, layer["wgu"][:hid], layer["wgu"][hid:], s["act"],
                                     norm_w=layer["mlp_norm"], eps=eps, prefetch=layer["wd"])
            gpu.linear_f64acc(s["act"], layer["wd"], x, resid=x, prefetch=nxt)
        gpu.linear_f64acc(x, s["head"], s["logits"], norm_w=s["final_norm"], eps=eps)
        gpu.argmax_rows(s["logits"], s["tokens"], b, VOCAB)

    if graph:
        s["graph"] = _graph(step)
    return s


def _run_step(s):
    s["graph"].replay()
    return {k: s[k] for k in ("logits", "x", "k_pool", "v_pool")}


def _prompts(case, host):
    lens = host.integers(case["lo"], case["hi"] + 1, size=case["prompts"])
    return [host.integers(0, VOCAB, size=int(n)).tolist() for n in lens]


def _prepare_model(case, seed, graph=True):
    r, cfg = _Seeded(seed), _config(case)
    w = {k: v.cpu().numpy() for k, v in _weights(cfg, r).items()}
    return {"case": case, "prompts": _prompts(case, r.host),
            "model": GpuModel(cfg, w, max_batch=case["prompts"], capacity=1024)}


def _run_model(s):
    return {"logits": s["model"].prefill_logits(s["prompts"])}


_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "chunk": _prepare_chunk,
            "proj": _prepare_proj, "step": _prepare_step, "model": _prepare_model}
_RUN = {"decode": _run_decode, "prefill": _run_prefill, "chunk": _run_chunk, "proj": _run_proj,
        "step": _run_step, "model": _run_model}


def prepare(case, seed):
    return _PREPARE[case["op"]](case, seed)


def run(state):
    return _RUN[state["case"]["op"]](state)


# ------------------------------------------------------------------------------- necessary work

def _size(name):
    return 2 if name == "f16" else 4


def work(case):
    """Bytes (inputs read once, outputs written once) and floating-point operations."""
    op = case["op"]
    if op == "decode":
        b, hd, kv = case["batch"], case["head_dim"], case["n_kv"] * case["head_dim"]
        qd, mean = case["n_head"] * hd, (case["lo"] + case["hi"]) / 2
        rows = b * qd * ((4 if case["entry"] == "qkv" else _size(case["q"])) + _size(case["out"]))
        if case["entry"] != "decode":
            rows += b * 2 * kv * (4 + 2)
        return {"bytes": case["layers"] * (rows + b * mean * 2 * kv * 2),
                "flops": case["layers"] * 4.0 * qd * b * mean}
    if op == "prefill":
        lens, hd = _ints(case["lens"]).astype(float), case["head_dim"]
        qd, kv, rows = case["n_head"] * hd, case["n_kv"] * hd, lens.sum()
        return {"bytes": float(case["layers"] * rows * (qd * (_size(case["q"]) + 4) + 2 * kv * 2)),
                "flops": float(case["layers"] * 4.0 * qd * (lens * (lens + 1) / 2).sum())}
    if op == "chunk":
        a, n = _ints(case["starts"]).astype(float), _ints(case["lens"]).astype(float)
        qd, kv = case["n_head"] * 64, case["n_kv"] * 64
        pairs = (n * a + n * (n + 1) / 2).sum()
        return {"bytes": float(case["layers"] * (n.sum() * (qd * 8 + 2 * kv * 6)
                                                 + a.sum() * 2 * kv * 2)),
                "flops": float(case["layers"] * 4.0 * qd * pairs)}
    if op == "proj":
        rows, d, hid = case["rows"], case["n_embd"], case["hidden"]
        width = d + 2 * case["n_kv"] * (d // case["n_head"])
        weights = d * (width + d + 3 * hid)
        return {"bytes": 2.0 * weights + 4.0 * rows * (2 * d + width + 2 * d + hid),
                "flops": 2.0 * rows * weights}
    cfg = _config(case)
    d, kv = cfg.n_embd, cfg.kv_dim
    weights = cfg.n_layer * d * (2 * d + 2 * kv + 3 * cfg.hidden)
    if op == "step":
        b, mean = case["batch"], (case["lo"] + case["hi"]) / 2
        return {"bytes": 2.0 * (weights + VOCAB * d) + b * (cfg.n_layer * mean * 4 * kv
                                                            + 4 * VOCAB),
                "flops": 2.0 * b * (weights + VOCAB * d) + cfg.n_layer * 4.0 * d * b * mean}
    n, mean = case["prompts"], (case["lo"] + case["hi"]) / 2
    return {"bytes": 2.0 * (weights + VOCAB * d) + n * (mean * (4 * d + cfg.n_layer * 4 * kv)
                                                        + 4 * VOCAB),
            "flops": 2.0 * n * (mean * weights + VOCAB * d)
            + cfg.n_layer * 4.0 * d * n * mean * (mean + 1) / 2}


def tolerance(case):
    """Attention: f32 sums over fp16 products, the softmax weights carried to about 22 bits.
    Projections: one f32 rounding of a 64-bit sum. Whole decoder: those differences pass
    through every layer, and a K or V value between two fp16 numbers may round to either."""
    op = case["op"]
    if op == "decode":
        return {"rel": 1e-3 if case["out"] == "f16" else 2e-6}
    if op in ("prefill", "chunk"):
        return {"rel": 2e-6}
    if op == "proj":
        return {"rel": 4e-7}
    return {"rel": 1e-4}


# ------------------------------------------------------------------------------- 64-bit reference

def _history(s, pages, n, layer):
    """K and V rows [n][n_kv][hd] of a sequence in f64, from its page ids."""
    case = s["case"]
    layers, hd, n_kv = case["layers"], case.get("head_dim", 64), case.get("n_kv", 3)
    kv = n_kv * hd
    k = s["k_pool"].view(s["n_pages"], layers, PAGE, kv)[pages, layer]
    v = s["v_pool"].view(s["n_pages"], layers, kv, PAGE)[pages, layer].transpose(1, 2)
    return (k.reshape(-1, n_kv, hd)[:n].double(), v.reshape(-1, n_kv, hd)[:n].double())


def _store(s, table, position, layer, k, v):
    """One K and one V row into the pools as fp16."""
    layers, kv = s["case"]["layers"], k.numel()
    page, slot = int(table[position // PAGE]), position % PAGE
    s["k_pool"].view(s["n_pages"], layers, PAGE, kv)[page, layer, slot] = k.half()
    s["v_pool"].view(s["n_pages"], layers, kv, PAGE)[page, layer, :, slot] = v.half()


def _attend(q, k, v, first):
    """q [rows][heads][hd] at positions first, first + 1, ... over k, v [n][n_kv][hd]: f64."""
    rows, heads, hd = q.shape
    rep = heads // k.shape[1]
    out = torch.empty((rows, heads, hd), dtype=torch.float64, device=q.device)
    at = torch.arange(k.shape[0], device=q.device)
    for h in range(heads):
        kh, vh = k[:, h // rep].contiguous(), v[:, h // rep].contiguous()
        for r0 in range(0, rows, 2048):
            r1 = min(rows, r0 + 2048)
            sc = torch.mm(q[r0:r1, h].contiguous(), kh.t().contiguous()) / math.sqrt(hd)
            sc.masked_fill_(at[None, :] > (first + torch.arange(r0, r1, device=q.device))[:, None],
                            -math.inf)
            out[r0:r1, h] = torch.mm(torch.softmax(sc, dim=-1), vh)
    return out.reshape(rows, heads * hd)


def _rotate(x, cos, sin):
    """Half-split RoPE of x [..., hd] by rows cos, sin [..., hd / 2]."""
    half = x.shape[-1] // 2
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * cos - hi * sin, lo * sin + hi * cos], dim=-1)


def _exact_decode(case, seed):
    s = _prepare_decode(case, seed, graph=False)
    hd, n_head, n_kv = case["head_dim"], case["n_head"], case["n_kv"]
    kv, qd = n_kv * hd, n_head * hd
    tables = s["tables"].cpu().numpy()
    out = torch.zeros(s["out"].shape, dtype=torch.float64, device="cuda")
    for i in range(case["layers"]):
        for b, n in enumerate(int(x) for x in s["seq_lens"]):
            if case["entry"] == "qkv":
                row = s["qkv"][i, b].double()
                c, t = s["cos"][n - 1].double(), s["sin"][n - 1].double()
                q = _rotate(row[:qd].view(n_head, hd), c, t)
                _store(s, tables[b], n - 1, i,
                       _rotate(row[qd:qd + kv].view(n_kv, hd), c, t).reshape(-1), row[qd + kv:])
            else:
                q = s["q"][i, b].double().view(n_head, hd)
                if case["entry"] == "append":
                    _store(s, tables[b], n - 1, i, s["k_new"][i, b], s["v_new"][i, b])
            pages = s["tables"][b, :-(-n // PAGE)].long()
            k, v = _history(s, pages, n, i)
            rep = n_head // n_kv
            for g in range(n_kv):
                sc = torch.mm(q[g * rep:(g + 1) * rep], k[:, g].t().contiguous()) / math.sqrt(hd)
                o = torch.mm(torch.softmax(sc, -1), v[:, g].contiguous())
                out[i, b, g * rep * hd:(g + 1) * rep * hd] = o.reshape(-1)
    if case["entry"] == "decode":
        return {"out": out}
    return {"out": out, "k_pool": s["k_pool"], "v_pool": s["v_pool"]}


def _exact_prefill(case, seed):
    s = _prepare_prefill(case, seed, graph=False)
    hd = case["head_dim"]
    out = torch.zeros(s["out"].shape, dtype=torch.float64, device="cuda")
    for i in range(case["layers"]):
        at = 0
        for b, n in enumerate(int(x) for x in s["seq_lens"]):
            k, v = _history(s, s["tables"][b, :-(-n // PAGE)].long(), n, i)
            q = s["q"][i, at:at + n].double().view(n, case["n_head"], hd)
            out[i, at:at + n] = _attend(q, k, v, 0)
            at += n
    return {"out": out}


def _exact_chunk(case, seed):
    s = _prepare_chunk(case, seed)
    tables = s["tables"].cpu().numpy()
    kv, layers = case["n_kv"] * 64, case["layers"]
    out = torch.zeros(s["out"].shape, dtype=torch.float64, device="cuda")
    at = 0
    for b, (a, n) in enumerate(zip(map(int, s["starts"]), map(int, s["seq_lens"]))):
        where = np.arange(a, a + n)
        page = torch.from_numpy(tables[b, where // PAGE].astype(np.int64)).cuda()
        slot = torch.from_numpy((where % PAGE).astype(np.int64)).cuda()
        for i in range(layers):
            s["k_pool"].view(s["n_pages"], layers, PAGE, kv)[page, i, slot] = \
                s["k"][i, at:at + n].half()
            s["v_pool"].view(s["n_pages"], layers, kv, PAGE)[page, i, :, slot] = \
                s["v"][i, at:at + n].half()
            k, v = _history(s, s["tables"][b, :-(-(a + n) // PAGE)].long(), a + n, i)
            q = s["q"][i, at:at + n].double().view(n, case["n_head"], 64)
            out[i, at:at + n] = _attend(q, k, v, a)
        at += n
    return {"out": out, "k_pool": s["k_pool"], "v_pool": s["v_pool"]}


def _norm64(x, w, eps=float(np.float32(1e-6))):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _mul64(x, w):
    return torch.mm(x, w.double().t().contiguous())


def _swiglu64(x, wg, wu):
    g = _mul64(x, wg)
    return g / (1.0 + torch.exp(-g)) * _mul64(x, wu)


def _exact_proj(case, seed):
    s = _prepare_proj(case, seed, graph=False)
    x = s["x"].double()
    h = x + _mul64(s["attn"].double(), s["wo"])
    act = _swiglu64(_norm64(h, s["norm2"]), s["wg"], s["wu"])
    return {"qkv": _mul64(_norm64(x, s["norm1"]), s["wqkv"]), "h": h, "act": act,
            "y": h + _mul64(act, s["wd"])}


def _exact_step(case, seed):
    s = _prepare_step(case, seed, graph=False)
    cfg, hid = s["cfg"], s["cfg"].hidden
    d, kv = cfg.n_embd, cfg.kv_dim
    tables = s["tables"].cpu().numpy()
    x = s["emb"].double().index_select(0, s["tokens_in"])
    for i, layer in enumerate(s["layers"]):
        qkv = _mul64(_norm64(x, layer["attn_norm"]), layer["wqkv"])
        attn = torch.empty_like(x)
        for b, n in enumerate(int(v) for v in s["seq_lens"]):
            c, t = s["cos"][n - 1].double(), s["sin"][n - 1].double()
            q = _rotate(qkv[b, :d].view(1, cfg.n_head, 64), c, t)
            _store(s, tables[b], n - 1, i,
                   _rotate(qkv[b, d:d + kv].view(cfg.n_kv_head, 64), c, t).reshape(-1),
                   qkv[b, d + kv:])
            k, v = _history(s, s["tables"][b, :-(-n // PAGE)].long(), n, i)
            attn[b] = _attend(q, k, v, n - 1)
        x = x + _mul64(attn, layer["wo"])
        act = _swiglu64(_norm64(x, layer["mlp_norm"]), layer["wgu"][:hid], layer["wgu"][hid:])
        x = x + _mul64(act, layer["wd"])
    return {"logits": _mul64(_norm64(x, s["final_norm"]), s["head"]), "x": x,
            "k_pool": s["k_pool"], "v_pool": s["v_pool"]}


def _exact_model(case, seed):
    r, cfg = _Seeded(seed), _config(case)
    w = _weights(cfg, r)
    prompts = _prompts(case, r.host)
    d, kv = cfg.n_embd, cfg.kv_dim
    cos, sin = (r.to(t).double() for t in rope_tables(64, 1024, cfg.rope_theta))
    lens = [len(p) for p in prompts]
    pos = torch.cat([torch.arange(n, device=r.dev) for n in lens])
    c, t = cos[pos][:, None, :], sin[pos][:, None, :]
    x = w["tok_emb.weight"][torch.tensor(sum(prompts, []), device=r.dev)].double()
    for i in range(cfg.n_layer):
        p = f"blocks.{i}."
        h = _norm64(x, w[p + "attn_norm.weight"])
        q, k, v = (_mul64(h, w[p + f"attn.{a}_proj.weight"]) for a in "qkv")
        q = _rotate(q.view(-1, cfg.n_head, 64), c, t)
        k = _rotate(k.view(-1, cfg.n_kv_head, 64), c, t).half().double()
        v = v.view(-1, cfg.n_kv_head, 64).half().double()
        attn, at = torch.empty_like(x), 0
        for n in lens:
            attn[at:at + n] = _attend(q[at:at + n], k[at:at + n], v[at:at + n], 0)
            at += n
        x = x + _mul64(attn, w[p + "attn.o_proj.weight"])
        h = _norm64(x, w[p + "mlp_norm.weight"])
        act = _swiglu64(h, w[p + "mlp.gate_proj.weight"], w[p + "mlp.up_proj.weight"])
        x = x + _mul64(act, w[p + "mlp.down_proj.weight"])
    last = torch.tensor(np.cumsum(lens) - 1, device=r.dev)
    return {"logits": _mul64(_norm64(x[last], w["final_norm.weight"]), w["tok_emb.weight"])}


_EXACT = {"decode": _exact_decode, "prefill": _exact_prefill, "chunk": _exact_chunk,
          "proj": _exact_proj, "step": _exact_step, "model": _exact_model}


def exact(case, seed):
    return _EXACT[case["op"]](case, seed)
