"""The workloads whose time is tracked: each is a dict of plain values naming one use of the library
at one size, prepared once (inputs, weights, workspaces, a captured graph where a program would
keep one) and then run as a user's program calls it.

The kinds, and what each stands for in use:

* ``attend``: one decode attention call of the reference's own API (``flash_attn.attend``), eager,
  one f32 query row per head over f32 or f16 K/V with K transposed: a program that steps one
  sequence and lets the binding allocate. Key counts are whatever the sequence has, odd ones too.
* ``merged``: one encoder layer of the reference's own API (``flash_attn.attend_merged``), f32.
* ``encoder``: one encoder layer over a batch of windows through the general call, 16-bit, K
  transposed as the projections leave it; ``ragged`` windows end at their own lengths.
* ``block``: the encoder's attention block (projections, attention, out-projection), 16-bit.
* ``prefill``: a causal prompt with grouped K/V heads, 16-bit, K as rows.
* ``prompt``: a decoder's prompt step: every layer appends the prompt's rows to its cache,
  attends causally over it and then over the window's encoder frames; a captured graph.
* ``decode_attention``: the attention calls of one beam-search step, every layer: self-attention
  over ragged caches and cross-attention over frames the beams share; a captured graph.
* ``projections``: the single-row projections of one beam-search step, every layer, and the int8
  vocabulary logits; a captured graph.
* ``decode_step``: one whole beam-search step of a small decoder, from the reorder of the caches by
  parent beam to the logits; a captured graph.
* ``cross_build``: the cross-attention caches of every layer, once per window, eager.
"""

from __future__ import annotations

import math

import torch

from ffai_amd import flash_attn as fa
from ffai_amd.encoder import EncoderAttention
from ffai_amd.gemv import F16Gemv, Int8Vocab
from ffai_amd.kv_cache import KVCache, cross_kv_build, self_attention_step

HEAD_DIM = 64     # every whisper size
SCALE = 0.125     # HEAD_DIM ** -0.5
VOCAB = 51865     # the multilingual vocabulary
CAPACITY = 448    # a decoder cache's positions
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # a tiny decoder early in a sequence, stepped through the reference's call: the smallest
        # call there is, and an odd key count
        {"name": "attend_h6_k37", "kind": "attend", "heads": 6, "keys": 37, "kv": "f32"},
        # whisper-tiny's encoder layer as the reference runs it
        {"name": "merged_h6_t1500", "kind": "merged", "heads": 6, "frames": 1500},
        # a wider f32 layer over a window cut short at an odd frame
        {"name": "merged_h16_t1037", "kind": "merged", "heads": 16, "frames": 1037},
        # whisper-large-v3's attention block, one window: the latency of a single request
        {"name": "block_n1280_t1500", "kind": "block", "dtype": "bf16", "batch": 1,
         "frames": 1500, "heads": 20},
        # whisper-large-v3's encoder layer over 16 windows: throughput serving, the headline shape
        {"name": "encoder_b16_h20_t1500", "kind": "encoder", "dtype": "bf16", "batch": 16,
         "heads": 20, "frames": 1500, "ragged": False},
        # whisper-small's encoder layer over 8 windows of an odd length
        {"name": "encoder_b8_h12_t1037", "kind": "encoder", "dtype": "f16", "batch": 8,
         "heads": 12, "frames": 1037, "ragged": False},
        # the causal grouped-head prefill of a 4096-token prompt
        {"name": "prefill_d128_s4096", "kind": "prefill", "dtype": "bf16", "heads_q": 12,
         "heads_kv": 2, "head_dim": 128, "tokens": 4096, "past": 0},
        # whisper-medium's prompt step with the previous window's text, an odd token count
        {"name": "prompt_h16_p227", "kind": "prompt", "layers": 24, "heads": 16, "tokens": 227,
         "frames": 1500},
        # whisper-medium's beam-5 step, attention only
        {"name": "decode_attention_h16_b5", "kind": "decode_attention", "dtype": "bf16",
         "layers": 24, "beams": 5, "heads": 16, "frames": 1500, "longest": 448, "k_rows": True},
        # whisper-medium's beam-5 step, projections and logits only
        {"name": "projections_n1024_b5", "kind": "projections", "layers": 24, "beams": 5,
         "heads": 16},
        # whisper-small's whole beam-5 step
        {"name": "decode_step_n768_b5", "kind": "decode_step", "layers": 12, "beams": 5,
         "heads": 12, "frames": 1500, "longest": 448},
        # whisper-medium's cross-attention caches, once per window
        {"name": "cross_build_h16_t1500", "kind": "cross_build", "dtype": "bf16", "layers": 24,
         "heads": 16, "frames": 1500, "k_rows": True},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], its logarithm uniform."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_HEADS = (6, 8, 12, 16, 20)  # the whisper sizes' heads (widths 384 .. 1280)


def draw(rng):
    kind = rng.choice(("attend", "merged", "encoder", "block", "prefill", "prompt",
                       "decode_attention", "projections", "decode_step", "cross_build"))
    heads = rng.choice(_HEADS)
    if kind == "attend":
        return {"kind": kind, "heads": heads, "keys": _log(rng, 8, 1500),
                "kv": rng.choice(("f32", "f16"))}
    frames = rng.choice((1500, rng.randint(256, 1500), rng.randint(256, 1500)))
    if kind == "merged":
        return {"kind": kind, "heads": heads, "frames": rng.randint(256, 1500)}
    dtype = rng.choice(("bf16", "f16"))
    if kind == "encoder":
        return {"kind": kind, "dtype": dtype, "batch": _log(rng, 1, 16), "heads": heads,
                "frames": frames, "ragged": rng.random() < 0.3}
    if kind == "block":
        return {"kind": kind, "dtype": dtype, "batch": rng.randint(1, 4), "frames": frames,
                "heads": heads}
    if kind == "prefill":
        hkv = rng.choice((1, 2, 4))
        return {"kind": kind, "dtype": dtype, "heads_q": hkv * rng.choice((1, 3, 6)),
                "heads_kv": hkv, "head_dim": rng.choice((64, 128)),
                "tokens": _log(rng, 64, 3500), "past": rng.choice((0, 0, rng.randint(1, 400)))}
    if kind == "prompt":
        return {"kind": kind, "layers": rng.randint(4, 16), "heads": heads,
                "tokens": _log(rng, 3, 400), "frames": frames}
    beams = rng.randint(1, 10)
    if kind == "decode_attention":
        return {"kind": kind, "dtype": dtype, "layers": rng.randint(4, 16), "beams": beams,
                "heads": heads, "frames": frames, "longest": _log(rng, 4, 448),
                "k_rows": rng.random() < 0.5}
    if kind == "projections":
        return {"kind": kind, "layers": rng.randint(2, 12), "beams": beams, "heads": heads}
    if kind == "decode_step":
        return {"kind": kind, "layers": rng.randint(2, 6), "beams": beams, "heads": heads,
                "frames": frames, "longest": rng.randint(20, 448)}
    return {"kind": kind, "dtype": dtype, "layers": rng.randint(4, 16), "heads": heads,
            "frames": frames, "k_rows": rng.random() < 0.5}


# ------------------------------------------------------------------------------------------
# Inputs: what exists before a call, made on the GPU from the seed alone. Queries, keys and values
# are N(0, 1) per element, so that scaled scores are N(0, 1) too.
# ------------------------------------------------------------------------------------------

def _rand(gen):
    dev = torch.device("cuda:0")

    def make(*shape, dtype=torch.float32, std=1.0):
        x = torch.randn(*shape, generator=gen, device=dev)
        return (x * std if std != 1.0 else x).to(dtype)
    return make


def _lens(gen, n, longest):
    """n sequence lengths in [1, longest]: beams of one search differ little, so most are close to
    the longest."""
    u = torch.rand(n, generator=gen, device="cuda:0")
    return (longest - (u * u * (longest - 1)).floor()).to(torch.int32)


def _inputs(case, seed):
    gen = torch.Generator(device="cuda:0").manual_seed(int(seed))
    r = _rand(gen)
    kind, d = case["kind"], HEAD_DIM
    if kind == "attend":
        h, k = case["heads"], case["keys"]
        kv = DT[case["kv"]]
        return {"q": r(1, h, 1, d, std=SCALE), "kt": r(1, h, d, k, dtype=kv),
                "v": r(1, h, k, d, dtype=kv)}
    if kind == "merged":
        h, t = case["heads"], case["frames"]
        return {"q": r(1, h, t, d, std=SCALE), "kt": r(1, h, d, t), "v": r(1, h, t, d)}
    if kind == "encoder":
        b, h, t, dt = case["batch"], case["heads"], case["frames"], DT[case["dtype"]]
        s = {"q": r(b, h, t, d, dtype=dt), "kt": r(b, h, d, t, dtype=dt),
             "v": r(b, h, t, d, dtype=dt), "lens": None}
        if case["ragged"]:
            u = torch.rand(b, generator=gen, device="cuda:0")
            s["lens"] = (t * (0.25 + 0.75 * u)).ceil().to(torch.int32)
        return s
    if kind == "block":
        n, dt = case["heads"] * d, DT[case["dtype"]]
        w = {k: r(n, n, dtype=dt, std=n ** -0.5) for k in ("wq", "wk", "wv", "wo")}
        w.update({k: r(n, dtype=dt, std=0.1) for k in ("bq", "bv", "bo")})
        # activations behind a layer norm; queries and keys a few times wider, so that the
        # attention weights are not uniform
        w["wq"] *= 2
        return {"w": w, "x": r(case["batch"], case["frames"], n, dtype=dt)}
    if kind == "prefill":
        hq, hkv, hd, s = case["heads_q"], case["heads_kv"], case["head_dim"], case["tokens"]
        dt, keys = DT[case["dtype"]], case["tokens"] + case["past"]
        return {"q": r(1, hq, s, hd, dtype=dt), "k": r(1, hkv, keys, hd, dtype=dt),
                "v": r(1, hkv, keys, hd, dtype=dt)}
    if kind == "prompt":
        l, h, p, t = case["layers"], case["heads"], case["tokens"], case["frames"]
        bf = torch.bfloat16
        return {"q": r(l, 1, h, p, d, dtype=bf), "k_new": r(l, 1, p, h * d),
                "v_new": r(l, 1, p, h * d), "qx": r(l, 1, h, p, d, dtype=bf),
                "kx": r(l, 1, h, t, d, dtype=bf), "vx": r(l, 1, h, t, d, dtype=bf)}
    if kind == "decode_attention":
        l, b, h, t = case["layers"], case["beams"], case["heads"], case["frames"]
        dt = DT[case["dtype"]]
        kx = (l, 1, h, t, d) if case["k_rows"] else (l, 1, h, d, t)
        return {"q": r(l, b, h, 1, d, dtype=dt), "k": r(l, b, h, CAPACITY, d, dtype=dt),
                "v": r(l, b, h, CAPACITY, d, dtype=dt), "lens": _lens(gen, b, case["longest"]),
                "qx": r(l, 1, h, b, d, dtype=dt), "kx": r(*kx, dtype=dt),
                "vx": r(l, 1, h, t, d, dtype=dt)}
    if kind == "projections":
        l, b, n = case["layers"], case["beams"], case["heads"] * d
        f16 = torch.float16
        shapes = _projection_shapes(n)
        return {"w": [[r(o, i, dtype=f16, std=i ** -0.5) for o, i in shapes] for _ in range(l)],
                "x": {n: r(b, n), 4 * n: r(b, 4 * n)},
                "emb": r(VOCAB, n, std=n ** -0.5)}
    if kind == "decode_step":
        l, b, h, t = case["layers"], case["beams"], case["heads"], case["frames"]
        n, f16, bf = h * d, torch.float16, torch.bfloat16
        shapes = _projection_shapes(n)
        return {"w": [[r(o, i, dtype=f16, std=i ** -0.5) for o, i in shapes] for _ in range(l)],
                "bias": [r(3 * n, std=0.1) for _ in range(l)],
                "emb": r(VOCAB, n, std=n ** -0.5), "x": r(b, n),
                "k": r(l, b, h, CAPACITY, d, dtype=bf), "v": r(l, b, h, CAPACITY, d, dtype=bf),
                # the step appends one row to every beam
                "lens": _lens(gen, b, max(1, case["longest"] - 1)),
                "parent": torch.randint(0, b, (b,), generator=gen, device="cuda:0",
                                        dtype=torch.int32),
                "kx": r(l, 1, h, t, d, dtype=bf), "vx": r(l, 1, h, t, d, dtype=bf)}
    if kind == "cross_build":
        l, t, n = case["layers"], case["frames"], case["heads"] * d
        return {"k": r(l, t, n), "v": r(l, t, n)}
    raise ValueError(kind)


def _projection_shapes(n):
    """(out, in) of one decoder layer: packed q/k/v, self-attention out, cross-attention q and
    out, and the MLP."""
    return [(3 * n, n), (n, n), (n, n), (n, n), (4 * n, n), (n, 4 * n)]


# ------------------------------------------------------------------------------------------
# prepare and run
# ------------------------------------------------------------------------------------------

def _captured(step):
    """`step` as a graph to replay, as a decode loop keeps one (after one eager pass)."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


def _zeroed(nbytes):
    return torch.zeros(max(1, nbytes), dtype=torch.uint8, device="cuda:0")


def prepare(case, seed):
    s = _inputs(case, seed)
    kind, d, dev = case["kind"], HEAD_DIM, torch.device("cuda:0")
    s["kind"] = kind
    if kind == "encoder":
        s["out"] = torch.empty_like(s["q"])
        s["ws"] = _zeroed(fa.workspace_bytes(s["q"], s["kt"], s["v"], s["out"], k_transposed=True,
                                             scale=SCALE, kv_lens=s["lens"]))
    elif kind == "block":
        n = case["heads"] * d
        s["block"] = EncoderAttention.load(n, case["heads"], **s.pop("w"))
        s["out"] = torch.empty_like(s["x"])
    elif kind == "prefill":
        s["out"], s["past"] = torch.empty_like(s["q"]), case["past"]
        s["scale"] = case["head_dim"] ** -0.5
        s["ws"] = _zeroed(fa.workspace_bytes(s["q"], s["k"], s["v"], s["out"], scale=s["scale"],
                                             causal=True, q_offset=s["past"]))
    elif kind == "prompt":
        l, h, p = case["layers"], case["heads"], case["tokens"]
        cache = KVCache(1, h, CAPACITY, d, torch.bfloat16, dev, layers=l)
        o = torch.empty(l, 1, h, p, d, device=dev)
        ox = torch.empty_like(o)
        ws = _zeroed(max(
            fa.workspace_bytes(s["q"][0], cache.k[0], cache.v[0], o[0], scale=SCALE,
                               kv_lens=cache.lens[0], causal=p > 1),
            fa.workspace_bytes(s["qx"][0], s["kx"][0], s["vx"][0], ox[0], scale=SCALE)))

        def step():
            cache.lens.zero_()  # a new window: the cache starts empty
            for i in range(l):
                self_attention_step(cache.layer(i), s["q"][i], s["k_new"][i], s["v_new"][i], 0,
                                    SCALE, out=o[i], workspace=ws)
                fa.attention(s["qx"][i], s["kx"][i], s["vx"][i], scale=SCALE, out=ox[i],
                             workspace=ws)
        s["graph"] = _captured(step)
        s["keep"] = ws
        s["result"] = {"self": o, "cross": ox, "k": cache.k, "v": cache.v, "lens": cache.lens}
    elif kind == "decode_attention":
        l, kt = case["layers"], not case["k_rows"]
        o = torch.empty(s["q"].shape, device=dev)
        ox = torch.empty(s["qx"].shape, device=dev)
        ws = _zeroed(max(
            fa.workspace_bytes(s["q"][0], s["k"][0], s["v"][0], o[0], scale=SCALE,
                               kv_lens=s["lens"]),
            fa.workspace_bytes(s["qx"][0], s["kx"][0], s["vx"][0], ox[0], scale=SCALE,
                               k_transposed=kt)))

        def step():
            for i in range(l):
                fa.attention(s["q"][i], s["k"][i], s["v"][i], scale=SCALE, kv_lens=s["lens"],
                             out=o[i], workspace=ws)
                fa.attention(s["qx"][i], s["kx"][i], s["vx"][i], scale=SCALE, k_transposed=kt,
                             out=ox[i], workspace=ws)
        s["graph"] = _captured(step)
        s["keep"] = ws
        s["result"] = {"self": o, "cross": ox}
    elif kind == "projections":
        b, l, n = case["beams"], case["layers"], case["heads"] * d
        mats = [[F16Gemv(w) for w in layer] for layer in s.pop("w")]
        vocab = Int8Vocab(s.pop("emb"))
        ys = [torch.empty(l, b, o, device=dev) for o, _ in _projection_shapes(n)]
        logits = torch.empty(b, VOCAB, device=dev)
        ws = torch.empty(vocab.workspace_bytes(b), dtype=torch.uint8, device=dev)

        def step():
            for i, layer in enumerate(mats):
                for m, y in zip(layer, ys):
                    m(s["x"][m.in_dim], out=y[i])
            vocab(s["x"][n], out=logits, workspace=ws)
        s["graph"] = _captured(step)
        s["keep"] = (mats, vocab, ws)
        s["result"] = {"y": ys, "logits": logits}
    elif kind == "decode_step":
        s["graph"], s["keep"], s["result"] = _decode_step(case, s)
    elif kind == "cross_build":
        l, h, t = case["layers"], case["heads"], case["frames"]
        s["dt"], s["heads"], s["k_rows"] = DT[case["dtype"]], h, case["k_rows"]
        s["kx"] = torch.empty((l, h, t, d) if s["k_rows"] else (l, h, d, t), dtype=s["dt"],
                              device=dev)
        s["vx"] = torch.empty(l, h, t, d, dtype=s["dt"], device=dev)
    return s


def _decode_step(case, s):
    """One beam-search step: the caches reordered by parent beam into the other stack, one row
    opened in every layer, the layers, the logits. The source stack is not written, so that every
    replay is the same step."""
    l, b, h, d, dev = case["layers"], case["beams"], case["heads"], HEAD_DIM, torch.device("cuda:0")
    n, bf = h * d, torch.bfloat16
    mats = [[F16Gemv(w) for w in layer] for layer in s.pop("w")]
    vocab = Int8Vocab(s.pop("emb"))
    src = KVCache(b, h, CAPACITY, d, bf, dev, layers=l)
    src.k.copy_(s.pop("k"))
    src.v.copy_(s.pop("v"))
    src.lens.copy_(s["lens"].expand(l, b))
    dst = KVCache(b, h, CAPACITY, d, bf, dev, layers=l)
    logits = torch.empty(b, VOCAB, device=dev)
    vws = torch.empty(vocab.workspace_bytes(b), dtype=torch.uint8, device=dev)
    q = torch.empty(b, n, device=dev)
    o = torch.empty(b, h, 1, d, device=dev)
    ox = torch.empty(b, h, 1, d, device=dev).permute(2, 1, 0, 3)  # (1, h, b, d) over the beams' rows
    qb = torch.empty(b, h, 1, d, dtype=bf, device=dev)
    ws = _zeroed(max(
        fa.workspace_bytes(qb, dst.k[0], dst.v[0], o, scale=SCALE, kv_lens=dst.lens[0]),
        fa.workspace_bytes(qb.permute(2, 1, 0, 3), s["kx"][0], s["vx"][0], ox, scale=SCALE)))
    norm = lambda x: torch.nn.functional.layer_norm(x, (n,))  # noqa: E731

    def step():
        x = s["x"]
        dst.gather_from(src, s["parent"])
        dst.advance()
        for i in range(l):
            qkv, out, xq, xout, up, down = mats[i]
            cache = dst.layer(i)
            qkv.qkv_into_cache(norm(x), q, cache, s["bias"][i])
            fa.attention(q.to(bf).view(b, h, 1, d), cache.k, cache.v, scale=SCALE,
                         kv_lens=cache.lens, out=o, workspace=ws)
            x = x + out(o.view(b, n))
            qx = xq(norm(x)).to(bf).view(b, h, 1, d)
            fa.attention(qx.permute(2, 1, 0, 3), s["kx"][i], s["vx"][i], scale=SCALE, out=ox,
                         workspace=ws)
            x = x + xout(ox.permute(2, 1, 0, 3).reshape(b, n))
            x = x + down(torch.nn.functional.gelu(up(norm(x))))
        vocab(norm(x), out=logits, workspace=vws)
    graph = _captured(step)
    return (graph, (mats, vocab, src, dst, ws, vws, q, o, ox, qb),
            {"logits": logits, "k": dst.k, "v": dst.v, "lens": dst.lens})


def run(s):
    kind = s["kind"]
    if kind == "attend":
        return fa.attend(s["q"], s["kt"], s["v"])
    if kind == "merged":
        return fa.attend_merged(s["q"], s["kt"], s["v"])
    if kind == "encoder":
        return fa.attention(s["q"], s["kt"], s["v"], k_transposed=True, scale=SCALE,
                            kv_lens=s["lens"], out=s["out"], workspace=s["ws"])
    if kind == "block":
        return s["block"](s["x"], out=s["out"])
    if kind == "prefill":
        return fa.attention(s["q"], s["k"], s["v"], scale=s["scale"], causal=True,
                            q_offset=s["past"], out=s["out"], workspace=s["ws"])
    if kind == "cross_build":
        for i in range(s["k"].shape[0]):
            cross_kv_build(s["k"][i], s["v"][i], s["heads"], s["dt"], not s["k_rows"],
                           out=(s["kx"][i], s["vx"][i]))
        return {"k": s["kx"], "v": s["vx"]}
    s["graph"].replay()
    return s["result"]


# ------------------------------------------------------------------------------------------
# What a pass cannot do without: each input read once, each output written once.
# ------------------------------------------------------------------------------------------

def work(case):
    kind, d = case["kind"], HEAD_DIM
    es = {"f32": 4, "f16": 2, "bf16": 2}
    h = case.get("heads", 0)
    if kind == "attend":
        k = case["keys"]
        return {"bytes": h * d * (2 * k * es[case["kv"]] + 8), "flops": 4 * h * k * d}
    if kind == "merged":
        t = case["frames"]
        return {"bytes": h * t * d * 16, "flops": 4 * h * t * t * d}
    if kind == "encoder":
        b, t = case["batch"], case["frames"]
        share = 0.625 if case["ragged"] else 1.0  # mean length of the ragged windows
        return {"bytes": int(b * h * t * d * 2 * (2 + 2 * share)),
                "flops": int(4 * b * h * t * t * d * share)}
    if kind == "block":
        b, t, n = case["batch"], case["frames"], h * d
        return {"bytes": 2 * (2 * b * t * n + 4 * n * n + 4 * n),
                "flops": b * (8 * t * n * n + 4 * t * t * n)}
    if kind == "prefill":
        hq, hkv, hd, s, past = (case[k] for k in ("heads_q", "heads_kv", "head_dim", "tokens",
                                                  "past"))
        return {"bytes": 2 * hd * (2 * hq * s + 2 * hkv * (s + past)),
                "flops": 4 * hd * hq * (s * (s + 1) // 2 + s * past)}
    if kind == "prompt":
        l, p, t = case["layers"], case["tokens"], case["frames"]
        row = h * d
        return {"bytes": l * row * (2 * p * (4 + 2) + 2 * p * (2 + 4) + 2 * t * 2),
                "flops": l * 4 * row * (p * (p + 1) // 2 + p * t)}
    if kind == "decode_attention":
        l, b, t = case["layers"], case["beams"], case["frames"]
        keys = b * (1 + case["longest"] * 2) // 3  # mean of the lengths' distribution
        return {"bytes": l * h * d * (2 * 2 * (t + keys) + 2 * b * (2 + 4)),
                "flops": l * 4 * h * d * (b * t + keys)}
    if kind in ("projections", "decode_step"):
        l, b, n = case["layers"], case["beams"], h * d
        macs = l * sum(o * i for o, i in _projection_shapes(n))
        rows = l * sum(o + i for o, i in _projection_shapes(n))
        w = {"bytes": 2 * macs + VOCAB * (n + n // 8 + 4) + 4 * b * (rows + n + VOCAB),
             "flops": 2 * b * (macs + VOCAB * n)}
        if kind == "decode_step":
            t, keys = case["frames"], b * (1 + case["longest"] * 2) // 3
            # caches read and written by the reorder, read once by the attention
            w["bytes"] += l * n * 2 * 2 * (t + 3 * keys)
            w["flops"] += l * 4 * n * (b * t + keys)
        return w
    if kind == "cross_build":
        return {"bytes": case["layers"] * 2 * case["frames"] * h * d * (4 + 2), "flops": 0}
    raise ValueError(kind)


def tolerance(case):
    kind = case["kind"]
    if kind == "cross_build":
        return "exact"  # a conversion and a layout
    if kind in ("attend", "merged"):
        return {"rel": 2e-6, "max": 2e-5}  # 32-bit sums
    if kind == "projections":
        return {"rel": 2e-6, "max": 4e-5}  # 32-bit sums; the logits' integer sums are exact
    if kind == "decode_step":
        # 16-bit queries and caches in every layer, and an int8 rounding before the logits: 4.9e-3
        # off the 64-bit result
        return {"rel": 2e-2, "max": 0.2}
    # 16-bit softmax weights, and outputs where they are 16-bit: up to 2.9e-3 off the 64-bit result
    # in bf16 (4.7e-3 through the block's projections), up to 6.2e-4 in f16
    if case.get("dtype") == "f16":
        return {"rel": 2.5e-3, "max": 0.025}
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------------------------------
# The same results in 64 bits, in plain torch.
# ------------------------------------------------------------------------------------------

def _softmax_attention(q, k, v, scale, hidden=None):
    """q (..., m, d), k and v (..., keys, d), all float64; `hidden`: a mask (m, keys) or None."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if hidden is not None:
        s.masked_fill_(hidden, float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v)


def _causal(m, keys, past):
    i = torch.arange(m, device="cuda:0")[:, None]
    return torch.arange(keys, device="cuda:0")[None, :] > i + past


def _half_away(x):
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _int8_logits(emb, x, blk=32):
    """Block-scaled int8 weights and 7-bit activations, as the vocabulary projection defines them,
    with every sum in 64 bits."""
    v, n = emb.shape
    w = emb.double().view(v, n // blk, blk)
    scale = w.abs().amax(-1, keepdim=True) / 127
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    wq = (_half_away(w / scale).clamp(-127, 127) * scale).view(v, n)
    sx = x.abs().amax(-1, keepdim=True) / 63
    sx = torch.where(sx == 0, torch.ones_like(sx), sx)
    return torch.matmul(_half_away(x / sx).clamp(-64, 63), wq.t().contiguous()) * sx


def exact(case, seed):
    s = _inputs(case, seed)
    kind, d = case["kind"], HEAD_DIM
    f8 = torch.float64
    if kind in ("attend", "merged"):
        o = _softmax_attention(s["q"].to(f8), s["kt"].to(f8).transpose(2, 3), s["v"].to(f8), 1.0)
        return o if kind == "attend" else o.transpose(1, 2).reshape(1, o.shape[2], -1)
    if kind == "encoder":
        o = torch.empty(s["q"].shape, dtype=f8, device="cuda:0")
        for b in range(o.shape[0]):
            end = None if s["lens"] is None else int(s["lens"][b])
            o[b] = _softmax_attention(s["q"][b].to(f8), s["kt"][b, :, :, :end].to(f8).transpose(1, 2),
                                      s["v"][b, :, :end].to(f8), SCALE)
        return o
    if kind == "block":
        h = case["heads"]
        w = {k: t.to(f8) for k, t in s["w"].items()}
        x = s["x"].to(f8)
        split = lambda t: t.reshape(x.shape[0], x.shape[1], h, d).transpose(1, 2)  # noqa: E731
        lin = lambda t, m, b: torch.matmul(t, m.t().contiguous()) + b  # noqa: E731
        o = _softmax_attention(split(lin(x, w["wq"], w["bq"])), split(lin(x, w["wk"], 0.0)),
                               split(lin(x, w["wv"], w["bv"])), SCALE)
        return lin(o.transpose(1, 2).reshape(x.shape), w["wo"], w["bo"])
    if kind == "prefill":
        hq, hkv = case["heads_q"], case["heads_kv"]
        q = s["q"][0].to(f8).view(hkv, hq // hkv, case["tokens"], -1)
        hidden = _causal(case["tokens"], s["k"].shape[2], case["past"])
        o = torch.stack([_softmax_attention(q[j], s["k"][0, j].to(f8), s["v"][0, j].to(f8),
                                            case["head_dim"] ** -0.5, hidden)
                         for j in range(hkv)])
        return o.reshape(s["q"].shape)
    if kind == "prompt":
        l, h, p = case["layers"], case["heads"], case["tokens"]
        bf = torch.bfloat16
        heads = lambda t: t.to(bf).view(l, 1, p, h, d).transpose(2, 3)  # noqa: E731
        k, v = heads(s["k_new"]), heads(s["v_new"])
        hidden = _causal(p, p, 0)
        one = lambda q, k, v, m: _softmax_attention(q.to(f8), k.to(f8), v.to(f8), SCALE, m)  # noqa: E731
        out = {"self": torch.stack([one(s["q"][i], k[i], v[i], hidden) for i in range(l)]),
               "cross": torch.stack([one(s["qx"][i], s["kx"][i], s["vx"][i], None)
                                     for i in range(l)])}
        for name, t in (("k", k), ("v", v)):
            full = torch.zeros(l, 1, h, CAPACITY, d, dtype=f8, device="cuda:0")
            full[:, :, :, :p] = t
            out[name] = full
        return {**out, "lens": None}
    if kind == "decode_attention":
        l, b = case["layers"], case["beams"]
        o = torch.empty(s["q"].shape, dtype=f8, device="cuda:0")
        ox = torch.empty(s["qx"].shape, dtype=f8, device="cuda:0")
        for i in range(l):
            for j in range(b):
                n = int(s["lens"][j])
                o[i, j] = _softmax_attention(s["q"][i, j].to(f8), s["k"][i, j, :, :n].to(f8),
                                             s["v"][i, j, :, :n].to(f8), SCALE)
            kx = s["kx"][i].to(f8)
            ox[i] = _softmax_attention(s["qx"][i].to(f8), kx if case["k_rows"] else
                                       kx.transpose(2, 3), s["vx"][i].to(f8), SCALE)
        return {"self": o, "cross": ox}
    if kind == "projections":
        shapes = _projection_shapes(case["heads"] * d)
        ys = [torch.stack([torch.matmul(s["x"][i].to(f8), layer[j].to(f8).t().contiguous())
                           for layer in s["w"]]) for j, (_, i) in enumerate(shapes)]
        return {"y": ys, "logits": _int8_logits(s["emb"], s["x"][case["heads"] * d].to(f8))}
    if kind == "decode_step":
        return _exact_step(case, s)
    if kind == "cross_build":
        l, t, h, dt = case["layers"], case["frames"], case["heads"], DT[case["dtype"]]
        heads = lambda x: x.to(dt).to(f8).view(l, t, h, d).transpose(1, 2)  # noqa: E731
        k = heads(s["k"])
        return {"k": k if case["k_rows"] else k.transpose(2, 3), "v": heads(s["v"])}
    raise ValueError(kind)


def _exact_step(case, s):
    l, b, h, d, f8 = case["layers"], case["beams"], case["heads"], HEAD_DIM, torch.float64
    n, bf = h * d, torch.bfloat16
    norm = lambda x: torch.nn.functional.layer_norm(x, (n,))  # noqa: E731
    lin = lambda x, w: torch.matmul(x, w.to(f8).t().contiguous())  # noqa: E731
    x = s["x"].to(f8)
    ck = torch.zeros(l, b, h, CAPACITY, d, dtype=f8, device="cuda:0")
    cv = torch.zeros_like(ck)
    for i in range(l):
        wqkv, out, xq, xout, up, down = s["w"][i]
        q, k, v = (lin(norm(x), wqkv) + s["bias"][i].to(f8)).view(b, 3, h, 1, d).unbind(1)
        o = torch.empty(b, h, 1, d, dtype=f8, device="cuda:0")
        for j in range(b):
            p = int(s["parent"][j])
            m = int(s["lens"][p])
            for cache, old, new in ((ck, s["k"], k), (cv, s["v"], v)):
                cache[i, j, :, :m] = old[i, p, :, :m]
                cache[i, j, :, m] = new[j, :, 0].to(bf)
            o[j] = _softmax_attention(q[j], ck[i, j, :, :m + 1], cv[i, j, :, :m + 1], SCALE)
        x = x + lin(o.view(b, n), out)
        qx = lin(norm(x), xq).view(b, h, d).transpose(0, 1)
        ox = _softmax_attention(qx, s["kx"][i, 0].to(f8), s["vx"][i, 0].to(f8), SCALE)
        x = x + lin(ox.transpose(0, 1).reshape(b, n), xout)
        x = x + lin(torch.nn.functional.gelu(lin(norm(x), up)), down)
    return {"logits": _int8_logits(s["emb"], norm(x)), "k": ck, "v": cv, "lens": None}
