"""The work that a program hands to this backend, as cases to time: single quantized products, the layer pieces of a
Qwen3.5-style hybrid decoder (FFN block, Gated DeltaNet layer, attention over a long cache, a batched projection) and
whole calls of the model driver (greedy decode, prompt processing, several sequences in lockstep), in the weight
formats and both arithmetics that the package offers. Sizes are those of the benchmark configurations (README.md,
bench.py), with whole models cut to 4 of 32 layers and an eighth of the vocabulary, so that every part keeps its share.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, weights, captured lists
    run(state)          one pass; its outputs
    work(case)          bytes and operations that a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the outputs in 64 bits, where they are a function of a few products
"""
from __future__ import annotations

import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "fpga-llama-gguf_amd"))

import gemvq as gq  # noqa: E402
import qwen35 as q35  # noqa: E402

TYPES = {"q4_0": gq.Q4_0, "q4_1": gq.Q4_1, "q8_0": gq.Q8_0, "q5_K": gq.Q5_K, "q6_K": gq.Q6_K}
S = 128  # DeltaNet head size
N_ROT, ROPE_BASE = 64, 1e7
EPS = 1e-6


def listed() -> list[dict]:
    return [
        # the smallest call: one product of a list run now, its input written and its output read (a ggml split)
        {"name": "gemv q4_0 9728x2560", "kind": "gemv", "fmt": "q4_0", "rows": 9728, "cols": 2560},
        # an output head: the largest single product of a token
        {"name": "head q6_K 151936x4096", "kind": "gemv", "fmt": "q6_K", "rows": 151936, "cols": 4096},
        # four feed-forward blocks of a Q8_0 model in one captured list (norm, gate/up, SwiGLU, down, residual)
        {"name": "ffn q8_0 2560-9728 x4", "kind": "ffn", "fmt": "q8_0", "embd": 2560, "ff": 9728, "layers": 4},
        # the recurrent half of eight DeltaNet layers: conv, step, gated norm, output projection
        {"name": "deltanet q4_0 x8", "kind": "gdn", "fmt": "q4_0", "hk": 16, "hv": 32, "layers": 8},
        # one token's attention at the end of a long cache
        {"name": "attention at 8191", "kind": "attn", "heads": 16, "kv_heads": 4, "dim": 256, "pos": 8191, "tokens": 1},
        # a projection pair over the rows of 16 tokens (prompt chunks, several sequences)
        {"name": "gate/up q4_0 16 tokens", "kind": "gemm", "fmt": "q4_0", "rows": 12288, "cols": 4096, "tokens": 16},
        # ordinary greedy decode of one sequence
        {"name": "decode q4_0", "kind": "decode", "fmt": "q4_0", "prompt": 16, "steps": 64, "reference": False},
        # the same in the arithmetic of the reference's CPU path (checking a build against it)
        {"name": "decode q4_0 reference", "kind": "decode", "fmt": "q4_0", "prompt": 16, "steps": 32,
         "reference": True},
        # an ordinary prompt up to its first generated token
        {"name": "prompt 512 q4_0", "kind": "prompt", "fmt": "q4_0", "prompt": 512},
        # a long prompt of ragged length, Q8_0 layers
        {"name": "prompt 1983 q8_0", "kind": "prompt", "fmt": "q8_0", "prompt": 1983},
        # a few and many sequences decoded in lockstep
        {"name": "lockstep 4 q4_0", "kind": "batch", "fmt": "q4_0", "seqs": 4, "steps": 32},
        {"name": "lockstep 32 q4_0", "kind": "batch", "fmt": "q4_0", "seqs": 32, "steps": 32},
    ]


def _spread(rng, lo: int, hi: int) -> int:
    """A whole number whose logarithm is spread evenly over lo..hi."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng) -> dict:
    kind = rng.choice(["gemv", "ffn", "gdn", "attn", "gemm", "decode", "prompt", "batch"])
    if kind == "gemv":
        fmt = rng.choice(list(TYPES))
        step = 256 if fmt.endswith("_K") else 32
        return {"kind": kind, "fmt": fmt, "rows": _spread(rng, 512, 40000), "cols": _spread(rng, 1024, 12288) // step * step}
    if kind == "ffn":
        return {"kind": kind, "fmt": rng.choice(["q4_0", "q8_0"]), "embd": _spread(rng, 1024, 4096) // 256 * 256,
                "ff": _spread(rng, 2048, 12288) // 256 * 256, "layers": rng.randint(1, 4)}
    if kind == "gdn":
        hk = rng.choice([2, 4, 8, 16])
        return {"kind": kind, "fmt": rng.choice(["q4_0", "q8_0"]), "hk": hk, "hv": 2 * hk, "layers": rng.randint(1, 8)}
    if kind == "attn":
        heads, kv_heads, dim = rng.choice([(16, 4, 256), (8, 2, 256), (16, 4, 128)])
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "dim": dim, "pos": _spread(rng, 32, 8191),
                "tokens": rng.choice([1, 1, 1, rng.randint(2, 32)])}
    if kind == "gemm":
        return {"kind": kind, "fmt": rng.choice(["q4_0", "q4_1", "q8_0"]), "rows": _spread(rng, 512, 12288),
                "cols": 512 * rng.randint(2, 24), "tokens": rng.randint(2, 32)}
    if kind == "decode":
        return {"kind": kind, "fmt": rng.choice(["q4_0", "q8_0", "q4_1"]), "prompt": _spread(rng, 1, 64),
                "steps": _spread(rng, 8, 64), "reference": rng.random() < 0.25}
    if kind == "prompt":
        return {"kind": kind, "fmt": rng.choice(["q4_0", "q8_0", "q4_1"]), "prompt": _spread(rng, 18, 1983)}
    return {"kind": kind, "fmt": rng.choice(["q4_0", "q8_0", "q4_1"]), "seqs": rng.randint(2, 32),
            "steps": _spread(rng, 8, 32)}


# ---- inputs ---------------------------------------------------------------------------------------------------
def _weights(fmt: int, rows: int, cols: int, seed: int, stream: int) -> np.ndarray:
    """N(0, 0.02^2) quantized, as GGUF bytes; past 512 rows the first 512 come again (their bytes are what is read)."""
    pool = gq.matrix(fmt, min(rows, 512), cols, seed, stream, std=0.02)
    return np.resize(pool, rows * gq.row_bytes(fmt, cols))


def _config(case: dict, n_ctx: int) -> q35.Config:
    return q35.Config(n_layer=4, n_vocab=18992, n_ctx=n_ctx, wtype=TYPES[case["fmt"]])


def _blob(cfg: q35.Config, seed: int) -> q35.Blob:
    """A model's tensors from the seed, matrices as _weights gives them (a row pool per type and width, every matrix
    from a row of its own on)."""
    specs = q35.tensor_specs(cfg)
    table, off = (q35.TensorDesc * len(specs))(), 0
    for i, (name, t, ne0, ne1, _) in enumerate(specs):
        nb = q35.tensor_bytes(t, ne0, ne1)
        table[i] = q35.TensorDesc(name.encode(), t, ne0, ne1, 0, off, nb)
        off += (nb + 255) // 256 * 256
    data = np.zeros(off, np.uint8)
    pools: dict[tuple[int, int], np.ndarray] = {}
    for i, (name, t, ne0, ne1, init) in enumerate(specs):
        view = data[table[i].offset:table[i].offset + table[i].nbytes]
        if t == q35.F32:
            v = {"ones": np.ones, "zeros": np.zeros, "neg1": lambda n, d: -np.ones(n, d)}.get(init)
            view[:] = (v(ne0 * ne1, np.float32) if v else gq.normal(seed, 1000 + i, ne0 * ne1, 0.0, 0.5)).view(np.uint8)
            continue
        if (t, ne0) not in pools:
            pools[t, ne0] = gq.matrix(t, 1031, ne0, seed, 1000 + i, std=0.02)
        pool, at = pools[t, ne0], 37 * i % 1031 * gq.row_bytes(t, ne0)
        done = min(view.size, pool.size - at)
        view[:done] = pool[at:at + done]
        if view.size > done:
            view[done:] = np.resize(pool, view.size - done)
    return q35.Blob(cfg, table, data, len(specs))


def _rope_table(n: int) -> np.ndarray:
    ang = np.arange(n)[:, None] * ROPE_BASE ** (-2.0 * np.arange(N_ROT // 2) / N_ROT)
    return np.stack([np.cos(ang), np.sin(ang)], -1).reshape(-1).astype(np.float32)


def _pad(n: int) -> int:
    return (n + 15) // 16 * 16


def _layout(**sizes: int) -> tuple[dict[str, int], int]:
    """Offsets of the named vectors in the activation buffer, each a multiple of 16 floats, and its size."""
    at, off = {}, 16
    for k, n in sizes.items():
        at[k] = off
        off += _pad(n)
    return at, off + 64


def _inputs(case: dict, seed: int) -> dict[str, np.ndarray]:
    """The vectors and weights of the single-layer kinds."""
    k, n, u = case["kind"], gq.normal, gq.uniform
    if k == "gemv":
        return {"w": _weights(TYPES[case["fmt"]], case["rows"], case["cols"], seed, 1), "x": n(seed, 2, case["cols"])}
    if k == "gemm":
        t, r, c = TYPES[case["fmt"]], case["rows"], case["cols"]
        return {"wg": _weights(t, r, c, seed, 1), "wu": _weights(t, r, c, seed, 2), "nw": u(seed, 3, c, 0.5, 1.5),
                "x": n(seed, 4, c * case["tokens"])}
    if k == "ffn":
        t, e, f, L = TYPES[case["fmt"]], case["embd"], case["ff"], case["layers"]
        d = {"x": n(seed, 2, e)}
        for i in range(L):
            d.update({f"wg{i}": _weights(t, f, e, seed, 10 * i + 3), f"wu{i}": _weights(t, f, e, seed, 10 * i + 4),
                      f"wd{i}": _weights(t, e, f, seed, 10 * i + 5), f"nw{i}": u(seed, 10 * i + 6, e, 0.5, 1.5)})
        return d
    if k == "gdn":
        hk, hv, L = case["hk"], case["hv"], case["layers"]
        ch, e = (2 * hk + hv) * S, hv * S
        d = {"qkv": n(seed, 2, L * ch), "x": n(seed, 3, e), "cw": n(seed, 4, L * 4 * ch, 0.0, 0.5),
             "cst": n(seed, 5, L * 3 * ch), "z": n(seed, 6, L * hv * S), "ba": n(seed, 7, L * 2 * _pad(hv)),
             "dt": n(seed, 8, L * _pad(hv)), "a": -np.abs(n(seed, 9, L * _pad(hv))), "sw": u(seed, 10, L * S, 0.5, 1.5),
             "state": n(seed, 11, L * hv * S * S, 0.0, 0.1)}
        d.update({f"wo{i}": _weights(TYPES[case["fmt"]], e, hv * S, seed, 20 + i) for i in range(L)})
        return d
    h, kv, dim, hist, nt = case["heads"], case["kv_heads"], case["dim"], case["pos"], case["tokens"]
    m = hist + nt  # keys and values of the history, then the new tokens'
    return {"q": n(seed, 2, nt * 2 * h * dim), "k": n(seed, 3, m * kv * dim), "v": n(seed, 4, m * kv * dim),
            "qn": u(seed, 5, dim, 0.5, 1.5), "kn": u(seed, 6, dim, 0.5, 1.5), "cs": _rope_table(m)}


# ---- the program's side: what it holds, and one pass -------------------------------------------------------------
class _State:
    """What a program keeps between passes: a context or a model, and what a pass needs."""

    def __init__(self, run, owner):
        self.run, self.owner = run, owner

    def __del__(self):
        self.owner.close()


def prepare(case: dict, seed: int) -> _State:
    return {"gemv": _prepare_gemv, "gemm": _prepare_gemm, "ffn": _prepare_ffn, "gdn": _prepare_gdn,
            "attn": _prepare_attn, "decode": _prepare_decode, "prompt": _prepare_prompt,
            "batch": _prepare_batch}[case["kind"]](case, seed)


def run(state: _State):
    return state.run()


def _prepare_gemv(case, seed):
    d, t, r, c = _inputs(case, seed), TYPES[case["fmt"]], case["rows"], case["cols"]
    at, size = _layout(x=c, y=r)
    ctx = gq.Context(act_floats=size, weight_bytes=d["w"].size + 4096)
    cmds = np.array(gq.gemv(t, r, c, ctx.upload(t, r, c, d["w"]), at["x"], at["y"]), np.uint32)

    def run():  # the list runs now, uncaptured
        ctx.write(at["x"], d["x"])
        if ctx.run(cmds):
            raise RuntimeError(ctx.error())
        return ctx.read(at["y"], r)
    return _State(run, ctx)


def _prepare_gemm(case, seed):
    d, t, r, c, nt = _inputs(case, seed), TYPES[case["fmt"]], case["rows"], case["cols"], case["tokens"]
    ys = _pad(r)
    at, size = _layout(x=c * nt, nw=c, y=ys * nt)
    ctx = gq.Context(act_floats=size, weight_bytes=2 * d["wg"].size + 8192)
    ctx.write(at["nw"], d["nw"])
    norm = dict(norm_w=at["nw"], eps=EPS, norm_flags=gq.NORM_DEFER)
    g = ctx.graph(gq.gemm(t, r, c, ctx.upload(t, r, c, d["wg"]), at["x"], at["y"], nt, c, ys, gq.GEMV_SWIGLU, **norm) +
                  gq.gemm(t, r, c, ctx.upload(t, r, c, d["wu"]), at["x"], at["y"], nt, c, ys, **norm))

    def run():
        ctx.write(at["x"], d["x"])
        ctx.replay(g)
        return ctx.read(at["y"], ys * nt).reshape(nt, ys)[:, :r]
    return _State(run, ctx)


def _prepare_ffn(case, seed):
    d, t, e, f, L = _inputs(case, seed), TYPES[case["fmt"]], case["embd"], case["ff"], case["layers"]
    at, size = _layout(x=e, h=e, xn=e, act=f, tmp=e, **{f"nw{i}": e for i in range(L)})
    ctx = gq.Context(act_floats=size, weight_bytes=sum(v.size + 512 for k, v in d.items() if k[:2] in ("wg", "wu", "wd")))
    cmds, src = [], at["x"]
    for i in range(L):
        ctx.write(at[f"nw{i}"], d[f"nw{i}"])
        off = [ctx.upload(t, rows, cols, d[k + str(i)]) for k, rows, cols in (("wg", f, e), ("wu", f, e), ("wd", e, f))]
        cmds += (gq.rmsnorm(e, src, at[f"nw{i}"], at["xn"], EPS, flags=gq.NORM_DEFER) +
                 gq.gemv(t, f, e, off[0], at["xn"], at["act"], gq.GEMV_SWIGLU) + gq.gemv(t, f, e, off[1], at["xn"], at["act"]) +
                 gq.gemv(t, e, f, off[2], at["act"], at["tmp"], gq.GEMV_ADD) + gq.add(e, at["tmp"], src, at["h"]))
        src = at["h"]
    g = ctx.graph(cmds)

    def run():
        ctx.write(at["x"], d["x"])
        ctx.replay(g)
        return ctx.read(at["h"], e)
    return _State(run, ctx)


def _prepare_gdn(case, seed):
    d, t, hk, hv, L = _inputs(case, seed), TYPES[case["fmt"]], case["hk"], case["hv"], case["layers"]
    ch, e, hp = (2 * hk + hv) * S, hv * S, _pad(hv)
    at, size = _layout(**{k: v.size for k, v in d.items() if k != "state" and k[:2] != "wo"}, cqkv=ch, y=e, tmp=e, out=L * e)
    ctx = gq.Context(act_floats=size, weight_bytes=L * (d["wo0"].size + 512), state_rows=L * hv * S)
    for k in ("cw", "cst", "z", "ba", "dt", "a", "sw", "x"):
        ctx.write(at[k], d[k])
    ctx.state_write(0, d["state"])
    cmds, flags, res = [], gq.GDN_L2_QK | gq.GDN_GATED | gq.GDN_GATES, at["x"]
    for i in range(L):
        st, ba, out = at["cst"] + 3 * ch * i, at["ba"] + 2 * hp * i, at["out"] + e * i
        cmds += (gq.conv(ch, at["qkv"] + ch * i, at["cw"] + 4 * ch * i, at["cqkv"], st, st) +
                 gq.gdn(hv, hk, at["cqkv"], at["cqkv"] + hk * S, at["cqkv"] + 2 * hk * S, ba + hp, ba, at["y"],
                        i * hv * S, i * hv * S, 1 / np.sqrt(S), flags, EPS, EPS, at["sw"] + S * i, at["z"] + e * i,
                        at["dt"] + hp * i, at["a"] + hp * i) +
                 gq.gemv(t, e, hv * S, ctx.upload(t, e, hv * S, d[f"wo{i}"]), at["y"], at["tmp"], gq.GEMV_ADD) +
                 gq.add(e, at["tmp"], res, out))
        res = out
    g = ctx.graph(cmds)

    def run():  # every pass is one more token: the windows and states move on
        ctx.write(at["qkv"], d["qkv"])
        ctx.replay(g)
        return ctx.read(at["out"], L * e).reshape(L, e)
    return _State(run, ctx)


def _prepare_attn(case, seed):
    d, h, kv, dim, hist, nt = (_inputs(case, seed), case["heads"], case["kv_heads"], case["dim"], case["pos"],
                               case["tokens"])
    m, row = hist + nt, kv * dim
    chunks = -(-hist // 32)
    at, size = _layout(**{k: v.size for k, v in d.items()}, y=32 * h * dim, fill=32 * 2 * h * dim, slots=16 * (chunks + 1))
    ctx = gq.Context(act_floats=size, weight_bytes=1 << 12)
    slots = np.zeros(16 * (chunks + 1), np.int32)
    slots[0:16 * chunks:16] = np.arange(0, hist, 32)
    slots[16 * chunks] = hist
    for k, v in {**d, "slots": slots}.items():
        ctx.write(at[k], v)
    cache = ctx.kv_create(-(-m // 64) * 64, kv, dim)

    def attn(q, first, slot, n):
        return gq.attn(h, kv, q, cache, at["y"], dim, N_ROT, at["slots"] + 16 * slot, at["k"] + first * row,
                       at["v"] + first * row, 1 / np.sqrt(dim), EPS, at["qn"], at["kn"], at["cs"], gate=q + dim, n_tok=n)
    # the history's keys and values, in batches (their queries do not matter)
    if ctx.run(sum((attn(at["fill"], 32 * i, i, min(32, hist - 32 * i)) for i in range(chunks)), [])):
        raise RuntimeError(ctx.error())
    g = ctx.graph(attn(at["q"], hist, chunks, nt))

    def run():
        ctx.write(at["q"], d["q"])
        ctx.replay(g)
        return ctx.read(at["y"], nt * h * dim).reshape(nt, h * dim)
    return _State(run, ctx)


def _prepare_decode(case, seed):
    cfg = _config(case, case["prompt"] + case["steps"])
    m = q35.Model(_blob(cfg, seed))
    if case["reference"]:
        m.set_arith(gq.ARITH_REFERENCE)
    ids = q35.prompt_ids(cfg, case["prompt"], seed)

    def run():
        return {"tokens": m.generate(ids, case["steps"]), "logits": m.logits(), "hidden": m.hidden()}
    return _State(run, m)


def _prepare_prompt(case, seed):
    n = case["prompt"]
    cfg = _config(case, n + 1)
    m = q35.Model(_blob(cfg, seed))
    ids = q35.prompt_ids(cfg, n, seed)

    def run():
        m.reset(ids)
        m.prefill(n - 1)
        m.step(1)
        return {"tokens": m.tokens(n + 1), "logits": m.logits(), "hidden": m.hidden()}
    return _State(run, m)


def _prepare_batch(case, seed):
    ns, steps = case["seqs"], case["steps"]
    cfg = _config(case, steps + 16)
    m = q35.BatchModel(_blob(cfg, seed), ns)
    ids = q35.prompt_ids(cfg, 16 * ns, seed)
    prompts = [ids[16 * s:16 * s + 1 + 5 * s % 16] for s in range(ns)]  # ragged prompts of 1 to 16 ids

    def run():
        m.reset(prompts)
        m.step(steps)
        return {"tokens": np.stack([m.tokens(s, steps + 1) for s in range(ns)]),
                "logits": np.stack([m.logits(s) for s in range(ns)])}
    return _State(run, m)


# ---- what a pass cannot do without -----------------------------------------------------------------------------
def work(case: dict) -> dict:
    k = case["kind"]
    if k == "gemv":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * gq.row_bytes(TYPES[case["fmt"]], c) + 4 * (r + c), "flops": 2 * r * c}
    if k == "gemm":
        r, c, nt = case["rows"], case["cols"], case["tokens"]
        return {"bytes": 2 * r * gq.row_bytes(TYPES[case["fmt"]], c) + 4 * (c + nt * (r + c)), "flops": 4 * r * c * nt}
    if k == "ffn":
        t, e, f, L = TYPES[case["fmt"]], case["embd"], case["ff"], case["layers"]
        return {"bytes": L * (2 * f * gq.row_bytes(t, e) + e * gq.row_bytes(t, f) + 4 * e) + 8 * e, "flops": 6 * L * e * f}
    if k == "gdn":
        hk, hv, L = case["hk"], case["hv"], case["layers"]
        ch, e = (2 * hk + hv) * S, hv * S
        per = 2 * 4 * e * S + 4 * ch * (1 + 4 + 2 * 3) + 4 * (e + 4 * hv + S) + e * gq.row_bytes(TYPES[case["fmt"]], e) + 4 * e
        return {"bytes": L * per + 4 * e, "flops": L * (2 * e * e + 7 * e * S + 8 * ch)}
    if k == "attn":
        h, kv, dim, nt, m = case["heads"], case["kv_heads"], case["dim"], case["tokens"], case["pos"] + case["tokens"]
        return {"bytes": 4 * m * kv * dim + 4 * nt * (3 * h + 2 * kv) * dim, "flops": 4 * nt * m * h * dim}
    # whole models: per token row the layers' products, states and keys; the weights once a step
    n_seq = case.get("seqs", 1)
    if k == "decode":
        steps, rows, heads, ctx_sum = case["prompt"] - 1 + case["steps"], 1, case["prompt"] - 1 + case["steps"], None
    elif k == "prompt":
        steps, rows, heads, ctx_sum = 1, case["prompt"], 1, None
    else:
        steps, rows, heads, ctx_sum = case["steps"], n_seq, case["steps"] * n_seq, None
    cfg = _config(case, 64)
    total = steps * rows
    per_seq = total // n_seq
    ctx_sum = n_seq * per_seq * (per_seq + 1) // 2  # positions read over all tokens
    layer_elems = sum(a * b for n, t, a, b, _ in q35.tensor_specs(cfg) if t != q35.F32 and n.startswith("blk."))
    layer_bytes = sum(q35.tensor_bytes(t, a, b) for n, t, a, b, _ in q35.tensor_specs(cfg) if n.startswith("blk."))
    head_elems, head_bytes = cfg.n_vocab * cfg.n_embd, q35.tensor_bytes(cfg.etype, cfg.n_embd, cfg.n_vocab)
    head_steps = 1 if k == "prompt" else steps
    gdn = sum(not cfg.is_attn(i) for i in range(cfg.n_layer))
    att, kv_row = cfg.n_layer - gdn, cfg.n_head_kv * cfg.head_dim
    state = 2 * 4 * cfg.ssm_v_heads * S * S + 2 * 4 * 3 * cfg.conv_ch
    passes = 1 if k == "prompt" else per_seq  # a prompt's keys and states need to be read once in all
    return {"bytes": steps * layer_bytes + head_steps * head_bytes + gdn * state * n_seq * passes +
            att * 4 * kv_row * (total if k == "prompt" else ctx_sum) + 4 * heads * cfg.n_vocab,
            "flops": 2 * total * layer_elems + 2 * heads * head_elems + gdn * total * 7 * cfg.ssm_v_heads * S * S +
            att * 4 * ctx_sum * cfg.n_head * cfg.head_dim}


def tolerance(case: dict):
    """Each about four times what was measured: the single layers against exact(), whole models as the logits of one
    prompt in this package's two arithmetics (the same products with their sums in another order and in other
    precisions, 0.018 apart)."""
    kind = case["kind"]
    if kind == "gemv":
        return {"rel": 1e-5}
    if kind == "attn":
        return {"rel": 3e-5}  # a query or key on the edge of two 16-bit values
    if kind == "gdn":
        return {"rel": 2e-4}  # an activation on the edge of two 8-bit values, as below
    if kind in ("ffn", "gemm"):
        return {"rel": 5e-4}
    return {"rel": 0.03}  # every layer's 8-bit roundings decide what the next one sees; the token ids are the same


# ---- the outputs in 64 bits ------------------------------------------------------------------------------------
def _half(b: np.ndarray) -> np.ndarray:
    return np.ascontiguousarray(b).view(np.float16)[..., 0].astype(np.float64)


def _dequantize(fmt: str, w: np.ndarray, rows: int, cols: int) -> np.ndarray:
    """GGUF blocks as 64-bit values, [rows, cols] (the block layouts of ggml-common.h)."""
    b = w.reshape(rows, -1, {"q4_0": 18, "q4_1": 20, "q8_0": 34, "q5_K": 176, "q6_K": 210}[fmt])
    if fmt == "q8_0":
        return (_half(b[..., :2])[..., None] * b[..., 2:].view(np.int8)).reshape(rows, cols)
    if fmt in ("q4_0", "q4_1"):
        qs = b[..., 2 if fmt == "q4_0" else 4:]
        q = np.concatenate([qs & 15, qs >> 4], -1).astype(np.float64)
        d = _half(b[..., :2])[..., None]
        return (d * (q - 8) if fmt == "q4_0" else d * q + _half(b[..., 2:4])[..., None]).reshape(rows, cols)
    if fmt == "q5_K":
        s = b[..., 4:16]
        sc = np.concatenate([s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6 << 4)], -1).astype(np.float64)
        mn = np.concatenate([s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6 << 4)], -1).astype(np.float64)
        qh, qs = b[..., 16:48], b[..., 48:]
        q = np.stack([((qs[..., 32 * (j // 2):32 * (j // 2) + 32] >> 4 * (j % 2)) & 15) + ((qh >> j & 1) << 4)
                      for j in range(8)], -2)
        d, dm = _half(b[..., :2])[..., None, None], _half(b[..., 2:4])[..., None, None]
        return (d * sc[..., None] * q - dm * mn[..., None]).reshape(rows, cols)
    ql, qh, sc, d = b[..., :128], b[..., 128:192], b[..., 192:208].view(np.int8).astype(np.float64), _half(b[..., 208:210])
    q = np.concatenate([((ql[..., 64 * n + 32 * (j % 2):64 * n + 32 * (j % 2) + 32] >> 4 * (j // 2)) & 15) |
                        ((qh[..., 32 * n:32 * n + 32] >> 2 * j & 3) << 4) for n in range(2) for j in range(4)], -1)
    scale = (d[..., None] * sc).repeat(16, -1)
    return (scale * (q.astype(np.float64) - 32)).reshape(rows, cols)


def _quantized(fmt: str, x: np.ndarray) -> np.ndarray:
    """The activation as a product of this format sees it: rounded to Q8_0 (Q8_1, Q8_K) blocks, in ggml's FP32 steps."""
    x = x.astype(np.float32)
    if fmt.endswith("_K"):
        b = x.reshape(-1, 256)
        top = np.take_along_axis(b, np.abs(b).argmax(1)[:, None], 1)
        scale = np.float32(-127) / top
        return (np.minimum(np.rint(scale * b), 127).astype(np.float64) * (np.float32(1) / scale)).reshape(x.shape)
    b = x.reshape(-1, 32)
    d = np.abs(b).max(1, keepdims=True) / np.float32(127)
    v = b * np.where(d > 0, np.float32(1) / np.where(d > 0, d, np.float32(1)), np.float32(0))
    q = np.trunc(v + np.copysign(np.float32(0.5), v)).astype(np.float64)
    return (q * d.astype(np.float16).astype(np.float64)).reshape(x.shape)


def _product(fmt: str, w: np.ndarray, rows: int, cols: int, x: np.ndarray) -> np.ndarray:
    """The rows' products with the token rows x [tokens, cols]: [tokens, rows]. Rows past 512 repeat (_weights)."""
    xq, n = torch.from_numpy(_quantized(fmt, x)), min(rows, 512)
    y = xq @ torch.from_numpy(_dequantize(fmt, w[:n * (w.size // rows)], n, cols)).T
    if fmt == "q4_1":  # Q8_1 keeps a block's weighted sum as fp16 of its own
        b = x.astype(np.float32).reshape(len(x), -1, 32)
        d = np.abs(b).max(-1, keepdims=True) / np.float32(127)
        q = np.rint(_quantized(fmt, x).reshape(b.shape) / np.where(d > 0, d.astype(np.float16), 1).astype(np.float64))
        s = (q.sum(-1) * d[..., 0]).astype(np.float32).astype(np.float16).astype(np.float64)
        ws = w[:n * (w.size // rows)].reshape(n, -1, 20)
        m = _half(ws[..., 2:4])
        y = y + torch.from_numpy((s - _quantized(fmt, x).reshape(b.shape).sum(-1)) @ m.T)
    return np.tile(y.numpy(), (1, -(-rows // n)))[:, :rows]


def _silu(v):
    return v / (1 + np.exp(-v))


def _rms(x, w):
    return x / np.sqrt((x * x).mean(-1, keepdims=True) + EPS) * w


def _exact_attn(case, d):
    h, kv, dim, hist, nt = case["heads"], case["kv_heads"], case["dim"], case["pos"], case["tokens"]
    cs = d["cs"].astype(np.float64).reshape(-1, 1, N_ROT // 2, 2)

    def rope(x, t):
        a, b = x[..., :N_ROT // 2], x[..., N_ROT // 2:N_ROT]
        return np.concatenate([a * t[..., 0] - b * t[..., 1], a * t[..., 1] + b * t[..., 0], x[..., N_ROT:]], -1)

    def half(x):  # queries, keys and values are held in 16 bits
        return torch.from_numpy(x.astype(np.float32).astype(np.float16).astype(np.float64))
    q = d["q"].astype(np.float64).reshape(nt, h, 2, dim)
    qh = half(rope(_rms(q[:, :, 0], d["qn"].astype(np.float64)), cs[hist:]))
    kh = half(rope(_rms(d["k"].astype(np.float64).reshape(-1, kv, dim), d["kn"].astype(np.float64)), cs))
    vh = half(d["v"].astype(np.float64).reshape(-1, kv, dim))
    out = np.empty((nt, h, dim))
    for t in range(nt):
        n = hist + t + 1
        for i in range(h):
            p = torch.softmax(kh[:n, i * kv // h] @ qh[t, i] / np.sqrt(dim), 0)
            out[t, i] = (p @ vh[:n, i * kv // h]).numpy()
    return (out / (1 + np.exp(-q[:, :, 1]))).reshape(nt, h * dim)


def _exact_gdn(case, d):
    hk, hv, L, fmt = case["hk"], case["hv"], case["layers"], case["fmt"]
    ch, e, hp = (2 * hk + hv) * S, hv * S, _pad(hv)
    f = {k: v.astype(np.float64) for k, v in d.items() if k[:2] != "wo"}
    res, out = f["x"], []
    for i in range(L):
        win = np.concatenate([f["cst"].reshape(L, ch, 3)[i], f["qkv"].reshape(L, ch, 1)[i]], 1)
        c = _silu((win * f["cw"].reshape(L, ch, 4)[i]).sum(1)).reshape(-1, S)
        qk = c[:2 * hk] / np.maximum(np.linalg.norm(c[:2 * hk], axis=1, keepdims=True), EPS)
        at = np.arange(hv) % hk
        q, k, v = qk[:hk][at], qk[hk:][at], c[2 * hk:]
        ba = f["ba"].reshape(L, 2, hp)[i, :, :hv]
        g = np.log1p(np.exp(ba[1] + f["dt"].reshape(L, hp)[i, :hv])) * f["a"].reshape(L, hp)[i, :hv]
        X = f["state"].reshape(L, hv, S, S)[i] * np.exp(g)[:, None, None]
        delta = (v - (X * k[:, None]).sum(-1)) / (1 + np.exp(-ba[0]))[:, None]
        y = ((X + delta[..., None] * k[:, None]) * q[:, None]).sum(-1) / np.sqrt(S)
        y = _rms(y, f["sw"].reshape(L, S)[i]) * _silu(f["z"].reshape(L, hv, S)[i])
        res = res + _product(fmt, d[f"wo{i}"], e, e, y.reshape(1, e))[0]
        out.append(res)
    return np.stack(out)


def exact(case: dict, seed: int):
    k = case["kind"]
    if k not in ("gemv", "gemm", "ffn", "gdn", "attn"):
        return None  # a whole model: every layer's 8-bit rounding decides what the next one sees
    d, fmt = _inputs(case, seed), case.get("fmt")
    if k == "attn":
        return _exact_attn(case, d)
    if k == "gdn":
        return _exact_gdn(case, d)
    if k == "gemv":
        return _product(fmt, d["w"], case["rows"], case["cols"], d["x"][None])[0]
    if k == "gemm":
        r, c = case["rows"], case["cols"]
        x = _rms(d["x"].astype(np.float64).reshape(-1, c), d["nw"].astype(np.float64))
        return _silu(_product(fmt, d["wg"], r, c, x)) * _product(fmt, d["wu"], r, c, x)
    h, e, f = d["x"].astype(np.float64), case["embd"], case["ff"]
    for i in range(case["layers"]):
        x = _rms(h, d[f"nw{i}"].astype(np.float64))[None]
        a = _silu(_product(fmt, d[f"wg{i}"], f, e, x)) * _product(fmt, d[f"wu{i}"], f, e, x)
        h = h + _product(fmt, d[f"wd{i}"], e, f, a)[0]
    return h
