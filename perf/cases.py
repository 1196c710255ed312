"""What this framework is used for, as cases that can be timed: decoding, prompts and training steps through the public entry points.

A case is a dict of plain values.  `kind`:
  decode        a Qwen3-shaped model with quantised layers generates: `steps` tokens of each of `seqs` sequences standing behind `pos` tokens (one sequence: Qwen3.run_steps,
                several: XcdReplicas.run_steps, as its request queue runs them)
  prefill       the same models read prompts: one (Qwen3.prefill) or several as one batch (XcdReplicas.prefill_batch)
  rows_decode   a design described layer by layer (Tizusun, Bolopel) generates for one sequence or several requests in slots
  rows_prefill  the same designs read the prompts of one or several requests as one ragged batch and give the logits of some rows (XcdReplicas.run)
  train         one training step of a GPT-2-shaped model in hybrid precision: forward, loss, backward, AdamW, re-quantisation (GPT2Step.step)
Decoding runs along ids that are set beforehand (set_forced), so that two runs see the same tokens whatever a near-tie picks; the picks are made all the same.
`exact` states every model in 64 bits in plain torch, without this repository's code.
"""
import math

import numpy as np
import torch
import torch.utils.checkpoint

from koifish_amd import lib as L
from koifish_amd import runtime as R
from koifish_amd import synth
from koifish_amd.train_step import GPT2Step

DEVICE = "cuda:0"
STORAGE = {"q4": L.Q4, "q1": L.BOOL1}


def listed():
    return [
        # a chat's next token, shortly behind the prompt: the smallest call, one launch
        dict(name="token", kind="decode", model="qwen3-0.6b", layers=28, storage="q4", seqs=1, pos=130, steps=1),
        # one sequence near the end of its context, a run of tokens as Generate makes them
        dict(name="decode", kind="decode", model="qwen3-0.6b", layers=28, storage="q4", seqs=1, pos=2030, steps=16),
        # a server's full house: 32 sequences of the small model sharing the weights
        dict(name="decode_32", kind="decode", model="qwen3-0.6b", layers=28, storage="q4", seqs=32, pos=2030, steps=4),
        # one sequence of a 32B-sized model (a slice of its 64 equal layers), 4k context
        dict(name="decode_wide", kind="decode", model="qwen3-32b", layers=8, storage="q4", seqs=1, pos=4030, steps=4),
        # a chat prompt
        dict(name="prompt", kind="prefill", model="qwen3-0.6b", layers=28, storage="q4", prompts=1, tokens=128),
        # a document as the prompt
        dict(name="prompt_long", kind="prefill", model="qwen3-0.6b", layers=28, storage="q4", prompts=1, tokens=2047),
        # prompts of unequal length waiting in the server's queue, read together
        dict(name="prompts", kind="prefill", model="qwen3-0.6b", layers=28, storage="q4", prompts=16, tokens=131),
        # a long prompt through recurrent layers and windowed attention
        dict(name="rows_prompt", kind="rows_prefill", design="bolopel", size="2k", dtype="bfloat16", spans=1, tokens=8190),
        # prompts of four requests through routed experts
        dict(name="rows_prompts_routed", kind="rows_prefill", design="tizusun", size="2k-moe", dtype="bfloat16", spans=4, tokens=509),
        # scoring in true 32-bit storage
        dict(name="rows_prompt_f32", kind="rows_prefill", design="tizusun", size="2k", dtype="float32", spans=1, tokens=512),
        # 32 requests of recurrent layers generating together
        dict(name="rows_decode_32", kind="rows_decode", design="bolopel", size="2k", dtype="bfloat16", seqs=32, pos=1024, steps=4),
        # a training step of the 1558M shapes, 8 x 1024 tokens
        dict(name="train", kind="train", width=1600, heads=25, layers=48, batch=8, tokens=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "rows_prefill", "rows_prefill", "rows_decode", "train"])
    if kind == "decode":
        model = rng.choice(["qwen3-0.6b", "qwen3-0.6b", "qwen3-1.7b", "qwen3-32b"])
        seqs = 1 if model == "qwen3-32b" else rng.choice([1, rng.randint(2, 8), rng.randint(9, 32 if model == "qwen3-0.6b" else 16)])
        storage = rng.choice(["q4", "q4", "q1"]) if model == "qwen3-0.6b" else "q4"
        return dict(kind=kind, model=model, layers=6 if model == "qwen3-32b" else 28, storage=storage, seqs=seqs, pos=_log_int(rng, 16, 4060 if model == "qwen3-32b" else 2020), steps=rng.randint(1, 16))
    if kind == "prefill":
        model = rng.choice(["qwen3-0.6b", "qwen3-0.6b", "qwen3-1.7b", "qwen3-32b"])
        prompts = 1 if model == "qwen3-32b" else rng.choice([1, 1, _log_int(rng, 2, 16)])
        return dict(kind=kind, model=model, layers=6 if model == "qwen3-32b" else 28, storage="q4", prompts=prompts, tokens=_log_int(rng, 8, 2040 if prompts == 1 else 8100 // (prompts + prompts // 4)))
    if kind == "rows_decode":
        design = rng.choice(["tizusun", "bolopel"])
        return dict(kind=kind, design=design, size=rng.choice(["2k", "4k"] + ["2k-moe"] * (design == "tizusun")), dtype="bfloat16", seqs=rng.choice([1, _log_int(rng, 2, 32)]), pos=_log_int(rng, 16, 3000),
                    steps=rng.randint(2, 8))
    if kind == "rows_prefill":
        design, dtype = rng.choice(["tizusun", "bolopel"]), rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"])
        spans = rng.choice([1, 1, _log_int(rng, 2, 8)])
        size = "2k" if dtype == "float32" else rng.choice(["2k", "4k"] + ["2k-moe"] * (design == "tizusun"))
        return dict(kind=kind, design=design, size=size, dtype=dtype, spans=spans, tokens=_log_int(rng, 8, (700 if dtype == "float32" else 8100) // spans))
    width, heads = rng.choice([(768, 12), (1600, 25)])
    return dict(kind=kind, width=width, heads=heads, layers=rng.randint(2, 12), batch=rng.randint(1, 8), tokens=_log_int(rng, 64, 1024))


# ---------------------------------------------------------------- inputs, from the seed alone

def _generator(seed):
    R.stream(0)   # this thread's torch work goes on the stream that the framework launches on
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _ids(seed, shape, vocab):
    return np.random.default_rng([int(seed), 17]).integers(0, vocab, size=shape).astype(np.int32)


def _lengths(n, tokens):
    """n unequal lengths around `tokens`, at most a quarter more"""
    return [max(1, tokens + ((i * 7) % 5 - 2) * tokens // 8) if n > 1 else tokens for i in range(n)]


def _qwen3_config(case):
    c = dict(synth.CONFIGS[case["model"]], name=case["model"], n_layer=case["layers"])
    if case["kind"] == "decode":
        c["max_seq"] = min(c["max_seq"], case["pos"] + case["steps"] + 1 + 128)
    return c


def _qwen3_tensors(c, seed):
    """(layer, name, bf16 tensor): weights and norms as models start out, the products into the residual stream smaller by the square root of their number"""
    g, back = _generator(seed), 0.02 / (2 * synth.CONFIGS[c["name"]]["n_layer"]) ** 0.5

    def mat(rows, cols, std=0.02):
        return torch.randn(rows, cols, generator=g, device=DEVICE).mul_(std).to(torch.bfloat16)

    def norm(n):
        return torch.randn(n, generator=g, device=DEVICE).mul_(0.01).add_(1.0).to(torch.bfloat16)
    q, kv = c["n_head"] * c["head_dim"], c["n_kv"] * c["head_dim"]
    yield -1, "embed", mat(c["vocab"], c["dim"])
    if not c["tied"]:
        yield -1, "head", mat(c["vocab"], c["dim"])
    yield -1, "norm", norm(c["dim"])
    for i in range(c["n_layer"]):
        for name, rows, cols in (("q", q, c["dim"]), ("k", kv, c["dim"]), ("v", kv, c["dim"]), ("o", c["dim"], q), ("gate", c["ffn"], c["dim"]), ("up", c["ffn"], c["dim"]), ("down", c["dim"], c["ffn"])):
            yield i, name, mat(rows, cols, back if name in ("o", "down") else 0.02)
        for name, n in (("norm_in", c["dim"]), ("norm_post", c["dim"]), ("qn", c["head_dim"]), ("kn", c["head_dim"])):
            yield i, name, norm(n)


def _hot(case, c, layer):
    """the feed-forward rows that the sparse forward of the 1-bit storage computes: one in five"""
    return (np.random.default_rng([5, layer]).random(c["ffn"]) < 0.2).astype(np.int32) if case["storage"] == "q1" else None


def _qwen3(case, seed):
    c = _qwen3_config(case)
    ctx, m = R.Context(0), R.Qwen3(c, 0)
    m._ctx = ctx
    for i, name, w in _qwen3_tensors(c, seed):
        if name == "embed":
            m.set_weight(-1, 0, ctx.quantize(w, L.BF16))
            if c["tied"]:
                m.tie_head()
        elif name == "head":
            m.set_weight(-1, 1, ctx.quantize(w, L.BF16))
        elif name == "norm":
            m.set_norm(-1, 0, w)
        elif name in synth.SLOTS:
            m.set_weight(i, synth.SLOTS.index(name), ctx.quantize(w, STORAGE[case["storage"]]))
        else:
            m.set_norm(i, synth.NORMS.index(name), w)
    for i in range(c["n_layer"]):
        if case["storage"] == "q1":
            m.set_hot(i, _hot(case, c, i))
    ctx.sync()
    return c, m


class _Memory:
    """device memory that `owner` owns, for torch.as_tensor: a tensor on it keeps its owner alive"""

    def __init__(self, owner, address, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<i2", data=(int(address), False), version=2)


def _bf16_view(owner, address, shape):
    return torch.as_tensor(_Memory(owner, address, shape), device=DEVICE).view(torch.bfloat16)


def _cache_views(owner, c, key, val, rows):
    shape = (c["n_layer"], c["max_seq"], c["n_kv"] * c["head_dim"])
    return _bf16_view(owner, key, shape)[:, :rows], _bf16_view(owner, val, shape)[:, :rows]


def _prepare_decode(case, seed):
    c, m = _qwen3(case, seed)
    n, p = case["seqs"], case["pos"]
    lens = [p - (3 * s) % min(p, 48) if n > 1 else p for s in range(n)]   # sequences stand at positions of their own
    ids = _ids(seed, (n, p + case["steps"]), c["vocab"])
    state = dict(case=case, model=m, at=[(int(ids[s, lens[s]]), lens[s]) for s in range(n)])
    if n == 1:
        m.set_forced(ids[0])
        m.prefill(ids[0, :p], want_logits=False)
        logits = _bf16_view(m, m.host.kfh_logits(m.h), (1, c["vocab"]))
        k, v = _cache_views(m, c, m.host.kfh_kcache(m.h), m.host.kfh_vcache(m.h), p + case["steps"])
        state["out"] = dict(logits=logits, k=k, v=v)
        return state
    x = R.XcdReplicas(m, n)
    for s in range(n):
        x.set_forced(s, ids[s])
        x.prefill(s, ids[s, :lens[s]])
    last = lens[-1] + case["steps"]
    k, v = _cache_views((x, m), c, x.host.kfh_xr_kcache(x.h, n - 1), x.host.kfh_xr_vcache(x.h, n - 1), last)
    state.update(slots=x, out=dict(logits=_bf16_view((x, m), x.host.kfh_xr_logits(x.h, 0), (n, c["vocab"])), k=k, v=v))
    return state


def _run_decode(s):
    n = s["case"]["steps"]
    if "slots" in s:
        for i, (token, pos) in enumerate(s["at"]):
            s["slots"].set_state(i, token, pos)
        s["slots"].run_steps(n)
    else:
        (token, pos), = s["at"]
        s["model"].set_state(token, pos)
        s["model"].run_steps(pos, n)
    return s["out"]


def _prepare_prefill(case, seed):
    c, m = _qwen3(case, seed)
    n, lens = case["prompts"], _lengths(case["prompts"], case["tokens"])
    ids = _ids(seed, (n, max(lens)), c["vocab"])
    state = dict(case=case, model=m, prompts=[ids[i, :lens[i]].copy() for i in range(n)], vocab=c["vocab"])
    if n > 1:
        x = R.XcdReplicas(m, n)
        k, v = _cache_views((x, m), c, x.host.kfh_xr_kcache(x.h, n - 1), x.host.kfh_xr_vcache(x.h, n - 1), lens[-1])
        state.update(slots=x, order=list(range(n)), out=dict(logits=_bf16_view((x, m), x.host.kfh_xr_logits(x.h, 0), (n, c["vocab"])), k=k, v=v))
    else:
        m.prefill(np.zeros(1, np.int32), want_logits=False)   # allocates the cache that the views below look at
        k, v = _cache_views(m, c, m.host.kfh_kcache(m.h), m.host.kfh_vcache(m.h), lens[0])
        state["cache"] = dict(k=k, v=v)
    return state


def _run_prefill(s):
    if "slots" in s:
        s["slots"].prefill_batch(s["order"], s["prompts"])
        return s["out"]
    _, logits = s["model"].prefill(s["prompts"][0])
    return dict(s["cache"], logits=torch.from_numpy(logits.view(np.int16)).view(torch.bfloat16)[None])


def _rows_config(case):
    """(config, {tensor: shape}, the tensors' shapes that the config leaves open)"""
    if case["design"] == "tizusun":
        _, cfg = synth.tizusun_sizes(case["size"])
        return cfg, _tizusun_shapes(cfg), None
    _, cfg, open_shapes = synth.bolopel_sizes(case["size"])
    return cfg, _bolopel_shapes(cfg, open_shapes), open_shapes


def _dense_shapes(p, ff, width):
    return {p + "gate": (ff, width), p + "up": (ff, width), p + "down": (width, ff)}


def _tizusun_shapes(cfg):
    w = cfg["width"]
    out = {"embed": (cfg["vocab"], w), "head": (cfg["vocab"], w), "final.norm": (w,)}
    for i, layer in enumerate(cfg["layers"]):
        p, m, f = "l%d." % i, layer["mixer"], layer["mlp"]
        q, k = m["heads"] * m["dim"], m["kv_heads"] * m["dim"]
        out.update({p + "mix.q": (q, w), p + "mix.k": (k, w), p + "mix.g": (q, w), p + "mix.o": (w, q), p + "mix.q.norm": (m["dim"],), p + "mix.k.norm": (m["dim"],), p + "norm1": (w,), p + "norm2": (w,)})
        if f["kind"] == "dense":
            out.update(_dense_shapes(p + "mlp.", f["ff"], w))
            continue
        n = f["router"]["experts"]
        out.update({p + "mlp.router": (n, w), p + "mlp.router.b": (n,)})
        for e in range(n):
            out.update(_dense_shapes(p + "mlp.e%d." % e, f["expert"]["ff"], w))
    return out


def _bolopel_shapes(cfg, ranks):
    w = cfg["width"]
    out = {"embed": (cfg["vocab"], w), "embed.norm": (w,), "head": (cfg["vocab"], w), "final.norm": (w,)}
    for i, layer in enumerate(cfg["layers"]):
        p, m = "l%d.mix." % i, layer["mixer"]
        if layer["type"] == "channel_delta":
            k, h, v, a, g = m["kv_heads"] * m["dim"], m["heads"] * m["dim"], m["heads"] * m["vdim"], ranks[p + "a1"][0], ranks[p + "g1"][0]
            out.update({p + "q": (k, w), p + "k": (k, w), p + "v": (v, w), p + "q.conv": (k, m["conv"]), p + "k.conv": (k, m["conv"]), p + "v.conv": (v, m["conv"]), p + "b": (m["heads"], w),
                        p + "A_log": (m["heads"],), p + "norm": (m["vdim"],), p + "a1": (a, w), p + "a2": (h, a), p + "dt_bias": (h,), p + "g1": (g, w), p + "g2": (v, g), p + "o": (w, v)})
        else:
            a, b = m["left"], m["right"]
            q, k, v, bq, bv = a["heads"] * a["dim"], a["kv_heads"] * a["dim"], a["heads"] * a["vdim"], b["heads"] * b["dim"], b["heads"] * b["vdim"]
            out.update({p + "left.q": (q, w), p + "left.k": (k, w), p + "left.v": (a["kv_heads"] * a["vdim"], w), p + "left.o": (w, v), p + "right.q": (bq, w), p + "right.k": (bq, w), p + "right.v": (bv, w),
                        p + "right.g": (bv, w), p + "right.o": (w, bv), p + "right.norm": (bv,)})
        out.update({"l%d.norm1" % i: (w,), "l%d.norm2" % i: (w,)})
        out.update(_dense_shapes("l%d.mlp." % i, layer["mlp"]["ff"], w))
    return out


def _rows_tensors(shapes, seed):
    """(name, bf16 tensor): unit-gain matrices, norms around 1, decays of a channel from slow to fast, routers with a clear choice"""
    g = _generator(seed)
    for name, shape in shapes.items():
        w = torch.randn(shape, generator=g, device=DEVICE)
        leaf = name.split(".")[-1]
        if leaf.startswith("norm"):
            w.mul_(0.1).add_(1.0)
        elif leaf == "A_log":
            w.sub_(0.5)
        elif leaf == "dt_bias":
            w.sub_(3.0)
        elif leaf == "router":
            w.mul_(2.0 / shape[1] ** 0.5)
        elif leaf != "embed" and len(shape) == 2:
            w.mul_(1.0 / shape[1] ** 0.5)
        yield name, w.to(torch.bfloat16)


def _rows(case, seed, max_seq):
    cfg, shapes, open_shapes = _rows_config(case)
    _generator(seed)
    cls = R.Tizusun if case["design"] == "tizusun" else R.Bolopel
    m = cls(cfg, case["dtype"], max_seq, 0, open_shapes)
    for name, w in _rows_tensors(shapes, seed):
        m.set_tensor(name, w)
    return cfg, m


def _prepare_rows_prefill(case, seed):
    lens = _lengths(case["spans"], case["tokens"])
    cfg, m = _rows(case, seed, max(lens) + 64)
    ids = _ids(seed, (case["spans"], max(lens)), cfg["vocab"])
    x = R.XcdReplicas(m, case["spans"])
    slots = [x.acquire() for _ in lens]
    return dict(case=case, model=m, slots=x, spans=[(slots[i], 0, ids[i, :n]) for i, n in enumerate(lens)], want=_wanted(lens))


def _wanted(lens):
    """the rows whose logits are asked for: the last of every span and seven before it, spread"""
    return [(i, r) for i, n in enumerate(lens) for r in sorted({n - 1 - j * n // 8 for j in range(8)})]


def _run_rows_prefill(s):
    return s["slots"].run(s["spans"], s["want"])


def _prepare_rows_decode(case, seed):
    n, p, k = case["seqs"], case["pos"], case["steps"]
    cfg, m = _rows(case, seed, p + k + 64)
    lens = [p - (3 * s) % min(p, 48) for s in range(n)]
    ids = _ids(seed, (n, p + k), cfg["vocab"])
    x = R.XcdReplicas(m, n)
    slots = [x.acquire() for _ in range(n)]
    for i in range(n):
        x.set_forced(slots[i], ids[i])
        x.run([(slots[i], 0, ids[i, :lens[i]])])
    last = [(slots[i], lens[i] + k - 1, ids[i, lens[i] + k - 1:lens[i] + k]) for i in range(n)]
    return dict(case=case, model=m, slots=x, at=[(slots[i], int(ids[i, lens[i]]), lens[i]) for i in range(n)], last=last, want=[(i, 0) for i in range(n)])


def _run_rows_decode(s):
    for slot, token, pos in s["at"]:
        s["slots"].set_state(slot, token, pos)
    s["slots"].run_steps(s["case"]["steps"] - 1)
    return s["slots"].run(s["last"], s["want"])   # the last step gives the logits of every request


VOCAB, PADDED = 50257, 50304
HYPER = dict(lr=3e-4, beta1=0.9, beta2=0.95, eps=1e-8, wd=0.1, seed=7)


def _gpt2_masters(case, seed):
    g, w, back = _generator(seed), case["width"], 0.02 / (2 * case["layers"]) ** 0.5

    def mat(*shape, std=0.02, mean=0.0):
        return torch.randn(*shape, generator=g, device=DEVICE).mul_(std).add_(mean).to(torch.bfloat16)
    wte = mat(PADDED, w)
    wte[VOCAB:] = 0
    blocks = []
    for _ in range(case["layers"]):
        b = {name: (mat(rows, cols, std=back if rows == w else 0.02), mat(rows)) for name, rows, cols in (("qkv", 3 * w, w), ("proj", w, w), ("fc", 4 * w, w), ("proj2", w, 4 * w))}
        b["ln"] = (mat(w, std=0.05, mean=1.0), mat(w), mat(w, std=0.05, mean=1.0), mat(w))
        blocks.append(b)
    return dict(wte=wte, wpe=mat(case["tokens"], w, std=0.01), lnf=(mat(w, std=0.05, mean=1.0), mat(w)), blocks=blocks)


def _prepare_train(case, seed):
    masters = _gpt2_masters(case, seed)
    ctx = R.Context(0)
    step = GPT2Step(ctx, case["width"], case["heads"], case["layers"], VOCAB, PADDED, case["batch"], case["tokens"], masters=masters)
    n = case["batch"] * case["tokens"]
    ids, tgt = (torch.from_numpy(a).to(DEVICE) for a in _ids(seed, (2, n), VOCAB))
    shown = [step.wte, step.wpe, step.lnf_w, step.lnf_b] + [step.blocks[i][k] for i in sorted({0, case["layers"] - 1}) for k in step.blocks[0]]
    out = {"%s %s" % (e["name"], k): e[k] for e in shown for k in ("p", "m")}
    return dict(case=case, ctx=ctx, step=step, ids=ids, tgt=tgt, out=dict(out, losses=step.losses))


def _run_train(s):
    s["step"].step(s["ids"], s["tgt"], **HYPER)
    return s["out"]   # the losses; the weights and the first moments (which hold the gradients) of the embeddings and of the outer blocks


def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "rows_prefill": _prepare_rows_prefill, "rows_decode": _prepare_rows_decode, "train": _prepare_train}[case["kind"]](case, seed)


def run(state):
    return {"decode": _run_decode, "prefill": _run_prefill, "rows_prefill": _run_rows_prefill, "rows_decode": _run_rows_decode, "train": _run_train}[state["case"]["kind"]](state)


# ---------------------------------------------------------------- what a pass cannot do without

def _attended(lens, window=0):
    """(query, key) pairs of causal attention over prompts of these lengths"""
    return sum(n * (n + 1) / 2 if not window or n <= window else window * (window + 1) / 2 + (n - window) * window for n in lens)


def _qwen3_work(c, storage, rows, pairs, kv_rows, heads_out, passes):
    q, kv = c["n_head"] * c["head_dim"], c["n_kv"] * c["head_dim"]
    weights = c["n_layer"] * c["dim"] * (2 * q + 2 * kv + 3 * c["ffn"])
    if storage == "q1":   # one gate / up row in five
        weights -= c["n_layer"] * c["dim"] * 2 * c["ffn"] * 4 // 5
    per = {"q4": 0.5, "q1": 0.125}[storage] + 4.0 / 128
    head = c["vocab"] * c["dim"]
    return {"bytes": passes * (weights * per + head * 2) + c["n_layer"] * 4.0 * kv * kv_rows + 2.0 * c["vocab"] * heads_out,
            "flops": 2.0 * weights * rows + 4.0 * c["n_layer"] * q * pairs + 2.0 * head * heads_out}


def _rows_work(case, rows, lens, heads_out, passes, old):
    """old: tokens in front of each sequence's rows"""
    cfg, shapes, _ = _rows_config(case)
    size = 4 if case["dtype"] == "float32" else 2
    weights = active = 0.0
    for name, s in shapes.items():
        if len(s) != 2 or name == "embed":
            continue
        n, routed, layer = s[0] * s[1], ".mlp.e" in name, None
        if routed:
            layer = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            share = layer["top"] / layer["experts"]
            weights += n * (1 - (1 - share) ** (rows / passes))
            active += n * share * rows
        else:
            weights += n
            active += n * (heads_out if name == "head" else rows)
    flops, state = 2.0 * active, 0.0
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer.get("type") == "channel_delta":
            flops += 8.0 * m["heads"] * m["dim"] * m["vdim"] * rows
            state += passes * 8.0 * m["heads"] * m["dim"] * m["vdim"] * len(lens)
            continue
        a = m["left"] if "left" in m else m
        window = a["mask"]["size"]
        flops += 4.0 * a["heads"] * a["dim"] * sum(_attended([o + n], window) - _attended([o], window) for o, n in zip(old, lens))
        state += 2.0 * size * a["kv_heads"] * a["dim"] * sum(min(window, o + n) * (passes if o else 1) for o, n in zip(old, lens))
        if "right" in m:
            b = m["right"]
            flops += 6.0 * b["heads"] * b["dim"] * b["vdim"] * rows
            state += passes * 8.0 * b["heads"] * b["dim"] * b["vdim"] * len(lens)
    return {"bytes": passes * weights * size + state + 4.0 * cfg["vocab"] * heads_out, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        c, n, k = _qwen3_config(case), case["seqs"], case["steps"]
        pairs = n * k * (case["pos"] + k / 2)
        return _qwen3_work(c, case["storage"], n * k, pairs, pairs, n * k, k)
    if kind == "prefill":
        lens = _lengths(case["prompts"], case["tokens"])
        return _qwen3_work(_qwen3_config(case), case["storage"], sum(lens), _attended(lens), sum(lens), len(lens), 1)
    if kind == "rows_prefill":
        lens = _lengths(case["spans"], case["tokens"])
        return _rows_work(case, sum(lens), lens, len(_wanted(lens)), 1, [0] * len(lens))
    if kind == "rows_decode":
        n, k = case["seqs"], case["steps"]
        return _rows_work(case, n * k, [k] * n, n * k, k, [case["pos"]] * n)
    w, n = case["width"], case["batch"] * case["tokens"]
    blocks, vocab = case["layers"] * 12 * w * w, PADDED * w
    forward = 2.0 * n * (blocks + vocab) + case["layers"] * 4.0 * w * _attended([case["tokens"]]) * case["batch"]
    return {"bytes": 14.0 * (blocks + vocab) + 2.0 * n * w * case["layers"] * 16 * 2, "flops": 3.0 * forward}


def tolerance(case):
    if case.get("dtype") == "float32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 0.03, "max": 0.9}


# ---------------------------------------------------------------- the same in 64 bits, in plain torch

def _f64(w):
    return w.to(torch.float64)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _stored(w, storage):
    """the values that the quantised storage of w holds: groups of 128, every step of the reconstruction rounded to bf16"""
    a = w.float().reshape(-1, 128)
    if storage == "q4":
        lo, hi = a.amin(1, keepdim=True), a.amax(1, keepdim=True)
        step, zero = (hi - lo) / torch.full_like(hi, 15), -lo   # (a division, not a product with the reciprocal: many codes are ties)
        q = (a + zero) / step
        q = (torch.floor(q) + (q - torch.floor(q) >= 0.5)).clamp_(0, 15)
    else:
        step = torch.sqrt((torch.where(a < 0, 0.0, a).double().square().sum(1, keepdim=True)) / 128).float().clamp_min(1e-5)
        zero = torch.zeros_like(step)
        q = torch.floor(a / step + 0.5).clamp_(0, 1)
    step, zero = step.bfloat16().float(), zero.bfloat16().float()
    return _f64(((step * q).bfloat16().float() - zero).bfloat16()).reshape(w.shape)


def _causal(q, k, v, scale, seen, sink=False):
    """q [T, H, D], k and v [T, G, .] -> [T, H, V]; the scores of one key head's queries at a time"""
    T, H, _ = q.shape
    G = k.shape[1]
    out = []
    for g in range(G):
        s = torch.matmul(q[:, g * (H // G):(g + 1) * (H // G)].permute(1, 0, 2).contiguous(), k[:, g].t().contiguous()) * scale
        s.masked_fill_(~seen, -math.inf)
        m = s.amax(-1, keepdim=True)
        if sink:
            m = m.clamp_min(0.0)
        s = torch.exp(s - m)
        total = s.sum(-1, keepdim=True) + (torch.exp(-m) if sink else 0.0)
        out.append(torch.matmul(s, v[:, g].contiguous()) / total)
    return torch.cat(out, 0).permute(1, 0, 2)


def _rotate(x, cos, sin):
    n = cos.shape[-1]
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * cos - v * sin, v * cos + u * sin, x[..., 2 * n:]], -1)


def _exact_qwen3(case, seed, ids, show, steps=0):
    """ids: token arrays, the last `steps` of each generated; show: the sequence whose K / V rows are wanted"""
    c = _qwen3_config(case)
    lens = [len(t) for t in ids]
    generated = torch.cat([torch.arange(n, device=DEVICE) >= n - steps for n in lens])[:, None]
    tensors = _qwen3_tensors(c, seed)
    top = {}
    for i, name, w in tensors:
        top[name] = w
        if name == "norm":
            break
    H, G, D = c["n_head"], c["n_kv"], c["head_dim"]
    x = _f64(top["embed"][torch.from_numpy(np.concatenate(ids)).long().to(DEVICE)])
    freq = c["theta"] ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEVICE) / D)
    at = torch.cat([torch.arange(n, dtype=torch.float64, device=DEVICE) for n in lens])[:, None, None] * freq
    cos, sin = torch.cos(at), torch.sin(at)
    keys, values = [], []
    for i in range(c["n_layer"]):
        W = {}
        for _ in range(11):
            _, name, w = next(tensors)
            W[name] = _stored(w, case["storage"]) if w.dim() == 2 else _f64(w)
        h = _rms(x, W["norm_in"], 1e-6)
        q, k, v = (torch.matmul(h, W[n].t()).reshape(len(h), -1, D) for n in ("q", "k", "v"))
        q, k = _rotate(_rms(q, W["qn"], 1e-6), cos, sin), _rotate(_rms(k, W["kn"], 1e-6), cos, sin)
        out, o = [], 0
        for s, n in enumerate(lens):
            seen = torch.ones(n, n, dtype=torch.bool, device=DEVICE).tril()
            out.append(_causal(q[o:o + n], k[o:o + n], v[o:o + n], D ** -0.5, seen).reshape(n, H * D))
            if s == show:
                keys.append(k[o:o + n].reshape(n, G * D).clone())
                values.append(v[o:o + n].reshape(n, G * D).clone())
            o += n
        x = x + torch.matmul(torch.cat(out), W["o"].t())
        h = _rms(x, W["norm_post"], 1e-6)
        act = torch.nn.functional.silu(torch.matmul(h, W["gate"].t())) * torch.matmul(h, W["up"].t())
        if case["storage"] == "q1":
            act = torch.where(generated, act * torch.from_numpy(_hot(case, c, i)).to(DEVICE), act)   # prompts are read densely
        x = x + torch.matmul(act, W["down"].t())
        del W, q, k, v, h, act
    ends = torch.tensor([sum(lens[:s + 1]) - 1 for s in range(len(lens))], device=DEVICE)
    head = _f64(top["embed" if c["tied"] else "head"])
    return dict(logits=torch.matmul(_rms(x[ends], _f64(top["norm"]), 1e-6), head.t()), k=torch.stack(keys), v=torch.stack(values))


def _rope_angles(rot, T):
    f = []
    for i in range(rot["dims"] // 2):
        w = float(rot["base"]) ** (-2.0 * i / rot["dims"])
        s = rot.get("scaling")
        if s:
            turns = s["original"] * w / (2 * math.pi)
            if turns < s["low"]:
                w /= s["factor"]
            elif turns <= s["high"]:
                kept = (turns - s["low"]) / (s["high"] - s["low"])
                w = kept * w + (1 - kept) * w / s["factor"]
        f.append(w)
    return torch.arange(T, dtype=torch.float64, device=DEVICE)[:, None, None] * torch.tensor(f, dtype=torch.float64, device=DEVICE)


def _each(x, fn):
    """fn over the sequences of x [S, T, ...]"""
    return torch.stack([fn(s) for s in range(x.shape[0])])


def _tizusun_mixer(x, W, p, m, eps, n_heads_dim):
    S, T, _ = x.shape
    H, G, D = n_heads_dim
    a = _rope_angles(m["rot"], T)
    q, v = torch.matmul(x, W(p + "q").t()).reshape(S, T, H, D), torch.matmul(x, W(p + "k").t()).reshape(S, T, G, D)
    gate = torch.sigmoid(torch.matmul(x, W(p + "g").t()))
    q, k = (_rotate(_rms(z, W(p + n), eps), torch.cos(a), torch.sin(a)) for z, n in ((q, "q.norm"), (v, "k.norm")))
    t = torch.arange(T, device=DEVICE)
    seen = (t[None] <= t[:, None]) & (t[None] // m["mask"]["size"] == t[:, None] // m["mask"]["size"])
    return torch.matmul(_each(x, lambda s: _causal(q[s], k[s], v[s], m["scale"], seen).reshape(T, H * D)) * gate, W(p + "o").t())


def _ff(h, W, p, act):
    return torch.matmul(act(torch.matmul(h, W(p + "gate").t())) * torch.matmul(h, W(p + "up").t()), W(p + "down").t())


def _experts(x, W, p, f):
    h = x.reshape(-1, x.shape[-1])
    best, chosen = (torch.matmul(h, W(p + "router").t()) + W(p + "router.b")).topk(f["router"]["top"], -1)
    weight, out = torch.softmax(best, -1), torch.zeros_like(h)
    for e in range(f["router"]["experts"]):
        row, pick = (chosen == e).nonzero(as_tuple=True)
        if len(row):
            out.index_add_(0, row, weight[row, pick][:, None] * _ff(h[row], W, p + "e%d." % e, torch.nn.functional.silu))
    return out.reshape(x.shape)


def _layer_norm(x, w, eps):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], eps=eps) * w


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _conv(x, taps):
    n = taps.shape[1]
    y = torch.zeros_like(x)
    for j in range(min(n, x.shape[1])):
        y[:, j:] += taps[:, n - 1 - j] * x[:, :x.shape[1] - j]
    return torch.nn.functional.silu(y)


def _delta_mixer(x, W, p, m, eps):
    S, T, _ = x.shape
    H, D, V = m["heads"], m["dim"], m["vdim"]
    q, k, v = (_conv(torch.matmul(x, W(p + n).t()), W(p + n + ".conv")) for n in ("q", "k", "v"))
    rep = H // m["kv_heads"]
    q, k = (_unit(z.reshape(S, T, -1, D)).repeat_interleave(rep, 2) for z in (q, k))
    q, v = q * D ** -0.5, v.reshape(S, T, H, V)
    z = torch.matmul(torch.matmul(x, W(p + "a1").t()), W(p + "a2").t()) + W(p + "dt_bias")
    g = torch.exp(-torch.exp(W(p + "A_log"))[:, None] * torch.nn.functional.softplus(z, threshold=1e9).reshape(S, T, H, D))
    beta = torch.sigmoid(torch.matmul(x, W(p + "b").t()))
    state, out = torch.zeros(S, H, D, V, dtype=torch.float64, device=DEVICE), torch.empty_like(v)
    for t in range(T):
        state.mul_(g[:, t, :, :, None])
        kt = k[:, t, :, :, None]
        u = (v[:, t] - (kt * state).sum(2)).mul_(beta[:, t, :, None])
        state.addcmul_(kt, u[:, :, None])
        out[:, t] = (q[:, t, :, :, None] * state).sum(2)
    gate = torch.sigmoid(torch.matmul(torch.matmul(x, W(p + "g1").t()), W(p + "g2").t()))
    return torch.matmul(_rms(out, W(p + "norm"), eps).reshape(S, T, H * V) * gate, W(p + "o").t())


def _parallel_mixer(x, W, p, m, eps):
    S, T, _ = x.shape
    a, b = m["left"], m["right"]
    q, k, v = (torch.matmul(x, W(p + "left." + n).t()).reshape(S, T, a["heads" if n == "q" else "kv_heads"], -1) for n in ("q", "k", "v"))
    q, k = _rms(q, 1.0, eps), _rms(k, 1.0, eps)
    t = torch.arange(T, device=DEVICE)
    d = t[:, None] - t[None]
    seen = (d >= 0) & (d < a["mask"]["size"])
    left = _each(x, lambda s: _causal(q[s], k[s], v[s], a["scale"], seen, sink=True).reshape(T, -1))
    H = b["heads"]
    q, k, v = (torch.nn.functional.silu(torch.matmul(x, W(p + "right." + n).t())).reshape(S, T, H, -1) for n in ("q", "k", "v"))
    decay = torch.tensor(b["decay"], dtype=torch.float64, device=DEVICE)
    out = torch.empty_like(v)
    for s in range(S):   # o_t = sum over j <= t of decay^(t - j) (q_t . k_j) v_j
        for h in range(H):
            w = torch.where(d >= 0, decay[h] ** d.clamp_min(0), 0.0).to(torch.float64)
            out[s, :, h] = torch.matmul(torch.matmul(q[s, :, h], k[s, :, h].t()) * w, v[s, :, h])
    right = _rms(out.reshape(S, T, -1), W(p + "right.norm"), eps)
    right = right * torch.sigmoid(torch.matmul(x, W(p + "right.g").t()))
    return m["left_scale"] * torch.matmul(left, W(p + "left.o").t()) + m["right_scale"] * torch.matmul(right, W(p + "right.o").t())


def _exact_rows(case, seed, ids):
    """the stream behind the last layer, normed, [S, T, width], and the head; ids [S, T] (what stands behind a sequence's end does not reach its rows)"""
    cfg, shapes, _ = _rows_config(case)
    P = dict(_rows_tensors(shapes, seed))
    W = lambda n: _f64(P[n])
    eps = cfg["norm"]["eps"]
    x = _f64(P["embed"][torch.from_numpy(ids).long().to(DEVICE)])
    if case["design"] == "bolopel":
        i = torch.arange(cfg["width"], device=DEVICE)
        a = torch.arange(x.shape[1], dtype=torch.float64, device=DEVICE)[:, None] * 10000.0 ** (-2.0 * (i // 2).double() / cfg["width"])
        x = _layer_norm(x + torch.where(i % 2 == 0, torch.sin(a), torch.cos(a)), W("embed.norm"), eps)
    for i, layer in enumerate(cfg["layers"]):
        p, m, f = "l%d." % i, layer["mixer"], layer["mlp"]
        if case["design"] == "tizusun":
            x = _rms(cfg["postln_alpha"] * x + _tizusun_mixer(x, W, p + "mix.", m, eps, (m["heads"], m["kv_heads"], m["dim"])), W(p + "norm1"), eps)
            y = _ff(x, W, p + "mlp.", torch.relu) if f["kind"] == "dense" else _experts(x, W, p + "mlp.", f)
            x = _rms(cfg["postln_alpha"] * x + y, W(p + "norm2"), eps)
        else:
            mixer = _delta_mixer if layer["type"] == "channel_delta" else _parallel_mixer
            x = x + _layer_norm(mixer(x, W, p + "mix.", m, eps), W(p + "norm1"), eps)
            x = x + _layer_norm(_ff(x, W, p + "mlp.", torch.nn.functional.silu), W(p + "norm2"), eps)
    return (_rms if case["design"] == "tizusun" else _layer_norm)(x, W("final.norm"), eps), W("head")


def _exact_train(case, seed):
    M = _gpt2_masters(case, seed)
    w, H, B, T = case["width"], case["heads"], case["batch"], case["tokens"]
    ids, tgt = (torch.from_numpy(a).long().to(DEVICE) for a in _ids(seed, (2, B * T), VOCAB))
    seen = torch.ones(T, T, dtype=torch.bool, device=DEVICE).tril()
    F, grads = torch.nn.functional, {}

    def leaf(name, value):
        grads[name] = _f64(value).requires_grad_()
        return grads[name]

    def f8(x):   # float8 e5m2: the upper byte of the half
        return ((x.float().half().view(torch.int16) & -256)).view(torch.float16)
    blocks = []
    for i, b in enumerate(M["blocks"]):
        p = {}
        for k in ("qkv", "proj", "fc", "proj2"):
            W, bias = b[k]
            p[k] = leaf("h%d.%s.w" % (i, k), f8(W) if k in ("qkv", "proj") else _stored(W, "q4"))
            p[k + "_b"] = leaf("h%d.%s.b" % (i, k), bias)
        for n, v in zip(("ln1.w", "ln1.b", "ln2.w", "ln2.b"), b["ln"]):
            p[n] = leaf("h%d.%s" % (i, n), v)
        blocks.append(p)
    wte, wpe, lw, lb = leaf("wte", M["wte"]), leaf("wpe", M["wpe"]), leaf("lnf.w", M["lnf"][0]), leaf("lnf.b", M["lnf"][1])

    def block(x, p):
        h = F.layer_norm(x, (w,), p["ln1.w"], p["ln1.b"], 1e-5)
        q, k, v = (torch.matmul(h, p["qkv"].t()) + p["qkv_b"]).reshape(B, T, 3, H, w // H).permute(2, 0, 3, 1, 4).contiguous()
        s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * (w // H) ** -0.5
        a = torch.matmul(torch.softmax(s.masked_fill(~seen, -math.inf), -1), v).permute(0, 2, 1, 3).reshape(B * T, w)
        x = x + torch.matmul(a, p["proj"].t()) + p["proj_b"]
        h = F.layer_norm(x, (w,), p["ln2.w"], p["ln2.b"], 1e-5)
        return x + torch.matmul(F.gelu(torch.matmul(h, p["fc"].t()) + p["fc_b"], approximate="tanh"), p["proj2"].t()) + p["proj2_b"]
    x = wte[ids] + wpe.repeat(B, 1)
    for p in blocks:
        x = torch.utils.checkpoint.checkpoint(block, x, p, use_reentrant=False)
    logits = torch.matmul(F.layer_norm(x, (w,), lw, lb, 1e-5), wte[:VOCAB].t())
    losses = F.cross_entropy(logits, tgt, reduction="none")
    losses.mean().backward()
    first = {"%s m" % n: (1 - HYPER["beta1"]) * g.grad for n, g in grads.items() if not n.startswith("h") or n.startswith(("h0.", "h%d." % (case["layers"] - 1)))}
    out = {n[:-1] + "p": None for n in first}   # the weights are rounded at random
    return dict(out, losses=losses.detach(), **first)


def exact(case, seed):
    _generator(seed)
    with torch.set_grad_enabled(case["kind"] == "train"):
        if case["kind"] == "decode":
            c, n, p, k = _qwen3_config(case), case["seqs"], case["pos"], case["steps"]
            ids = _ids(seed, (n, p + k), c["vocab"])
            lens = [p - (3 * s) % min(p, 48) + k if n > 1 else p + k for s in range(n)]
            return _exact_qwen3(case, seed, [ids[s, :lens[s]] for s in range(n)], n - 1, k)
        if case["kind"] == "prefill":
            c, lens = _qwen3_config(case), _lengths(case["prompts"], case["tokens"])
            ids = _ids(seed, (len(lens), max(lens)), c["vocab"])
            return _exact_qwen3(case, seed, [ids[s, :n] for s, n in enumerate(lens)], len(lens) - 1)
        if case["kind"] == "train":
            return _exact_train(case, seed)
        cfg, _, _ = _rows_config(case)
        if case["kind"] == "rows_prefill":
            lens = _lengths(case["spans"], case["tokens"])
            x, head = _exact_rows(case, seed, _ids(seed, (len(lens), max(lens)), cfg["vocab"]))
            return torch.stack([torch.matmul(head, x[i, r]) for i, r in _wanted(lens)])
        n, p, k = case["seqs"], case["pos"], case["steps"]
        x, head = _exact_rows(case, seed, _ids(seed, (n, p + k), cfg["vocab"]))
        return torch.stack([torch.matmul(head, x[s, p - (3 * s) % min(p, 48) + k - 1]) for s in range(n)])
