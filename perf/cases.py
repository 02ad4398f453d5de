"""What a user of this framework has it do, as cases that can be timed and checked.

The engine runs a step as a list of layers.  A case is one layer's part of such a step, or a whole step:

* ``attention`` -- one layer's attention node (``host.paged_attention`` on a bound step: the KV write, then split-K
  decode, causal prefill or the mixed step), over paged pools that hold each sequence's history;
* ``qkv``  -- the block before it: RMSNorm, the q / k / v projections, q/k norm + RoPE + KV write;
* ``mlp``  -- the SwiGLU block: RMSNorm, gate and up projections, SiLU, product, down projection, residual add;
* ``head`` -- the end of a step: final RMSNorm, gather of each sequence's last row, LM head, sampling;
* ``model`` -- a whole engine step of the Qwen3 forward (``Qwen3.forward``), which gives the step's logits.

Everything is bf16 with f32 norm gains and f32 RoPE tables, as the engine stores them.  A case holds plain sizes;
sequence lengths come from its ``lens`` number, tensors from the seed given to :func:`prepare`.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from llmgen_amd import attention as A
from llmgen_amd import host as H
from llmgen_amd import step as stepmod
from llmgen_amd._lib import lib
from llmgen_amd.qwen3 import Qwen3, Qwen3Config, weight_shapes

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
HD = 128  # head size of every supported model shape
EPS = 1e-6
THETA = 1_000_000.0


# ------------------------------------------------------------------------------------------------ the cases
def _attention(name, nq, nkv, block, max_len, lens, rows=0, row_lo=1, row_hi=1, first=0, chunks=0, chunk_lo=1,
               chunk_hi=1, past_lo=0, past_hi=0):
    """``rows`` decode rows with contexts in [row_lo, row_hi]; a fresh prompt of ``first`` tokens (0: none);
    ``chunks`` prefill chunks of [chunk_lo, chunk_hi] tokens behind [past_lo, past_hi] cached ones."""
    return {"name": name, "kind": "attention", "nq": nq, "nkv": nkv, "block": block, "max_len": max_len, "lens": lens,
            "rows": rows, "row_lo": row_lo, "row_hi": row_hi, "first": first, "chunks": chunks, "chunk_lo": chunk_lo,
            "chunk_hi": chunk_hi, "past_lo": past_lo, "past_hi": past_hi}


def listed():
    return [
        # one user, one token: the smallest call there is, 2 MB of cache
        _attention("decode_single", 16, 8, 256, 1024, 1, rows=1, row_lo=512, row_hi=512),
        # the ordinary decode step of a small server: 32 sequences of very different lengths
        _attention("decode_batch", 16, 8, 256, 1024, 2, rows=32, row_lo=128, row_hi=1024),
        # long-context decode, 2 GB of cache per layer
        _attention("decode_long", 32, 8, 256, 32768, 5, rows=16, row_lo=32768, row_hi=32768),
        # prompts arriving together: one long, eight short and ragged
        _attention("prefill_prompts", 16, 8, 256, 4096, 3, first=3584, chunks=8, chunk_lo=128, chunk_hi=512),
        # one very long prompt
        _attention("prefill_long", 32, 8, 256, 32768, 6, first=16384),
        # continuous batching: prefill chunks beside many decode rows
        _attention("mixed_batch", 16, 8, 256, 2048, 4, rows=248, row_lo=100, row_hi=2048, chunks=8, chunk_lo=512,
                   chunk_hi=512, past_lo=100, past_hi=1536),
        # the block before attention for a prefill step of ragged prompts
        {"name": "qkv_prefill", "kind": "qkv", "hidden": 1024, "nq": 16, "nkv": 8, "block": 16, "tokens": 2051},
        # the MLP of a decode step, and of a prefill step with an odd number of tokens
        {"name": "mlp_decode", "kind": "mlp", "hidden": 1024, "ffn": 3072, "tokens": 32},
        {"name": "mlp_prefill", "kind": "mlp", "hidden": 1024, "ffn": 3072, "tokens": 997},
        # the end of a decode step: a third of the sequences sample with a temperature, the others are greedy
        {"name": "head_decode", "kind": "head", "hidden": 1024, "vocab": 151936, "tokens": 32, "seqs": 32},
        # whole steps of the 28-layer model: eight sequences decoding, and three prompts prefilled together
        {"name": "model_decode", "kind": "model", "layers": 28, "rows": 8, "row_lo": 60, "row_hi": 900, "chunks": 0,
         "chunk_lo": 1, "chunk_hi": 1, "past_hi": 0, "lens": 8},
        {"name": "model_prefill", "kind": "model", "layers": 28, "rows": 0, "row_lo": 1, "row_hi": 1, "chunks": 3,
         "chunk_lo": 90, "chunk_hi": 250, "past_hi": 0, "lens": 9},
    ]


def _log_int(rng, lo, hi):
    """A whole number whose logarithm is even over [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_attention(rng):
    nq, nkv = rng.choice([(16, 8), (16, 8), (32, 8), (32, 8), (8, 8), (64, 8), (32, 2)])
    block = rng.choice([16, 16, 32, 48, 256, 256])
    lens = rng.randrange(1 << 30)
    what = rng.choice(["decode", "decode", "prefill", "chunk", "mixed"])
    if what == "decode":
        rows = _log_int(rng, 1, 256)
        # at most the cached tokens of the largest listed decode step
        hi = _log_int(rng, 32, min(32768, 524288 // rows))
        return _attention("", nq, nkv, block, hi, lens, rows=rows, row_lo=max(1, hi // rng.choice([1, 2, 8])), row_hi=hi)
    if what == "prefill":
        first = _log_int(rng, 33, 8192)
        n = rng.choice([0, 0, 1, 5, 12])
        hi = _log_int(rng, 17, 900)
        return _attention("", nq, nkv, block, max(first, hi), lens, first=first, chunks=n, chunk_lo=max(2, hi // 4),
                          chunk_hi=hi)
    past = _log_int(rng, 64, 16384)
    size = _log_int(rng, 16, 1024)
    n = rng.choice([1, 1, 2, 4])
    if what == "chunk":
        return _attention("", nq, nkv, block, past + size, lens, chunks=n, chunk_lo=max(2, size // 2), chunk_hi=size,
                          past_lo=past // 2, past_hi=past)
    rows = _log_int(rng, 1, 200)
    hi = _log_int(rng, 64, 3000)
    return _attention("", nq, nkv, block, max(past + size, hi), lens, rows=rows, row_lo=max(1, hi // 8), row_hi=hi,
                      chunks=n, chunk_lo=max(2, size // 2), chunk_hi=size, past_lo=past // 2, past_hi=past)


def draw(rng):
    kind = rng.choice(["attention"] * 5 + ["mlp", "mlp", "qkv", "head", "model"])
    if kind == "attention":
        c = _draw_attention(rng)
    elif kind == "mlp":
        hidden, ffn = rng.choice([(1024, 3072), (1024, 3072), (2048, 6144), (1536, 4104)])
        c = {"kind": "mlp", "hidden": hidden, "ffn": ffn, "tokens": _log_int(rng, 1, 2048)}
    elif kind == "qkv":
        hidden, nq, nkv = rng.choice([(1024, 16, 8), (1024, 16, 8), (2048, 16, 8), (2560, 32, 8), (1000, 8, 8)])
        c = {"kind": "qkv", "hidden": hidden, "nq": nq, "nkv": nkv, "block": rng.choice([16, 256]),
             "tokens": _log_int(rng, 1, 3000)}
    elif kind == "head":
        hidden, vocab = rng.choice([(1024, 151936), (1024, 151936), (2048, 151936), (1024, 32003)])
        seqs = _log_int(rng, 1, 100)
        c = {"kind": "head", "hidden": hidden, "vocab": vocab, "seqs": seqs, "tokens": seqs * rng.choice([1, 1, 7])}
    else:
        c = {"kind": "model", "layers": 28, "rows": rng.choice([0, 1, 2, 5, 16, 31]), "row_lo": 20,
             "row_hi": _log_int(rng, 40, 1000), "chunks": rng.choice([0, 1, 2]), "chunk_lo": 8,
             "chunk_hi": _log_int(rng, 16, 250), "past_hi": rng.choice([0, 300]), "lens": rng.randrange(1 << 30)}
        if c["rows"] + c["chunks"] == 0:
            c["rows"] = 3
    c.pop("name", None)
    return c


# ------------------------------------------------------------------------------------------------ shared pieces
def _lengths(c):
    """[(cached tokens, this step's tokens)] of the step's sequences."""
    r = np.random.default_rng(c["lens"])
    spec = [(0, c["first"])] if c.get("first") else []
    for _ in range(c["chunks"]):
        n = int(r.integers(c["chunk_lo"], c["chunk_hi"] + 1))
        spec.append((int(r.integers(c.get("past_lo", 0), c["past_hi"] + 1)), n))
    for _ in range(c["rows"]):
        spec.append((int(r.integers(c["row_lo"], c["row_hi"] + 1)) - 1, 1))
    return [spec[i] for i in r.permutation(len(spec))]


def _tables(spec, block, seed):
    """Block tables over shuffled physical blocks, and how many blocks they use."""
    need = [-(-(a + b) // block) for a, b in spec]
    ids = np.random.default_rng(seed).permutation(sum(need))
    ends = np.cumsum([0] + need)
    return [[int(i) for i in ids[ends[j]:ends[j + 1]]] for j in range(len(need))], int(ends[-1])


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape, std=1.0):
    """N(0, std) rounded to bf16, made in slices so that large pools need no f32 copy of themselves."""
    out = torch.empty(shape, dtype=BF16, device="cuda")
    flat, step = out.view(-1), 1 << 27
    for i in range(0, flat.numel(), step):
        part = flat[i:i + step]
        part.copy_(torch.randn(part.numel(), generator=gen, device="cuda") * std)
    return out


def _gains(gen, n):
    return 1 + 0.1 * torch.randn(n, generator=gen, device="cuda")


def _angles(n):
    inv = torch.pow(torch.tensor(THETA, dtype=F64, device="cuda"),
                    -torch.arange(0, HD, 2, dtype=F64, device="cuda") / HD)
    return torch.arange(n, dtype=F64, device="cuda")[:, None] * inv[None, :]


def _rope_tables(n):
    """cos / sin as the engine lays them out: [n, HD] f32, each half of a row the same."""
    a = _angles(n)
    return (torch.cat([a.cos(), a.cos()], 1).to(F32).contiguous(), torch.cat([a.sin(), a.sin()], 1).to(F32).contiguous())


def _token_slots(c, seed):
    """Positions and cache slots of a step's tokens: prompts of at most 1024 tokens, on shuffled blocks."""
    spec, left = [], c["tokens"]
    while left:
        n = min(left, 1024)
        spec.append((0, n))
        left -= n
    tables, nblocks = _tables(spec, c["block"], seed)
    pos = np.concatenate([np.arange(n) for _, n in spec])
    slots = np.concatenate([np.asarray(t)[np.arange(n) // c["block"]] * c["block"] + np.arange(n) % c["block"]
                            for (_, n), t in zip(spec, tables)])
    up = lambda x: torch.from_numpy(x.astype(np.int32)).cuda()  # noqa: E731
    return up(pos), up(slots), nblocks


def _p(t):
    return t.data_ptr()


# ------------------------------------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    A.init_device()
    return {"kind": case["kind"], **_PREPARE[case["kind"]](case, seed)}


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_attention(c, seed):
    gen, spec = _gen(seed), _lengths(c)
    tables, nblocks = _tables(spec, c["block"], seed)
    entries = [stepmod.Entry(a, b, t) for (a, b), t in zip(spec, tables)]
    mb = -(-c["max_len"] // c["block"])
    ws = A.Workspace.allocate(c["nq"], HD, len(spec), c["max_len"], A.meta_bytes(entries, mb))
    pool = (nblocks, c["nkv"], c["block"], HD)
    kc, vc = _normal(gen, *pool), _normal(gen, *pool)
    n = sum(b for _, b in spec)
    q, k, v = _normal(gen, n, c["nq"], HD), _normal(gen, n, c["nkv"], HD), _normal(gen, n, c["nkv"], HD)
    g = A.bind_step(entries, ws, c["nq"], c["nkv"], HD, c["block"], mb, c["max_len"])
    return {"ws": ws, "step": g, "q": q, "k": k, "v": v, "kc": kc, "vc": vc, "out": torch.zeros_like(q),
            "spec": spec, "tables": tables}


def _run_attention(s):
    H.paged_attention(s["step"], s["out"], s["q"], s["k"], s["v"], s["kc"], s["vc"])
    return {"out": s["out"], "k": s["kc"], "v": s["vc"]}


def _prepare_qkv(c, seed):
    gen = _gen(seed)
    T, D, nq, nkv = c["tokens"], c["hidden"], c["nq"], c["nkv"]
    pos, slots, nblocks = _token_slots(c, seed)
    cos, sin = _rope_tables(1024)
    s = {"x": _normal(gen, T, D), "norm": _gains(gen, D), "q_norm": _gains(gen, HD), "k_norm": _gains(gen, HD),
         "wq": _normal(gen, nq * HD, D, std=0.03), "wk": _normal(gen, nkv * HD, D, std=0.03),
         "wv": _normal(gen, nkv * HD, D, std=0.03), "cos": cos, "sin": sin, "pos": pos, "slots": slots}
    pool = (nblocks, nkv, c["block"], HD)
    s.update(kc=torch.zeros(pool, dtype=BF16, device="cuda"), vc=torch.zeros(pool, dtype=BF16, device="cuda"),
             xn=torch.empty_like(s["x"]), q=torch.empty((T, nq, HD), dtype=BF16, device="cuda"),
             k=torch.empty((T, nkv, HD), dtype=BF16, device="cuda"), v=torch.empty((T, nkv, HD), dtype=BF16, device="cuda"))
    return s


def _run_qkv(s):
    L = lib()
    T, D = s["x"].shape
    nq, nkv, block = s["q"].shape[1], s["k"].shape[1], s["kc"].shape[2]
    L.hip_rmsnorm(_p(s["xn"]), _p(s["x"]), _p(s["norm"]), T, D, EPS)
    L.hip_linear(_p(s["q"]), 0, _p(s["xn"]), _p(s["wq"]), T, nq * HD, D)
    L.hip_linear(_p(s["k"]), 0, _p(s["xn"]), _p(s["wk"]), T, nkv * HD, D)
    L.hip_linear(_p(s["v"]), 0, _p(s["xn"]), _p(s["wv"]), T, nkv * HD, D)
    L.hip_qk_norm_rope_store_kv(_p(s["q"]), _p(s["kc"]), _p(s["vc"]), _p(s["q"]), _p(s["k"]), _p(s["v"]),
                                _p(s["q_norm"]), _p(s["k_norm"]), EPS, _p(s["cos"]), _p(s["sin"]), _p(s["pos"]),
                                _p(s["slots"]), T, nq, nkv, HD, block)
    return {"q": s["q"], "k": s["kc"], "v": s["vc"]}


def _prepare_mlp(c, seed):
    gen = _gen(seed)
    T, D, F = c["tokens"], c["hidden"], c["ffn"]
    s = {"x": _normal(gen, T, D), "norm": _gains(gen, D), "gate": _normal(gen, F, D, std=0.03),
         "up": _normal(gen, F, D, std=0.03), "down": _normal(gen, D, F, std=0.03)}
    s.update(xn=torch.empty_like(s["x"]), o=torch.empty_like(s["x"]), y=torch.empty_like(s["x"]),
             g=torch.empty((T, F), dtype=BF16, device="cuda"), u=torch.empty((T, F), dtype=BF16, device="cuda"))
    return s


def _run_mlp(s):
    L = lib()
    (T, D), F = s["x"].shape, s["gate"].shape[0]
    L.hip_rmsnorm(_p(s["xn"]), _p(s["x"]), _p(s["norm"]), T, D, EPS)
    L.hip_linear(_p(s["g"]), 0, _p(s["xn"]), _p(s["gate"]), T, F, D)
    L.hip_linear(_p(s["u"]), 0, _p(s["xn"]), _p(s["up"]), T, F, D)
    L.hip_silu(_p(s["g"]), _p(s["g"]), T * F)
    L.hip_mul(_p(s["g"]), _p(s["g"]), _p(s["u"]), T * F)
    L.hip_linear(_p(s["o"]), 0, _p(s["g"]), _p(s["down"]), T, D, F)
    L.hip_add(_p(s["y"]), _p(s["x"]), _p(s["o"]), T * D)
    return s["y"]


def _prepare_head(c, seed):
    gen = _gen(seed)
    T, D, V, S = c["tokens"], c["hidden"], c["vocab"], c["seqs"]
    ends = np.linspace(T / S, T, S).astype(np.int32) - 1
    temps = torch.tensor([0.8 if i % 3 == 1 else 0.0 for i in range(S)], dtype=F32, device="cuda")
    s = {"x": _normal(gen, T, D), "norm": _gains(gen, D), "w": _normal(gen, V, D, std=0.03),
         "last": torch.from_numpy(ends).cuda(), "temps": temps,
         "seed": torch.tensor([seed * 7919 + 11], dtype=torch.int64, device="cuda")}
    s.update(xn=torch.empty_like(s["x"]), rows=torch.empty((S, D), dtype=BF16, device="cuda"),
             logits=torch.empty((S, V), dtype=BF16, device="cuda"), ids=torch.empty(S, dtype=torch.int32, device="cuda"))
    return s


def _run_head(s):
    L = lib()
    (T, D), (S, V) = s["x"].shape, s["logits"].shape
    L.hip_rmsnorm(_p(s["xn"]), _p(s["x"]), _p(s["norm"]), T, D, EPS)
    L.hip_gather_rows(_p(s["rows"]), _p(s["xn"]), _p(s["last"]), S, D)
    L.hip_linear(_p(s["logits"]), 0, _p(s["rows"]), _p(s["w"]), S, V, D)
    L.hip_sample(_p(s["ids"]), _p(s["logits"]), _p(s["temps"]), _p(s["seed"]), S, V, None)
    return {"logits": s["logits"], "ids": s["ids"]}


def _model_inputs(c, seed):
    """Weights, KV history and token ids of a whole-model case, all from the seed."""
    cfg, gen, spec = Qwen3Config(n_layers=c["layers"]), _gen(seed), _lengths(c)
    weights = {}
    for name, shape in weight_shapes(cfg).items():
        weights[name] = _gains(gen, shape[0]) if len(shape) == 1 else _normal(gen, *shape, std=0.02)
    tables, nblocks = _tables(spec, cfg.block_size, seed)
    kv = [[_normal(gen, nblocks, cfg.n_kv_head, cfg.block_size, HD, std=sd) for sd in (1.0, 0.6)]
          for _ in range(cfg.n_layers)]
    ids = np.random.default_rng(seed).integers(0, cfg.vocab, sum(b for _, b in spec))
    return cfg, spec, tables, nblocks, weights, kv, [int(i) for i in ids]


def _prepare_model(c, seed):
    cfg, spec, tables, nblocks, weights, kv, ids = _model_inputs(c, seed)
    host = {}
    for name, w in weights.items():  # the model takes its weights from host arrays, bf16 as bit patterns
        w = w.view(torch.int16) if w.dtype == BF16 else w
        host[name] = w.cpu().numpy().view(np.uint16) if w.dtype == torch.int16 else w.cpu().numpy()
    model = Qwen3(cfg, host, nblocks, max_seqs=max(8, len(spec)), max_tokens=1024)
    for layer, (k, v) in zip(model.kv, kv):
        layer.k.copy_(k)
        layer.v.copy_(v)
    return {"model": model, "entries": [stepmod.Entry(a, b, t) for (a, b), t in zip(spec, tables)], "ids": ids}


def _run_model(s):
    s["model"].forward(s["entries"], s["ids"])
    return s["model"].last_logits.view(BF16)


_PREPARE = {"attention": _prepare_attention, "qkv": _prepare_qkv, "mlp": _prepare_mlp, "head": _prepare_head,
            "model": _prepare_model}
_RUN = {"attention": _run_attention, "qkv": _run_qkv, "mlp": _run_mlp, "head": _run_head, "model": _run_model}


# ------------------------------------------------------------------------------------------------ work and tolerance
def _attention_work(spec, nq, nkv):
    cached = sum(a for a, _ in spec)
    new = sum(b for _, b in spec)
    # history read; this step's k and v read and written; q read and out written
    nbytes = 2 * HD * (2 * nkv * cached + 4 * nkv * new + 2 * nq * new)
    pairs = sum(b * a + b * (b + 1) // 2 for a, b in spec)
    return nbytes, 4 * HD * nq * pairs


def work(case):
    c, kind = case, case["kind"]
    if kind == "attention":
        nbytes, flops = _attention_work(_lengths(c), c["nq"], c["nkv"])
    elif kind == "qkv":
        T, D, n = c["tokens"], c["hidden"], (c["nq"] + 2 * c["nkv"]) * HD
        nbytes, flops = 2 * (T * D + n * D + T * n) + 8 * T * HD, 2 * T * D * n
    elif kind == "mlp":
        T, D, F = c["tokens"], c["hidden"], c["ffn"]
        nbytes, flops = 2 * (2 * T * D + 3 * F * D), 6 * T * D * F
    elif kind == "head":
        T, D, V, S = c["tokens"], c["hidden"], c["vocab"], c["seqs"]
        nbytes, flops = 2 * (S * D + V * D + S * V) + 4 * S, 2 * S * D * V
    else:
        cfg, spec = Qwen3Config(n_layers=c["layers"]), _lengths(c)
        T, S = sum(b for _, b in spec), len(spec)
        per = sum(s[0] * s[1] for n, s in weight_shapes(cfg).items() if n.startswith("blk.0.") and len(s) == 2)
        ab, af = _attention_work(spec, cfg.n_head, cfg.n_kv_head)
        kv = ab - 4 * HD * cfg.n_head * T  # q and out stay inside the layer
        nbytes = cfg.n_layers * (2 * per + kv) + 2 * (T * cfg.hidden + cfg.vocab * cfg.hidden + S * cfg.vocab)
        flops = cfg.n_layers * (2 * T * per + af) + 2 * S * cfg.vocab * cfg.hidden
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Four times what the path shows against 64-bit results: bf16 outputs are rounded once after f32 sums; blocks
    # round their inner tensors to bf16 too; 28 layers amplify such roundings.
    return {"attention": {"rel": 8e-3, "max": 0.05}, "qkv": {"rel": 1e-2, "max": 0.1}, "mlp": {"rel": 1e-2, "max": 0.1},
            "head": {"rel": 1e-2, "max": 0.1, "differ": 0.01}, "model": {"rel": 0.03, "max": 0.3}}[case["kind"]]


# ------------------------------------------------------------------------------------------------ 64-bit results
def exact(case, seed):
    A.init_device()
    return _EXACT[case["kind"]](case, seed)


def _attend64(q, kc, vc, spec, tables, block):
    """Causal attention of every sequence over its pages, in 64 bits: q [T, nq, HD] -> [T, nq, HD]."""
    nq, nkv = q.shape[1], kc.shape[1]
    out, t = torch.empty(q.shape, dtype=F64, device="cuda"), 0
    for (past, n), table in zip(spec, tables):
        blocks = torch.tensor(table, device="cuda")
        for h in range(nkv):
            k = kc[blocks, h].reshape(-1, HD)[:past + n].to(F64)
            v = vc[blocks, h].reshape(-1, HD)[:past + n].to(F64)
            kt = k.t().contiguous()
            for q0 in range(0, n, 2048):
                rows = min(2048, n - q0)
                end = past + q0 + rows  # later keys are hidden from all of these rows
                hidden = None
                if rows > 1:
                    at = past + q0 + torch.arange(rows, device="cuda")
                    hidden = torch.arange(end, device="cuda")[None, :] > at[:, None]
                for head in range(h * (nq // nkv), (h + 1) * (nq // nkv)):
                    s = q[t + q0:t + q0 + rows, head].to(F64) @ kt[:, :end]
                    s *= 1 / math.sqrt(HD)
                    if hidden is not None:
                        s.masked_fill_(hidden, -math.inf)
                    out[t + q0:t + q0 + rows, head] = torch.softmax(s, -1) @ v[:end]
        t += n
    return out


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.to(F64)


def _rope64(x, pos):
    a = _angles(int(pos.max()) + 1)[pos.long()][:, None, :]
    x0, x1 = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x1 * a.cos() + x0 * a.sin()], -1)


def _put64(pool, slots, rows):
    """The pool in 64 bits with ``rows`` [T, nkv, HD] at their slots."""
    out, block = pool.to(F64), pool.shape[2]
    slots = slots.long()
    out[slots // block, :, slots % block] = rows.to(F64)
    return out


def _exact_attention(c, seed):
    s = _prepare_attention(c, seed)
    slots = torch.tensor([tb[p // c["block"]] * c["block"] + p % c["block"]
                          for (a, b), tb in zip(s["spec"], s["tables"]) for p in range(a, a + b)], device="cuda")
    for pool, new in ((s["kc"], s["k"]), (s["vc"], s["v"])):  # the KV write moves bits
        pool[slots // c["block"], :, slots % c["block"]] = new
    return {"out": _attend64(s["q"], s["kc"], s["vc"], s["spec"], s["tables"], c["block"]), "k": None, "v": None}


def _exact_qkv(c, seed):
    s = _prepare_qkv(c, seed)
    T = c["tokens"]
    xn = _norm64(s["x"].to(F64), s["norm"])
    q, k, v = ((xn @ s[w].to(F64).t()).view(T, -1, HD) for w in ("wq", "wk", "wv"))
    q, k = _rope64(_norm64(q, s["q_norm"]), s["pos"]), _rope64(_norm64(k, s["k_norm"]), s["pos"])
    return {"q": q, "k": _put64(s["kc"], s["slots"], k), "v": _put64(s["vc"], s["slots"], v)}


def _mlp64(x, norm, gate, up, down):
    xn = _norm64(x, norm)
    g = xn @ gate.to(F64).t()
    return x + (g * torch.sigmoid(g) * (xn @ up.to(F64).t())) @ down.to(F64).t()


def _exact_mlp(c, seed):
    s = _prepare_mlp(c, seed)
    return _mlp64(s["x"].to(F64), s["norm"], s["gate"], s["up"], s["down"])


def _exact_head(c, seed):
    s = _prepare_head(c, seed)
    rows = _norm64(s["x"].to(F64), s["norm"])[s["last"].long()]
    return {"logits": rows @ s["w"].to(F64).t(), "ids": None}


def _exact_model(c, seed):
    cfg, spec, tables, _, w, kv, ids = _model_inputs(c, seed)
    pos = torch.tensor([p for a, b in spec for p in range(a, a + b)], device="cuda")
    slots = torch.tensor([tb[p // cfg.block_size] * cfg.block_size + p % cfg.block_size
                          for (a, b), tb in zip(spec, tables) for p in range(a, a + b)], device="cuda")
    T, last = len(ids), torch.tensor(np.cumsum([b for _, b in spec]) - 1, device="cuda")
    x = w["token_embd.weight"][torch.tensor(ids, device="cuda")].to(F64)
    for i in range(cfg.n_layers):
        m = lambda n: w["blk.%d.%s.weight" % (i, n)]  # noqa: E731,B023
        xn = _norm64(x, m("attn_norm"))
        q, k, v = ((xn @ m("attn_" + n).to(F64).t()).view(T, -1, HD) for n in "qkv")
        q, k = _rope64(_norm64(q, m("attn_q_norm")), pos), _rope64(_norm64(k, m("attn_k_norm")), pos)
        kc, vc = _put64(kv[i][0], slots, k), _put64(kv[i][1], slots, v)
        o = _attend64(q, kc, vc, spec, tables, cfg.block_size).reshape(T, -1)
        x = x + o @ m("attn_output").to(F64).t()
        x = _mlp64(x, m("ffn_norm"), m("ffn_gate"), m("ffn_up"), m("ffn_down"))
    return _norm64(x, w["output_norm.weight"])[last] @ w["token_embd.weight"].to(F64).t()


_EXACT = {"attention": _exact_attention, "qkv": _exact_qkv, "mlp": _exact_mlp, "head": _exact_head,
          "model": _exact_model}
