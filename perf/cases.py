"""What the engine is timed on: dense decoders served through Engine.prefill / prefill_batch / replay.

The two model shapes are the repository's own (Qwen3-0.6B and Llama-3-8B, llm/synthetic.py) at full depth, with random weights whose
scale keeps the residual stream and the logits where a trained model has them: unit-variance projections, small contributions of the
layers, logits with one clear favourite over a flat tail (which also makes every greedy chain the same on every correct implementation).

  decode         `steps` tokens for each of `batch` sequences, one captured step per token, contexts from `context` down to
                 `shortest` of it; greedy, or drawn with temperature, top-k and top-p
  prefill        one prompt of `tokens` into an empty cache
  chunk          `tokens` more of a prompt whose first `context` positions are cached
  prefill_batch  `batch` prompts of different lengths, the longest `tokens`, in one call

Formats: bf16, and fp8 (e4m3 weights, bf16 activations).  The third, fp8a8, rounds activations to e4m3 too: over a whole model that doubles
any difference in the order of a sum until the results of two correct programs are over a tenth apart, so there is nothing to compare."""

from __future__ import annotations

import math

import numpy as np
import torch

from pygpukit_amd.core.array import GPUArray
from pygpukit_amd.core.dtypes import bfloat16, uint8
from pygpukit_amd.llm.engine import Engine
from pygpukit_amd.llm.synthetic import LLAMA3_8B, QWEN3_0_6B

MODELS = {"qwen3-0.6b": QWEN3_0_6B, "llama3-8b": LLAMA3_8B}
MATS = ("w_qkv", "w_o", "w_gate_up", "w_down")


def _case(kind, model, fmt, *, batch=1, tokens=0, context=0, shortest=1.0, steps=0, sampled=False, name=None):
    c = {"kind": kind, "model": model, "format": fmt, "batch": batch, "tokens": tokens, "context": context, "shortest": shortest, "steps": steps, "sampled": sampled}
    return dict(c, name=name) if name else c


def listed():
    q, l = "qwen3-0.6b", "llama3-8b"
    return [
        # one token for one user: the smallest call, nothing but launches and latency
        _case("decode", q, "bf16", context=131, steps=1, name="q06 decode 1 token"),
        # one user deep into a conversation, quantised weights
        _case("decode", q, "fp8", context=2048, steps=16, name="q06 fp8 decode ctx 2048"),
        # a handful of users, sampled as chat front ends do
        _case("decode", q, "bf16", batch=5, context=300, shortest=0.3, steps=8, sampled=True, name="q06 decode 5 sampled"),
        # a full batch of fresh conversations
        _case("decode", q, "bf16", batch=64, context=190, shortest=0.7, steps=8, name="q06 decode 64"),
        # a serving batch in its steady state: contexts of every length up to the cache's
        _case("decode", q, "fp8", batch=37, context=3900, shortest=0.05, steps=4, name="q06 fp8 decode 37 long"),
        # a short question
        _case("prefill", q, "bf16", tokens=93, name="q06 prefill 93"),
        # a document
        _case("prefill", q, "bf16", tokens=1531, name="q06 prefill 1531"),
        # requests that arrived together: system prompt and a question each
        _case("prefill_batch", q, "bf16", batch=16, tokens=400, shortest=0.05, name="q06 prefill 16 prompts"),
        # the next turn of a long conversation, or a piece of a prompt that is prefilled in pieces
        _case("chunk", q, "fp8", tokens=384, context=3201, name="q06 fp8 chunk at 3201"),
        # the larger model, one user
        _case("decode", l, "fp8", context=700, steps=4, name="l8b fp8 decode ctx 700"),
        # the larger model, a few users (it decodes at most seven sequences together)
        _case("decode", l, "bf16", batch=6, context=1100, shortest=0.1, steps=2, name="l8b decode 6"),
        # the larger model, a long prompt
        _case("prefill", l, "fp8", tokens=4096, name="l8b fp8 prefill 4096"),
    ]


def draw(rng):
    def log(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))

    model = rng.choice(("qwen3-0.6b", "qwen3-0.6b", "llama3-8b"))
    large = model == "llama3-8b"
    kind = rng.choice(("decode", "decode", "decode", "prefill", "prefill_batch", "chunk"))
    if kind == "decode":
        most = 7 if large else 64
        batch = rng.choice((1, log(2, most), log(2, most)))
        return _case(kind, model, rng.choice(("bf16", "fp8")), batch=batch, context=log(32, 1500 if large else 3900), shortest=round(rng.uniform(0.05, 1.0), 3),
                     steps=rng.randint(1, 2 if large else 4), sampled=rng.random() < 0.3)
    if kind == "prefill":
        return _case(kind, model, rng.choice(("bf16", "fp8")), tokens=log(8, 2000 if large else 4000))
    if kind == "chunk":
        return _case(kind, model, rng.choice(("bf16", "fp8")), tokens=log(16, 1000), context=log(100, 3000))
    return _case(kind, model, rng.choice(("bf16", "fp8")), batch=log(2, 8 if large else 24), tokens=log(24, 512), shortest=round(rng.uniform(0.05, 1.0), 3))


# ---------------------------------------------------------------------------------------------- inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _config(case):
    cfg = dict(MODELS[case["model"]])
    cfg["qk_norm"] = case["model"] == "qwen3-0.6b"
    return cfg


def _spread(n, longest, shortest):
    """`n` lengths from longest * shortest up to longest, in an order that is not sorted."""
    lo = max(1, int(longest * shortest))
    v = [longest - (longest - lo) * i // max(1, n - 1) for i in range(n)]
    return [v[i * 7 % n] if n % 7 else v[(i * 5 + 1) % n if n % 5 else i] for i in range(n)]


def _lengths(case):
    """(lengths of the new prompts, positions cached before the call), a value per sequence"""
    b = case["batch"]
    if case["kind"] == "decode":
        return [0] * b, _spread(b, case["context"], case["shortest"])
    if case["kind"] == "prefill_batch":
        return _spread(b, case["tokens"], case["shortest"]), [0] * b
    return [case["tokens"]], [case["context"]]


def _rows(case):
    new, old = _lengths(case)
    return (max(n + o for n, o in zip(new, old)) + case["steps"] + 15) // 8 * 8


def _quantised(w):
    """e4m3 codes and bf16 scales of 128 x 128 blocks"""
    n, k = w.shape
    blocks = w.float().view(n // 128, 128, k // 128, 128)
    scale = (blocks.abs().amax(dim=(1, 3)) / 448).to(torch.bfloat16)
    codes = (blocks / scale.float()[:, None, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return codes.view(n, k).view(torch.uint8), scale


def _weights(case, gen):
    """embed, final norm, and each layer's matrices (a pair of codes and scales each for fp8) and norms, layer by layer"""
    c = _config(case)
    H, D, F, L = c["hidden_size"], c["head_dim"], c["intermediate_size"], c["num_layers"]
    qd, nqkv = c["num_heads"] * D, (c["num_heads"] + 2 * c["num_kv_heads"]) * D

    def normal(*shape, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=torch.bfloat16, device=_device()).normal_(mean, std, generator=gen)

    out = 0.5 / math.sqrt(2 * L)
    yield normal(c["vocab_size"], H, std=2 / math.sqrt(H)), normal(H, mean=1.0, std=0.05)
    for _ in range(L):
        lw = {"w_qkv": normal(nqkv, H, std=H**-0.5), "w_o": normal(H, qd, std=out * qd**-0.5), "w_gate_up": normal(2 * F, H, std=H**-0.5), "w_down": normal(H, F, std=out * F**-0.5)}
        if case["format"] != "bf16":
            lw = {k: _quantised(w) for k, w in lw.items()}
        lw.update(attn_norm=normal(H, mean=1.0, std=0.1), mlp_norm=normal(H, mean=1.0, std=0.1))
        if c["qk_norm"]:
            lw.update(q_norm=normal(D, mean=1.0, std=0.1), k_norm=normal(D, mean=1.0, std=0.1))
        yield lw


def _generators(seed):
    gens = [torch.Generator(device=_device()) for _ in range(2)]
    for i, g in enumerate(gens):
        g.manual_seed(seed * 2 + i + 1)
    return gens


def _token_ids(case, seed):
    """prompts (or, decoding, the one token each sequence goes on from)"""
    rng = np.random.default_rng(seed)
    return [rng.integers(0, _config(case)["vocab_size"], max(1, n)).astype(np.int32) for n in _lengths(case)[0]]


class _Wrapped:
    def __init__(self, address, shape, kind):
        self.__cuda_array_interface__ = {"data": (address, False), "shape": tuple(shape), "typestr": kind, "version": 2}


def _tensor(a, kind, copies=1):
    """The memory of a GPUArray, or of `copies` arrays like it that lie end to end"""
    return torch.as_tensor(_Wrapped(a.data_ptr(), a.shape if copies == 1 else (copies, *a.shape), kind), device="cuda")


def _array(t):
    return GPUArray(tuple(t.shape), uint8 if t.dtype == torch.uint8 else bfloat16, t.data_ptr(), owns_memory=False)


def prepare(case, seed):
    c = _config(case)
    gen, gen_kv = _generators(seed)
    new, old = _lengths(case)
    parts = _weights(case, gen)
    embed, final = next(parts)
    keep, layers = [embed, final], []
    for lw in parts:
        arrays = {"q_norm": None, "k_norm": None}
        for k, w in lw.items():
            if isinstance(w, tuple):
                arrays[k], arrays["s" + k[1:]] = _array(w[0]), _array(w[1])
            else:
                arrays[k] = _array(w)
            keep.append(w)
        layers.append(arrays)
    torch.cuda.synchronize()
    engine = Engine(c, _array(embed), layers, _array(final), None, max_seq_len=_rows(case), max_batch=case["batch"], weight_format=case["format"], use_qk_norm=c["qk_norm"])
    # the engine's whole cache, all layers of it
    caches = [_tensor(a, "<i2", c["num_layers"]).view(torch.bfloat16) for a in engine.kv_cache(0)]
    engine.synchronize()
    if max(old):
        for k, v in zip(*caches):    # what earlier turns left; rows beyond a sequence's context are never read
            k.normal_(generator=gen_kv)
            v.normal_(generator=gen_kv)
    state = {"case": dict(case), "engine": engine, "keep": keep, "tokens": _token_ids(case, seed), "old": old, "caches": caches}
    if case["kind"] == "decode":
        state["first"] = np.concatenate(state["tokens"])
        state["positions"] = np.asarray(old, np.int32)
        if case["sampled"]:
            engine.set_sampling(0.7, 50, 0.9, n_steps=max(16, case["steps"]), seed=seed)
        engine.capture(case["batch"])
        state["logits"] = _tensor(engine.logits(case["batch"]), "<f4")
    torch.cuda.synchronize()
    return state


def run(state):
    engine, case = state["engine"], state["case"]
    if case["kind"] == "decode":
        engine.reset_log()
        engine.set_state(state["first"], state["positions"])
        engine.replay(case["steps"])
        return {"tokens": engine.read_tokens(case["batch"], case["steps"]), "logits": state["logits"]}
    if case["kind"] == "prefill_batch":
        logits = engine.prefill_batch(state["tokens"])
    else:
        logits = engine.prefill(state["tokens"][0], seq=0, start_pos=state["old"][0])
    return {"logits": logits, "keys": state["caches"][0], "values": state["caches"][1]}


# ---------------------------------------------------------------------------------------------- what it is measured against

def _sizes(case):
    c = _config(case)
    H, D, F, L = c["hidden_size"], c["head_dim"], c["intermediate_size"], c["num_layers"]
    qd, kvd = c["num_heads"] * D, c["num_kv_heads"] * D
    return c, L, L * (H * (qd + 2 * kvd) + qd * H + 3 * H * F), 2 * kvd * 2 * L, 4 * qd * L      # linear weights, cache bytes a position, flops a (query, key)


def work(case):
    c, L, linear, row, pair = _sizes(case)
    H, V = c["hidden_size"], c["vocab_size"]
    weights = linear * 2 if case["format"] == "bf16" else linear + linear // 16384 * 2
    new, old = _lengths(case)
    if case["kind"] == "decode":
        n, b = case["steps"], case["batch"]
        seen = sum(n * o + n * (n + 1) // 2 for o in old)
        return {"bytes": n * (weights + V * H * 2 + b * V * 4) + row * (sum(n * o for o in old) + n * b), "flops": 2 * n * b * (linear + V * H) + pair * seen}
    pairs = sum(n * o + n * (n + 1) // 2 for n, o in zip(new, old))
    rows = sum(new)
    return {"bytes": weights + V * H * 2 + len(new) * V * 4 + row * (sum(old) + rows), "flops": 2 * rows * linear + 2 * len(new) * V * H + pair * pairs}


def tolerance(case):
    # measured against exact(): 0.0004 to 0.0015 where one sequence decodes on fp32 activations, 0.007 to 0.015 where bf16 ones are multiplied
    return {"rel": 0.006 if case["kind"] == "decode" and case["batch"] == 1 else 0.03}


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _turn(x, positions, theta):
    """[rows, heads, D] by the angles of the rows' positions, column i against i + D / 2"""
    half = x.shape[-1] // 2
    freq = theta ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    a = positions.double()[:, None, None] * freq
    x0, x1 = x[..., :half], x[..., half:]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x1 * a.cos() + x0 * a.sin()], -1)


def _wide(w):
    if not isinstance(w, tuple):
        return w.double()
    codes, scale = w
    n, k = codes.shape
    x = codes.view(torch.float8_e4m3fn).float().view(n // 128, 128, k // 128, 128) * scale.float()[:, None, :, None]
    return x.view(n, k).double()


def _layer(c, lw, h, k, v, spans, old):
    """One layer on the rows of all sequences; spans: rows of each sequence; k, v: its cache, written in place."""
    Hq, G, D, F, eps = c["num_heads"], c["num_kv_heads"], c["head_dim"], c["intermediate_size"], c["norm_eps"]
    x = _norm(h, lw["attn_norm"], eps) @ _wide(lw["w_qkv"]).T
    q, kk, vv = (t.reshape(len(h), -1, D) for t in x.split([Hq * D, G * D, G * D], 1))
    if c["qk_norm"]:
        q, kk = _norm(q, lw["q_norm"], eps), _norm(kk, lw["k_norm"], eps)
    att = torch.empty(len(h), Hq * D, dtype=torch.float64, device=h.device)
    for b, (lo, hi) in enumerate(spans):
        n, o = hi - lo, old[b]
        at = torch.arange(o, o + n, device=h.device)
        k[b, :, o:o + n] = _turn(kk[lo:hi], at, c["rope_theta"]).transpose(0, 1)
        v[b, :, o:o + n] = vv[lo:hi].transpose(0, 1)
        qs = _turn(q[lo:hi], at, c["rope_theta"])
        hidden = torch.arange(o + n, device=h.device)[None, :] > at[:, None]
        for g in range(G):
            ks, vs, m = k[b, g, :o + n].double(), v[b, g, :o + n].double(), Hq // G
            for i in range(g * m, (g + 1) * m):
                s = (qs[:, i] @ ks.T / math.sqrt(D)).masked_fill_(hidden, -math.inf)
                att[lo:hi, i * D:(i + 1) * D] = s.softmax(-1) @ vs
    h = h + att @ _wide(lw["w_o"]).T
    gate, up = (_norm(h, lw["mlp_norm"], eps) @ _wide(lw["w_gate_up"]).T).split(F, 1)
    return h + (torch.nn.functional.silu(gate) * up) @ _wide(lw["w_down"]).T


def _one_each(c, lw, h, k, v, old):
    """_layer for one row a sequence, all sequences at once; k, v: the bf16 rows before this call and, last, a list of the rows since"""
    Hq, G, D, F, eps = c["num_heads"], c["num_kv_heads"], c["head_dim"], c["intermediate_size"], c["norm_eps"]
    B, done, dev = len(h), len(k[1]), h.device
    at = torch.tensor(old, device=dev) + done
    x = _norm(h, lw["attn_norm"], eps) @ _wide(lw["w_qkv"]).T
    q, kk, vv = (t.reshape(B, -1, D) for t in x.split([Hq * D, G * D, G * D], 1))
    if c["qk_norm"]:
        q, kk = _norm(q, lw["q_norm"], eps), _norm(kk, lw["k_norm"], eps)
    q, kk = _turn(q, at, c["rope_theta"]), _turn(kk, at, c["rope_theta"])
    k[1].append(kk)
    v[1].append(vv)
    att = torch.empty(B, Hq, D, dtype=torch.float64, device=dev)
    for b in range(B):
        ks = torch.cat([k[0][b, :, :old[b]].double(), torch.stack([r[b] for r in k[1]], 1)], 1)
        vs = torch.cat([v[0][b, :, :old[b]].double(), torch.stack([r[b] for r in v[1]], 1)], 1)
        att[b] = ((q[b].view(G, Hq // G, D) @ ks.transpose(1, 2) / math.sqrt(D)).softmax(-1) @ vs).reshape(Hq, D)
    h = h + att.reshape(B, -1) @ _wide(lw["w_o"]).T
    gate, up = (_norm(h, lw["mlp_norm"], eps) @ _wide(lw["w_gate_up"]).T).split(F, 1)
    return h + (torch.nn.functional.silu(gate) * up) @ _wide(lw["w_down"]).T


def _head(c, h, embed, final):
    x = _norm(h, final, c["norm_eps"])
    return torch.cat([x @ part.double().T for part in embed.split(32768)], 1)


def exact(case, seed):
    """The weights of a quantised format are the numbers their codes stand for; activations are never rounded.  The sampled cases' nucleus
    holds the favourite alone, so that a draw is what greedy decoding gives."""
    c, dev = _config(case), _device()
    gen, gen_kv = _generators(seed)
    parts = list(_weights(case, gen))
    (embed, final), layers = parts[0], parts[1:]
    new, old = _lengths(case)
    tokens = _token_ids(case, seed)
    shape = (case["batch"], c["num_kv_heads"], _rows(case), c["head_dim"])
    rows = []
    for _ in layers:
        kv = [torch.zeros(shape, dtype=torch.bfloat16, device=dev) for _ in range(2)]
        if max(old):
            for x in kv:
                x.normal_(generator=gen_kv)
        rows.append(kv)
    if case["kind"] == "decode":
        caches = [((k, []), (v, [])) for k, v in rows]
        cur, log = torch.as_tensor(np.concatenate(tokens), device=dev), []
        for _ in range(case["steps"]):
            h = embed[cur.long()].double()
            for lw, (k, v) in zip(layers, caches):
                h = _one_each(c, lw, h, k, v, old)
            logits = _head(c, h, embed, final)
            cur = logits.argmax(1).to(torch.int32)
            log.append(cur)
        return {"tokens": torch.stack(log).cpu().numpy(), "logits": logits}
    edges = np.concatenate([[0], np.cumsum(new)])
    spans = [(int(a), int(b)) for a, b in zip(edges, edges[1:])]
    h = embed[torch.as_tensor(np.concatenate(tokens), device=dev).long()].double()
    for i, lw in enumerate(layers):
        kv = [x.double() for x in rows[i]]
        h = _layer(c, lw, h, kv[0], kv[1], spans, old)
        rows[i] = kv
    logits = _head(c, h[torch.as_tensor([b - 1 for _, b in spans], device=dev)], embed, final)
    return {"logits": (logits if case["kind"] == "prefill_batch" else logits[0]).cpu().numpy(), "keys": torch.stack([k for k, _ in rows]), "values": torch.stack([v for _, v in rows])}
