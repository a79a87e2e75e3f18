"""The work that is measured: what a program that serves GGUF models through this backend asks of it, call by call.

Every case is one `mi355_decode` of a batch and the reading of its output rows (a prompt longer than n_batch: one call per n_batch chunk), on the models
of `gguf_synth.CONFIGS`:

  step     one token of one conversation: what a user waits for, token by token
  slots    one tick of a server with several conversations, one token each (n_parallel), their contexts of different lengths
  prompt   a prompt, or the next turn of a conversation behind what its cache holds already, up to the logits of its last token
  embed    a text through the encoder, up to its tokens' embeddings

A model file is written once per process tree with fixed weights (random valid blocks of the file type's mix, `gguf_synth`) and stays loaded, as a server's
model does; the seed makes the conversations.  `layers` cuts a model's depth (0: all of them): every layer does the same work, and an int8 rounding of an
activation that falls the other way (see `tolerance`) grows with every layer that it passes, with a router's choice behind it to a row of its own.  The cut
models' weights are still larger than what the last level of cache holds.
"""
import ctypes
import dataclasses
import math
import os
import tempfile

import numpy as np
import torch

from __graft_entry__ import load_pkg

pkg = load_pkg()
synth = pkg.gguf_synth

CACHE = {"f16": 1, "q8_0": 8}
N_BATCH = 2048                 # n_batch = n_ubatch of the engine and of bench.py
# file type, cache type and layers each model is run with
MODELS = {
    "tinyllama-1.1b": ("q8_0", "f16", 6),
    "llama-2-7b": ("q5_k_m", "f16", 8),
    "llama-3-8b": ("q4_k_m", "q8_0", 8),
    "mixtral-8x7b": ("q5_k_m", "q8_0", 2),
    "nomic-embed": ("f16", "f16", 0),
}


def _case(name, do, model, **sizes):
    ftype, cache, layers = MODELS[model]
    c = {"do": do, "model": model, "ftype": ftype, "cache": cache, "layers": layers, "n": 1, "past": 0, "spread": 0}
    c.update(sizes)
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest model that is served, early in a conversation: launches and latency
        _case("step small model", "step", "tinyllama-1.1b", past=93),
        # the benchmark's decode step: one user, half a thousand tokens into the conversation
        _case("step", "step", "llama-3-8b", past=515),
        # the same with the context nearly full: the cache's bytes beside the weights'
        _case("step full context", "step", "llama-3-8b", past=3970),
        # as many kv heads as query heads, an f16 cache, 5-bit weights: the other common file
        _case("step 7b", "step", "llama-2-7b", past=1201),
        # a mixture of experts: two of eight experts' weights per token
        _case("step experts", "step", "mixtral-8x7b", past=700),
        # a small server's tick: four conversations
        _case("slots 4", "slots", "llama-3-8b", n=4, past=180, spread=211),
        # a busy server's tick
        _case("slots 16", "slots", "llama-3-8b", n=16, past=90, spread=61),
        # the next user turn of a conversation: a few words behind a cached prefix
        _case("prompt turn", "prompt", "llama-3-8b", n=37, past=640),
        # the benchmark's prompt
        _case("prompt", "prompt", "llama-3-8b", n=512),
        # a document: more than one batch
        _case("prompt long", "prompt", "llama-3-8b", n=3967),
        # a prompt through experts
        _case("prompt experts", "prompt", "mixtral-8x7b", n=611),
        # a paragraph for a vector store
        _case("embed", "embed", "nomic-embed", n=187),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["step", "step", "slots", "slots", "prompt", "prompt", "prompt", "embed"])
    if do == "embed":
        return _case(None, do, "nomic-embed", n=_log(rng, 3, 2000))
    model = rng.choice(["llama-3-8b", "llama-3-8b", "llama-2-7b", "tinyllama-1.1b", "mixtral-8x7b"])
    if do == "slots" and model == "mixtral-8x7b":   # one expert chosen otherwise is another row, and a tick has many rows (see `tolerance`)
        model = "llama-3-8b"
    most = 2000 if model == "tinyllama-1.1b" else 3968
    if do == "step":
        return _case(None, do, model, past=_log(rng, 4, most))
    if do == "slots":
        n = _log(rng, 2, 32)
        return _case(None, do, model, n=n, past=_log(rng, 8, 400), spread=rng.randrange(0, 1 + 1500 // n))
    n = _log(rng, 2, most)
    return _case(None, do, model, n=n, past=rng.choice([0, rng.randrange(0, most - n + 1)]))


def _config(case):
    cfg = synth.CONFIGS[case["model"]]
    return dataclasses.replace(cfg, n_layer=case["layers"]) if case["layers"] else cfg


def _file(case):
    """The model's file: written by the first process that needs it."""
    cfg = _config(case)
    path = os.path.join(tempfile.gettempdir(), "perf_%s_%s_%d_%d.gguf" % (case["model"], case["ftype"], cfg.n_layer, os.getuid()))
    if not os.path.exists(path):
        part = "%s.%d" % (path, os.getpid())
        synth.write_synthetic_llama(part, cfg, case["ftype"])
        os.replace(part, path)
    return path


_kept = {}


def _model(case):
    """The loaded model; one at a time is kept, as long as its conversations live."""
    key = (case["model"], case["ftype"], case["layers"])
    if key not in _kept:
        _kept.clear()
        _kept[key] = _Model(_file(case))
    return _kept[key]


class _Model(pkg.Model):
    def __del__(self):
        if getattr(self, "h", None):
            self.close()


def _conversations(case, seed):
    """[(tokens, past)]: `past` of the tokens are in the cache before the call, the others are its batch."""
    rng = np.random.default_rng([int(seed), 7])
    lo = 5 if case["do"] == "embed" else 3
    out = []
    for s in range(case["n"] if case["do"] == "slots" else 1):
        past = case["past"] + s * case["spread"] if case["do"] == "slots" else case["past"]
        new = case["n"] if case["do"] in ("prompt", "embed") else 1
        out.append((rng.integers(lo, synth.CONFIGS[case["model"]].n_vocab, past + new).astype(np.int32), past))
    return out


class _State:
    """A context of the model with its conversations' pasts in the cache, and the batches of the call that follows."""

    def __init__(self, case, seed):
        self.model = _model(case)
        self.lib = self.model.lib
        self.embed = case["do"] == "embed"
        talks = _conversations(case, seed)
        cells = sum(len(t) for t, _ in talks)
        kv = CACHE[case["cache"]]
        self.ctx = pkg.Context(self.model, n_ctx=max(4096, -(-cells // 256) * 256), n_batch=N_BATCH, n_ubatch=N_BATCH, n_seq_max=len(talks), type_k=kv, type_v=kv)
        for s, (toks, past) in enumerate(talks):
            for i in range(0, past, N_BATCH):
                part = toks[i:min(past, i + N_BATCH)]
                if self.ctx.decode(part, np.arange(i, i + part.size), s) != 0:
                    raise RuntimeError("no cells for the conversation's past")
        self.cut = [(s, past) for s, (_, past) in enumerate(talks)]
        self.batches, self.held = [], []
        if len(talks) > 1:
            self._add([(toks[past], past, s, True) for s, (toks, past) in enumerate(talks)])
        else:
            toks, past = talks[0]
            for i in range(past, len(toks), N_BATCH):
                self._add([(toks[p], p, 0, self.embed or p == len(toks) - 1) for p in range(i, min(len(toks), i + N_BATCH))])
        self.rows = [i for i in range(len(talks))] if len(talks) > 1 else [-1]
        self.ctx.synchronize()

    def _add(self, entries):
        b = self.lib.mi355_batch_init(len(entries), 0, 1)
        b.n_tokens = len(entries)
        for i, (tok, pos, seq, flag) in enumerate(entries):
            b.token[i], b.pos[i], b.n_seq_id[i], b.logits[i] = int(tok), int(pos), 1, int(flag)
            b.seq_id[i][0] = seq
        self.batches.append(b)

    def __del__(self):
        for b in getattr(self, "batches", []):
            self.lib.mi355_batch_free(b)
        if getattr(self, "ctx", None) is not None:
            self.ctx.close()


def prepare(case, seed):
    return _State(case, seed)


def _rows(state, first, *shape):
    """The context's output rows as they lie on the host; they keep the context."""
    buf = (ctypes.c_float * math.prod(shape)).from_address(ctypes.addressof(first.contents))
    buf.state = state
    return np.frombuffer(buf, np.float32).reshape(shape)


def run(state):
    lib, h = state.lib, state.ctx.h
    for seq, past in state.cut:                     # the call's tokens are new ones behind the past, in every pass
        lib.mi355_kv_cache_seq_rm(h, seq, past, -1)
    for b in state.batches:
        if lib.mi355_decode(h, b) != 0:
            raise RuntimeError("mi355_decode failed: %s" % lib.mi355_last_error())
    if state.embed:                                 # the tokens' rows lie one behind the other
        n, e = state.batches[0].n_tokens, state.model.n_embd
        first, last = (lib.mi355_get_embeddings_ith(h, i) for i in (0, n - 1))
        if ctypes.addressof(last.contents) - ctypes.addressof(first.contents) != 4 * e * (n - 1):
            raise RuntimeError("the embeddings' rows are apart")
        return [_rows(state, first, n, e)]
    return [_rows(state, lib.mi355_get_logits_ith(h, i), state.model.n_vocab) for i in state.rows]


def work(case):
    cfg = _config(case)
    E, kv, hd = cfg.n_embd, cfg.n_head_kv * cfg.head_dim, cfg.head_dim
    talks = [(case["past"] + s * case["spread"], 1) for s in range(case["n"])] if case["do"] == "slots" else [(case["past"], case["n"] if case["do"] in ("prompt", "embed") else 1)]
    T, rows = sum(n for _, n in talks), sum(n for _, n in talks) if case["do"] == "embed" else len(talks)
    cell = 2 * kv * cfg.n_layer * (2.0 if case["cache"] == "f16" else 34 / 32)
    nbytes = flops = 0.0
    for name, ne, t, _ in synth.model_tensors(cfg, case["ftype"]):
        rb, n = synth.row_bytes(t, ne[0]), int(np.prod(ne))
        if name == "token_embd.weight":
            nbytes += rb * T
        elif name == "output.weight":
            nbytes += rb * ne[1]
            flops += 2.0 * n * rows
        elif "_exps." in name:
            used = min(cfg.n_expert, cfg.n_expert_used * T)
            nbytes += rb * ne[1] * used
            flops += 2.0 * n / cfg.n_expert * cfg.n_expert_used * T
        else:
            nbytes += rb * (n // ne[0])
            flops += 2.0 * n * T if len(ne) > 1 else 0.0
    nbytes += 4.0 * rows * (E if case["do"] == "embed" else cfg.n_vocab)
    for past, n in talks:
        nbytes += cell * (past + n)
        seen = n * n if case["do"] == "embed" else n * past + n * (n + 1) // 2
        flops += 4.0 * seen * cfg.n_head * hd * cfg.n_layer
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Activations (and a q8_0 cache) are rounded to int8 blocks: where sums in another order move a value over a rounding's edge, a whole code changes and every
    layer behind adds its own.  The same token as a step, in a tick, as a prompt's end and as a turn's end (four kernels that differ only in the order of their
    f32 sums) is up to 0.019 apart over these models (largest difference: 0.085 of the row's root mean square); against `exact`, which rounds nothing, it is 0.02
    to 0.03.  The encoder has no such rounding: 4e-4 against `exact`."""
    return {"rel": 1.6e-3, "max": 0.02} if case["do"] == "embed" else {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits: plain torch on the file's bytes, no rounding of activations or of the cache

def _k_scales(s):
    s = s.to(torch.int32)
    return (torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double(),
            torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double())


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _dequantised(raw, t, shape):
    """The weights of a tensor's bytes."""
    if t == synth.F32:
        return raw.view(torch.float32).double().reshape(shape)
    if t == synth.F16:
        return raw.view(torch.float16).double().reshape(shape)
    b = raw.reshape(-1, synth.BLOCK_BYTES[t])
    if t == synth.Q8_0:
        return (b[:, 2:].contiguous().view(torch.int8).double() * _half(b[:, :2])).reshape(shape)
    if t in (synth.Q4_K, synth.Q5_K):
        d, dmin = _half(b[:, 0:2]), _half(b[:, 2:4])
        sc, mn = _k_scales(b[:, 4:16])
        qs = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        if t == synth.Q5_K:
            bit = torch.arange(8, device=raw.device, dtype=torch.uint8).reshape(1, 8, 1)
            q = q + (((b[:, 16:48].reshape(-1, 1, 32) >> bit) & 1) << 4)
        return (q.double() * (d * sc)[:, :, None] - (dmin * mn)[:, :, None]).reshape(shape)
    if t == synth.Q6_K:
        ql, qh = b[:, 0:128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)                                              # [blocks, half, four runs of 32, 32]
        shift = torch.arange(0, 8, 2, device=raw.device, dtype=torch.uint8).reshape(1, 1, 4, 1)
        q = (low | (((qh >> shift) & 3) << 4)).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _half(b[:, 208:210])
        return (q.reshape(-1, 16, 16) * sc[:, :, None]).reshape(shape)
    raise ValueError("type %d" % t)


class _Weights:
    def __init__(self, case):
        self.bytes = np.memmap(_file(case), np.uint8, "r")
        self.at, off = {}, 0
        for name, ne, t, _ in synth.model_tensors(_config(case), case["ftype"]):
            size = synth.row_bytes(t, ne[0]) * (int(np.prod(ne)) // ne[0])
            self.at[name] = (off, size, t, ne)
            off += -(-size // 32) * 32
        self.start = self.bytes.size - off                                                  # the tensors are the file's end

    def __call__(self, name, part=None, rows=None):
        off, size, t, ne = self.at[name]
        shape = tuple(reversed(ne))
        if part is not None:                                                                # one expert of a stack
            size //= shape[0]
            off, shape = off + part * size, shape[1:]
        raw = self.bytes[self.start + off:self.start + off + size]
        if rows is not None:
            raw, shape = raw.reshape(shape[0], -1)[rows].reshape(-1), (len(rows),) + shape[1:]
        return _dequantised(torch.from_numpy(np.array(raw)).cuda(), t, shape)


def _rope(x, pos, base, halves):
    """x [tokens, heads, D]: pairs of neighbours, or (halves) of an element of each half."""
    D = x.shape[-1]
    th = pos[:, None] * base ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    c, s = torch.cos(th)[:, None], torch.sin(th)[:, None]
    a, b = (x[..., : D // 2], x[..., D // 2:]) if halves else (x[..., 0::2], x[..., 1::2])
    y = (a * c - b * s, a * s + b * c)
    return torch.cat(y, -1) if halves else torch.stack(y, -1).reshape(x.shape)


def _attention(q, k, v, causal):
    """One sequence: q [T, H, D], k and v [T, G, D]."""
    T, H, D = q.shape
    R = H // k.shape[1]
    out = torch.empty_like(q)
    hide = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1) if causal else None
    for h in range(H):
        s = q[:, h].contiguous() @ k[:, h // R].t().contiguous() / math.sqrt(D)
        if causal:
            s.masked_fill_(hide, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // R].contiguous()
    return out.reshape(T, H * D)


def _linear(x, w):
    return x @ w.t()


def _layer_norm(x, w, b, eps):
    return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, keepdim=True, unbiased=False) + eps) * w + b


def exact(case, seed):
    cfg, W = _config(case), _Weights(case)
    talks = [t for t, _ in _conversations(case, seed)]
    H, G, D, E = cfg.n_head, cfg.n_head_kv, cfg.head_dim, cfg.n_embd
    ends = np.cumsum([len(t) for t in talks])
    spans = [(int(e) - len(t), int(e)) for t, e in zip(talks, ends)]
    toks = np.concatenate(talks)
    pos = torch.cat([torch.arange(len(t), device="cuda", dtype=torch.float64) for t in talks])
    x = W("token_embd.weight", rows=toks)
    if case["do"] == "embed":
        x = _layer_norm(x + W("token_types.weight")[0], W("token_embd_norm.weight"), W("token_embd_norm.bias"), cfg.eps)
        for il in range(cfg.n_layer):
            w = lambda n: W("blk.%d.%s" % (il, n))  # noqa: E731
            q, k, v = _linear(x, w("attn_qkv.weight")).split([E, E, E], 1)
            q, k, v = (y.reshape(-1, H, D) for y in (q, k, v))
            a = _attention(_rope(q, pos, cfg.rope_base, True), _rope(k, pos, cfg.rope_base, True), v, False)
            x = _layer_norm(x + _linear(a, w("attn_output.weight")), w("attn_output_norm.weight"), w("attn_output_norm.bias"), cfg.eps)
            f = torch.nn.functional.silu(_linear(x, w("ffn_gate.weight"))) * _linear(x, w("ffn_up.weight"))
            x = _layer_norm(x + _linear(f, w("ffn_down.weight")), w("layer_output_norm.weight"), w("layer_output_norm.bias"), cfg.eps)
        return [x]

    def norm(y, w):
        return y * torch.rsqrt((y * y).mean(-1, keepdim=True) + cfg.eps) * w

    def feed(y, p, e=None):
        s = "_exps" if e is not None else ""
        gate, up, down = (lambda: W(p + "ffn_gate%s.weight" % s, e)), (lambda: W(p + "ffn_up%s.weight" % s, e)), (lambda: W(p + "ffn_down%s.weight" % s, e))
        return _linear(torch.nn.functional.silu(_linear(y, gate())) * _linear(y, up()), down())

    last = torch.tensor([j - 1 for _, j in spans], device="cuda")
    sure = torch.ones(len(spans), dtype=torch.bool, device="cuda")
    for il in range(cfg.n_layer):
        p = "blk.%d." % il
        y = norm(x, W(p + "attn_norm.weight"))
        q, k, v = (_linear(y, W(p + "attn_%s.weight" % n)).reshape(len(toks), -1, D) for n in "qkv")
        q, k = _rope(q, pos, cfg.rope_base, False), _rope(k, pos, cfg.rope_base, False)
        a = torch.cat([_attention(q[i:j], k[i:j], v[i:j], True) for i, j in spans])
        x = x + _linear(a, W(p + "attn_output.weight"))
        y = norm(x, W(p + "ffn_norm.weight"))
        if cfg.n_expert:
            choice = _linear(y, W(p + "ffn_gate_inp.weight"))
            order = choice[last].sort(-1, descending=True).values
            sure &= order[:, cfg.n_expert_used - 1] - order[:, cfg.n_expert_used] > 0.06    # the router's logits are of unit size and 0.02 off: with less between, either choice is right
            share = torch.softmax(choice, -1)
            best, who = share.topk(cfg.n_expert_used, -1)
            best = best / best.sum(-1, keepdim=True)
            z = torch.zeros_like(x)
            for e in range(cfg.n_expert):
                at, rank = (who == e).nonzero(as_tuple=True)
                if len(at):
                    z.index_add_(0, at, feed(y[at], p, e) * best[at, rank][:, None])
            x = x + z
        else:
            x = x + feed(y, p)
    logits = _linear(norm(x[last], W("output_norm.weight")), W("output.weight"))
    rows = [row if ok else None for row, ok in zip(logits, sure.tolist())]
    return rows if bool(sure.any()) else None
