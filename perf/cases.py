"""Timed workloads of the engine: prompts, chat turns, sessions decoded
together, prompt scoring and the device sampler, on the three models that
bench.py measures (the 4B shape in Q4_K_M, the 1.7B shape in Q8_0 and in
Q4_K_M; random weights).

A case is a dict of plain values with a "kind":

* ``prefill`` -- a session holding `history` tokens takes `n` more; the result
  is the next-token logits.
* ``score``   -- the same with the logits of every one of the `n` positions.
* ``chat``    -- one turn: prefill the user's `n` tokens after `history`,
  generate a reply of `new` tokens, prefill the `follow` tokens that come
  after it (a tool result, the next message).
* ``batch``   -- `sessions` such conversations, the replies decoded together.
* ``sample``  -- one draw from `vocab` logits held on the device.

`exact` restates the network in float64 from the model file's own blocks.
"""

from __future__ import annotations

import math
import mmap
import os
import struct
import tempfile

import numpy as np
import torch

import rpgbarengine_amd as eng
from rpgbarengine_amd import synth

# name -> (preset, weight mix, weight seed): bench.py's models
MODELS = {
    "4b-q4km": ("s4", "q4_k_m", 1),
    "1.7b-q8": ("s17", "q8_0", 2),
    "1.7b-q4km": ("s17", "q4_k_m", 3),
}
CAPACITY = 4096  # positions a session of the chat ABI holds unless told otherwise


def listed():
    return [
        # A host that samples from logits of its own in its serving loop: the
        # chat ABI's defaults (no top-k, top-p 0.95). The smallest call.
        {"name": "sample default", "kind": "sample", "vocab": 151936, "temperature": 0.7, "top_k": 0, "top_p": 0.95},
        # The same at bench.py's sampled-decode parameters.
        {"name": "sample top-k", "kind": "sample", "vocab": 151936, "temperature": 0.8, "top_k": 40, "top_p": 0.95},
        # A short greeting to a fresh session of the small model, and its reply.
        {"name": "chat 1.7b q8 greeting", "kind": "chat", "model": "1.7b-q8", "history": 0, "n": 32, "new": 64,
         "follow": 1, "temperature": 0.0, "top_k": 0, "top_p": 1.0, "capacity": 160},
        # The headline decode: sampled reply behind a 512-token prompt.
        {"name": "chat 4b top-k", "kind": "chat", "model": "4b-q4km", "history": 500, "n": 12, "new": 64,
         "follow": 5, "temperature": 0.8, "top_k": 40, "top_p": 0.95, "capacity": 776},
        # An ordinary turn of a running conversation through a session of the
        # default capacity, at a low temperature without top-k.
        {"name": "chat 4b default", "kind": "chat", "model": "4b-q4km", "history": 1337, "n": 29, "new": 48,
         "follow": 11, "temperature": 0.2, "top_k": 0, "top_p": 0.95, "capacity": CAPACITY},
        # The end of a long conversation: the cache nearly full.
        {"name": "chat 1.7b long", "kind": "chat", "model": "1.7b-q4km", "history": 3950, "n": 50, "new": 64,
         "follow": 3, "temperature": 0.0, "top_k": 0, "top_p": 1.0, "capacity": CAPACITY},
        # A user's message after a cached prefix: what a reply waits for.
        {"name": "prefill 4b turn", "kind": "prefill", "model": "4b-q4km", "history": 611, "n": 37,
         "capacity": CAPACITY},
        # A pasted paragraph or a tool's result, no multiple of any tile.
        {"name": "prefill 4b paragraph", "kind": "prefill", "model": "4b-q4km", "history": 1500, "n": 203,
         "capacity": CAPACITY},
        # The headline prompt.
        {"name": "prefill 4b 512", "kind": "prefill", "model": "4b-q4km", "history": 0, "n": 512, "capacity": 776},
        # A system prompt with its tool list on the Q8_0 model.
        {"name": "prefill 1.7b q8 prompt", "kind": "prefill", "model": "1.7b-q8", "history": 0, "n": 777,
         "capacity": CAPACITY},
        # A document that fills the context.
        {"name": "prefill 1.7b long", "kind": "prefill", "model": "1.7b-q4km", "history": 0, "n": 3999,
         "capacity": CAPACITY},
        # Eight players' sessions served together, chat defaults.
        {"name": "batch 4b 8 sessions", "kind": "batch", "model": "4b-q4km", "sessions": 8, "history": 1000, "n": 24,
         "new": 48, "follow": 2, "temperature": 0.2, "top_k": 0, "top_p": 0.95, "capacity": 1152},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sample", "prefill", "prefill", "prefill", "score", "chat", "chat", "chat", "batch"])
    top_k, top_p = rng.choice([(0, 0.95), (40, 0.95), (20, 0.8), (0, 0.9)])
    if kind == "sample":
        return {"kind": kind, "vocab": _log(rng, 1000, 151936), "temperature": round(rng.uniform(0.1, 1.5), 2),
                "top_k": top_k, "top_p": top_p}
    model = rng.choice(sorted(MODELS))
    if kind in ("prefill", "score"):
        n = _log(rng, 2, 64) if rng.random() < 0.4 else _log(rng, 65, 1500 if model == "4b-q4km" else 3900)
        if kind == "score":
            n = _log(rng, 8, 300)
        history = rng.choice([0, rng.randrange(1, CAPACITY - n)])
        return {"kind": kind, "model": model, "history": history, "n": n, "capacity": CAPACITY}
    n, new, follow = _log(rng, 1, 60), rng.randrange(8, 49), rng.randrange(1, 13)
    temperature = rng.choice([0.0, 0.0, 0.2])
    if kind == "chat":
        history = _log(rng, 1, 3900)
        tight = 32 * -(-(history + n + new + follow) // 32)
        return {"kind": kind, "model": model, "history": history, "n": n, "new": new, "follow": follow,
                "temperature": temperature, "top_k": top_k if temperature else 0, "top_p": top_p if temperature else 1.0,
                "capacity": rng.choice([CAPACITY, tight])}
    history = _log(rng, 16, 1000)
    return {"kind": kind, "model": model, "sessions": rng.randrange(2, 9), "history": history, "n": n,
            "new": rng.randrange(8, 41), "follow": follow, "temperature": temperature,
            "top_k": top_k if temperature else 0, "top_p": top_p if temperature else 1.0, "capacity": 1152}


# ---- models and inputs

_paths, _models = {}, {}


def _spec(name):
    preset, mix, seed = MODELS[name]
    return synth.PRESETS[preset].with_(mix=synth.MIXES[mix], seed=seed)


def _path(name):
    """The model's GGUF file, written once per machine."""
    if name not in _paths:
        folder = os.path.join(tempfile.gettempdir(), "rpg-cases-%d" % os.getuid())
        os.makedirs(folder, exist_ok=True)
        path = os.path.join(folder, name + ".gguf")
        if not os.path.exists(path):
            part = "%s.%d" % (path, os.getpid())
            synth.write_gguf(part, _spec(name), threads=min(16, os.cpu_count() or 1))
            os.replace(part, path)
        _paths[name] = path
    return _paths[name]


def _model(name):
    """The loaded model: a program loads its weights once."""
    if name not in _models:
        _models[name] = eng.Model(_path(name), max_pos=CAPACITY)
    return _models[name]


def _inputs(case, seed):
    """Per session: history, turn and follow-up ids, uniform over the vocabulary."""
    vocab = _spec(case["model"]).vocab
    out = []
    for i in range(case.get("sessions", 1)):
        rng = np.random.default_rng([int(seed), i])
        out.append([rng.integers(0, vocab, size=int(k), dtype=np.int32)
                    for k in (case["history"], case["n"], case.get("follow", 0))])
    return out


def _logits(case, seed):
    """Logits as the models give them: standard normal values."""
    return np.random.default_rng(int(seed)).standard_normal(case["vocab"]).astype(np.float32)


def prepare(case, seed):
    if case["kind"] == "sample":
        dev = torch.device("cuda")
        return {"case": case, "seed": seed, "logits": torch.from_numpy(_logits(case, seed)).to(dev),
                "token": torch.zeros(1, dtype=torch.int32, device=dev),
                "probs": torch.zeros(case["vocab"], dtype=torch.float32, device=dev)}
    model = _model(case["model"])
    ids = _inputs(case, seed)
    sessions = []
    for history, _, _ in ids:
        s = model.session(case["capacity"])
        if history.size:
            s.prefill(history)
        sessions.append(s)
    return {"case": case, "seed": seed, "ids": ids, "sessions": sessions, "eos": model.eos_id}


def run(state):
    case, seed = state["case"], int(state["seed"]) & 0xFFFFFFFF
    kind = case["kind"]
    if kind == "sample":
        rc = eng.lib().rpg_hip_sample_noalloc(
            state["logits"].data_ptr(), case["vocab"], case["temperature"], case["top_k"], case["top_p"], seed, 7,
            state["token"].data_ptr(), state["probs"].data_ptr(), None)
        if rc != 0:
            raise RuntimeError(eng.lib().rpg_hip_last_error().decode())
        return {"token": state["token"], "probs": state["probs"]}
    sessions = state["sessions"]
    first = []
    for s, (_, turn, _) in zip(sessions, state["ids"]):
        s.set_len(case["history"])
        first.append(s.prefill(turn, all_logits=kind == "score"))
    if kind in ("prefill", "score"):
        return {"logits": first[0]}
    if kind == "chat":
        reply = sessions[0].generate(case["new"], case["temperature"], case["top_k"], case["top_p"], seed,
                                     stop_ids=(state["eos"],))
    else:
        reply, _ = eng.generate_batch(sessions, case["new"], case["temperature"], case["top_k"], case["top_p"],
                                      [seed + i for i in range(len(sessions))])
    after = [s.prefill(follow) for s, (_, _, follow) in zip(sessions, state["ids"])]
    return {"first": first, "reply": reply, "after": after}


# ---- what a pass cannot do without

def _shape(name):
    """(weights of the layers, their bytes, lm_head bytes, KV bytes per position)."""
    s = _spec(name)
    qd, kvd = s.n_heads * s.head_dim, s.n_kv_heads * s.head_dim
    wide, down, v = s.hidden * (2 * qd + kvd + 2 * s.ffn), s.hidden * s.ffn, s.hidden * kvd
    body = s.n_layers * (wide + down + v)
    if s.mix == synth.MIX_Q8_0:
        per, more, head = 34 / 32, 34 / 32, 34 / 32
    else:  # Q4_K; down and v are Q6_K in half of the layers, the embedding is Q6_K
        per, more, head = 144 / 256, (144 + 210) / 512, 210 / 256
    size = s.n_layers * (wide * per + (down + v) * more + 4 * (2 * s.hidden + 2 * s.head_dim))
    return body, size, s.vocab * s.hidden * head, 2 * 4 * s.n_layers * kvd


def _segment(case, pos, n, rows=1):
    """Bytes and operations of forwarding n tokens of one session behind pos others."""
    s = _spec(case["model"])
    body, size, head, kv = _shape(case["model"])
    pairs = n * pos + n * (n + 1) / 2
    return (size + head + kv * (pos + n) + 4 * (n * s.hidden + rows * s.vocab),
            2 * body * n + 4 * s.n_layers * s.n_heads * s.head_dim * pairs + 2 * s.hidden * s.vocab * rows)


def work(case):
    if case["kind"] == "sample":
        return {"bytes": 8 * case["vocab"] + 4, "flops": 8 * case["vocab"]}
    rows = case["n"] if case["kind"] == "score" else 1
    b, f = _segment(case, case["history"], case["n"], rows)
    if case["kind"] in ("prefill", "score"):
        return {"bytes": b, "flops": f}
    sessions = case.get("sessions", 1)
    start = case["history"] + case["n"]
    b, f = b * sessions, f * sessions
    _, size, head, _ = _shape(case["model"])
    for t in range(case["new"]):
        one = _segment(case, start + t, 1)
        b += one[0] * sessions - (sessions - 1) * (size + head)  # a step reads the weights once for all
        f += one[1] * sessions
    end = _segment(case, start + case["new"], case["follow"])
    return {"bytes": b + end[0] * sessions, "flops": f + end[1] * sessions}


def tolerance(case):
    # The engine computes in fp32 (or fp32-equivalent split products)
    # throughout. Against float64, a layer's rounding carried through the rest
    # shows in the logits as a few 1e-6 of their norm; another order of sums
    # moves as much.
    if case["kind"] == "sample":
        return {"rel": 1e-6, "max": 1e-5}  # specified bit for bit
    return {"rel": 2e-5, "max": 2e-4}


# ---- float64

def _read_gguf(path):
    """{tensor name: (type, dims, bytes)} of a GGUF file."""
    with open(path, "rb") as f:
        mm = mmap.mmap(f.fileno(), 0, access=mmap.ACCESS_READ)
    at = 24
    n_tensors, n_keys = struct.unpack_from("<QQ", mm, 8)
    plain = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}

    def text():
        nonlocal at
        (n,) = struct.unpack_from("<Q", mm, at)
        at += 8 + n
        return mm[at - n:at].decode()

    def skip(kind):
        nonlocal at
        if kind == 8:
            (n,) = struct.unpack_from("<Q", mm, at)
            at += 8 + n
        elif kind == 9:
            inner, n = struct.unpack_from("<IQ", mm, at)
            at += 12
            if inner in plain:
                at += n * plain[inner]
            else:
                for _ in range(n):
                    skip(inner)
        else:
            at += plain[kind]

    for _ in range(n_keys):
        text()
        (kind,) = struct.unpack_from("<I", mm, at)
        at += 4
        skip(kind)
    heads = []
    for _ in range(n_tensors):
        name = text()
        (nd,) = struct.unpack_from("<I", mm, at)
        dims = struct.unpack_from("<%dQ" % nd, mm, at + 4)
        kind, off = struct.unpack_from("<IQ", mm, at + 4 + 8 * nd)
        at += 16 + 8 * nd
        heads.append((name, kind, dims, off))
    base = -(-at // 32) * 32
    block = {0: (1, 4), 8: (32, 34), 12: (256, 144), 14: (256, 210)}
    out = {}
    for name, kind, dims, off in heads:
        per, size = block[kind]
        n = math.prod(dims) // per * size
        out[name] = (kind, dims, np.frombuffer(mm, dtype=np.uint8, count=n, offset=base + off))
    return out


def _half(b):
    """fp16 values from byte pairs [..., 2]."""
    return b.contiguous().view(torch.float16).double()


def _wide(kind, dims, raw, dev):
    """A tensor's values in float64, from its blocks as the format defines them."""
    b = torch.from_numpy(raw.copy()).to(dev)
    shape = tuple(reversed(dims))
    if kind == 0:
        return b.view(torch.float32).double().reshape(shape)
    if kind == 8:  # d, 32 signed quants
        b = b.reshape(-1, 34)
        return (_half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(shape)
    if kind == 12:  # d, dmin, 8 six-bit (scale, min) pairs, 128 bytes of nibbles
        b = b.reshape(-1, 144)
        s = b[:, 4:16]
        low = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mins = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = (_half(b[:, :2]) * low).unsqueeze(2) * q - (_half(b[:, 2:4]) * mins).unsqueeze(2)
        return w.reshape(shape)
    # Q6_K: low nibbles (128 B), high bit pairs (64 B), 16 signed scales, d
    b = b.reshape(-1, 210)
    lo, hi = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
    lo = torch.cat([lo & 15, lo >> 4], 2)
    hi = torch.cat([hi & 3, (hi >> 2) & 3, (hi >> 4) & 3, hi >> 6], 2)
    q = (lo | (hi << 4)).reshape(-1, 16, 16).double() - 32
    scale = b[:, 192:208].contiguous().view(torch.int8).double() * _half(b[:, 208:])
    return (scale.unsqueeze(2) * q).reshape(shape)


class _Wide:
    """The network in float64 over one model file; weights are unpacked once."""

    def __init__(self, name):
        self.s = _spec(name)
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.w = {k: _wide(*v, self.dev) for k, v in _read_gguf(_path(name)).items()}

    def norm(self, x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.s.rms_eps) * self.w[name]

    def rope(self, x, pos):
        """x [tokens, heads, 128], rotated in pairs (i, i + 64)."""
        half = self.s.head_dim // 2
        freq = self.s.rope_theta ** (-torch.arange(half, dtype=torch.float64, device=self.dev) / half)
        a = (pos.double().unsqueeze(1) * freq).unsqueeze(1)
        u, v = x[..., :half], x[..., half:]
        return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)

    def forward(self, cache, ids, every=False):
        """Appends ids to cache (per layer keys, values [kv heads, positions,
        128]) and gives the last position's logits, or every one's."""
        s, w = self.s, self.w
        n, d = len(ids), s.head_dim
        x = w["token_embd.weight"][torch.as_tensor(np.asarray(ids), dtype=torch.long, device=self.dev)]
        before = cache[0][0].shape[1] if cache else 0
        pos = torch.arange(before, before + n, device=self.dev)
        hidden = torch.arange(before + n, device=self.dev).unsqueeze(0) > pos.unsqueeze(1)
        for l in range(s.n_layers):
            p = "blk.%d." % l
            h = self.norm(x, p + "attn_norm.weight")
            q, k, v = ((h @ w[p + "attn_%s.weight" % c].T).reshape(n, -1, d) for c in "qkv")
            q = self.rope(self.norm(q, p + "attn_q_norm.weight"), pos).transpose(0, 1).contiguous()
            k = self.rope(self.norm(k, p + "attn_k_norm.weight"), pos).transpose(0, 1).contiguous()
            v = v.transpose(0, 1).contiguous()
            if l < len(cache):
                k, v = torch.cat([cache[l][0], k], 1), torch.cat([cache[l][1], v], 1)
                cache[l] = (k, v)
            else:
                cache.append((k, v))
            group = s.n_heads // s.n_kv_heads
            o = []
            for g in range(s.n_kv_heads):
                score = q[g * group:(g + 1) * group].reshape(group * n, d) @ k[g].T.contiguous() / math.sqrt(d)
                score = score.reshape(group, n, -1).masked_fill(hidden, -math.inf)
                o.append((torch.softmax(score, -1).reshape(group * n, -1) @ v[g]).reshape(group, n, d))
            o = torch.cat(o, 0).transpose(0, 1).reshape(n, -1)
            x = x + o @ w[p + "attn_output.weight"].T
            h = self.norm(x, p + "ffn_norm.weight")
            act = torch.nn.functional.silu(h @ w[p + "ffn_gate.weight"].T) * (h @ w[p + "ffn_up.weight"].T)
            x = x + act @ w[p + "ffn_down.weight"].T
        x = self.norm(x if every else x[-1], "output_norm.weight")
        return x @ w["token_embd.weight"].T


_wides = {}


def exact(case, seed):
    if case["kind"] == "sample":
        p = torch.softmax(torch.from_numpy(_logits(case, seed)).double() / case["temperature"], 0)
        if case["top_k"] > 1:
            p = torch.where(p < torch.topk(p, min(case["top_k"], p.numel())).values[-1], 0.0, p)
        order = torch.argsort(p / p.sum())
        drop = torch.cumsum((p / p.sum())[order], 0) <= 1.0 - case["top_p"]
        p[order[drop]] = 0.0
        return {"token": None, "probs": p / p.sum()}
    name = case["model"]
    if name not in _wides:
        _wides.clear()
        _wides[name] = _Wide(name)
    net = _wides[name]
    first, reply, after = [], [], []
    for history, turn, follow in _inputs(case, seed):
        cache = []
        if history.size:
            net.forward(cache, history)
        logits = net.forward(cache, turn, every=case["kind"] == "score")
        first.append(logits.cpu())
        if case["kind"] in ("prefill", "score"):
            return {"logits": first[0]}
        if case["temperature"] > 0:  # the draws depend on the seed: the turn's logits only
            after.append(None)
            continue
        ids = []
        for _ in range(case["new"]):
            ids.append(int(torch.argmax(logits)))
            logits = net.forward(cache, ids[-1:])
        reply.append(ids)
        after.append(net.forward(cache, follow).cpu())
    if not reply:
        return {"first": first, "reply": None, "after": after}
    reply = np.array(reply[0] if case["kind"] == "chat" else reply, dtype=np.int32)
    return {"first": first, "reply": reply, "after": after}
