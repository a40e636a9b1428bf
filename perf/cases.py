"""What this framework is used for, as cases to time: the section-6b kvdecode
backend under a serving program, from one decode step behind a short prompt to a
2048-token prefill and a 64-session batched step.

The models keep the layer sizes of the shapes spkv.SHAPES names with fewer layers
(Gemma-3-12B: one period of its layer pattern, five window layers and a global
one) and a smaller vocabulary, so that the layers, not the LM head, are most of
a pass, as in the whole models.  Weights are seeded random-init OK_Q4B files; the
tokens of prompts and steps come from a state's seed.
"""
import ctypes
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "shannon-prime-system_amd"))
import spkv  # noqa: E402

# layers kept of each named shape, and the vocabulary
MODELS = {
    "qwen3-0.6b": dict(n_layers=4, vocab=32768),
    "qwen3-8b": dict(n_layers=2, vocab=16384),
    "gemma3-12b": dict(n_layers=6, vocab=16384),
}
RECALL = dict(B=1024, W=64, sink=4, r=16)     # the recall budget of the long-context records
CONTEXT_MAX = 32768
WINDOW_BASE = 10000.0                         # RoPE base of Gemma-3's window layers


def listed():
    return [
        # the first step after a short question: nothing but latency and launches
        dict(name="decode 0.6b after 24, exact", op="decode", model="qwen3-0.6b", mode="exact", ctx=24),
        # a chat at the small model's usual context, reference (float) arithmetic
        dict(name="decode 0.6b at 4k, float", op="decode", model="qwen3-0.6b", mode="float", ctx=4095),
        # the headline configuration: one long-context session
        dict(name="decode 12b at 32k, exact", op="decode", model="gemma3-12b", mode="exact", ctx=32767),
        # a session with the compressed K/V codec at an odd length
        dict(name="decode 12b at 6k, spinor", op="decode", model="gemma3-12b", mode="spinor", ctx=6001),
        # sparse recall over a long context
        dict(name="decode 12b at 16k, recall", op="decode", model="gemma3-12b", mode="recall", ctx=16001),
        # the device-resident greedy loop of an offline generation
        dict(name="greedy 12b 16 tokens, exact", op="greedy", model="gemma3-12b", mode="exact", ctx=777, n=16),
        # a full server step: 64 sessions of ragged contexts
        dict(name="batch 8b 64 sessions, exact", op="batch", model="qwen3-8b", mode="exact", sessions=64, lo=256, hi=4096),
        # a quiet server: a handful of short sessions
        dict(name="batch 0.6b 7 sessions, float", op="batch", model="qwen3-0.6b", mode="float", sessions=7, lo=100, hi=900),
        # a short prompt
        dict(name="prefill 0.6b 61 tokens, exact", op="prefill", model="qwen3-0.6b", mode="exact", ctx=0, n=61),
        # a document's prompt
        dict(name="prefill 12b 2048 tokens, exact", op="prefill", model="gemma3-12b", mode="exact", ctx=0, n=2048),
        # the next turn of a conversation, float arithmetic, ragged
        dict(name="prefill 12b 777 at 1500, float", op="prefill", model="gemma3-12b", mode="float", ctx=1500, n=777),
        # one chunk of a long document's prefill
        dict(name="prefill 8b 512 at 8k, float", op="prefill", model="qwen3-8b", mode="float", ctx=8192, n=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "decode", "greedy", "batch", "prefill", "prefill"])
    model = rng.choice(sorted(MODELS))
    if op == "decode":
        mode = rng.choice(["exact", "float", "spinor", "recall"])
        return dict(op=op, model=model, mode=mode, ctx=_log_int(rng, 16, CONTEXT_MAX if mode == "exact" else 16384))
    if op == "greedy":
        return dict(op=op, model=model, mode=rng.choice(["exact", "float"]), ctx=_log_int(rng, 16, 4096), n=_log_int(rng, 2, 16))
    if op == "batch":
        lo = _log_int(rng, 16, 256)
        return dict(op=op, model=model, mode=rng.choice(["exact", "float"]),
                    sessions=_log_int(rng, 2, 64 if model != "gemma3-12b" else 16), lo=lo, hi=lo + _log_int(rng, 16, 1800))
    mode = rng.choice(["exact", "exact", "float", "float", "spinor"])
    start = rng.choice([0, _log_int(rng, 16, 8192)])
    return dict(op=op, model=model, mode=mode, ctx=start, n=_log_int(rng, 2, 2048 if start == 0 and mode == "exact" else 640))


# ---------------------------------------------------------------- models
_models = {}


class _File:
    """The tensors of a written .sp-model file, for the 64-bit results."""

    def __init__(self, path):
        self.raw = np.memmap(path, dtype=np.uint8, mode="r")
        head = self.raw[:512].tobytes()
        count = int.from_bytes(head[24 + 256 + 32 + 4:24 + 256 + 32 + 8], "little")
        table, data = np.frombuffer(head, np.uint64, 2, 24 + 256 + 32 + 8)
        self.at = {}
        for i in range(count):
            e = self.raw[int(table) + 256 * i:int(table) + 256 * (i + 1)].tobytes()
            off, size = np.frombuffer(e, np.uint64, 2, 80 + 8 + 64)
            self.at[e[:80].split(b"\0")[0].decode()] = (int(data) + int(off), int(size))

    def bytes(self, name):
        off, size = self.at[name]
        return torch.from_numpy(np.array(self.raw[off:off + size])).cuda()

    def matrix(self, name, cols, rows=None):
        """Rows of an OK_Q4B matrix in 64 bits: nibble (low first) times its 32-column block's f16 step."""
        c = self.bytes(name).view(-1, cols // 2)
        s = self.bytes(name + ".bscale").view(torch.float16).view(-1, cols // 32)
        if rows is not None:
            c, s = c[rows], s[rows]
        v = torch.stack((c & 15, c >> 4), dim=-1).to(torch.int16)
        v = torch.where(v > 7, v - 16, v).double().view(-1, cols // 32, 32)
        return (v * s.double().unsqueeze(-1)).view(-1, cols)


def _shape(model):
    return dict(spkv.SHAPES[model], **MODELS[model])


def _model(model):
    """A program loads its model once: the file is written, mapped, and its name given up."""
    if model not in _models:
        with tempfile.TemporaryDirectory() as d:
            spm, spt = spkv.write_model(os.path.join(d, "m"), model, max_context=2 * CONTEXT_MAX, **MODELS[model])
            _models[model] = (spkv.Model(spm, spt), _File(spm))
    return _models[model]


# ---------------------------------------------------------------- states
def _tokens(case, seed, what, n):
    return spkv.splitmix_tokens(n, MODELS[case["model"]]["vocab"], seed=(seed * 1000003 + what) & 0x7FFFFFFFFFFF)


def _contexts(case, seed):
    """Context lengths of a batch's sessions: uniform in [lo, hi]."""
    u = spkv.splitmix_u64(case["sessions"], seed * 7919 + 2)
    return [int(case["lo"] + x % np.uint64(case["hi"] - case["lo"] + 1)) for x in u]


class State:
    """The sessions, tokens and buffers a program holds; closed with its last reference."""

    def __init__(self):
        self.sessions, self.backend = [], None

    def __del__(self):
        for s in self.sessions:
            s.close()
        if self.backend is not None:
            self.backend.close()


def prepare(case, seed):
    m, _ = _model(case["model"])
    vocab, mode = MODELS[case["model"]]["vocab"], case["mode"]
    st = State()
    st.op, st.logits = case["op"], np.zeros(vocab, np.float32)

    def session(ctx, room, what):
        s = spkv.Session(m, ctx + room, flags=spkv.SP_KV_SPINOR if mode == "spinor" else 0)
        st.sessions.append(s)
        s.attach(ctx + room, exact=mode in ("exact", "recall"))
        if mode == "recall":
            spkv.check(spkv.kv().sp_hipkv_set_recall(s.backend_handle(), *(RECALL[k] for k in ("B", "W", "sink", "r"))),
                       "sp_hipkv_set_recall")
        if ctx:
            spkv.check(s.prefill(_tokens(case, seed, what, ctx), st.logits), "sp_prefill_chunk")
        return s

    if case["op"] == "decode":
        session(case["ctx"], 64, 0)
        st.token = int(_tokens(case, seed, 1, 1)[0])
    elif case["op"] == "prefill":
        session(case["ctx"], case["n"] + 64, 0)
        st.tokens = _tokens(case, seed, 1, case["n"])
    elif case["op"] == "batch":
        lengths = _contexts(case, seed)
        for i, c in enumerate(lengths):
            session(c, case["hi"] + 64 - c, 2 + i)
        n = st.n = len(lengths)
        st.tokens = _tokens(case, seed, 1, n)
        st.handles = (ctypes.c_void_p * n)(*[s.h.value for s in st.sessions])
        st.logits, st.next = np.zeros((n, vocab), np.float32), np.zeros(n, np.int32)
    else:
        qm = spkv.l1().sp_session_qwen3_model
        st.sessions.append(spkv.Session(m, 64))
        st.backend = spkv.Backend(qm(st.sessions[0].h), case["ctx"] + case["n"] + 64, exact=mode == "exact")
        st.backend.prefill(_tokens(case, seed, 0, case["ctx"]))
        st.token, st.n = int(_tokens(case, seed, 1, 1)[0]), case["n"]
    return st


def run(st):
    """One pass; the sessions go back to where they were (an O(1) rewind)."""
    if st.op == "decode":
        spkv.check(st.sessions[0].decode(st.token, st.logits), "sp_decode_step")
        spkv.check(st.sessions[0].rewind(1), "sp_session_rewind")
        return st.logits
    if st.op == "prefill":
        spkv.check(st.sessions[0].prefill(st.tokens, st.logits), "sp_prefill_chunk")
        spkv.check(st.sessions[0].rewind(len(st.tokens)), "sp_session_rewind")
        return st.logits
    if st.op == "batch":
        spkv.check(spkv.l1().spx_decode_batch(st.handles, st.n, spkv.ptr(st.tokens), spkv.ptr(st.logits),
                                              st.logits.size, spkv.ptr(st.next)), "spx_decode_batch")
        for s in st.sessions:
            spkv.check(s.rewind(1), "sp_session_rewind")
        return {"logits": st.logits, "next": st.next}
    out, _ = st.backend.greedy(st.token, st.n)
    st.backend.decode(int(out[-1]), st.logits)
    spkv.check(st.backend.rewind(st.n + 1), "sp_hipkv_rewind")
    return {"tokens": out, "logits": st.logits}


# ---------------------------------------------------------------- what a pass needs
def _is_global(d, layer):
    return d["swa_window"] == 0 or layer % 6 == 5


def work(case):
    d = _shape(case["model"])
    qd, kvd, e, ff = d["n_heads"] * d["head_dim"], d["n_kv_heads"] * d["head_dim"], d["hidden"], d["n_ff"]
    layer, head = e * (qd + 2 * kvd) + qd * e + 3 * e * ff, d["vocab"] * e
    row = 2 * kvd * 4 if case["mode"] != "spinor" else 2 * d["n_kv_heads"] * (d["head_dim"] + 4 * -(-d["head_dim"] // 55))
    if case["op"] == "decode":
        spans, heads = [[case["ctx"]]], 1
    elif case["op"] == "greedy":
        spans, heads = [[case["ctx"] + i] for i in range(case["n"] + 1)], case["n"] + 1
    elif case["op"] == "batch":
        spans, heads = [_contexts(case, 1)], case["sessions"]
    else:
        spans, heads = [list(range(case["ctx"], case["ctx"] + case["n"]))], 1
    # bytes: each matrix once a pass over it, each K/V row that some token attends once, each new row written
    # (a prefill's rows serve all its tokens); flops: two a weight and token, and four a dimension and attended row
    nbytes = flops = 0.0
    for step in spans:
        nbytes += 0.5625 * (d["n_layers"] * layer + head)
        flops += 2.0 * d["n_layers"] * layer * len(step)
        for l in range(d["n_layers"]):
            span = [p + 1 if _is_global(d, l) else min(p + 1, d["swa_window"]) for p in step]
            if case["mode"] == "recall" and _is_global(d, l):
                span = [min(s, RECALL["B"]) for s in span]
            if case["op"] == "prefill":
                seen = step[-1] + 1 if _is_global(d, l) else min(step[-1] + 1, d["swa_window"] + len(step) - 1)
                nbytes += row * (seen + len(step))
            else:
                nbytes += row * (sum(span) + len(step))
            flops += 4.0 * qd * sum(span)
    flops += 2.0 * head * heads
    return {"bytes": nbytes + 4.0 * d["vocab"] * heads, "flops": flops}


def tolerance(case):
    # the exact-integer modes are bit-reproducible by definition
    if case["mode"] in ("exact", "recall"):
        return "exact"
    # float: 1.1e-5 to 6.3e-5 off 64 bits; 1.2e-6 between the batched prefill and
    # one decode step per token, which add in other orders in part of the layers.
    # The codec rounds K/V to 8 bits, and another order flips codes: 9.5e-5
    # between the same two.
    return {"rel": 5e-4 if case["mode"] == "spinor" else 4e-5}


# ---------------------------------------------------------------- 64 bits
def _rms(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)          # every norm weight of these models is one


def _rope(x, pos, base):
    half = x.shape[-1] // 2
    th = pos.double().view(-1, 1, 1) * torch.pow(torch.tensor(float(base), dtype=torch.float64, device=x.device),
                                                 -torch.arange(half, dtype=torch.float64, device=x.device) / half)
    c, s, a, b = torch.cos(th), torch.sin(th), x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, a * s + b * c), -1)


def _attend(q, k, v, first, window):
    """q [n][heads][d] at positions first.., k and v [len][kv heads][d]."""
    n, nh, hd = q.shape
    g = nh // k.shape[1]
    out = torch.empty_like(q)
    for t0 in range(0, n, 512):
        t1 = min(n, t0 + 512)
        lo = max(0, first + t0 - window + 1) if window else 0
        hi = first + t1
        kk, vv = k[lo:hi].permute(1, 2, 0).contiguous(), v[lo:hi].permute(1, 0, 2).contiguous()
        p = torch.arange(lo, hi, device=q.device)
        t = torch.arange(first + t0, hi, device=q.device).view(-1, 1)
        dead = (p > t) | (p <= t - window) if window else p > t
        for i in range(g):                                                 # query head h g + i reads kv head h
            sc = torch.bmm(q[t0:t1, i::g].permute(1, 0, 2).contiguous(), kk) / math.sqrt(hd)
            out[t0:t1, i::g] = torch.bmm(torch.softmax(sc.masked_fill(dead, -math.inf), -1), vv).permute(1, 0, 2)
    return out


def _logits64(case, f, sequences):
    """The last position's logits of each token sequence."""
    d = _shape(case["model"])
    e, ff, hd, nh, nkv = d["hidden"], d["n_ff"], d["head_dim"], d["n_heads"], d["n_kv_heads"]
    gemma, eps = d["swa_window"] > 0, 1e-6
    xs = [f.matrix("token_embd.weight", e, torch.from_numpy(t.astype(np.int64)).cuda()) * (math.sqrt(e) if gemma else 1.0)
          for t in sequences]
    act = (lambda y: torch.nn.functional.gelu(y, approximate="tanh")) if gemma else torch.nn.functional.silu
    post = (lambda y: _rms(y, eps)) if gemma else (lambda y: y)
    for l in range(d["n_layers"]):
        w = {n: f.matrix("blk.%d.%s.weight" % (l, n), c).t().contiguous() for n, c in (
            ("attn_q", e), ("attn_k", e), ("attn_v", e), ("attn_output", nh * hd), ("ffn_gate", e), ("ffn_up", e), ("ffn_down", ff))}
        glob = _is_global(d, l)
        base, last = d["rope_base"] if glob else WINDOW_BASE, l == d["n_layers"] - 1
        for i, x in enumerate(xs):
            n, pos = x.shape[0], torch.arange(x.shape[0], device=x.device)
            hs = _rms(x, eps)
            k = _rope(_rms((hs @ w["attn_k"]).view(n, nkv, hd), eps), pos, base)
            v = (hs @ w["attn_v"]).view(n, nkv, hd)
            if last:                                                       # only the last position goes on
                x, hs, pos = x[-1:], hs[-1:], pos[-1:]
            q = _rope(_rms((hs @ w["attn_q"]).view(len(pos), nh, hd), eps), pos, base)
            o = _attend(q, k, v, n - len(pos), 0 if glob else d["swa_window"]).view(len(pos), nh * hd)
            x = x + post(o @ w["attn_output"])
            y = torch.empty_like(x)
            for r in range(0, len(x), 4096):
                hs = _rms(x[r:r + 4096], eps)
                y[r:r + 4096] = (act(hs @ w["ffn_gate"]) * (hs @ w["ffn_up"])) @ w["ffn_down"]
            xs[i] = x + post(y)
    out = f.matrix("output.weight" if "output.weight" in f.at else "token_embd.weight", e).t().contiguous()
    return [(_rms(x, eps) @ out)[0] for x in xs]


def exact(case, seed):
    # the codec's rounding, the recall's choice of rows and greedy tokens are
    # steps of which 64 bits has no nearby value
    if case["mode"] in ("spinor", "recall") or case["op"] == "greedy":
        return None
    _, f = _model(case["model"])
    if case["op"] == "batch":
        steps = _tokens(case, seed, 1, case["sessions"])
        rows = _logits64(case, f, [np.append(_tokens(case, seed, 2 + i, c), steps[i]) for i, c in enumerate(_contexts(case, seed))])
        return {"logits": torch.stack(rows), "next": None}
    tail = _tokens(case, seed, 1, case.get("n", 1))
    return _logits64(case, f, [np.concatenate((_tokens(case, seed, 0, case["ctx"]), tail))])[0]
