"""The work that programs have this library do, as cases that can be timed and
compared: greedy decoding of one sequence (resident launches and one call per
token), batched decoding of up to 16 sequences, and prompt prefill, each
through the Python entry points (``MegakernelEngine``, ``BatchEngine``).

Every case runs the whole 28-layer model with its 151,936-token tied head on
synthetic weights (``DeviceWeights``: N(0, 0.02) matrices, gains 1 + N(0, 0.1))
and, where it starts inside a conversation, a synthetic N(0, 1) KV prefix
(``fill_kv_synthetic``).  Activations are fp32 throughout, so the logits of a
whole model are comparable to about 1e-4.

Kinds:
  stream    one engine, ``decode_token`` per token (what ``generate`` does when
            there is an EOS token or a listener): fixed tokens go in, as a
            program that samples or constrains them would feed
  resident  one engine, all tokens in one resident launch (``decode_many``)
  request   one engine with a prefill context, a whole request as it arrives:
            ``generate_ids`` resets, prefills the prompt, decodes the answer
  batch     ``BatchEngine``: one ``decode`` call per step of all sequences
  prefill   ``BatchEngine.prefill``: prompt tokens at a position, logits back

The decode kinds end with one validation forward (``debug_forward``,
``debug_logits``), so that what comes back is the logits, which every position
appended before them has entered.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from megakernel_amd import BASELINE, QWEN3_06B
from megakernel_amd.batch import BatchEngine
from megakernel_amd.bridge import MegakernelEngine
from megakernel_amd.weights import DeviceWeights

SHAPES = {"baseline": BASELINE, "qwen3_06b": QWEN3_06B}
GAIN_STD = 0.1
MAX_SEQ = 33024  # the engine's default KV capacity
ANSWER = 12  # tokens of a request's answer
BATCH_SEQ = 4224  # KV capacity of a batch handle: 4,096 cached positions and some steps


def _case(kind, preset="baseline", seqs=1, lo=0, hi=0, n=1, kv8=False, lm8=False, w8=False):
    """lo .. hi: cached positions (one engine: lo); n: tokens, steps or prompt
    tokens; kv8 / lm8 / w8: FP8 KV cache, LM head, layer weights."""
    return {"kind": kind, "preset": preset, "seqs": seqs, "lo": lo, "hi": max(lo, hi), "n": n,
            "kv8": kv8, "lm8": lm8, "w8": w8}


def listed():
    named = [
        # the first tokens of an answer, streamed: a launch and a wait per token
        ("stream_ctx9", _case("stream", lo=9, n=12)),
        # the benchmark's context length, tokens of one resident launch
        ("resident_ctx1024", _case("resident", lo=1024, n=24)),
        # a long conversation, more attention splits than the role tables hold
        ("resident_ctx6001", _case("resident", lo=6001, n=16)),
        # the longest contexts, with the formats that are meant for them
        ("resident_ctx32000_fp8", _case("resident", lo=32000, n=16, kv8=True, lm8=True)),
        # the released 0.6B shape (head_dim 128, ffn 3072)
        ("resident_qwen3_ctx700", _case("resident", "qwen3_06b", lo=700, n=24)),
        # a short question and its answer, from an empty cache
        ("request_150", _case("request", lo=0, n=150)),
        # a full batch of ragged lengths (the batched benchmark's range)
        ("batch16_ctx512_4096", _case("batch", seqs=16, lo=512, hi=4096, n=8)),
        # a few short sequences on the FP8 formats
        ("batch3_fp8_ctx40_900", _case("batch", seqs=3, lo=40, hi=900, n=8, kv8=True, lm8=True)),
        # a one-line prompt, not a multiple of 16
        ("prefill_23", _case("prefill", lo=0, n=23)),
        # the next turn of a conversation on an FP8 cache
        ("prefill_200_at_1500_fp8", _case("prefill", lo=1500, n=200, kv8=True)),
        # the benchmark's prompt: one pass over the weights
        ("prefill_1024", _case("prefill", lo=0, n=1024)),
        # a document, several passes
        ("prefill_4000", _case("prefill", lo=0, n=4000)),
    ]
    return [dict(c, name=name) for name, c in named]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _one_split_count(at, tokens):
    """A start near `at` from which `tokens` positions pass no multiple of 512,
    where the attention's split count grows inside a resident launch (a thing
    of its own, for a test)."""
    over = at // 512 != (at + tokens - 1) // 512
    return max(1, (at + tokens - 1) // 512 * 512 - tokens) if over else at


def draw(rng):
    # FP8 rows only behind a prefix: on an empty cache every row is its own
    # rounding to 3 bits, and a rounding that falls the other way in one layer
    # moves the next layer's
    kind = rng.choice(("stream", "resident", "resident", "request", "batch", "batch", "prefill", "prefill", "prefill"))
    if kind == "stream":
        ctx = _log(rng, 1, 4000)
        return _case(kind, lo=ctx, n=rng.randint(8, 16), kv8=ctx >= 256 and rng.random() < 0.4, lm8=rng.random() < 0.25)
    if kind == "resident":
        if rng.random() < 0.3:
            n = rng.randint(8, 24)
            return _case(kind, "qwen3_06b", lo=_one_split_count(_log(rng, 16, 6000), n), n=n)
        n = rng.randint(8, 16)
        ctx = _one_split_count(_log(rng, 100, 32000), n)
        # FP8 layer weights are served up to about 4,000 positions
        return _case(kind, lo=ctx, n=n, kv8=ctx >= 256 and rng.random() < 0.4, lm8=rng.random() < 0.4,
                     w8=ctx < 3500 and rng.random() < 0.3)
    if kind == "request":
        return _case(kind, n=_one_split_count(_log(rng, 2, 2000), ANSWER), lm8=rng.random() < 0.25)
    if kind == "batch":
        lo = _log(rng, 1, 3000)
        return _case(kind, seqs=rng.randint(1, 16), lo=lo, hi=rng.randint(lo, 4096), n=rng.randint(4, 8),
                     kv8=lo >= 32 and rng.random() < 0.5, lm8=rng.random() < 0.3)
    ctx = rng.choice((0, _log(rng, 1, 1000)))
    return _case(kind, lo=ctx, n=_log(rng, 1, 3000), kv8=ctx >= 256 and rng.random() < 0.7, lm8=rng.random() < 0.2)


def _inputs(case, seed):
    """Cached positions per sequence, and the tokens that go in: [n] or [n][seqs]."""
    rng = random.Random(f"{seed} {case['kind']}")
    ctx = [rng.randint(case["lo"], case["hi"]) for _ in range(case["seqs"])]
    if case["kind"] == "batch":
        return ctx, [[rng.randrange(BASELINE.vocab) for _ in ctx] for _ in range(case["n"])]
    return ctx, [rng.randrange(BASELINE.vocab) for _ in range(case["n"])]


def prepare(case, seed):
    shape = SHAPES[case["preset"]]
    ctx, tokens = _inputs(case, seed)
    dw = DeviceWeights(shape, seed, gain_std=GAIN_STD)
    if case["kind"] in ("batch", "prefill"):
        eng = BatchEngine(dw, case["seqs"], BATCH_SEQ, shape)
    else:
        eng = MegakernelEngine(shape=shape, max_seq=MAX_SEQ, device_weights=dw, prefill=case["kind"] == "request")
    dw.free()  # the engines keep their own layouts
    if case["kv8"]:
        eng.set_kv_fp8(True)
    if case["lm8"]:
        eng.set_lmhead_fp8(True)
    if case["w8"]:
        eng.set_layer_fp8(True)
    for b, c in enumerate(ctx):
        if c:
            eng.fill_kv_synthetic(b, c, seed + b) if isinstance(eng, BatchEngine) else eng.fill_kv_synthetic(c, seed)
    return {"kind": case["kind"], "eng": eng, "ctx": ctx, "tokens": tokens, "n": case["n"]}


def run(state):
    eng, ctx, tokens, n = state["eng"], state["ctx"], state["tokens"], state["n"]
    if state["kind"] == "stream":
        eng.set_pos(ctx[0])
        for t in tokens[:-1]:
            eng.decode_token(t)
        nxt, layers, logits = eng.debug_forward(tokens[-1])
        return {"next": nxt, "layers": layers, "logits": logits}
    if state["kind"] == "resident":
        eng.set_pos(ctx[0])
        ids = eng.decode_many(tokens[0], n)
        nxt, layers, logits = eng.debug_forward(ids[-1])
        return {"ids": ids + [nxt], "layers": layers, "logits": logits}
    if state["kind"] == "request":
        ids, _rate = eng.generate_ids(tokens, max_tokens=ANSWER)
        nxt, layers, logits = eng.debug_forward(ids[-1])
        return {"ids": ids + [nxt], "layers": layers, "logits": logits}
    if state["kind"] == "batch":
        for b, c in enumerate(ctx):
            eng.set_pos(b, c)
        for step in tokens[:-1]:
            eng.decode(step)
        nxt, logits = eng.debug_logits(tokens[-1])
        return {"next": nxt, "logits": logits}
    eng.set_pos(0, ctx[0])
    nxt, logits = eng.prefill(0, tokens, with_logits=True)
    return {"next": nxt, "logits": logits}


def work(case):
    """Weights once per dependent step (a prefill: once, whatever its passes),
    the K / V rows that the step attends to read once, the appended rows
    written, the logits that come back written."""
    s = SHAPES[case["preset"]]
    L, n, B = s.n_layers, case["n"], case["seqs"]
    q, kv = s.n_q_heads * s.head_dim, s.n_kv_heads * s.head_dim
    mats = L * ((q + 2 * kv) * s.hidden + s.hidden * q + 3 * s.ffn * s.hidden)
    head = s.vocab * s.hidden
    wbytes = mats * (1 if case["w8"] else 2) + head * (1 if case["lm8"] else 2)
    row = L * 2 * (kv * (1 if case["kv8"] else 2) + (4 * s.n_kv_heads if case["kv8"] else 0))  # one position's K and V
    attn = 4 * L * q  # flops per query and position
    ctx = (case["lo"] + case["hi"]) / 2
    out = 4 * s.vocab * B

    def sweep(tokens, at):  # one pass over the weights for `tokens` consecutive tokens of one sequence
        return (wbytes + row * (at + 2 * tokens),
                2 * mats * tokens + 2 * head + attn * tokens * (at + (tokens + 1) / 2))

    if case["kind"] == "prefill":
        b, f = sweep(n, ctx)
    elif case["kind"] == "batch":
        b = n * (wbytes + B * row * (ctx + n / 2 + 1))
        f = n * B * (2 * (mats + head) + attn * (ctx + n / 2))
    else:
        steps = {"stream": n, "resident": n + 1, "request": ANSWER}[case["kind"]]
        at = n if case["kind"] == "request" else ctx
        b = steps * (wbytes + row * (at + steps / 2 + 1))
        f = steps * (2 * (mats + head) + attn * (at + steps / 2))
        if case["kind"] == "request":
            pb, pf = sweep(n, 0)
            b, f = b + pb, f + pf
    return {"bytes": b + out, "flops": f}


def tolerance(case):
    """About four times what a pass differs from 64 bits with the same cache
    format.  Behind a prefix the fp32 arithmetic shows (2e-5 .. 2e-4, with a
    few hundred appended FP8 roundings 1.2e-3); from a short or empty cache the appended
    rows' own bf16 roundings do, which fall either way after a few layers
    (up to 2.4e-3 for a two-token prompt)."""
    if case["lo"] < 100:
        return {"rel": 0.01, "max": 0.05}
    return {"rel": 0.005, "max": 0.02} if case["kv8"] else {"rel": 0.001, "max": 0.005}


# ------------------------------------------------------------------ 64 bits
# The model in float64 torch, from the documented synthetic streams.
_GOLD = 0x9E3779B97F4A7C15
_M64 = (1 << 64) - 1
_KV_STREAM = 0x40000000


def _mix(z):
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
    return z ^ (z >> 31)


def _key(seed, tensor):
    return _mix((seed + (tensor + 1) * _GOLD) & _M64)


def _signed(v):
    return v - (1 << 64) if v >> 63 else v


def _stream(key, count, std, add_one, device):
    """bf16 values 0 .. count - 1 of a splitmix64 stream: the sum of each
    output's four 16-bit fields, centred and scaled."""
    out = torch.empty(count, dtype=torch.bfloat16, device=device)
    c = torch.tensor(np.float32(std * math.sqrt(3.0) / 65536.0), device=device)
    for at in range(0, count, 1 << 25):
        m = min(1 << 25, count - at)
        z = torch.arange(at + 1, at + 1 + m, dtype=torch.int64, device=device) * _signed(_GOLD) + _signed(key)
        z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * _signed(0xBF58476D1CE4E5B9)
        z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * _signed(0x94D049BB133111EB)
        z = z ^ ((z >> 31) & ((1 << 33) - 1))
        s = (z & 0xFFFF) + ((z >> 16) & 0xFFFF) + ((z >> 32) & 0xFFFF) + ((z >> 48) & 0xFFFF)
        f = (s - 131070).float() * c
        out[at:at + m] = (1.0 + f if add_one else f).to(torch.bfloat16)
    return out


def _e4m3_rows(x):
    """Rows through OCP e4m3 with the smallest power-of-two scale that fits."""
    amax = x.abs().amax(-1, keepdim=True).float()
    m, ex = torch.frexp(amax)
    e = torch.where(amax > 0, ex - 9 + (m > 0.875).int(), torch.zeros_like(ex))
    scale = torch.ldexp(torch.ones_like(amax), e).double()
    return (x.double() / scale).float().to(torch.float8_e4m3fn).double() * scale


class _Exact:
    def __init__(self, case, seed):
        self.s = s = SHAPES[case["preset"]]
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.kv8 = case["kv8"]
        q, kv, h = s.n_q_heads * s.head_dim, s.n_kv_heads * s.head_dim, s.hidden
        dims = [("attn_norm", (h,)), ("q", (q, h)), ("k", (kv, h)), ("v", (kv, h)), ("q_norm", (s.head_dim,)),
                ("k_norm", (s.head_dim,)), ("o", (h, q)), ("ffn_norm", (h,)), ("gate", (s.ffn, h)),
                ("up", (s.ffn, h)), ("down", (h, s.ffn))]

        def tensor(ident, shape):
            norm = len(shape) == 1
            return _stream(_key(seed, ident), math.prod(shape), GAIN_STD if norm else 0.02, norm, self.dev).view(shape)

        self.embed = tensor(0, (s.vocab, h))
        self.final = tensor(1, (h,)).double()
        self.layers = []
        for i in range(s.n_layers):
            w = {name: tensor(2 + 11 * i + j, shape) for j, (name, shape) in enumerate(dims)}
            self.layers.append({k: _e4m3_rows(v).to(torch.bfloat16) if case["w8"] and v.ndim == 2 else v
                                for k, v in w.items()})
        self.head = _e4m3_rows(self.embed).to(torch.bfloat16) if case["lm8"] else self.embed

    def stored(self, x):
        """What the cache holds of K / V rows."""
        return _e4m3_rows(x.float()) if self.kv8 else x.to(torch.bfloat16).double()

    def fill(self, seed, ctx, room):
        """A cache of `ctx` synthetic positions with room for more."""
        s = self.s
        self.kv = torch.zeros(s.n_layers, 2, s.n_kv_heads, ctx + room, s.head_dim, dtype=torch.float64, device=self.dev)
        self.pos = ctx
        for i in range(s.n_layers):
            for j in range(2):
                if ctx:
                    rows = _stream(_key(seed, _KV_STREAM + 2 * i + j), ctx * s.n_kv_heads * s.head_dim, 1.0, False, self.dev)
                    self.kv[i, j, :, :ctx] = self.stored(rows.view(ctx, s.n_kv_heads, s.head_dim).transpose(0, 1))

    def norm(self, x, gain):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * gain.double()

    def forward(self, tokens):
        """Consumes tokens at the position: the last one's layers and logits."""
        s, D, n, p = self.s, self.s.head_dim, len(tokens), self.pos
        freq = 1.0 / (1e6 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))  # angles in fp32, as the model defines them
        angle = (torch.arange(p, p + n, dtype=torch.float32)[:, None] * freq).double().to(self.dev)
        cos, sin = torch.cat((angle, angle), -1).cos(), torch.cat((angle, angle), -1).sin()

        def rope(x):  # [heads][n][D]
            return x * cos + torch.cat((-x[..., D // 2:], x[..., :D // 2]), -1) * sin

        def heads(x):
            return x.view(n, -1, D).transpose(0, 1)

        x = self.embed[torch.tensor(tokens, device=self.dev)].double()
        layers = [x[-1]]
        causal = torch.arange(p + n, device=self.dev)[None] > torch.arange(p, p + n, device=self.dev)[:, None]
        for i, w in enumerate(self.layers):
            a = self.norm(x, w["attn_norm"])
            qh = rope(self.norm(heads(a @ w["q"].double().T), w["q_norm"]))
            self.kv[i, 0, :, p:p + n] = self.stored(rope(self.norm(heads(a @ w["k"].double().T), w["k_norm"])))
            self.kv[i, 1, :, p:p + n] = self.stored(heads(a @ w["v"].double().T))
            out = []
            for g in range(s.n_kv_heads):
                k, v = self.kv[i, 0, g, :p + n], self.kv[i, 1, g, :p + n]
                for j in range(s.n_q_heads // s.n_kv_heads):
                    sc = (qh[g * (s.n_q_heads // s.n_kv_heads) + j] @ k.T / math.sqrt(D)).masked_fill_(causal, -math.inf)
                    out.append(torch.softmax(sc, -1) @ v)
            x = x + torch.cat(out, -1) @ w["o"].double().T
            f = self.norm(x, w["ffn_norm"])
            x = x + (torch.nn.functional.silu(f @ w["gate"].double().T) * (f @ w["up"].double().T)) @ w["down"].double().T
            layers.append(x[-1])
        self.pos += n
        hid = self.norm(x[-1], self.final)
        logits = torch.cat([part.double() @ hid for part in self.head.split(1 << 14)])
        return torch.stack(layers), logits


def exact(case, seed):
    ctx, tokens = _inputs(case, seed)
    m = _Exact(case, seed)
    if case["kind"] == "batch":
        rows = []
        for b, c in enumerate(ctx):
            m.fill(seed + b, c, len(tokens))
            rows.append(m.forward([step[b] for step in tokens])[1])
        logits = torch.stack(rows)
        return {"next": logits.argmax(-1).tolist(), "logits": logits}
    m.fill(seed, ctx[0], len(tokens) + 64)
    if case["kind"] in ("stream", "prefill"):
        layers, logits = m.forward(tokens)
        out = {"next": int(logits.argmax()), "logits": logits}
        return dict(out, layers=layers) if case["kind"] == "stream" else out
    layers, logits = m.forward(tokens if case["kind"] == "request" else tokens[:1])
    ids = [int(logits.argmax())]
    for _ in range(ANSWER if case["kind"] == "request" else case["n"]):
        layers, logits = m.forward(ids[-1:])
        ids.append(int(logits.argmax()))
    return {"ids": ids, "layers": layers, "logits": logits}
