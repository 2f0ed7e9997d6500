"""The work that programs have this device do, as cases to be timed and compared.

Two kinds of program use it. One drives the model: it feeds a prompt or a
chat's next turn, lets the device decode a reply, and reads logits
(`Model.forward`, `Model.decode`). The other drives the operations one by one,
as the reference's `Model<D: Device>` does (model/model.rs:93-149). A
"session" case is the first kind, over the fused path or the trait's
operations; "matmul", "attention" and "norm" are single calls of the second.

Sessions run the Qwen3-0.6B and Qwen3-4B layer shapes and the tiny one. Two of
them are the whole Qwen3-0.6B; the others stack fewer layers over a smaller
vocabulary, so that their time is the layers'. Weights are drawn once per
shape (a program loads its model once); tokens, caches and activations come
from a case's seed.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from titania_amd import QWEN3_0_6B, QWEN3_4B, TH_KV_BF16, TH_KV_F32, TH_PATH_FUSED, TH_PATH_TRAIT
from titania_amd.config import QWEN3_TINY, Config
from titania_amd.device import Hip, Tensor
from titania_amd.model import Model, State
from titania_amd.sampler import Sampler
from titania_amd.synth import shapes

EPS = 1e-6
SHAPES = {"0.6b": QWEN3_0_6B, "4b": QWEN3_4B, "tiny": QWEN3_TINY}


def _session(name, shape, layers, vocab, pos, n, steps=0, follow=0, kv="f32", path="fused", temperature=0.0, top_k=1,
             top_p=1.0):
    """`pos` tokens are in the caches; a pass feeds `n` tokens, then (with
    steps) decodes a reply of `steps` tokens and feeds a next turn of `follow`
    tokens, and reads the logits after the last token fed."""
    c = dict(kind="session", shape=shape, layers=layers, vocab=vocab, pos=pos, n=n, steps=steps, follow=follow, kv=kv,
             path=path, temperature=temperature, top_k=top_k, top_p=top_p)
    return dict(c, name=name) if name else c


def listed():
    return [
        # A chat at temperature 0 with the whole Qwen3-0.6B: a 16-token
        # prompt, 32 tokens of reply, and the user's next turn of 6 tokens.
        _session("chat", "0.6b", 28, 151936, 0, 16, 32, 6),
        # A sampled reply (temperature 0.7, as the reference's command line
        # draws), the caller looking at the logits after one more token.
        _session("chat sampled", "0.6b", 12, 151936, 0, 40, 24, 1, temperature=0.7, top_k=20, top_p=0.8),
        # The prefill workload: a 512-token prompt, the whole Qwen3-0.6B.
        _session("prompt", "0.6b", 28, 151936, 0, 512),
        # A chat's next user turn, of an odd and small length, in a
        # conversation of some length; wider layers.
        _session("turn", "4b", 4, 8192, 700, 11),
        # A caller that picks every token itself, over bf16 caches: one token
        # in, logits out.
        _session("token", "0.6b", 12, 16384, 100, 1, kv="bf16"),
        # A document of 8192 tokens: the largest prompt fed at once.
        _session("long prompt", "4b", 2, 8192, 0, 8192),
        # A reply far into a long context.
        _session("long context", "4b", 4, 8192, 8192, 1, 16, 1),
        # The same model through the trait's operations (in batches of 64).
        _session("trait prompt", "0.6b", 12, 16384, 0, 100, path="trait"),
        # A projection of one batch of the trait's forward (down_proj, 4B).
        {"name": "matmul batch", "kind": "matmul", "n": 64, "rows": 2560, "cols": 9728},
        # A projection of sizes that are whole tiles in no direction.
        {"name": "matmul ragged", "kind": "matmul", "n": 50, "rows": 1000, "cols": 1096},
        # Decode attention of the trait over a long cache.
        {"name": "attention", "kind": "attention", "n": 1, "pos": 32767, "heads": 16, "kv_heads": 8, "head_dim": 128},
        # The smallest call: one token's residual add and norm.
        {"name": "norm", "kind": "norm", "rows": 1, "dim": 1024},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49)))))))


def draw(rng):
    pick = rng.random()
    if pick < 0.6:
        shape, layers, vocab = rng.choice([("0.6b", 12, 16384), ("0.6b", 12, 151936), ("4b", 2, 8192), ("4b", 4, 8192),
                                           ("tiny", 2, 1000)])
        what = rng.random()
        if what < 0.25:  # a prompt through the trait's operations
            return _session(None, shape, layers, vocab, 0, _log_int(rng, 1, 400), path="trait")
        pos = rng.choice([0, _log_int(rng, 1, 4000)])
        if what < 0.7:  # a prompt or a turn
            return _session(None, shape, layers, vocab, pos, _log_int(rng, 1, 3000), kv=rng.choice(["f32", "f32", "bf16"]))
        # A reply, over f32 caches: in bf16 a key that rounds the other way
        # moves the logits by 1e-3, enough to change a drawn token and with it
        # all that follow.
        warm = rng.random() < 0.5  # drawn, or greedy
        return _session(None, shape, layers, vocab, pos, _log_int(rng, 1, 200), rng.randint(2, 32),
                        _log_int(rng, 1, 40), temperature=round(rng.uniform(0.5, 1.2), 2) if warm else 0.0,
                        top_k=_log_int(rng, 2, 256) if warm else 1, top_p=round(rng.uniform(0.6, 1.0), 2) if warm else 1.0)
    if pick < 0.8:
        # The projections of the two models, or any matrix of rows of whole
        # 16-byte chunks.
        rows, cols = rng.choice([(2048, 1024), (1024, 1024), (1024, 2048), (3072, 1024), (1024, 3072), (4096, 2560),
                                 (2560, 4096), (9728, 2560), (2560, 9728),
                                 (_log_int(rng, 40, 8000), 8 * _log_int(rng, 8, 600)),
                                 (_log_int(rng, 40, 8000), 8 * _log_int(rng, 8, 600))])
        return {"kind": "matmul", "n": _log_int(rng, 1, 2000), "rows": rows, "cols": cols}
    if pick < 0.93:
        heads, kv_heads, hd = rng.choice([(16, 8, 128), (32, 8, 128), (4, 2, 128), (4, 4, 64), (8, 1, 128), (4, 2, 256)])
        n = rng.choice([1, _log_int(rng, 2, 64)])  # the trait's forward goes in batches of up to 64
        return {"kind": "attention", "n": n, "pos": _log_int(rng, 8, 32000), "heads": heads, "kv_heads": kv_heads,
                "head_dim": hd}
    return {"kind": "norm", "rows": _log_int(rng, 1, 4000), "dim": rng.choice([128, 512, 896, 1024, 2560, 4096])}


# ---- what a program has in hand ----

_device = None
_models: dict = {}


def _hip() -> Hip:
    global _device
    if _device is None:
        _device = Hip(0)
    return _device


def _config(case) -> Config:
    c = SHAPES[case["shape"]]
    return Config(c.hidden_size, c.intermediate_size, case["layers"], c.num_attention_heads, c.num_key_value_heads,
                  case["vocab"], EPS, c.rope_theta, True, c.head_dim())


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(shape, index: int) -> torch.Tensor:
    """N(0, 0.02) matrices and gains about 1, bf16, on the GPU."""
    t = torch.randn(shape, generator=_generator(1000 + index), device="cuda")
    return ((1 + 0.1 * t) if len(shape) == 1 else 0.02 * t).to(torch.bfloat16)


def _bits(t: torch.Tensor) -> Tensor:
    return Tensor(tuple(t.shape), t.view(torch.int16).cpu().numpy().view(np.uint16))


def _model(case) -> Model:
    key = (case["shape"], case["layers"], case["vocab"])
    if key not in _models:
        cfg = _config(case)
        _models[key] = Model(_hip(), cfg, {name: _bits(_weight(shape, i)) for i, (name, shape) in enumerate(shapes(cfg).items())})
    return _models[key]


def _tokens(case, seed: int) -> np.ndarray:
    """Every token of a session, in order: those in the caches, those fed, and
    the next turn's."""
    r = np.random.RandomState(seed % (1 << 32))
    return r.randint(case["vocab"], size=case["pos"] + case["n"] + case["follow"]).astype(np.uint32)


class _InPlace:
    """A buffer's memory, for torch to look at in place (which keeps the
    buffer): a handle points at the device address first."""

    def __init__(self, buf, shape: tuple):
        self.buf = buf
        address = ctypes.c_void_p.from_address(buf.handle).value
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False), "version": 2}


def _view(buf, *shape) -> torch.Tensor:
    """A buffer's values where they are. The outputs of the single operations
    are looked at this way, since a program that chains operations reads none
    of them back."""
    return torch.as_tensor(_InPlace(buf, shape), device="cuda")


def _buffer(values: torch.Tensor):
    b = _hip().alloc(values.numel())
    _view(b, values.numel()).copy_(values.reshape(-1))
    return b


class _Chat:
    """A session's model, state and tokens; the state is freed with it."""

    def __init__(self, case, seed):
        self.case, self.model = case, _model(case)
        self.tokens = _tokens(case, seed)
        self.seed = 1 + seed % 1000003
        self.path = TH_PATH_TRAIT if case["path"] == "trait" else TH_PATH_FUSED
        total = len(self.tokens) + case["steps"]
        self.state = State(self.model, total, TH_KV_BF16 if case["kv"] == "bf16" else TH_KV_F32)
        if case["pos"]:
            self.model.forward(self.state, self.tokens[:case["pos"]], 0, self.path, want_logits=False)

    def __del__(self):
        if getattr(self, "state", None) is not None:
            self.state.close()


def _norm_inputs(case, seed):
    g = _generator(seed)
    x, y = (torch.randn((case["rows"], case["dim"]), generator=g, device="cuda") for _ in range(2))
    return x, y, (1 + 0.1 * torch.randn(case["dim"], generator=g, device="cuda")).to(torch.bfloat16)


def _matmul_inputs(case, seed):
    g = _generator(seed)
    w = (0.02 * torch.randn((case["rows"], case["cols"]), generator=g, device="cuda")).to(torch.bfloat16)
    return w, torch.randn((case["n"], case["cols"]), generator=g, device="cuda")


def _attention_inputs(case, seed):
    """Queries and keys of unit scale per dimension, as the q/k norms leave them."""
    g = _generator(seed)
    ctx = case["pos"] + case["n"]
    q = torch.randn((case["n"], case["heads"], case["head_dim"]), generator=g, device="cuda")
    k, v = (torch.randn((ctx, case["kv_heads"], case["head_dim"]), generator=g, device="cuda") for _ in range(2))
    return q, k, v


def prepare(case, seed):
    hip = _hip()
    if case["kind"] == "session":
        return _Chat(case, seed)
    if case["kind"] == "matmul":
        w, x = _matmul_inputs(case, seed)
        out = hip.alloc(case["n"] * case["rows"])
        return case, hip.upload(_bits(w)), _buffer(x), out, _view(out, case["n"], case["rows"])
    if case["kind"] == "attention":
        q, k, v = _attention_inputs(case, seed)
        out = hip.alloc(q.numel())
        return case, _buffer(q), _buffer(k), _buffer(v), out, _view(out, *q.shape)
    x, y, gain = _norm_inputs(case, seed)
    x, y, xb = _buffer(x), _buffer(y), hip.alloc(x.numel())
    views = {"x": _view(x, case["rows"], case["dim"]), "xb": _view(xb, case["rows"], case["dim"])}
    return case, x, y, xb, hip.upload(_bits(gain)), views


def run(state):
    if isinstance(state, _Chat):
        c, m, s, t = state.case, state.model, state.state, state.tokens
        pos, n, steps = c["pos"], c["n"], c["steps"]
        if not steps:
            return m.forward(s, t[pos:], pos, state.path)
        m.forward(s, t[pos:pos + n], pos, state.path, want_logits=False)
        sampler = Sampler(c["temperature"], c["top_k"], c["top_p"], state.seed) if c["temperature"] else None
        reply = m.decode(s, pos + n, steps, sampler=sampler)
        return {"reply": reply, "logits": m.forward(s, t[pos + n:], pos + n + steps, state.path)}
    case, hip = state[0], _hip()
    if case["kind"] == "matmul":
        _, w, x, out, seen = state
        hip.matmul(out, w, x)
        return seen
    if case["kind"] == "attention":
        _, q, k, v, out, seen = state
        hip.attention(out, q, k, v, case["pos"], case["heads"], case["head_dim"], case["kv_heads"])
        return seen
    _, x, y, xb, gain, views = state
    hip.add_rmsnorm(x, y, xb, gain, EPS)
    return views


# ---- what a pass cannot do without ----

def work(case):
    if case["kind"] == "matmul":
        n, rows, cols = case["n"], case["rows"], case["cols"]
        return {"bytes": 2 * rows * cols + 4 * n * (rows + cols), "flops": 2 * n * rows * cols}
    if case["kind"] == "attention":
        n, ctx, hd = case["n"], case["pos"] + case["n"], case["head_dim"]
        seen = n * case["pos"] + n * (n + 1) // 2
        return {"bytes": 4 * (2 * ctx * case["kv_heads"] * hd + 2 * n * case["heads"] * hd),
                "flops": 4 * seen * case["heads"] * hd}
    if case["kind"] == "norm":
        return {"bytes": 16 * case["rows"] * case["dim"] + 2 * case["dim"], "flops": 6 * case["rows"] * case["dim"]}
    c = _config(case)
    qd, kvd = c.num_attention_heads * c.head_dim(), c.num_key_value_heads * c.head_dim()
    layer = c.hidden_size * (2 * qd + 2 * kvd + 3 * c.intermediate_size)
    head = c.hidden_size * c.vocab_size
    kv_size = 2 if case["kv"] == "bf16" else 4
    total = {"bytes": 0, "flops": 0}

    def feed(pos, n):
        seen = n * pos + n * (n + 1) // 2
        total["bytes"] += 2 * (c.num_hidden_layers * layer + head) + 4 * c.vocab_size
        total["bytes"] += c.num_hidden_layers * 2 * kvd * kv_size * (pos + 2 * n)
        total["flops"] += 2 * (c.num_hidden_layers * layer * n + head) + 4 * c.num_hidden_layers * seen * qd

    feed(case["pos"], case["n"])
    for i in range(case["steps"]):
        feed(case["pos"] + case["n"] + i, 1)
    if case["follow"]:
        feed(case["pos"] + case["n"] + case["steps"], case["follow"])
    return total


def tolerance(case):
    """About four times the distance from `exact` that was measured: sessions
    6e-6 to 1.4e-5 over f32 caches (activations enter the matrix cores as two
    bf16 terms) and 1e-3 over bf16 ones, products 2.5e-6, attention 2.5e-7 for
    one token and two-term products for more, norms 1e-7."""
    if case["kind"] == "session":
        return {"rel": 5e-3 if case["kv"] == "bf16" else 5e-5, "differ": 0.0}
    return {"rel": {"matmul": 1e-5, "attention": 2e-5, "norm": 1e-6}[case["kind"]]}


# ---- the same in 64 bits ----

def _rms64(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain.double()


def _attention64(q, k, v, pos):
    """Causal attention of q [n, heads, hd] at positions pos.. over k, v
    [ctx, kv_heads, hd], in 64 bits."""
    n, heads, hd = q.shape
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    step = max(1, (1 << 28) // (k.shape[0] * heads))
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    at = torch.arange(k.shape[0], device=q.device)
    for t in range(0, n, step):
        m = min(step, n - t)
        s = torch.matmul(q[t:t + m].reshape(m, -1, group, hd).permute(1, 2, 0, 3).reshape(-1, group * m, hd), kt)
        s = s.reshape(-1, group, m, k.shape[0]) / math.sqrt(hd)
        s.masked_fill_(at[None, :] > (pos + t + torch.arange(m, device=q.device))[:, None], -math.inf)
        p = torch.softmax(s, -1).reshape(-1, group * m, k.shape[0])
        out[t:t + m] = torch.matmul(p, vt).reshape(-1, group, m, hd).permute(2, 0, 1, 3).reshape(m, heads, hd)
    return out


class _Model64:
    """The model of model/model.rs:93-149 in 64 bits. The rotation angles are
    the 32-bit ones that the reference's table is made of."""

    def __init__(self, case):
        self.c = _config(case)
        self.bf16 = case["kv"] == "bf16"
        weights = [_weight(shape, i) for i, shape in enumerate(shapes(self.c).values())]
        self.layers = [weights[11 * i:11 * i + 11] for i in range(self.c.num_hidden_layers)]
        self.embed, self.norm = weights[11 * self.c.num_hidden_layers:][:2]
        self.keys = [None] * len(self.layers)
        self.values = [None] * len(self.layers)
        hd = self.c.head_dim()
        power = np.float64(np.float32(self.c.rope_theta)) ** (2 * np.arange(hd // 2) / hd)
        self.freq = torch.from_numpy(np.float32(1) / power.astype(np.float32)).cuda()

    def rope(self, x, pos):
        a = (torch.arange(pos, pos + x.shape[0], device="cuda").float()[:, None] * self.freq).double()[:, None]
        lo, hi = x.chunk(2, -1)
        return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)

    def forward(self, tokens, pos):
        c, n, hd = self.c, len(tokens), self.c.head_dim()
        x = self.embed[torch.from_numpy(np.asarray(tokens, dtype=np.int64)).cuda()].double()
        for i, (norm, wq, wk, wv, wo, q_norm, k_norm, mlp_norm, gate, up, down) in enumerate(self.layers):
            h = _rms64(x, norm)
            q, k, v = ((h @ w.double().T).reshape(n, -1, hd) for w in (wq, wk, wv))
            q, k = self.rope(_rms64(q, q_norm), pos), self.rope(_rms64(k, k_norm), pos)
            if self.bf16:
                k, v = (t.float().to(torch.bfloat16).double() for t in (k, v))
            if pos:
                k, v = torch.cat([self.keys[i][:pos], k]), torch.cat([self.values[i][:pos], v])
            self.keys[i], self.values[i] = k, v
            x = x + _attention64(q, k, v, pos).reshape(n, -1) @ wo.double().T
            h = _rms64(x, mlp_norm)
            x = x + (torch.nn.functional.silu(h @ gate.double().T) * (h @ up.double().T)) @ down.double().T
        return _rms64(x[-1], self.norm) @ self.embed.double().T


def _draw64(logits, case, state):
    """model/sampler.rs:21-76 in 64 bits: a token, and the generator's next state."""
    top, index = torch.topk(logits, min(case["top_k"], logits.numel()))
    p = torch.softmax(top / case["temperature"], 0).cpu().numpy()
    before = np.concatenate([[0.0], np.cumsum(p)[:-1]])
    p = p[before < case["top_p"]]
    mask = (1 << 64) - 1
    state ^= state >> 12
    state ^= (state << 25) & mask
    state ^= state >> 27
    r = (((state * 0x2545F4914F6CDD1D) & mask) >> 40) / float(1 << 24) * p.sum()
    at = np.nonzero(np.cumsum(p) >= r)[0]
    return int(index[at[0] if len(at) else len(p) - 1]), state


def exact(case, seed):
    if case["kind"] == "matmul":
        w, x = _matmul_inputs(case, seed)
        return x.double() @ w.double().T
    if case["kind"] == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        return _attention64(q, k, v, case["pos"])
    if case["kind"] == "norm":
        x, y, gain = _norm_inputs(case, seed)
        x = x.double() + y.double()
        return {"x": x, "xb": _rms64(x, gain)}
    m, t, pos, n = _Model64(case), _tokens(case, seed), case["pos"], case["n"]
    for at in range(0, pos, 2048):
        m.forward(t[at:min(pos, at + 2048)], at)
    for at in range(pos, pos + n, 2048):
        logits = m.forward(t[at:min(pos + n, at + 2048)], at)
    if not case["steps"]:
        return logits
    reply, state = [], 1 + seed % 1000003
    for i in range(case["steps"]):
        if case["temperature"]:
            token, state = _draw64(logits, case, state)
        else:
            token = int(logits.argmax())
        reply.append(token)
        logits = m.forward([token], pos + n + i)
    return {"reply": np.array(reply, dtype=np.uint32), "logits": m.forward(t[pos + n:], pos + n + case["steps"])}
