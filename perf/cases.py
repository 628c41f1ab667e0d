"""The workloads this framework's speed is measured on: what a program that serves or evaluates a Qwen3-shaped decoder
calls, through `QwenModel` (forward, decode_set / decode_run / decode_ids, read_logits).

A case is a model and one call on it:

  shape   "tiny" (hidden 64, 4/2 heads of 16, SwiGLU 192), "0.6b" (hidden 1024, 16/8 heads of 128, SwiGLU 3072) or
          "1.7b" (hidden 2048, 16/8 heads of 128, SwiGLU 6144): the configurations of this repository
  layers, vocab   28 layers and 151936 ids are the whole 0.6B model; fewer layers over a 4096-id vocabulary are a block
          of its decoder layers between an embedding and a head
  mode    "fp32" (the parity path: float32 activations and caches) or "fast" (fp16 operands and caches)
  op      "forward": t tokens at positions pos .. pos + t - 1, the last `rows` rows of logits returned
          "decode": one on-device step of `batch` sequences; sequence b stands at position pos - b * stagger, and the
          program reads the step's logits (a sampler's loop)
  chunk   rows per forward chunk the model is planned for

The contexts a call stands on are prefilled by the model itself in prepare(), as a program's are. Weights are
N(0, 0.02) in bf16, norm weights 1 + N(0, 0.1), ids uniform, all from the seed.
"""
import math

import numpy as np
import torch

from rosylnalive_amd.gpu_core import HipBackend
from rosylnalive_amd.qwen import LAYER_WEIGHTS, QwenConfig, QwenModel

SHAPES = {  # hidden, heads, kv heads, head_dim, intermediate
    "tiny": (64, 4, 2, 16, 192),
    "0.6b": (1024, 16, 8, 128, 3072),
    "1.7b": (2048, 16, 8, 128, 6144),
}
EPS = 1e-6


def _case(name, mode, shape, layers, vocab, op, **kw):
    c = {"name": name, "mode": mode, "shape": shape, "layers": layers, "vocab": vocab, "op": op, "t": 1, "pos": 0,
         "rows": 1, "batch": 1, "stagger": 0, "chunk": 512}
    c.update(kw)
    return c


def listed():
    return [
        # the plumbing model's decode step in the parity mode: the smallest call, all launches and host time
        _case("tiny_step_fp32", "fp32", "tiny", 2, 512, "forward", t=1, pos=40, chunk=64),
        # the parity path scoring a ragged prompt (every row's logits), two layers
        _case("prompt150_fp32", "fp32", "0.6b", 2, 4096, "forward", t=150, rows=150),
        # the parity path's decode step over a 700-token context, four layers
        _case("step700_fp32", "fp32", "0.6b", 4, 4096, "forward", t=1, pos=700),
        # a short ragged chat prompt, every row scored
        _case("prompt37", "fast", "0.6b", 4, 4096, "forward", t=37, rows=37),
        # a whole 0.6B prefill of 512 tokens, last row: the time to the first token
        _case("prefill512_0.6b", "fast", "0.6b", 28, 151936, "forward", t=512),
        # a long prompt in one chunk, the last 64 rows scored
        _case("prompt2048", "fast", "0.6b", 4, 4096, "forward", t=2048, rows=64, chunk=2048),
        # the last 512-token chunk of an 8K document: attention over the cached keys carries the weight
        _case("chunk512_at7680", "fast", "0.6b", 4, 4096, "forward", t=512, pos=7680),
        # an odd-length prompt on the larger layer
        _case("prompt777_1.7b", "fast", "1.7b", 4, 4096, "forward", t=777, chunk=1024),
        # one token of the whole 0.6B model for one sequence, its logits read by a sampler
        _case("step400_0.6b", "fast", "0.6b", 28, 151936, "decode", pos=400),
        # the same loop on the larger layer at a longer context
        _case("step1500_1.7b", "fast", "1.7b", 8, 4096, "decode", pos=1500),
        # a few sequences of uneven length decoded together
        _case("batch5_0.6b", "fast", "0.6b", 8, 4096, "decode", pos=1900, batch=5, stagger=411),
        # a full batch at 8K context, the serving workload
        _case("batch16_8k_1.7b", "fast", "1.7b", 4, 4096, "decode", pos=8192, batch=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("fp32", "fp32", "prompt", "prompt", "chunk", "step", "batch", "batch"))
    if kind == "fp32":
        if rng.random() < 0.5:  # a prompt, scored
            t = _log(rng, 2, 300)
            c = _case("", "fp32", "0.6b", rng.randint(1, 2), 4096, "forward", t=t, rows=rng.randint(1, t),
                      pos=rng.choice((0, 0, _log(rng, 1, 300))))
        else:  # a step
            c = _case("", "fp32", "0.6b", rng.randint(2, 6), 4096, "forward", pos=_log(rng, 8, 1500))
    elif kind == "prompt":
        shape = rng.choice(("0.6b", "0.6b", "1.7b"))
        t = _log(rng, 2, 2048)
        c = _case("", "fast", shape, rng.randint(2, 4), 4096, "forward", t=t, rows=rng.randint(1, min(t, 64)),
                  chunk=rng.choice((512, 1024, 2048)))
    elif kind == "chunk":
        t = _log(rng, 16, 512)
        c = _case("", "fast", "0.6b", rng.randint(2, 4), 4096, "forward", t=t, pos=_log(rng, 100, 7680))
    elif kind == "step":
        shape = rng.choice(("0.6b", "1.7b"))
        c = _case("", "fast", shape, rng.randint(4, 28 if shape == "0.6b" else 8), 4096, "decode",
                  pos=_log(rng, 16, 6000))
    else:
        shape, batch = rng.choice(("0.6b", "1.7b")), rng.randint(2, 16)
        pos = _log(rng, 64, 8000)
        c = _case("", "fast", shape, rng.randint(2, 4), 4096, "decode", pos=pos, batch=batch,
                  stagger=rng.randint(0, pos // batch))
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs

def _positions(case):
    """The position of each sequence's next token."""
    return [case["pos"] - b * case["stagger"] for b in range(case["batch"])]


def _inv_freq(head_dim):
    """float32 theta^(-2j/d), theta = 1e6."""
    return (1.0 / 1e6 ** (np.arange(0, head_dim, 2, dtype=np.float64) / head_dim)).astype(np.float32)


def _weights(case, seed, device):
    """{Hugging Face name: bf16 tensor} on `device`, from the seed."""
    H, QH, KVH, HD, I = SHAPES[case["shape"]]
    g = torch.Generator(device=device).manual_seed(seed)

    def matrix(*shape):
        return (torch.randn(shape, generator=g, device=device) * 0.02).to(torch.bfloat16)

    def norm(n):
        return (1 + 0.1 * torch.randn(n, generator=g, device=device)).to(torch.bfloat16)

    w = {"model.embed_tokens.weight": matrix(case["vocab"], H), "model.norm.weight": norm(H)}
    make = {"input_layernorm.weight": (H,), "post_attention_layernorm.weight": (H,), "self_attn.q_norm.weight": (HD,),
            "self_attn.k_norm.weight": (HD,), "self_attn.q_proj.weight": (QH * HD, H),
            "self_attn.k_proj.weight": (KVH * HD, H), "self_attn.v_proj.weight": (KVH * HD, H),
            "self_attn.o_proj.weight": (H, QH * HD), "mlp.gate_proj.weight": (I, H), "mlp.up_proj.weight": (I, H),
            "mlp.down_proj.weight": (H, I)}
    for i in range(case["layers"]):
        for n in LAYER_WEIGHTS:
            s = make[n]
            w["model.layers.%d.%s" % (i, n)] = norm(s[0]) if len(s) == 1 else matrix(*s)
    return w


def _ids(case, seed):
    """Per sequence: the ids of its context, then those of the call."""
    r = np.random.default_rng([seed, 7])
    return [r.integers(0, case["vocab"], p + case["t"]).astype(np.int32) for p in _positions(case)]


class State:
    """A resident model with its context prefilled, and the call's own ids. The device goes with the last reference."""

    def __init__(self, case, seed):
        H, QH, KVH, HD, I = SHAPES[case["shape"]]
        end = case["pos"] + case["t"]
        cfg = QwenConfig(case["layers"], H, QH, KVH, HD, I, case["vocab"], (end + 63) // 64 * 64, EPS)
        self.case = case
        self.backend = HipBackend(0)
        self.model = QwenModel(self.backend, cfg, mode=case["mode"], max_tokens=max(case["chunk"], case["batch"]),
                               inv_freq=_inv_freq(HD).view(np.uint32), batch=case["batch"])
        w = _weights(case, seed, "cuda")
        self.model.load_weights({k: v.view(torch.int16).cpu().numpy().view(np.uint16) for k, v in w.items()})
        ids, self.pos = _ids(case, seed), np.array(_positions(case), np.int32)
        self.ids = np.concatenate([s[p:] for s, p in zip(ids, self.pos)])
        for b, (s, p) in enumerate(zip(ids, self.pos)):  # (a context of no tokens: one, rewritten by the call)
            self.model.forward(s[: max(1, p)], 0, logits_rows=0, seq=b)
        if case["op"] == "decode":  # the step is recorded at its first run
            self.step()

    def step(self):
        m, n = self.model, self.case["batch"]
        m.decode_set(self.ids, self.pos)
        m.decode_run(1)
        return m.read_logits(n), m.decode_ids(n)

    def __del__(self):
        for o in ("model", "backend"):
            if hasattr(self, o):
                getattr(self, o).close()


def prepare(case, seed):
    return State(case, seed)


def run(state):
    """The call's logits, and the logit of the id it chose (equal for ids that tie)."""
    c = state.case
    if c["op"] == "decode":
        logits, ids = state.step()
        return {"logits": logits, "best": logits[np.arange(c["batch"]), ids]}
    logits, best = state.model.forward(state.ids, int(state.pos[0]), logits_rows=c["rows"])
    return {"logits": logits, "best": logits[-1, best]}


def work(case):
    """Every weight once (bf16; of the embedding, the head's read of it), the cached keys and values each sequence
    attends to once and the new ones written (float32 or fp16), the logits written; a multiply-add is two."""
    H, QH, KVH, HD, I = SHAPES[case["shape"]]
    L, V, T = case["layers"], case["vocab"], case["t"]
    per_layer = H * (QH + 2 * KVH) * HD + QH * HD * H + 3 * H * I
    tokens = T * case["batch"]
    rows = case["batch"] if case["op"] == "decode" else case["rows"]
    kv = 4 if case["mode"] == "fp32" else 2
    pairs = sum(T * p + T * (T + 1) // 2 for p in _positions(case))
    keys = sum(p + T for p in _positions(case))
    return {"bytes": 2 * (L * per_layer + V * H) + L * keys * 2 * KVH * HD * kv + 4 * rows * V,
            "flops": 2 * tokens * L * per_layer + L * pairs * QH * 4 * HD + 2 * rows * V * H}


def tolerance(case):
    """float32: sums in another order. fast: activations and caches rounded to fp16 (2^-11 each) at five places a
    layer, the error growing with the layers."""
    if case["mode"] == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 5e-3, "max": 5e-2}


# ---------------------------------------------------------------- the same in 64 bits

def _rms(x, w):
    return w.double() * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS))


def _forward64(case, w, ids, rows):
    """Logits [rows, vocab] of the last `rows` of `ids` (positions 0 ..), in float64."""
    H, QH, KVH, HD, I = SHAPES[case["shape"]]
    n = len(ids)
    dev = w["model.norm.weight"].device
    # the rotation's angle is the float32 product of position and frequency
    ang = (np.arange(n, dtype=np.float32)[:, None] * _inv_freq(HD)[None, :]).astype(np.float64)
    cos, sin = (torch.from_numpy(f(ang)).to(dev)[:, None, :] for f in (np.cos, np.sin))

    def rope(x):
        a, b = x[..., : HD // 2], x[..., HD // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x = w["model.embed_tokens.weight"][torch.from_numpy(ids.astype(np.int64)).to(dev)].double()
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        lin = lambda v, name: v @ w[p + name].double().t()  # noqa: E731
        h = _rms(x, w[p + "input_layernorm.weight"])
        q = rope(_rms(lin(h, "self_attn.q_proj.weight").view(n, QH, HD), w[p + "self_attn.q_norm.weight"]))
        k = rope(_rms(lin(h, "self_attn.k_proj.weight").view(n, KVH, HD), w[p + "self_attn.k_norm.weight"]))
        v = lin(h, "self_attn.v_proj.weight").view(n, KVH, HD)
        o = torch.empty_like(q)
        for hd in range(QH):
            kh, vh = (t[:, hd * KVH // QH].contiguous() for t in (k, v))
            for r0 in range(0, n, 2048):
                r1 = min(n, r0 + 2048)
                s = (q[r0:r1, hd].contiguous() @ kh[:r1].t()) * HD ** -0.5
                s.masked_fill_(torch.arange(r1, device=dev)[None, :] > torch.arange(r0, r1, device=dev)[:, None],
                               -math.inf)
                o[r0:r1, hd] = torch.softmax(s, -1) @ vh[:r1]
        x = x + lin(o.view(n, QH * HD), "self_attn.o_proj.weight")
        h = _rms(x, w[p + "post_attention_layernorm.weight"])
        a = torch.nn.functional.silu(lin(h, "mlp.gate_proj.weight")) * lin(h, "mlp.up_proj.weight")
        x = x + lin(a, "mlp.down_proj.weight")
    return _rms(x[n - rows:], w["model.norm.weight"]) @ w["model.embed_tokens.weight"].double().t()


def exact(case, seed):
    w = _weights(case, seed, "cuda")
    logits = torch.cat([_forward64(case, w, s, case["rows"]) for s in _ids(case, seed)])
    best = logits.max(-1).values
    return {"logits": logits.cpu().numpy(), "best": best.cpu().numpy() if case["op"] == "decode" else best[-1].item()}
