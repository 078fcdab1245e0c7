"""Performance cases of the token loop, through the package's public entry points.

What a user has this library do: answer requests (a new session reads a prompt in chunks,
then decodes, the logits read back after every token), decode on in a long conversation (one
token at a time over a primed session), and, below the model, the operator trait's calls on
prompt chunks and single tokens (`linear`, `attend`, `gla`). The models are the package's own
synthetic ones (`tiny`, `a86`, `g86`), in fp32 and in fp16 mode; operator sizes are those
models' or generic.

Kinds of case:
  request  session(loops), feed(n tokens), logits; then k times step + logits (a server's
           request; k = 0: reading a prompt)
  step     one step + logits of a session that has read `pos` tokens
  linear   y[m][rows] = x[m][cols] w^T
  attend   m queries at position pos over a ring of `cap` slots
  gla      m tokens of gated linear attention, the state carried on
"""

import importlib.util
import json
import math
import struct
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
FAR = 2 ** 64 - 1  # slm_attn.reach of a layer without a window


def _package():
    """The package (its folder's name is not an identifier) and its model generator."""
    if "slm_use_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "slm_use_amd", ROOT / "slm.use_amd" / "__init__.py",
            submodule_search_locations=[str(ROOT / "slm.use_amd")])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["slm_use_amd"] = mod
        spec.loader.exec_module(mod)
    import slm_use_amd
    from slm_use_amd import synth
    return slm_use_amd, synth


# What one program keeps for its lifetime: a backend per data type, and loaded models.
_BACKENDS = {}
_MODELS = {}
_SEEDS = {"tiny": 1, "a86": 2, "g86": 4}


def _backend(fp16):
    if fp16 not in _BACKENDS:
        hip = _package()[0].Hip(0)
        if fp16:
            hip.set_fp16(True)
        _BACKENDS[fp16] = hip
    return _BACKENDS[fp16]


def _folder(name):
    synth = _package()[1]
    return synth.write_model(Path(tempfile.gettempdir()) / "slm_models" / f"{name}-{_SEEDS[name]}", name,
                             _SEEDS[name])


def _model(name, fp16):
    if (name, fp16) not in _MODELS:
        # global caches grow on the device: the path a program that cares for speed asks for
        _MODELS[name, fp16] = _package()[0].Model(_backend(fp16), _folder(name), device_grow=True)
    return _MODELS[name, fp16]


def listed():
    return [
        # the smallest work there is: the fixture-sized model answers a short request; launches
        # and host work count
        dict(name="request-tiny", kind="request", model="tiny", n=12, k=4, loops=3, fp16=False),
        # the headline: one token of a long conversation, the window full
        dict(name="step-a86-r4", kind="step", model="a86", pos=4120, loops=4, fp16=False),
        # fp16 mode at the highest think level, a short conversation
        dict(name="step-a86-r16-fp16", kind="step", model="a86", pos=600, loops=16, fp16=True),
        # the model with global layers at the lowest think level, past its far distance
        dict(name="step-g86-r2", kind="step", model="g86", pos=9000, loops=2, fp16=False),
        # a 4096-token prompt in 256-token chunks
        dict(name="request-a86-4096", kind="request", model="a86", n=4096, k=0, loops=4, fp16=False),
        # a ragged long prompt of the model with global layers, the last chunks past `far`
        dict(name="request-g86-5001", kind="request", model="g86", n=5001, k=0, loops=4, fp16=False),
        # a chat turn in fp16 mode: a short ragged prompt, then a few tokens
        dict(name="request-a86-333-fp16", kind="request", model="a86", n=333, k=8, loops=8, fp16=True),
        # a chat turn of a few words, fp32, the answer's first tokens
        dict(name="request-a86-21", kind="request", model="a86", n=21, k=4, loops=4, fp16=False),
        # the up projection of a whole prompt chunk
        dict(name="linear-up-256", kind="linear", rows=6144, cols=768, m=256, fp16=False),
        # the down projection of a chunk's last few tokens
        dict(name="linear-down-5", kind="linear", rows=768, cols=3072, m=5, fp16=False),
        # a prompt chunk's queries over a full window
        dict(name="attend-window-256", kind="attend", pos=4400, m=256, reach=4096, cap=4352, heads=12,
             key_heads=12, dh=64, fp16=False),
        # a chunk of linear attention
        dict(name="gla-256", kind="gla", m=256, heads=12, dh=64, fp16=False),
    ]


def _spread(rng, lo, hi):
    """A whole number in lo..hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["request", "request", "step", "step", "linear", "attend", "gla"])
    fp16 = rng.random() < 0.35
    if kind == "request":
        model = rng.choice(["tiny", "a86", "a86", "g86"])
        loops = rng.randint(1, 6) if model == "tiny" else rng.choice([2, 3, 4, 4, 6, 8, 16])
        n = _spread(rng, 2, 600 if model == "tiny" else 16384 // loops)
        return dict(kind=kind, model=model, n=n, k=rng.randint(0, 8), loops=loops,
                    fp16=fp16 and model != "tiny")
    if kind == "step":
        return dict(kind=kind, model=rng.choice(["a86", "a86", "g86"]), pos=_spread(rng, 16, 7000),
                    loops=rng.choice([2, 3, 4, 4, 6, 8, 16]), fp16=fp16)
    if kind == "linear":
        if rng.random() < 0.5:
            rows, cols = rng.choice([(768, 768), (2304, 768), (3072, 768), (6144, 768), (768, 3072),
                                     (512, 768), (12, 768)])
        else:
            rows, cols = _spread(rng, 12, 8192), _spread(rng, 32, 4096)
            if fp16:  # fp16 mode takes multiples of 64 columns
                cols = 64 * max(1, cols // 64)
        return dict(kind=kind, rows=rows, cols=cols, m=_spread(rng, 1, 256), fp16=fp16)
    if kind == "attend":
        dh = rng.choice([64, 64, 64, 32, 128])
        heads, key_heads = rng.choice([(12, 12), (12, 4), (8, 2), (16, 16)])
        m, pos = _spread(rng, 1, 256), _spread(rng, 1, 12000)
        if key_heads == heads:
            window = rng.choice([512, 4096, 4096])
            reach, cap = window, window + 256
        else:
            reach, cap = 0, 8192 if pos + m <= 8192 else 16384
        return dict(kind=kind, pos=pos, m=m, reach=reach, cap=cap, heads=heads, key_heads=key_heads, dh=dh,
                    fp16=fp16)
    return dict(kind="gla", m=_spread(rng, 1, 256), heads=rng.choice([4, 8, 12, 12, 16]),
                dh=rng.choice([64, 64, 32, 128]), fp16=fp16)


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------

def _normal(rng, *shape, scale=1.0):
    return rng.standard_normal(shape, dtype=np.float32) * np.float32(scale)


def _inputs(case, seed):
    """The host arrays of an operator case, by name."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "linear":
        return dict(w=_normal(rng, case["rows"], case["cols"], scale=0.02),
                    x=_normal(rng, case["m"], case["cols"]))
    if case["kind"] == "attend":
        q = _normal(rng, case["m"], case["heads"], case["dh"], scale=0.55)
        k, v = (_normal(rng, case["key_heads"], case["cap"], case["dh"], scale=0.55) for _ in range(2))
        return dict(q=q, k=k, v=v)
    m, H, dh = case["m"], case["heads"], case["dh"]
    q, k = (_normal(rng, m, H, dh) for _ in range(2))
    q /= np.linalg.norm(q, axis=-1, keepdims=True)
    k /= np.linalg.norm(k, axis=-1, keepdims=True)
    u = 0.1 * 0.01 ** (np.arange(H) / max(H - 1, 1))
    return dict(q=q, k=k, v=_normal(rng, m, H, dh, scale=0.55), decay=_normal(rng, m, H, scale=0.55),
                bias=np.log(u / (1 - u)).astype(np.float32), s=_normal(rng, H, dh, dh, scale=0.1))


def _tokens(case, seed):
    """The prompt and the tokens of the steps after it."""
    vocab = 97 if case["model"] == "tiny" else 32000
    rng = np.random.default_rng(seed)
    n = case["n"] if case["kind"] == "request" else case["pos"]
    return (rng.integers(0, vocab, n).astype(np.uint32), rng.integers(0, vocab, 64).astype(np.uint32))


class _Buffers:
    """Device buffers that go back to the backend with the last view of them."""

    def __init__(self, hip):
        self.hip, self.held = hip, []

    def upload(self, a):
        self.held.append(self.hip.upload(a))
        return self.held[-1]

    def alloc(self, n):
        self.held.append(self.hip.alloc(n))
        return self.held[-1]

    def cache(self, a):
        heads, cap, dh = a.shape
        self.held.append(self.hip.alloc_cache(heads, cap, dh))
        self.hip.upload_into(self.held[-1], a)
        return self.held[-1]

    def __del__(self):
        if self.hip.ctx:
            for b in self.held:
                b.free()


class _View:
    """A device buffer as torch takes it, holding its owner."""

    def __init__(self, owner, buf, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(buf.ptr, False), version=2)


def _view(owner, buf, *shape):
    return torch.as_tensor(_View(owner, buf, shape), device="cuda")


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, s.kind = case, case["kind"]
    if s.kind in ("request", "step"):
        s.model = _model(case["model"], case["fp16"])
        s.prompt, s.next = _tokens(case, seed)
        if s.kind == "step":
            s.session, s.i = s.model.session(case["loops"]), 0
            s.session.feed(s.prompt)
            s.session.logits()
        return s
    hip = s.hip = _backend(case["fp16"])
    mem = s.mem = _Buffers(hip)
    a = _inputs(case, seed)
    if s.kind == "linear":
        s.w, s.x = mem.upload(a["w"]), mem.upload(a["x"])
        s.y = mem.alloc(case["m"] * case["rows"])
        s.out = _view(mem, s.y, case["m"], case["rows"])
    elif s.kind == "attend":
        s.q, s.k, s.v = mem.upload(a["q"]), mem.cache(a["k"]), mem.cache(a["v"])
        s.y = mem.alloc(a["q"].size)
        s.args = {n: case[n] for n in ("pos", "m", "cap", "heads", "key_heads", "dh")}
        s.args.update(reach=case["reach"] or FAR, gap=0, scale=1.0 / math.sqrt(case["dh"]))
        s.out = _view(mem, s.y, *a["q"].shape)
    else:
        s.q, s.k, s.v, s.decay, s.bias, s.s = (mem.upload(a[n]) for n in ("q", "k", "v", "decay", "bias", "s"))
        s.y = mem.alloc(a["q"].size)
        s.out = dict(y=_view(mem, s.y, *a["q"].shape), s=_view(mem, s.s, *a["s"].shape))
    return s


def run(s):
    c = s.case
    if s.kind == "request":
        se = s.model.session(c["loops"])
        se.feed(s.prompt)
        out = [se.logits()]
        for t in s.next[:c["k"]]:
            se.step(t)
            out.append(se.logits())
        return out
    if s.kind == "step":
        s.session.step(s.next[s.i % len(s.next)])
        s.i += 1
        return s.session.logits()
    if s.kind == "linear":
        s.hip.linear(s.y.ptr, s.w.ptr, c["rows"], c["cols"], s.x.ptr, c["m"])
    elif s.kind == "attend":
        s.hip.attend(s.y.ptr, s.q.ptr, s.k.ptr, s.v.ptr, **s.args)
    else:
        s.hip.gla(s.y.ptr, s.s.ptr, s.q.ptr, s.k.ptr, s.v.ptr, s.decay.ptr, s.bias.ptr, c["m"], c["heads"],
                  c["dh"])
    return s.out


# ---------------------------------------------------------------------------------------
# compulsory work
# ---------------------------------------------------------------------------------------

def _matrices(cfg, kind):
    """(rows, cols, products a token) of a block's matrices."""
    d, H = cfg["d_model"], cfg["n_heads"]
    hid, kd = int(round(cfg["mlp_mult"] * d)), cfg["global_kv_heads"] * (d // H)
    mix = {"S": [(3 * d, d, 1), (d, d, 1)], "L": [(4 * d, d, 1), (H, d, 1), (d, d, 1)],
           "G": [(d, d, 1), (2 * kd, d, 2 if cfg["global_kshift"] else 1), (d, d, 1)]}[kind]
    return mix + [(2 * hid, d, 1), (d, hid, 1)]


def _call_work(cfg, loops, start, count, heads_read, half, fresh):
    """Bytes and flops of reading `count` tokens from position `start`, the logits formed
    `heads_read` times. Every weight is read once (the tied embedding whole: the logits read
    it); each layer's keys, values and state once, what the call itself made not at all."""
    d, H, W, V = cfg["d_model"], cfg["n_heads"], cfg["window"], cfg["vocab_size"]
    dh, unit = d // H, 2 if half else 4
    kd = cfg["global_kv_heads"] * dh
    far = W if cfg["global_far"] else 0
    nbytes, flops = unit * V * d, 2 * V * d * heads_read
    if cfg["core"]:
        nbytes += unit * d * d
        flops += 2 * d * d * count
    pos = np.arange(start, start + count)
    for part, times in (("prelude", 1), ("core", loops), ("coda", 1)):
        for kind in cfg[part]:
            for r, c, products in _matrices(cfg, kind):
                nbytes += unit * r * c
                flops += 2 * r * c * products * count * times
            if kind == "S":
                old = 0 if fresh else min(start, W - 1)
                nbytes += times * unit * 2 * d * (old + count)
                flops += times * 4 * d * int(np.minimum(pos + 1, W).sum())
            elif kind == "G":
                old = 0 if fresh else max(start - far, 0)
                nbytes += times * unit * 2 * kd * (old + count)
                flops += times * 4 * d * int(np.maximum(pos + 1 - far, 0).sum())
            else:
                nbytes += times * 4 * H * dh * dh * (1 if fresh else 2)
                flops += times * 5 * H * dh * dh * count
    return dict(bytes=nbytes + 4 * V * heads_read, flops=flops)


def work(case):
    c = case
    if c["kind"] == "request":
        cfg = _package()[1].CONFIGS[c["model"]]
        return _call_work(cfg, c["loops"], 0, c["n"] + c["k"], 1 + c["k"], c["fp16"], True)
    if c["kind"] == "step":
        cfg = _package()[1].CONFIGS[c["model"]]
        return _call_work(cfg, c["loops"], c["pos"], 1, 1, c["fp16"], False)
    if c["kind"] == "linear":
        r, k, m = c["rows"], c["cols"], c["m"]
        return dict(bytes=(2 if c["fp16"] else 4) * r * k + 4 * m * (k + r), flops=2 * r * k * m)
    if c["kind"] == "attend":
        reach = c["reach"] or FAR
        p = c["pos"] + np.arange(c["m"])
        seen = np.array([min(int(i) + 1, reach) for i in p])
        span = int(p[-1]) + 1 - max(0, c["pos"] + 1 - reach)
        return dict(bytes=(2 if c["fp16"] else 4) * 2 * c["key_heads"] * c["dh"] * span
                    + 8 * c["m"] * c["heads"] * c["dh"],
                    flops=4 * c["heads"] * c["dh"] * int(seen.sum()))
    m, H, dh = c["m"], c["heads"], c["dh"]
    return dict(bytes=4 * (4 * m * H * dh + m * H + 2 * H * dh * dh), flops=5 * m * H * dh * dh)


def tolerance(case):
    """About four times the distance from the 64-bit results: whole fp32 models are 1e-6 to 6e-6
    off, single fp32 operators 1.6e-7 to 4.4e-7, fp16 operators 3.1e-4 to 3.6e-4 (half a step of
    the last rounding); a whole fp16 model is 3e-3 to 1.1e-2 off, and 2e-2 is that mode's bar."""
    if case["kind"] in ("request", "step"):
        return {"rel": 2e-2} if case["fp16"] else {"rel": 3e-5}
    return {"rel": 1.5e-3} if case["fp16"] else {"rel": 2e-6}


# ---------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------

_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_DEV).double()


def _weights64(name):
    """The model's weights (f32 safetensors: a JSON header, then the data)."""
    with open(_folder(name) / "model.safetensors", "rb") as f:
        n = struct.unpack("<Q", f.read(8))[0]
        head = json.loads(f.read(n))
        data = f.read()
    out = {}
    for k, v in head.items():
        if k != "__metadata__":
            a, b = v["data_offsets"]
            out[k] = _f64(np.frombuffer(data, np.float32, (b - a) // 4, a).reshape(v["shape"]).copy())
    return out


def _rms64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope64(x, base):
    """x [n, heads, dh] at positions 0..n-1; the angle is a 32-bit product, as the library
    defines it."""
    n, _, dh = x.shape
    inv = (1.0 / (np.float32(base) ** (np.arange(0, dh, 2, dtype=np.float32) / np.float32(dh)))).astype(np.float32)
    ang = _f64(np.arange(n, dtype=np.float32)[:, None] * inv[None])[:, None]
    lo, hi = x[..., :dh // 2], x[..., dh // 2:]
    return torch.cat([lo * ang.cos() - hi * ang.sin(), lo * ang.sin() + hi * ang.cos()], -1)


def _attend64(q, k, v, lo, hi):
    """q [m, H, dh] over k, v [n, KH, dh]; query i sees keys lo[i] <= j < hi[i] (none: zeros)."""
    m, H, dh = q.shape
    out = torch.zeros_like(q)
    j = torch.arange(k.shape[0], device=q.device)
    hid = (j[None] < lo[:, None]) | (j[None] >= hi[:, None])
    some = (hi > lo)[:, None]
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h] @ k[:, g].T.contiguous() / math.sqrt(dh)).masked_fill_(hid, -math.inf)
        s = torch.where(some, s, torch.zeros_like(s)).softmax(-1)
        out[:, h] = torch.where(some, s @ v[:, g], torch.zeros_like(out[:, h]))
    return out


def _gla64(q, k, v, decay, s):
    """Tokens in order over s [H, dh, dh]; decay [m, H] is the state's factor."""
    y = torch.empty_like(q)
    for t in range(q.shape[0]):
        s = s * decay[t, :, None, None] + k[t, :, :, None] * v[t, :, None, :]
        y[t] = (q[t, :, :, None] * s).sum(1)
    return y, s


def _block64(cfg, w, p, kind, x, e0):
    d, H = cfg["d_model"], cfg["n_heads"]
    dh, n, eps, W = d // H, x.shape[0], cfg["norm_eps"], cfg["window"]
    at = torch.arange(n, device=x.device)
    a = _rms64(x, w[p + ".norm1.weight"], eps)
    if kind == "S":
        q, k, v = ((a @ w[p + ".mixer.qkv.weight"].T).view(n, 3, H, dh)[:, i] for i in range(3))
        q, k = _rope64(q, cfg["rope_base"]), _rope64(k, cfg["rope_base"])
        y = _attend64(q, k, v, (at + 1 - W).clamp(min=0), at + 1).reshape(n, d)
    elif kind == "L":
        mix = (a @ w[p + ".mixer.qkvg.weight"].T).view(n, 4, H, dh)
        dec = torch.sigmoid(-(a @ w[p + ".mixer.decay.weight"].T + w[p + ".mixer.decay.bias"]))
        q, k = (mix[:, i] / mix[:, i].norm(dim=-1, keepdim=True).clamp(min=1e-12) for i in range(2))
        y, _ = _gla64(q, k, mix[:, 2], dec, torch.zeros(H, dh, dh, dtype=x.dtype, device=x.device))
        y = (torch.nn.functional.silu(mix[:, 3]) * _rms64(y, w[p + ".mixer.head_norm.weight"], eps)).reshape(n, d)
    else:
        KH = cfg["global_kv_heads"]
        if cfg["global_emb"]:
            a = a + _rms64(e0, w[p + ".mixer.norm_e.weight"], eps)
        q = a @ w[p + ".mixer.q.weight"].T
        if cfg["global_logn"]:
            q = q * (torch.log1p(at.double()) / math.log(cfg["global_logn"]))[:, None]
        kv = a @ w[p + ".mixer.kv.weight"].T
        k = kv[:, :KH * dh]
        if cfg["global_kshift"]:
            k = torch.cat([torch.zeros_like(k[:1]), k[:-1]])
        far = W if cfg["global_far"] else 0
        y = _attend64(q.view(n, H, dh), k.view(n, KH, dh), kv[:, KH * dh:].view(n, KH, dh),
                      torch.zeros_like(at), (at + 1 - far).clamp(min=0)).reshape(n, d)
    x = x + y @ w[p + ".mixer.o.weight"].T
    up = _rms64(x, w[p + ".norm2.weight"], eps) @ w[p + ".mlp.up.weight"].T
    g, u = up.chunk(2, -1)
    return x + (torch.nn.functional.silu(g) * u) @ w[p + ".mlp.down.weight"].T


def _logits64(name, loops, tokens, want):
    """The logits at the last `want` of the tokens' positions, read from the start."""
    cfg, w = _package()[1].CONFIGS[name], _weights64(name)
    e0 = w["embed.weight"][torch.from_numpy(tokens.astype(np.int64)).to(_DEV)]
    x = e0
    for i, kind in enumerate(cfg["prelude"]):
        x = _block64(cfg, w, f"prelude.{i}", kind, x, e0)
    if cfg["core"]:
        e, s = x @ w["inject_e.weight"].T, x
        for r in range(loops):
            x = s + e + w["loop_embed.weight"][r]
            for i, kind in enumerate(cfg["core"]):
                x = _block64(cfg, w, f"core.{i}", kind, x, e0)
            s = s + cfg["damp"] * (x - s)
        x = s
    for i, kind in enumerate(cfg["coda"]):
        x = _block64(cfg, w, f"coda.{i}", kind, x, e0)
    return _rms64(x[-want:], w["norm_f.weight"], cfg["norm_eps"]) @ w["embed.weight"].T


def exact(case, seed):
    c = case
    if c["kind"] in ("request", "step"):
        prompt, nxt = _tokens(c, seed)
        k = c["k"] if c["kind"] == "request" else 1
        out = _logits64(c["model"], c["loops"], np.concatenate([prompt, nxt[:k]]), k + 1).cpu().numpy()
        return out[-1] if c["kind"] == "step" else list(out)
    a = {n: _f64(v) for n, v in _inputs(c, seed).items()}
    if c["kind"] == "linear":
        return a["x"] @ a["w"].T
    if c["kind"] == "attend":
        reach, cap = c["reach"] or FAR, c["cap"]
        p = np.arange(c["pos"], c["pos"] + c["m"])
        first = max(0, c["pos"] + 1 - reach)
        slots = torch.arange(first, int(p[-1]) + 1, device=_DEV) % cap
        lo = torch.tensor([max(0, int(i) + 1 - reach) - first for i in p], device=_DEV)
        hi = torch.tensor([int(i) + 1 - first for i in p], device=_DEV)
        k, v = (a[n][:, slots].transpose(0, 1).contiguous() for n in "kv")
        return _attend64(a["q"], k, v, lo, hi)
    y, s = _gla64(a["q"], a["k"], a["v"], torch.sigmoid(-(a["decay"] + a["bias"])), a["s"])
    return dict(y=y, s=s)
