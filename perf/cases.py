"""The work that users of quicknn_amd have it do, as cases that can be timed and compared.

Every case is one pass through the public entry points of ``quicknn_amd.hip`` (the resident context of
``include/qnn_hip.h``), as the LLM engine calls them: weights resident, activations in context tensors, the
outputs left in context tensors.  Seven families, named by what the engine has in that place:

* ``mlp``        the gated MLP of a decoder in native INT4 (norm, gate/up, SwiGLU, down, residual)
* ``gguf``       the projections of a decoder layer in mixed GGUF encodings (q, k, v, o, gate/up, GEGLU, down)
* ``q8``         one Q8_0 projection of an image or text encoder's MLP over many rows
* ``head``       the output head over the vocabulary and the sampling of the next token
* ``moe``        a routed-expert layer: router, route, experts
* ``attention``  rotary embedding, KV-cache append and cached attention
* ``decoder``    whole decoder layers: everything of ``attention`` and ``mlp`` with the INT4 projections between

A case's numbers are plain sizes; ``prepare`` makes weights and activations from the seed on the GPU and hands
the packed weight bytes to the context as the engine hands it a checkpoint's.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from quicknn_amd import hip

DEV = "cuda"
EPS = 1e-6
THETA = 1000000.0

# Projections of a Gemma-2-9B-shaped layer: the mix of encodings of the repository's GGUF benchmark.
MIX = {"q": "Q4_K", "k": "Q3_K", "v": "Q3_K", "o": "Q4_K", "gate": "Q2_K", "up": "Q2_K", "down": "Q6_K"}


def listed():
    return [
        # One decoded token through the MLPs of a 4B model (the headline benchmark), four layers so that the
        # weights come from HBM as they do in a whole model.
        dict(name="int4_mlp_token", family="mlp", rows=1, hidden=2560, inter=9728, layers=4),
        # A batch of eight sequences, one token each.
        dict(name="int4_mlp_batch8", family="mlp", rows=8, hidden=2560, inter=9728, layers=4),
        # A prompt chunk: the most rows that the INT4 projection takes.
        dict(name="int4_mlp_prompt", family="mlp", rows=128, hidden=2560, inter=9728, layers=4),
        # One decoded token through the projections of a 9B GGUF checkpoint.
        dict(name="gguf_token", family="gguf", rows=1, hidden=3584, inter=14336, qdim=4096, kvdim=2048, layers=2,
             mix="gemma"),
        # A prompt of 200 tokens through one such layer.
        dict(name="gguf_prompt", family="gguf", rows=200, hidden=3584, inter=14336, qdim=4096, kvdim=2048, layers=1,
             mix="gemma"),
        # The MLP projection of an image model over 512 latent tokens.
        dict(name="q8_rows512", family="q8", rows=512, k=3072, n=12288, int8=False),
        # The next token of a 152k-token vocabulary: Q6_K head, then top-k sampling.
        dict(name="head_sample", family="head", vocab=151936, hidden=2560, top_k=40),
        # One decoded token through a 30B-A3B routed-expert layer.
        dict(name="moe_token", family="moe", rows=1, hidden=2048, inter=768, experts=128, topk=8),
        # A prompt chunk through the same layer.
        dict(name="moe_prompt", family="moe", rows=128, hidden=2048, inter=768, experts=128, topk=8),
        # One decoded token over a long context.
        dict(name="attention_token_32k", family="attention", rows=1, heads=32, kv=8, dim=128, capacity=32768,
             position=32767, window=0, softcap=0.0),
        # A prompt chunk over a 4k context.
        dict(name="attention_prompt", family="attention", rows=128, heads=32, kv=8, dim=128, capacity=4096,
             position=3968, window=0, softcap=0.0),
        # One decoded token through two whole decoder layers at a 4k context.
        dict(name="decoder_token", family="decoder", rows=1, hidden=2560, inter=9728, heads=32, kv=8, dim=128,
             capacity=4096, position=4000, layers=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most / 2:
            return c


def _draw(rng):
    family = rng.choice(["mlp", "mlp", "gguf", "q8", "head", "moe", "attention", "attention", "decoder"])
    if family == "mlp":
        # Widths of any size, most of them multiples of the quantisation group as checkpoints have them.
        unit = rng.choice([32, 32, 64, 4, 1])
        hidden, inter = (max(unit, _log(rng, 500, hi) // unit * unit) for hi in (4096, 12288))
        return dict(family="mlp", rows=_log(rng, 1, 128), hidden=hidden, inter=inter, layers=rng.randint(1, 3))
    if family == "gguf":
        hidden, inter, qdim, kvdim = (256 * max(1, _log(rng, 512, hi) // 256) for hi in (4096, 14336, 4096, 2048))
        return dict(family="gguf", rows=_log(rng, 1, 256), hidden=hidden, inter=inter, qdim=qdim, kvdim=kvdim, layers=1,
                    mix=rng.choice(["gemma", "Q4_K", "Q8_0", "Q6_K"]))
    if family == "q8":
        return dict(family="q8", rows=_log(rng, 2, 512), k=32 * _log(rng, 16, 128), n=_log(rng, 500, 12288),
                    int8=rng.random() < 0.3)
    if family == "head":
        return dict(family="head", vocab=_log(rng, 8000, 152000), hidden=256 * rng.randint(4, 14),
                    top_k=rng.randint(1, 64))
    if family == "moe":
        experts = rng.choice([8, 32, 60, 64, 128])
        return dict(family="moe", rows=_log(rng, 1, 128), hidden=4 * _log(rng, 128, 512), inter=4 * _log(rng, 64, 384),
                    experts=experts, topk=rng.randint(2, 8))
    if family == "attention":
        kv = rng.choice([1, 2, 4, 8])
        rows = _log(rng, 1, 128) if rng.random() < 0.6 else 1
        capacity = _log(rng, 256, 16384 if rows == 1 else 4096)
        rows = min(rows, capacity // 2)
        return dict(family="attention", rows=rows, heads=kv * rng.choice([1, 2, 4, 7]), kv=kv,
                    dim=rng.choice([64, 80, 128, 128, 256]), capacity=capacity,
                    position=rng.randint(0, capacity - rows), window=rng.choice([0, 0, capacity // 3]),
                    softcap=rng.choice([0.0, 0.0, 50.0]))
    rows = rng.choice([1, 1, 1, _log(rng, 2, 128)])
    capacity = _log(rng, 256, 4096)
    kv = rng.choice([2, 4, 8])
    return dict(family="decoder", rows=rows, hidden=32 * _log(rng, 24, 96), inter=32 * _log(rng, 64, 300),
                heads=kv * rng.choice([2, 4]), kv=kv, dim=rng.choice([64, 128]), capacity=capacity,
                position=rng.randint(0, capacity - rows), layers=1)


# ---------------------------------------------------------------------------------------------------------------
# Weights: packed bytes made on the GPU, and their values in 64 bits
# ---------------------------------------------------------------------------------------------------------------
class Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV, dtype=torch.float32) * std

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV, dtype=torch.int32)


def int4_pack(w):
    """fp32 [n, k] -> packed rows [n, ceil(k / 32) * 20]: per 32 weights an fp32 scale, then 16 bytes of nibbles."""
    n, k = w.shape
    groups = (k + 31) // 32
    w = torch.nn.functional.pad(w, (0, groups * 32 - k)).view(n, groups, 32)
    s = w.abs().amax(2) / 7
    q = (torch.round(w / s.clamp_min(1e-30)[..., None]).clamp(-8, 7) + 8).to(torch.uint8)
    out = torch.empty(n, groups, 20, dtype=torch.uint8, device=DEV)
    out[..., :4] = s.contiguous().view(torch.uint8).view(n, groups, 4)
    out[..., 4:] = q[..., 0::2] | (q[..., 1::2] << 4)
    return out.view(n, groups * 20)


def int4_values(p, k):
    n = p.shape[0]
    p = p.view(n, -1, 20)
    s = p[..., :4].contiguous().view(torch.float32)
    q = torch.stack([p[..., 4:] & 15, p[..., 4:] >> 4], -1).view(n, -1, 32)
    return ((q.float() - 8) * s).view(n, -1)[:, :k].double()


def _halfs(x):
    return x.to(torch.float16).contiguous().view(torch.uint8).view(*x.shape, 2)


def _unhalf(b):
    return b.contiguous().view(torch.float16)[..., 0].float()


def _codes(g, n, blocks, mid, spread, top):
    """256 codes per block around the middle of their range, as the weights of a trained layer fall."""
    return torch.round(g.normal(n, blocks, 256, std=spread) + mid).clamp(0, top).to(torch.uint8)


def gguf_pack(g, enc, n, k):
    """Blocks of [n, k] weights of standard deviation about 0.02 -> uint8 [n, bytes per row]."""
    if enc == "Q8_0":
        w = g.normal(n, k // 32, 32, std=0.02)
        d = (w.abs().amax(2) / 127).to(torch.float16)
        q = torch.round(w / d.float().clamp_min(1e-8)[..., None]).clamp(-127, 127).to(torch.int8)
        return torch.cat([_halfs(d), q.view(torch.uint8)], 2).view(n, -1)
    b = k // 256
    jitter = 1 + 0.2 * torch.rand(n, b, generator=g.g, device=DEV)
    if enc == "Q4_K":  # d, dmin, eight 6-bit scales and mins, 256 4-bit codes
        q = _codes(g, n, b, 7.5, 2.6, 15)
        sc = g.ints(32, 64, n, b, 8).to(torch.uint8)
        d = 0.02 / 2.6 / 48 * jitter
        s = torch.empty(n, b, 12, dtype=torch.uint8, device=DEV)
        s[..., :4] = (sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6)
        s[..., 4:8] = s[..., :4]  # the mins equal the scales, with dmin = 7.5 d
        s[..., 8:] = (sc[..., 4:] & 15) | ((sc[..., 4:] & 15) << 4)
        q = q.view(n, b, 4, 2, 32)
        return torch.cat([_halfs(d), _halfs(7.5 * d), s, (q[..., 0, :] | (q[..., 1, :] << 4)).reshape(n, b, 128)],
                         2).view(n, -1)
    if enc == "Q6_K":  # low nibbles, high bit pairs, sixteen int8 scales, d
        q = _codes(g, n, b, 32, 10, 63).view(n, b, 2, 4, 32)
        low = torch.cat([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)],
                        -1).reshape(n, b, 128)
        high = ((q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) |
                ((q[..., 3, :] >> 4) << 6)).reshape(n, b, 64)
        sc = g.ints(64, 128, n, b, 16).to(torch.uint8)
        return torch.cat([low, high, sc, _halfs(0.02 / 10 / 96 * jitter)], 2).view(n, -1)
    if enc == "Q3_K":  # high bits, low bit pairs, sixteen 6-bit scales, d
        q = _codes(g, n, b, 4, 1.5, 7).view(n, b, 2, 4, 32)
        bits = (q >> 2).reshape(n, b, 8, 32)
        hm = sum(bits[..., j, :] << j for j in range(8))
        qs = sum((q[..., j, :] & 3) << (2 * j) for j in range(4)).reshape(n, b, 64)
        sc = g.ints(48, 64, n, b, 16).to(torch.uint8)
        s = torch.empty(n, b, 12, dtype=torch.uint8, device=DEV)
        s[..., :8] = (sc[..., :8] & 15) | ((sc[..., 8:] & 15) << 4)
        s[..., 8:] = sum((sc[..., 4 * j:4 * j + 4] >> 4) << (2 * j) for j in range(4))
        return torch.cat([hm, qs, s, _halfs(0.02 / 1.5 / 24 * jitter)], 2).view(n, -1)
    if enc == "Q2_K":  # sixteen 4-bit scales and mins, low bit pairs, d, dmin
        q = _codes(g, n, b, 1.5, 0.9, 3).view(n, b, 2, 4, 32)
        qs = sum(q[..., j, :] << (2 * j) for j in range(4)).reshape(n, b, 64)
        sc = g.ints(8, 16, n, b, 16).to(torch.uint8)
        d = 0.02 / 0.9 / 12 * jitter
        return torch.cat([sc | (sc << 4), qs, _halfs(d), _halfs(1.5 * d)], 2).view(n, -1)
    raise ValueError(enc)


def gguf_values(enc, p, k):
    n = p.shape[0]
    if enc == "Q8_0":
        p = p.view(n, -1, 34)
        return (p[..., 2:].contiguous().view(torch.int8).float() * _unhalf(p[..., :2])[..., None]).view(n, k).double()
    b = k // 256
    p = p.view(n, b, -1)
    if enc == "Q4_K":
        s, q = p[..., 4:16], p[..., 16:].view(n, b, 4, 1, 32)
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], 2).float()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], 2).float()
        v = torch.cat([q & 15, q >> 4], 3).view(n, b, 8, 32).float()
        d, m = _unhalf(p[..., :2])[..., None] * sc, _unhalf(p[..., 2:4])[..., None] * mn
        return (v.double() * d.double()[..., None] - m.double()[..., None]).view(n, k)
    if enc == "Q6_K":
        low, high = p[..., :128].reshape(n, b, 2, 2, 32), p[..., 128:192].reshape(n, b, 2, 32)
        v = torch.stack([(low[..., j & 1, :] >> (4 * (j >> 1)) & 15) | ((high >> (2 * j) & 3) << 4) for j in range(4)], 3)
        sc = p[..., 192:208].contiguous().view(torch.int8).float() * _unhalf(p[..., 208:210])[..., None]
        return ((v.float() - 32).view(n, b, 16, 16).double() * sc.double()[..., None]).view(n, k)
    if enc == "Q3_K":
        hm, qs, s = p[..., :32], p[..., 32:96].reshape(n, b, 2, 32), p[..., 96:108]
        v = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], 3).view(n, b, 8, 32).float()
        v -= 4 * torch.stack([1 - ((hm >> j) & 1) for j in range(8)], 2).float()
        sc = torch.cat([s[..., :8] & 15, s[..., :8] >> 4], 2) | (torch.cat([(s[..., 8:] >> (2 * j)) & 3 for j in range(4)],
                                                                          2) << 4)
        d = (sc.float() - 32) * _unhalf(p[..., 108:110])[..., None]
        return (v.view(n, b, 16, 16).double() * d.double()[..., None]).view(n, k)
    if enc == "Q2_K":
        s, qs = p[..., :16], p[..., 16:80].reshape(n, b, 2, 32)
        v = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], 3).view(n, b, 16, 16).double()
        d, m = _unhalf(p[..., 80:82])[..., None] * (s & 15).float(), _unhalf(p[..., 82:84])[..., None] * (s >> 4).float()
        return (v * d.double()[..., None] - m.double()[..., None]).view(n, k)
    raise ValueError(enc)


ENCODING = {"Q8_0": hip.WE_Q8_0, "Q4_K": hip.WE_Q4_K, "Q6_K": hip.WE_Q6_K, "Q3_K": hip.WE_Q3_K, "Q2_K": hip.WE_Q2_K}


def gguf_bytes(enc, n, k):
    elements, size = hip.GGUF_BLOCK[ENCODING[enc]]
    return n * (k // elements) * size


def int4_bytes(n, k):
    return n * ((k + 31) // 32) * 20


# ---------------------------------------------------------------------------------------------------------------
# The context and what a state holds in it
# ---------------------------------------------------------------------------------------------------------------
_ctx = None


def context():
    """One context per process, as the engine has one."""
    global _ctx
    if _ctx is None:
        _ctx = hip.GPUContext(0)
    return _ctx


class View:
    """Device memory of a context tensor, for torch."""

    def __init__(self, tensor):
        self.__cuda_array_interface__ = dict(shape=(tensor.count,), typestr="<f4", data=(tensor.device_ptr, False),
                                             version=2)


def view(tensor, *shape):
    return torch.as_tensor(View(tensor), device=DEV).view(*shape)


class State:
    def __init__(self, case):
        self.case, self.ctx, self.tensors, self.weights, self.sets = case, context(), [], [], []

    def new(self, count):
        t = self.ctx.NewTensor(int(count))
        self.tensors.append(t)
        return t

    def put(self, values):
        t = self.new(values.numel())
        view(t, -1).copy_(values.reshape(-1))
        return t

    def int4(self, packed):
        return self.keep(hip.MemoryBlock.int4(packed.cpu().numpy()))

    def gguf(self, enc, packed, n, k):
        return self.keep(hip.MemoryBlock.gguf(packed.cpu().numpy(), n, k, ENCODING[enc]))

    def vector(self, values):
        return self.keep(hip.MemoryBlock.vector(values.cpu().numpy()))

    def bf16(self, bits):
        return self.keep(hip.MemoryBlock.matrix(bits.cpu().numpy().view(np.uint16)))

    def keep(self, block):
        self.weights.append(block)
        return block

    def ready(self):
        """Weights resident, everything that was queued done."""
        if self.weights:
            self.ctx.PreloadWeights(self.weights)
        torch.cuda.synchronize()
        self.ctx.Flush()
        return self

    def __del__(self):
        try:
            torch.cuda.synchronize()
            for s in self.sets:
                self.ctx.DestroyExpertSet(s)
            for t in self.tensors:
                self.ctx.Recycle(t)
        except Exception:  # the context has gone first
            pass


def norm_args(rows, dim):
    return [rows, dim, 0, 0, 0, 0, 0, hip.float_bits(EPS)]


ONE = hip.float_bits(1.0)


def norm_exact(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def silu(x):
    return x * torch.sigmoid(x)


def gelu(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


# ---- the INT4 MLP -------------------------------------------------------------------------------------------
def mlp_inputs(c, g):
    layers = [dict(gamma=1 + g.normal(c["hidden"], std=0.1),
                   gate=int4_pack(g.normal(c["inter"], c["hidden"], std=0.02)),
                   up=int4_pack(g.normal(c["inter"], c["hidden"], std=0.02)),
                   down=int4_pack(g.normal(c["hidden"], c["inter"], std=0.02))) for _ in range(c["layers"])]
    return g.normal(c["rows"], c["hidden"]), layers


def mlp_blocks(s, layer):
    return dict(gamma=s.vector(layer["gamma"]), **{n: s.int4(layer[n]) for n in ("gate", "up", "down")})


def mlp_tensors(s, c):
    n, i = c["rows"] * c["hidden"], c["rows"] * c["inter"]
    s.xn, s.h, s.g, s.u = s.new(n), s.new(i), s.new(i), s.new(i)


def mlp_run(s, c, w, dst, src):
    """dst = src + down(silu(gate(norm(src))) * up(norm(src))), as the engine records it."""
    ctx, rows, hidden, inter = s.ctx, c["rows"], c["hidden"], c["inter"]
    ctx.KernelWeights(hip.GO_NORM, rows * hidden, s.xn, src, w["gamma"], None, norm_args(rows, hidden))
    if rows == 1:
        ctx.TrySwiGLUVector(s.h, s.xn, w["gate"], w["up"], hidden, inter)
    else:
        ctx.Int4Linear(s.g, s.xn, w["gate"], rows, hidden, inter)
        ctx.Int4Linear(s.u, s.xn, w["up"], rows, hidden, inter)
        ctx.Kernel(hip.GO_SWIGLU, rows * inter, s.h, s.g, s.u, None, [inter, 0])
    ctx.Int4Linear(dst, s.h, w["down"], rows, inter, hidden)
    ctx.Kernel(hip.GO_ADD, rows * hidden, dst, src, None, None, [hidden, hidden, ONE, 0, 0])


def mlp_exact(x, layer, hidden, inter):
    xn = norm_exact(x, layer["gamma"])
    h = silu(xn @ int4_values(layer["gate"], hidden).T) * (xn @ int4_values(layer["up"], hidden).T)
    return x + h @ int4_values(layer["down"], inter).T


# ---- attention ----------------------------------------------------------------------------------------------
def attention_inputs(c, g):
    kv, dim, cap, rows = c["kv"], c["dim"], c["capacity"], c["rows"]
    return dict(q=g.normal(rows, c["heads"], dim), k=g.normal(rows, kv, dim), v=g.normal(rows, kv, dim),
                cache=g.normal(2 * kv * dim * cap))


def rope_exact(x, position):
    rows, _, dim = x.shape
    j = torch.arange(dim // 2, device=DEV, dtype=torch.float64)
    a = (position + torch.arange(rows, device=DEV, dtype=torch.float64))[:, None] * THETA ** (-2 * j / dim)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    x0, x1 = x[..., :dim // 2].double(), x[..., dim // 2:].double()
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)


def attention_exact(c, q, k, v, cache):
    """q, k, v before the rotation, in 64 bits -> (output, cache)."""
    kv, dim, cap, rows, at = c["kv"], c["dim"], c["capacity"], c["rows"], c["position"]
    cache = cache.double().clone()
    kt, vs = cache[:kv * dim * cap].view(kv, dim, cap), cache[kv * dim * cap:].view(kv, cap, dim)
    kt[:, :, at:at + rows] = rope_exact(k, at).permute(1, 2, 0)
    vs[:, at:at + rows] = v.double().permute(1, 0, 2)
    q = rope_exact(q, at)
    group, out = c["heads"] // kv, torch.empty_like(q)
    key = torch.arange(cap, device=DEV)[None]
    last = at + torch.arange(rows, device=DEV)[:, None]
    hidden = key > last
    if c.get("window"):
        hidden = hidden | (key <= last - c["window"])
    for h in range(c["heads"]):
        sc = q[:, h] @ kt[h // group] / math.sqrt(dim)
        if c.get("softcap"):
            sc = c["softcap"] * torch.tanh(sc / c["softcap"])
        out[:, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), -1) @ vs[h // group]
    return out, cache


def attention_run(s, c, dst, q, qr, k, kr, v, cache):
    ctx, rows, heads, kv, dim = s.ctx, c["rows"], c["heads"], c["kv"], c["dim"]
    theta = hip.float_bits(THETA)
    ctx.Kernel(hip.GO_LLM_ROPE, rows * heads * dim // 2, qr, q, None, None, [heads, dim, c["position"], theta])
    ctx.Kernel(hip.GO_LLM_ROPE, rows * kv * dim // 2, kr, k, None, None, [kv, dim, c["position"], theta])
    ctx.Kernel(hip.GO_LLM_CACHE_WRITE, rows * kv * dim, cache, kr, v, None,
               [rows, kv, dim, c["capacity"], c["position"]])
    ctx.CachedAttention(dst, qr, cache, rows, c["capacity"], heads, kv, dim, c["position"], c.get("window", 0),
                        c.get("softcap", 0.0))


# ---- whole layers -------------------------------------------------------------------------------------------
def decoder_inputs(c, g):
    hidden, qd, kd = c["hidden"], c["heads"] * c["dim"], c["kv"] * c["dim"]
    x, layers = mlp_inputs(c, g)
    for l in layers:
        l.update(gamma1=1 + g.normal(hidden, std=0.1), gq=1 + g.normal(c["dim"], std=0.1),
                 gk=1 + g.normal(c["dim"], std=0.1), q=int4_pack(g.normal(qd, hidden, std=0.02)),
                 k=int4_pack(g.normal(kd, hidden, std=0.02)), v=int4_pack(g.normal(kd, hidden, std=0.02)),
                 o=int4_pack(g.normal(hidden, qd, std=0.02)), cache=g.normal(2 * kd * c["capacity"]))
    return x, layers


# ---------------------------------------------------------------------------------------------------------------
# prepare, run
# ---------------------------------------------------------------------------------------------------------------
def moe_inputs(c, g):
    hidden, inter, experts = c["hidden"], c["inter"], c["experts"]
    x = g.normal(c["rows"], hidden)
    router = g.normal(experts, hidden, std=0.02).bfloat16().contiguous()
    packed = {}
    for name, (n, k) in dict(gate=(inter, hidden), up=(inter, hidden), down=(hidden, inter)).items():
        step = max(1, (1 << 26) // (n * k))
        packed[name] = torch.cat([int4_pack(g.normal(min(step, experts - e) * n, k, std=0.02))
                                  for e in range(0, experts, step)]).view(experts, n, -1)
    return x, router, packed


def gguf_shapes(c):
    hidden, inter, qd, kd = c["hidden"], c["inter"], c["qdim"], c["kvdim"]
    shapes = dict(q=(qd, hidden), k=(kd, hidden), v=(kd, hidden), o=(hidden, qd), gate=(inter, hidden),
                  up=(inter, hidden), down=(hidden, inter))
    return {name: (MIX[name] if c["mix"] == "gemma" else c["mix"], *nk) for name, nk in shapes.items()}


def gguf_inputs(c, g):
    x = [g.normal(c["rows"], c["hidden"]) for _ in range(c["layers"])]
    return x, [{name: gguf_pack(g, e, n, k) for name, (e, n, k) in gguf_shapes(c).items()} for _ in range(c["layers"])]


def prepare(case, seed):
    c, s, g = case, State(case), Gen(seed)
    f = c["family"]
    if f == "mlp":
        x, layers = mlp_inputs(c, g)
        s.x, s.layers = s.put(x), [mlp_blocks(s, l) for l in layers]
        s.ys = [s.new(x.numel()) for _ in layers]
        mlp_tensors(s, c)
    elif f == "decoder":
        x, layers = decoder_inputs(c, g)
        qd, kd, rows = c["heads"] * c["dim"], c["kv"] * c["dim"], c["rows"]
        s.x, s.layers = s.put(x), []
        for l in layers:
            b = mlp_blocks(s, l)
            b.update({n: s.int4(l[n]) for n in ("q", "k", "v", "o")})
            b.update({n: s.vector(l[n]) for n in ("gamma1", "gq", "gk")})
            b["cache"] = s.put(l["cache"])
            s.layers.append(b)
        s.ys, s.zs = ([s.new(x.numel()) for _ in layers] for _ in range(2))
        mlp_tensors(s, c)
        s.q, s.qn, s.qr, s.a = (s.new(rows * qd) for _ in range(4))
        s.k, s.kn, s.kr, s.v = (s.new(rows * kd) for _ in range(4))
    elif f == "gguf":
        x, layers = gguf_inputs(c, g)
        shapes = gguf_shapes(c)
        s.xs = [s.put(v) for v in x]
        s.layers = [{name: s.gguf(e, l[name], n, k) for name, (e, n, k) in shapes.items()} for l in layers]
        s.outs = [{name: s.new(c["rows"] * n) for name, (_, n, _) in shapes.items()} for _ in layers]
        s.h = s.new(c["rows"] * c["inter"])
    elif f == "q8":
        s.w = s.gguf("Q8_0", gguf_pack(g, "Q8_0", c["n"], c["k"]), c["n"], c["k"])
        s.x, s.y = s.put(g.normal(c["rows"], c["k"])), s.new(c["rows"] * c["n"])
    elif f == "head":
        s.w = s.gguf("Q6_K", gguf_pack(g, "Q6_K", c["vocab"], c["hidden"]), c["vocab"], c["hidden"])
        s.x, s.logits, s.token = s.put(g.normal(c["hidden"])), s.new(c["vocab"]), s.new(1)
        s.seen = s.new(c["vocab"])
        view(s.seen, -1).view(torch.int32).copy_((g.ints(0, 500, c["vocab"]) == 0).int())
        s.uniform = float(torch.rand(1, generator=g.g, device=DEV)) * 0.999
    elif f == "moe":
        x, router, packed = moe_inputs(c, g)
        host = {n: p.cpu().numpy() for n, p in packed.items()}
        mk = lambda n: [hip.MemoryBlock.int4(host[n][e]) for e in range(c["experts"])]  # noqa: E731
        s.sets.append(s.ctx.CreateExpertSet(mk("gate"), mk("up"), mk("down"), c["hidden"], c["inter"]))
        s.router = s.bf16(router.view(torch.int16))
        s.x, s.logits = s.put(x), s.new(c["rows"] * c["experts"])
        s.routes, s.y = s.new(2 * c["rows"] * c["topk"]), s.new(c["rows"] * c["hidden"])
    elif f == "attention":
        i = attention_inputs(c, g)
        s.q, s.k, s.v, s.cache = (s.put(i[n]) for n in ("q", "k", "v", "cache"))
        s.qr, s.kr, s.y = s.new(i["q"].numel()), s.new(i["k"].numel()), s.new(i["q"].numel())
    else:
        raise ValueError(f)
    return s.ready()


def run(s):
    c, ctx = s.case, s.ctx
    f, rows = c["family"], c.get("rows", 1)
    if f == "mlp":
        src = s.x
        for w, y in zip(s.layers, s.ys):
            mlp_run(s, c, w, y, src)
            src = y
        return {"y": view(src, rows, c["hidden"])}
    if f == "decoder":
        hidden, heads, kv, dim = c["hidden"], c["heads"], c["kv"], c["dim"]
        src = s.x
        for w, y, z in zip(s.layers, s.ys, s.zs):
            ctx.KernelWeights(hip.GO_NORM, rows * hidden, s.xn, src, w["gamma1"], None, norm_args(rows, hidden))
            ctx.Int4Linear(s.q, s.xn, w["q"], rows, hidden, heads * dim)
            ctx.Int4Linear(s.k, s.xn, w["k"], rows, hidden, kv * dim)
            ctx.Int4Linear(s.v, s.xn, w["v"], rows, hidden, kv * dim)
            ctx.KernelWeights(hip.GO_NORM, rows * heads * dim, s.qn, s.q, w["gq"], None, norm_args(rows * heads, dim))
            ctx.KernelWeights(hip.GO_NORM, rows * kv * dim, s.kn, s.k, w["gk"], None, norm_args(rows * kv, dim))
            attention_run(s, c, s.a, s.qn, s.qr, s.kn, s.kr, s.v, w["cache"])
            ctx.Int4Linear(z, s.a, w["o"], rows, heads * dim, hidden)
            ctx.Kernel(hip.GO_ADD, rows * hidden, z, src, None, None, [hidden, hidden, ONE, 0, 0])
            mlp_run(s, c, w, y, z)
            src = y
        return {"y": view(src, rows, hidden), "caches": [view(w["cache"], -1) for w in s.layers]}
    if f == "gguf":
        hidden, inter = c["hidden"], c["inter"]
        for x, w, o in zip(s.xs, s.layers, s.outs):
            for name in ("q", "k", "v"):
                ctx.Linear(o[name], x, w[name], None, None, rows, hidden, w[name].shape[0])
            ctx.Linear(o["o"], o["q"], w["o"], None, None, rows, c["qdim"], hidden)
            ctx.Linear(o["gate"], x, w["gate"], None, None, rows, hidden, inter)
            ctx.Linear(o["up"], x, w["up"], None, None, rows, hidden, inter)
            ctx.Kernel(hip.GO_GEGLU, rows * inter, s.h, o["gate"], o["up"], None, [inter, 0])
            ctx.Linear(o["down"], s.h, w["down"], None, None, rows, inter, hidden)
            ctx.Kernel(hip.GO_ADD, rows * hidden, o["down"], o["o"], None, None, [hidden, hidden, ONE, 0, 0])
        return [{n: view(o[n], rows, -1) for n in ("q", "k", "v", "o", "down")} for o in s.outs]
    if f == "q8":
        if c["int8"]:
            ctx.Q8GemmInt8(s.y, s.x, s.w, rows, c["k"], c["n"])
        else:
            ctx.Linear(s.y, s.x, s.w, None, None, rows, c["k"], c["n"])
        return {"y": view(s.y, rows, c["n"])}
    if f == "head":
        ctx.Linear(s.logits, s.x, s.w, None, None, 1, c["hidden"], c["vocab"])
        ctx.SampleToken(s.token, s.logits, s.seen, c["vocab"], c["top_k"], 0.8, 0.95, 1.1, s.uniform)
        return {"logits": view(s.logits, -1), "token": view(s.token, -1).view(torch.int32)}
    if f == "moe":
        hidden, experts, k = c["hidden"], c["experts"], c["topk"]
        if rows == 1:
            ctx.VectorLinear(s.logits, s.x, s.router, hidden, experts)
        else:
            ctx.Linear(s.logits, s.x, s.router, None, None, rows, hidden, experts)
        ctx.Kernel(hip.GO_MOE_ROUTE, 2 * rows * k, s.routes, s.logits, None, None, [rows, experts, k, 1])
        ctx.MoEExperts(s.sets[0], s.y, s.x, s.routes, rows, k)
        routes = view(s.routes, 2, rows, k)
        return {"logits": view(s.logits, rows, experts), "ids": routes[0].view(torch.int32), "p": routes[1],
                "y": view(s.y, rows, hidden)}
    attention_run(s, c, s.y, s.q, s.qr, s.k, s.kr, s.v, s.cache)
    return {"y": view(s.y, rows, c["heads"], c["dim"]), "cache": view(s.cache, -1)}


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without, how close its results are, and the results in 64 bits
# ---------------------------------------------------------------------------------------------------------------
def _matrices(shapes, rows, bytes_of):
    return (sum(bytes_of(*s) for s in shapes),
            2.0 * rows * sum(float(n) * k for *_, n, k in shapes))


def _attention_work(c):
    rows, at, window = c["rows"], c["position"], c.get("window", 0)
    lens = [min(at + r + 1, window) if window else at + r + 1 for r in range(rows)]
    span = min(at + rows, lens[-1] + rows - 1)
    return (8.0 * span * c["kv"] * c["dim"] + 8.0 * rows * (c["heads"] + c["kv"]) * c["dim"],
            4.0 * sum(lens) * c["heads"] * c["dim"])


def work(case):
    c, f, rows = case, case["family"], case.get("rows", 1)
    if f in ("mlp", "decoder"):
        hidden, inter = c["hidden"], c["inter"]
        shapes = [(inter, hidden), (inter, hidden), (hidden, inter)]
        if f == "decoder":
            qd, kd = c["heads"] * c["dim"], c["kv"] * c["dim"]
            shapes += [(qd, hidden), (kd, hidden), (kd, hidden), (hidden, qd)]
        b, fl = _matrices(shapes, rows, int4_bytes)
        if f == "decoder":
            ab, af = _attention_work(c)
            b, fl = b + ab, fl + af
        return {"bytes": c["layers"] * b + 8.0 * rows * hidden, "flops": c["layers"] * fl}
    if f == "gguf":
        shapes = list(gguf_shapes(c).values())
        b, fl = _matrices(shapes, rows, gguf_bytes)
        io = 4.0 * rows * (c["hidden"] + c["qdim"] + 2 * c["kvdim"] + 2 * c["hidden"])
        return {"bytes": c["layers"] * (b + io), "flops": c["layers"] * fl}
    if f == "q8":
        return {"bytes": gguf_bytes("Q8_0", c["n"], c["k"]) + 4.0 * rows * (c["k"] + c["n"]),
                "flops": 2.0 * rows * c["k"] * c["n"]}
    if f == "head":
        return {"bytes": gguf_bytes("Q6_K", c["vocab"], c["hidden"]) + 8.0 * c["vocab"] + 4.0 * c["hidden"],
                "flops": 2.0 * c["vocab"] * c["hidden"]}
    if f == "moe":
        hidden, inter, experts, k = c["hidden"], c["inter"], c["experts"], c["topk"]
        touched = experts * (1 - (1 - k / experts) ** rows)
        one = 2 * int4_bytes(inter, hidden) + int4_bytes(hidden, inter)
        return {"bytes": touched * one + 2.0 * experts * hidden + 4.0 * rows * (2 * hidden + experts + 2 * k),
                "flops": 2.0 * rows * (experts * hidden + 3.0 * k * hidden * inter)}
    b, fl = _attention_work(c)
    return {"bytes": b, "flops": fl}


def tolerance(case):
    """About four times what the path differed by from its results in 64 bits, when measured over these ranges."""
    f, rows = case["family"], case.get("rows", 1)
    if f == "mlp":  # activations in 16 bits of fixed point per group of 32 (7.9e-5 over four layers)
        return {"rel": 3.2e-4}
    if f in ("moe", "decoder"):  # the same (4.7e-5, 5.0e-5)
        return {"rel": 2e-4}
    if f == "gguf":
        # Few rows: as above (4.3e-5).  Many rows: operands rounded to fp16, twice where one projection feeds
        # another (4.9e-4).
        return {"rel": 2e-3} if rows > 2 else {"rel": 1.8e-4}
    if f == "q8":  # operands rounded to fp16 (2.9e-4); activations of 8 bits (5e-3)
        return {"rel": 2e-2} if case["int8"] else {"rel": 1.2e-3}
    if f == "head":  # 2.2e-5
        return {"rel": 9e-5}
    return {"rel": 2.4e-6}  # attention in 32 bits (5.8e-7)


@torch.no_grad()
def exact(case, seed):
    c, g = case, Gen(seed)
    f, rows = c["family"], c.get("rows", 1)
    if f == "mlp":
        x, layers = mlp_inputs(c, g)
        x = x.double()
        for l in layers:
            x = mlp_exact(x, l, c["hidden"], c["inter"])
        return {"y": x}
    if f == "decoder":
        x, layers = decoder_inputs(c, g)
        x, caches = x.double(), []
        hidden, dim = c["hidden"], c["dim"]
        for l in layers:
            xn = norm_exact(x, l["gamma1"])
            q, k, v = ((xn @ int4_values(l[n], hidden).T).view(rows, -1, dim) for n in ("q", "k", "v"))
            a, cache = attention_exact(c, norm_exact(q, l["gq"]), norm_exact(k, l["gk"]), v, l["cache"])
            caches.append(cache)
            x = x + a.reshape(rows, -1) @ int4_values(l["o"], c["heads"] * dim).T
            x = mlp_exact(x, l, hidden, c["inter"])
        return {"y": x, "caches": caches}
    if f == "gguf":
        xs, layers = gguf_inputs(c, g)
        got = []
        for x, l in zip(xs, layers):
            x = x.double()
            w = lambda name: gguf_values(gguf_shapes(c)[name][0], l[name], gguf_shapes(c)[name][2]).T  # noqa: E731
            o = {n: x @ w(n) for n in ("q", "k", "v")}
            o["o"] = o["q"] @ w("o")
            o["down"] = (gelu(x @ w("gate")) * (x @ w("up"))) @ w("down") + o["o"]
            got.append(o)
        return got
    if f == "q8":
        w = gguf_values("Q8_0", gguf_pack(g, "Q8_0", c["n"], c["k"]), c["k"])
        return {"y": g.normal(rows, c["k"]).double() @ w.T}
    if f == "head":
        p = gguf_pack(g, "Q6_K", c["vocab"], c["hidden"])
        x = g.normal(c["hidden"]).double()
        step = 16384
        return {"logits": torch.cat([gguf_values("Q6_K", p[i:i + step], c["hidden"]) @ x
                                     for i in range(0, c["vocab"], step)]), "token": None}
    if f == "moe":
        x, router, packed = moe_inputs(c, g)
        hidden, inter = c["hidden"], c["inter"]
        x = x.double()
        logits = x @ router.double().T
        p, ids = torch.topk(torch.softmax(logits, -1), c["topk"], -1)
        p = p / p.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(c["experts"]):
            t, j = torch.nonzero(ids == e, as_tuple=True)
            if t.numel():
                h = silu(x[t] @ int4_values(packed["gate"][e], hidden).T) * (x[t] @ int4_values(packed["up"][e], hidden).T)
                y[t] += p[t, j][:, None] * (h @ int4_values(packed["down"][e], inter).T)
        return {"logits": logits, "ids": None, "p": p, "y": y}
    i = attention_inputs(c, g)
    y, cache = attention_exact(c, i["q"], i["k"], i["v"], i["cache"])
    return {"y": y, "cache": cache}
