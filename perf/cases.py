"""Performance cases: the work that a user of this framework has it do, through the Layer
interface, over the range of sizes that it serves.

Each case is one kind of call:
  gpt      a whole character-level GPT forward: host-side launch count and latency
  vit      a whole ViT classifier forward on a batch of images
  block    one pre-LN transformer block over a batch of sequences (decoder: GPT prefill,
           encoder: ViT), in fp32 (the default FLOAT_TYPE) or bf16
  decode   one GPT decoder block, one new position per sequence, against its KV cache
  gemma    one multi-query rotary block over a prompt (prefill into the KV cache)
  gstep    one replayed step of that block, one new position per sequence
  head     final LayerNorm, tied LM head and vocabulary softmax
  ghead    final RMSNorm and tied LM head of a decode step
"""
import os
import sys

import torch

# the package's modules import each other by bare name; they come from the tree that this
# process runs in
_PKG = os.path.join(os.getcwd(), "torchless-nn_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
os.environ.setdefault("XP_RUNTIME", "MI355X")


def listed():
    return [
        # the character model on a batch of four windows: the smallest call, all latency
        dict(name="char_gpt_f32", kind="gpt", dtype="fp32", vocab=65, layers=4, heads=4,
             head_dim=32, batch=4, seq=128),
        # a GPT-2-small-shaped block on a full batch of full windows
        dict(name="gpt2_block_bf16", kind="block", dtype="bf16", decoder=True, act="gelu",
             heads=12, head_dim=64, batch=8, seq=1024),
        # the same block on a few prompts of an odd length
        dict(name="gpt2_block_ragged_bf16", kind="block", dtype="bf16", decoder=True, act="gelu",
             heads=12, head_dim=64, batch=3, seq=777),
        # the same block in the default FLOAT_TYPE
        dict(name="gpt2_block_f32", kind="block", dtype="fp32", decoder=True, act="gelu",
             heads=12, head_dim=64, batch=4, seq=1000),
        # batched generation with that block, windows nearly full
        dict(name="gpt2_decode_bf16", kind="decode", dtype="bf16", act="gelu", heads=12,
             head_dim=64, batch=24, pos=901, capacity=1024),
        # its last layers on a full batch: final norm, 50257-way head, softmax
        dict(name="gpt2_head_bf16", kind="head", dtype="bf16", vocab=50257, heads=12, head_dim=64,
             batch=8, seq=1024),
        # ViT-S/4 on a batch of 32x32 images
        dict(name="vit_s4_bf16", kind="vit", dtype="bf16", patch=4, heads=6, head_dim=64, layers=8,
             act="gelu", registers=0, hidden=0, batch=512),
        # the notebook's ViT (patch 2, four registers, 261 tokens) in the default FLOAT_TYPE
        dict(name="vit_notebook_f32", kind="vit", dtype="fp32", patch=2, heads=4, head_dim=64,
             layers=12, act="silu", registers=4, hidden=256, batch=50),
        # a 2B-class multi-query block over four long prompts
        dict(name="gemma_prefill_bf16", kind="gemma", heads=8, kv_heads=1, head_dim=256, d=2048,
             ffn=16384, batch=4, seq=2048),
        # that block in a replayed greedy step, few sequences
        dict(name="gemma_step_b4_bf16", kind="gstep", heads=8, kv_heads=1, head_dim=256, d=2048,
             ffn=16384, batch=4, pos=2050, capacity=2176),
        # and in a batched server's step
        dict(name="gemma_step_b48_bf16", kind="gstep", heads=8, kv_heads=1, head_dim=256, d=2048,
             ffn=16384, batch=48, pos=1500, capacity=2048),
        # the 256000-way head of a batched step
        dict(name="gemma_head_b20_bf16", kind="ghead", vocab=256000, d=2048, batch=20),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _rows(rng, most, longest, shortest=1):
    """(batch, seq) with at most `most` rows."""
    seq = _log(rng, shortest, longest)
    return _log(rng, 1, max(1, most // seq)), seq


def draw(rng):
    kind = rng.choice(["gpt", "vit", "block", "block", "decode", "gemma", "gstep", "head", "ghead"])
    dtype = rng.choice(["fp32", "bf16"])
    if kind == "gpt":
        batch, seq = _rows(rng, 2048, 256, 16)
        return dict(kind=kind, dtype=dtype, vocab=rng.choice([65, 96, 257]), layers=rng.randint(2, 6),
                    heads=rng.choice([4, 6, 8]), head_dim=32, batch=batch, seq=seq)
    if kind == "vit":
        patch = rng.choice([2, 4])
        return dict(kind=kind, dtype=dtype, patch=patch, heads=rng.choice([3, 4, 6]), head_dim=64,
                    layers=rng.randint(2, 8), act=rng.choice(["gelu", "silu"]),
                    registers=rng.choice([0, 4]), hidden=rng.choice([0, 256]),
                    batch=_log(rng, 1, 512 if patch == 4 else 96))
    if kind == "block":
        batch, seq = _rows(rng, 8192 if dtype == "bf16" else 4096, 1024, 16)
        return dict(kind=kind, dtype=dtype, decoder=rng.random() < 0.7,
                    act=rng.choice(["gelu", "silu"]), heads=rng.choice([4, 6, 8, 12, 16]),
                    head_dim=rng.choice([32, 64]), batch=batch, seq=seq)
    if kind == "decode":
        capacity = rng.choice([256, 512, 1024])
        return dict(kind=kind, dtype=dtype, act="gelu", heads=rng.choice([4, 6, 8, 12, 16]),
                    head_dim=rng.choice([32, 64]), batch=_log(rng, 1, 96),
                    pos=_log(rng, 8, capacity - 1), capacity=capacity)
    if kind == "gemma":
        batch, seq = _rows(rng, 8192, 2048, 64)
        heads, kv_heads, head_dim, d, ffn = rng.choice([(8, 1, 256, 2048, 16384), (4, 1, 256, 1024, 4096),
                                                        (8, 2, 128, 1024, 4096)])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, head_dim=head_dim, d=d, ffn=ffn,
                    batch=batch, seq=seq)
    if kind == "gstep":
        heads, kv_heads, head_dim, d, ffn = rng.choice([(8, 1, 256, 2048, 16384), (4, 1, 256, 1024, 4096),
                                                        (8, 2, 128, 1024, 4096)])
        capacity = rng.choice([512, 1024, 2048, 4096])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, head_dim=head_dim, d=d, ffn=ffn,
                    batch=_log(rng, 1, 96), pos=_log(rng, 16, capacity - 1), capacity=capacity)
    if kind == "head":
        batch, seq = _rows(rng, 8192 if dtype == "bf16" else 1024, 1024)
        return dict(kind=kind, dtype=dtype, vocab=rng.choice([50257, 32000, 10007]),
                    heads=rng.choice([4, 8, 12]), head_dim=64, batch=batch, seq=seq)
    return dict(kind="ghead", vocab=rng.choice([256000, 32000, 50257]), d=rng.choice([1024, 2048]),
                batch=_log(rng, 1, 96))


# ---- inputs and weights, from the seed alone ------------------------------------------
_IMAGE = (3, 32, 32)
_CLASSES = 10


class _Draw:
    """Seeded tensors on the GPU, rounded to the case's storage type."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))
        self.dtype = torch.bfloat16 if dtype == "bf16" else torch.float32

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.empty(shape, device="cuda", dtype=torch.float32)
        return t.normal_(mean, std, generator=self.g).to(self.dtype)

    def ids(self, high, *shape):
        return torch.randint(0, high, shape, device="cuda", generator=self.g)


def _dtype(c):
    return c.get("dtype", "bf16")  # the Gemma-style kinds are bf16


def _block_params(r, d):
    """A TransformerBlock's parameters in `layer.parameters` order, at initialisation scale."""
    return [r.normal(d, mean=1.0, std=0.1), r.normal(d, std=0.1),
            r.normal(d, 3 * d, std=(2 / d) ** 0.5), r.normal(3 * d, std=0.1),
            r.normal(d, d, std=(2 / d) ** 0.5), r.normal(d, std=0.1),
            r.normal(d, mean=1.0, std=0.1), r.normal(d, std=0.1),
            r.normal(d, 4 * d, std=(2 / d) ** 0.5), r.normal(4 * d, std=0.1),
            r.normal(4 * d, d, std=(0.5 / d) ** 0.5), r.normal(d, std=0.1)]


def _gemma_params(r, c):
    d, f, hd = c["d"], c["ffn"], c["heads"] * c["head_dim"]
    return [r.normal(d, std=0.1), r.normal(d, hd + 2 * c["kv_heads"] * c["head_dim"], std=d ** -0.5),
            r.normal(hd, d, std=hd ** -0.5), r.normal(d, std=0.1), r.normal(d, f, std=d ** -0.5),
            r.normal(d, f, std=d ** -0.5), r.normal(f, d, std=f ** -0.5)]


def _inputs(c, seed):
    """(parameters in the model's order, inputs by name), as torch tensors on the GPU."""
    r = _Draw(seed, _dtype(c))
    kind, b = c["kind"], c["batch"]
    if kind in ("gpt", "block", "decode", "head", "vit"):
        d = c["heads"] * c["head_dim"]
    if kind == "gpt":
        p = [r.normal(c["seq"], d, std=0.1), r.normal(c["vocab"], d)]
        for _ in range(c["layers"]):
            p += _block_params(r, d)
        p += [r.normal(d, mean=1.0, std=0.1), r.normal(d, std=0.1)]
        # logits of a few units: the notebook's table is drawn at unit scale, trained ones are not
        p[1] *= 4 / d ** 0.5
        return p, dict(ids=r.ids(c["vocab"], b, c["seq"]))
    if kind == "vit":
        patches = (32 // c["patch"]) ** 2
        k = 3 * c["patch"] ** 2
        p = [r.normal(k, d, std=k ** -0.5), r.normal(1 + c["registers"], d, std=d ** -0.5),
             r.normal(1 + c["registers"] + patches, d, std=0.1)]
        for _ in range(c["layers"]):
            p += _block_params(r, d)
        p += [r.normal(d, mean=1.0, std=0.1), r.normal(d, std=0.1)]
        if c["hidden"]:
            p += [r.normal(d, c["hidden"], std=d ** -0.5), r.normal(c["hidden"], std=0.1),
                  r.normal(c["hidden"], _CLASSES, std=c["hidden"] ** -0.5), r.normal(_CLASSES, std=0.1)]
        else:
            p += [r.normal(d, _CLASSES, std=d ** -0.5), r.normal(_CLASSES, std=0.1)]
        return p, dict(x=r.normal(b, *_IMAGE))
    if kind == "block":
        return _block_params(r, d), dict(x=r.normal(b, c["seq"], d))
    if kind == "decode":
        p = _block_params(r, d)
        k = r.normal(b, c["heads"], c["capacity"], c["head_dim"])
        vt = r.normal(b, c["heads"], c["head_dim"], c["capacity"])
        return p, dict(x=r.normal(b, 1, d), k=k, vt=vt)
    if kind == "gemma":
        return _gemma_params(r, c), dict(x=r.normal(b, c["seq"], c["d"]))
    if kind == "gstep":
        p = _gemma_params(r, c)
        k = r.normal(b, c["kv_heads"], c["capacity"], c["head_dim"])
        vt = r.normal(b, c["kv_heads"], c["head_dim"], c["capacity"])
        return p, dict(x=r.normal(b, 1, c["d"]), k=k, vt=vt)
    if kind == "head":
        p = [r.normal(d, mean=1.0, std=0.1), r.normal(d, std=0.1), r.normal(c["vocab"], d, std=2 / d ** 0.5)]
        return p, dict(x=r.normal(b, c["seq"], d))
    p = [r.normal(c["d"], std=0.1), r.normal(c["vocab"], c["d"], std=2 / c["d"] ** 0.5)]
    return p, dict(x=r.normal(b, 1, c["d"]))


# ---- device tensors as torch tensors (the same memory) --------------------------------
class _Memory:
    """A DeviceTensor's memory for torch.as_tensor; it keeps the tensor alive."""

    def __init__(self, t):
        es = t.dtype.itemsize
        # rows of the last dimension `pitch` elements apart, outer dimensions packed over rows
        strides, step = [es], t.pitch * es
        for n in reversed(t.shape[:-1]):
            strides.append(step)
            step *= n
        self.tensor = t
        self.__cuda_array_interface__ = {
            "shape": t.shape, "typestr": {"float32": "<f4", "bfloat16": "<i2", "int64": "<i8"}[t.dtype.name],
            "data": (t.ptr, False), "strides": tuple(reversed(strides)), "version": 2}


def _torch(t):
    v = torch.as_tensor(_Memory(t), device="cuda")
    return v.view(torch.bfloat16) if t.dtype.name == "bfloat16" else v


def _fill(tensors, values):
    """The seeded values into the framework's tensors."""
    torch.cuda.synchronize()  # the framework's own stream may still write its initial values
    for t, v in zip(tensors, values):
        assert tuple(t.shape) == tuple(v.shape), (t.shape, v.shape)
        _torch(t).copy_(v)
        t._version += 1
    torch.cuda.synchronize()


def prepare(case, seed):
    import backend
    import tl_hip as xp
    from activations import GeLU, SiLU, SoftMax
    from gpt import build_gpt
    from layers import DevicePosition, GemmaBlock, KVCache, LayerNorm, RMSNorm, TransformerBlock
    from transformer_adapters import GPTEmbedBack, GPTEmbeddingTable
    from vit import build_vit

    c = case
    kind, b = c["kind"], c["batch"]
    dt = backend.set_float_type(_dtype(c))
    values, inputs = _inputs(c, seed)
    acts = {"gelu": GeLU, "silu": SiLU}
    s = {"kind": kind}

    def device(v):
        t = xp.empty(tuple(v.shape), xp.int64 if v.dtype == torch.int64 else dt)
        _fill([t], [v])
        return t

    if kind == "gpt":
        net, _ = build_gpt(dict(vocab=c["vocab"], ctx=c["seq"], layers=c["layers"],
                                d=c["heads"] * c["head_dim"], heads=c["heads"]))
        _fill([p for layer in net.layers for p in layer.parameters], values)
        s.update(net=net, x=device(inputs["ids"]))
    elif kind == "vit":
        net = build_vit(dict(image=_IMAGE, patch=(c["patch"],) * 2, d=c["heads"] * c["head_dim"],
                             heads=c["heads"], layers=c["layers"], act=c["act"],
                             registers=c["registers"], classes=_CLASSES,
                             head_hidden=c["hidden"] or None, dropout=0.0))
        _fill(_vit_parameters(net), values)
        s.update(net=net, x=device(inputs["x"]))
    elif kind in ("block", "decode"):
        d = c["heads"] * c["head_dim"]
        blk = TransformerBlock(d, c.get("capacity", c.get("seq")), c["heads"], acts[c["act"]],
                               decoder=c.get("decoder", True))
        blk.set_eval(True)
        _fill(blk.parameters, values)
        s.update(block=blk, x=device(inputs["x"]))
        if kind == "decode":
            s.update(cache=KVCache(1, b, c["heads"], c["capacity"], c["head_dim"], dt), pos=c["pos"])
            _fill([s["cache"].k[0], s["cache"].vt[0]], [inputs["k"], inputs["vt"]])
    elif kind in ("gemma", "gstep"):
        cap = c.get("capacity", c.get("seq"))
        blk = GemmaBlock(c["d"], cap, c["heads"], c["kv_heads"], c["head_dim"], c["ffn"])
        _fill(blk.parameters, values)
        s.update(block=blk, x=device(inputs["x"]),
                 cache=KVCache(1, b, c["kv_heads"], cap, c["head_dim"], dt))
        if kind == "gstep":
            # a server's step is recorded once and replayed at the position in device memory
            pos = DevicePosition(c["pos"], 1, c["head_dim"])
            pos.refresh()
            blk.forward(s["x"], s["cache"], 0, pos)
            with xp.capture() as g:
                pos.refresh()
                s["y"] = blk.forward(s["x"], s["cache"], 0, pos)
            s.update(graph=g, position=pos)
            _fill([s["cache"].k[0], s["cache"].vt[0]], [inputs["k"], inputs["vt"]])
    else:
        d = c["d"] if kind == "ghead" else c["heads"] * c["head_dim"]
        table = GPTEmbeddingTable(c["vocab"], d)
        norm = RMSNorm(d, gamma_offset=1.0) if kind == "ghead" else LayerNorm(d)
        _fill([*norm.parameters, table.table], values)
        s.update(norm=norm, back=GPTEmbedBack(table), softmax=SoftMax() if kind == "head" else None,
                 x=device(inputs["x"]))
    torch.cuda.synchronize()
    return s


def _vit_parameters(net):
    """Every layer's parameters in order: the projector, the blocks, the norm, the head."""
    return [p for layer in net.layers for p in layer.parameters]


def run(state):
    s = state
    kind = s["kind"]
    if kind in ("gpt", "vit"):
        probs = s["net"].predict(s["x"])
        # the layer before the SoftMax keeps its output: the logits
        return _torch(s["net"].layers[-2].output), _torch(probs)
    if kind == "block":
        return _torch(s["block"].forward(s["x"]))
    if kind in ("decode", "gemma"):
        cache = s["cache"]
        y = s["block"].forward(s["x"], cache, 0, s.get("pos", 0))
        return _torch(y), _torch(cache.k[0]), _torch(cache.vt[0])
    if kind == "gstep":
        s["graph"].launch()
        return _torch(s["y"]), _torch(s["cache"].k[0]), _torch(s["cache"].vt[0])
    logits = s["back"].forward(s["norm"].forward(s["x"]))
    return _torch(s["softmax"].forward(logits)) if s["softmax"] is not None else _torch(logits)


# ---- what a pass cannot do without ----------------------------------------------------
def _block_work(b, t, d, keys):
    """flops of a block's products and its attention over `keys` (query, key) pairs in all."""
    return 24.0 * b * t * d * d + 4.0 * keys * d


def work(case):
    c = case
    kind, b = c["kind"], c["batch"]
    es = 4 if _dtype(c) == "fp32" else 2
    if kind in ("gpt", "vit", "block", "decode", "head"):
        d = c["heads"] * c["head_dim"]
        block_weights = 12.0 * d * d + 13 * d
    if kind == "gpt":
        t, v = c["seq"], c["vocab"]
        flops = c["layers"] * _block_work(b, t, d, b * t * (t + 1) / 2) + 2.0 * b * t * d * v
        weights = c["layers"] * block_weights + (v + t) * d
        return {"bytes": es * (weights + 2.0 * b * t * v) + 8 * b * t, "flops": flops}
    if kind == "vit":
        n, k = (32 // c["patch"]) ** 2, 3 * c["patch"] ** 2
        t = n + 1 + c["registers"]
        flops = c["layers"] * _block_work(b, t, d, b * t * t) + 2.0 * b * n * k * d
        weights = c["layers"] * block_weights + (k + t) * d
        return {"bytes": es * (weights + b * (3 * 32 * 32 + 2 * _CLASSES)), "flops": flops}
    if kind == "block":
        t = c["seq"]
        pairs = b * t * (t + 1) / 2 if c["decoder"] else b * t * t
        return {"bytes": es * (block_weights + 2.0 * b * t * d), "flops": _block_work(b, t, d, pairs)}
    if kind == "decode":
        keys = b * (c["pos"] + 1)
        return {"bytes": es * (block_weights + 2.0 * b * d + 2.0 * keys * d),
                "flops": _block_work(b, 1, d, keys)}
    if kind in ("gemma", "gstep"):
        d, hd, kd = c["d"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        weights = d * (hd + 2 * kd) + hd * d + 3.0 * d * c["ffn"]
        t = c.get("seq", 1)
        keys = t * (t + 1) / 2 if kind == "gemma" else c["pos"] + 1
        cached = t if kind == "gemma" else c["pos"] + 1
        return {"bytes": 2 * (weights + 2.0 * b * t * d + 2.0 * b * cached * kd),
                "flops": 2.0 * b * t * weights + 4.0 * b * keys * hd}
    d, t, v = (c["d"], 1, c["vocab"]) if kind == "ghead" else (d, c["seq"], c["vocab"])
    return {"bytes": es * (1.0 * v * d + b * t * d + 1.0 * b * t * v), "flops": 2.0 * b * t * d * v}


def tolerance(case):
    """About four times the error measured against `exact` over listed and drawn cases."""
    c = case
    if _dtype(c) == "fp32":
        return {"rel": 1e-5}
    if c["kind"] in ("gpt", "head"):
        return {"rel": 6e-2}  # probabilities: exp of bf16 logits of a few units (0.015 seen)
    if c["kind"] == "vit":
        return {"rel": 4e-2}  # up to eight layers of bf16 roundings (0.009 seen)
    return {"rel": 2e-2}  # one block (0.0044 seen)


# ---- the same in 64 bits --------------------------------------------------------------
def _act(x, name):
    if name == "silu":
        return x * ((1 + torch.tanh(x / 2)) / 2)
    return 0.5 * x * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (x + 0.044715 * x ** 3)))


def _layernorm(x, g, b):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / (v + 1e-5).sqrt() * g + b


def _rmsnorm(x, g):
    return x / ((x * x).mean(-1, keepdim=True) + 1e-6).sqrt() * (1 + g)


def _attend(q, k, v, offset, causal):
    """q [b, h, t, e] over k, v [b, h, n, e], query i at position offset + i."""
    out = torch.empty_like(q)
    t, n = q.shape[2], k.shape[2]
    keep = torch.arange(n, device=q.device)[None, :] <= torch.arange(t, device=q.device)[:, None] + offset
    for i in range(q.shape[0]):
        s = torch.matmul(q[i], k[i].transpose(-1, -2).contiguous()) / q.shape[-1] ** 0.5
        if causal:
            s = s.masked_fill(~keep, float("-inf"))
        out[i] = torch.matmul(torch.softmax(s, -1), v[i].contiguous())
    return out


def _heads(x, h):
    b, t, d = x.shape
    return x.reshape(b, t, h, d // h).transpose(1, 2)


def _block(x, p, heads, act, causal, cache=None, pos=0):
    b, t, d = x.shape
    q, k, v = (_heads(y, heads) for y in (_layernorm(x, p[0], p[1]) @ p[2] + p[3]).split(d, -1))
    if cache is not None:
        cache[0][:, :, pos:pos + t] = k
        cache[1][:, :, :, pos:pos + t] = v.transpose(2, 3)
        k, v = cache[0][:, :, :pos + t], cache[1][:, :, :, :pos + t].transpose(2, 3)
    a = _attend(q, k, v, pos, causal).transpose(1, 2).reshape(b, t, d)
    y = x + a @ p[4] + p[5]
    return y + _act(_layernorm(y, p[6], p[7]) @ p[8] + p[9], act) @ p[10] + p[11]


def _rope(x, pos):
    """Rotate-half RoPE of x [b, h, t, e] at positions pos .."""
    half = x.shape[-1] // 2
    inv = 10000.0 ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / x.shape[-1])
    a = (pos + torch.arange(x.shape[2], device=x.device, dtype=torch.float64))[:, None] * inv
    u, w = x[..., :half], x[..., half:]
    return torch.cat([u * a.cos() - w * a.sin(), w * a.cos() + u * a.sin()], -1)


def _gemma_block(x, p, c, cache, pos):
    b, t, _ = x.shape
    hq, hk, e = c["heads"], c["kv_heads"], c["head_dim"]
    q, k, v = (_rmsnorm(x, p[0]) @ p[1]).split([hq * e, hk * e, hk * e], -1)
    cache[0][:, :, pos:pos + t] = _rope(_heads(k, hk), pos)
    cache[1][:, :, :, pos:pos + t] = _heads(v, hk).transpose(2, 3)
    k, v = cache[0][:, :, :pos + t], cache[1][:, :, :, :pos + t].transpose(2, 3)
    g = hq // hk
    a = _attend(_rope(_heads(q, hq), pos), k.repeat_interleave(g, 1), v.repeat_interleave(g, 1), pos, True)
    y = x + a.transpose(1, 2).reshape(b, t, hq * e) @ p[2]
    z = _rmsnorm(y, p[3])
    return y + (_act(z @ p[4], "gelu") * (z @ p[5])) @ p[6]


def exact(case, seed):
    c = case
    kind = c["kind"]
    p, inputs = _inputs(c, seed)
    p = [v.double() for v in p]
    x = inputs["ids"] if kind == "gpt" else inputs["x"].double()
    if kind == "gpt":
        y = p[1][x] + p[0]
        for i in range(c["layers"]):
            y = _block(y, p[2 + 12 * i:14 + 12 * i], c["heads"], "gelu", True)
        logits = _layernorm(y, p[-2], p[-1]) @ p[1].T
        return logits, torch.softmax(logits, -1)
    if kind == "vit":
        b, n = c["batch"], 32 // c["patch"]
        tok = x.reshape(b, 3, n, c["patch"], n, c["patch"]).permute(0, 2, 4, 3, 5, 1).reshape(b, n * n, -1)
        y = torch.cat([p[1].expand(b, -1, -1), tok @ p[0]], 1) + p[2]
        for i in range(c["layers"]):
            y = _block(y, p[3 + 12 * i:15 + 12 * i], c["heads"], c["act"], False)
        tail = p[3 + 12 * c["layers"]:]
        z = _layernorm(y, tail[0], tail[1])[:, 0] @ tail[2] + tail[3]
        if c["hidden"]:
            z = _act(z, "silu") @ tail[4] + tail[5]
        return z, torch.softmax(z, -1)
    if kind == "block":
        return _block(x, p, c["heads"], c["act"], c["decoder"])
    if kind == "decode":
        cache = [inputs["k"].double(), inputs["vt"].double()]
        return _block(x, p, c["heads"], c["act"], True, cache, c["pos"]), cache[0], cache[1]
    if kind == "gemma":
        cache = [x.new_zeros(c["batch"], c["kv_heads"], -(-c["seq"] // 8) * 8, c["head_dim"]),
                 x.new_zeros(c["batch"], c["kv_heads"], c["head_dim"], -(-c["seq"] // 8) * 8)]
        return _gemma_block(x, p, c, cache, 0), cache[0], cache[1]
    if kind == "gstep":
        cache = [inputs["k"].double(), inputs["vt"].double()]
        return _gemma_block(x, p, c, cache, c["pos"]), cache[0], cache[1]
    if kind == "head":
        return torch.softmax(_layernorm(x, p[0], p[1]) @ p[2].T, -1)
    return _rmsnorm(x, p[0]) @ p[1].T
