"""The work whose speed is followed here, case by case.

A case is a plain dict. Its "kind" says which call of the library a user's
program makes:

* "matmul": one weight matrix times m activation rows on device pointers,
  hako_gpu_matmul for one token and hako_gpu_matmul_batch for more (the
  matmul of the reference's forward, once per weight and token).
* "layer": the seven matmuls of one transformer block for one token, each a
  hako_gpu_matmul call in the order the reference's forward makes them.
* "decode": n_seq sequences with `pos` cached positions each, one
  hako_gpu_decoder_step that returns the logits (the program samples from
  them) and then `steps` - 1 greedy tokens through hako_gpu_decoder_generate.
* "prompt": hako_gpu_decoder_prefill of m tokens at position `pos` of a
  sequence, with the logits of the last one.

Weights are random Q4_K / Q6_K blocks made on the GPU from the seed: uniform
quants and packed scales, block scales in the range of trained matrices.
Activations that come out of a norm are N(0, 1); those that come out of
SwiGLU (the inputs of a down projection) are products of two normals, whose
tails are as heavy as real ones.
"""
import ctypes as C
import math

import numpy as np
import torch

from hako_amd.decoder import Block, Model
from hako_amd.gpu import TYPE_Q4_K, TYPE_Q6_K, Gpu

BLOCK_BYTES = {"q4_k": 144, "q6_k": 210}
TYPE_ID = {"q4_k": TYPE_Q4_K, "q6_k": TYPE_Q6_K}

# The two model shapes of the benchmark (Qwen2.5-3B and Qwen2-7B).
SHAPE_3B = {"layers": 36, "heads": 16, "kv_heads": 2, "head_dim": 128, "ffn": 11008, "vocab": 151936, "tied": True}
SHAPE_7B = {"layers": 28, "heads": 28, "kv_heads": 4, "head_dim": 128, "ffn": 18944, "vocab": 152064, "tied": False}


def listed():
    def mm(name, qtype, n_out, n_in, m, bias=False):
        return {"name": name, "kind": "matmul", "type": qtype, "n_out": n_out, "n_in": n_in, "m": m, "bias": bias}

    blocks_7b = dict(SHAPE_7B, layers=4)
    return [
        # the smallest call of a forward: the 3B key projection with its bias, one token
        mm("k_proj_1", "q4_k", 256, 2048, 1, True),
        # a 3B block's seven matmuls for one token (the headline 11008 x 2048 matrix is two of them)
        {"name": "layer_3b_1", "kind": "layer", "d_model": 2048, "kv_dim": 256, "ffn": 11008},
        # the widest activation a token meets: the 7B down projection
        mm("down_7b_1", "q6_k", 3584, 18944, 1),
        # the 3B output matrix, the largest weight a token reads
        mm("vocab_3b_1", "q6_k", 151936, 2048, 1),
        # 16 sequences in step: a 7B up projection
        mm("up_7b_16", "q4_k", 18944, 3584, 16),
        # a short chat turn of 77 tokens through a 3B query projection
        mm("q_proj_77", "q4_k", 2048, 2048, 77, True),
        # a question of 200 tokens through a 3B down projection
        mm("down_3b_200", "q6_k", 2048, 11008, 200),
        # a full prompt pass of 512 tokens: the 7B up and down projections
        mm("up_7b_512", "q4_k", 18944, 3584, 512),
        mm("down_7b_512", "q6_k", 3584, 18944, 512),
        # a whole 3B model, one sequence, in the middle of a conversation
        dict(SHAPE_3B, name="decode_3b", kind="decode", n_seq=1, pos=1024, steps=8),
        # serving: 16 sequences with 4095 cached positions each through four 7B blocks and the output matrix
        dict(blocks_7b, name="decode_7b_blocks_16", kind="decode", n_seq=16, pos=4095, steps=4),
        # a 512-token prompt through the same four blocks
        dict(blocks_7b, name="prompt_7b_blocks_512", kind="prompt", m=512, pos=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: matmuls of one, a few (2..16) and many (17..512) tokens, and decoders of one to four blocks."""
    kind = rng.choice(["one", "one", "few", "few", "many", "many", "many", "decode", "prompt"])
    if kind in ("one", "few", "many"):
        m = 1 if kind == "one" else rng.randint(2, 16) if kind == "few" else _log_int(rng, 17, 512)
        n_in = 256 * _log_int(rng, 1, 74)
        # up to an output matrix for one or a few tokens (a prompt takes the last token's logits only), 7B blocks else
        most = 18944 if kind == "many" else 152064
        n_out = min(_log_int(rng, 64, most), (18944 if kind == "many" else 152064) * 3584 // n_in)
        return {"kind": "matmul", "type": rng.choice(["q4_k", "q6_k"]), "n_out": n_out, "n_in": n_in, "m": m,
                "bias": rng.random() < 0.3}
    head_dim = rng.choice([64, 128, 128])
    group = rng.choice([1, 2, 4, 6, 7, 8])
    kv_heads = rng.choice([k for k in (1, 2, 4, 8) if k * group * head_dim % 256 == 0 and k * group * head_dim <= 3584])
    d = {"layers": rng.randint(1, 4), "heads": group * kv_heads, "kv_heads": kv_heads, "head_dim": head_dim,
         "ffn": 256 * _log_int(rng, 4, 74), "vocab": _log_int(rng, 1000, 152064), "tied": rng.random() < 0.5}
    if kind == "decode":
        return dict(d, kind="decode", n_seq=rng.choice([1, 1, rng.randint(2, 16)]), pos=_log_int(rng, 1, 4095), steps=4)
    return dict(d, kind="prompt", m=_log_int(rng, 4, 512), pos=rng.choice([0, 0, _log_int(rng, 1, 1500)]))


# ── inputs ──

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _weight(g, qtype, n_out, n_in):
    """Random blocks [n_out * n_in / 256, block bytes]."""
    n = n_out * n_in // 256
    b = torch.randint(0, 256, (n, BLOCK_BYTES[qtype]), generator=g, device="cuda", dtype=torch.uint8)

    def f16(lo, hi):
        v = torch.rand(n, generator=g, device="cuda") * (hi - lo) + lo
        return v.to(torch.float16).view(torch.uint8).reshape(n, 2)

    if qtype == "q4_k":
        b[:, 0:2] = f16(1e-3, 2e-2)     # d
        b[:, 2:4] = f16(1e-3, 2e-2)     # dmin
    else:
        b[:, 208:210] = f16(2.5e-4, 2.5e-3)   # d; the 16 scales take every int8 value
    return b


def _activation(g, m, n_in, swiglu):
    x = _randn(g, m, n_in)
    return x * _randn(g, m, n_in) if swiglu else x


_gpu = None


def _lib():
    global _gpu
    if _gpu is None:
        _gpu = Gpu(0)
    return _gpu


def _layer_plan(case):
    """(name, type, n_out, n_in, input, bias) of a block's matmuls; the inputs are x, att, xf, h."""
    D, KV, F = case["d_model"], case["kv_dim"], case["ffn"]
    return [("q", "q4_k", D, D, "x", True), ("k", "q4_k", KV, D, "x", True), ("v", "q4_k", KV, D, "x", True),
            ("o", "q4_k", D, D, "att", False), ("gate", "q4_k", F, D, "xf", False), ("up", "q4_k", F, D, "xf", False),
            ("down", "q6_k", D, F, "h", False)]


def _model_plan(case):
    """Every tensor of a decoder's model: name -> (type, n_out, n_in); "f32" rows are norms and biases."""
    D, KV, F = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["ffn"]
    plan = {"tok_embd": ("q6_k" if case["tied"] else "q4_k", case["vocab"], D)}
    for l in range(case["layers"]):
        for role, n_out, n_in in (("wq", D, D), ("wk", KV, D), ("wv", KV, D), ("wo", D, D), ("gate", F, D), ("up", F, D)):
            plan["%d.%s" % (l, role)] = ("q4_k", n_out, n_in)
        plan["%d.down" % l] = ("q6_k", D, F)
        for role, n in (("attn_norm", D), ("ffn_norm", D), ("bq", D), ("bk", KV), ("bv", KV)):
            plan["%d.%s" % (l, role)] = ("f32", 1, n)
    plan["out_norm"] = ("f32", 1, D)
    if not case["tied"]:
        plan["output"] = ("q6_k", case["vocab"], D)
    return plan


def _model_tensors(case, seed):
    g, t = _gen(seed), {}
    for name, (qtype, n_out, n_in) in _model_plan(case).items():
        if qtype != "f32":
            t[name] = _weight(g, qtype, n_out, n_in)
        else:
            t[name] = (1.0 if name.endswith("norm") else 0.0) + 0.1 * _randn(g, n_in)
    return t


def _max_seq(case):
    return (case["pos"] + (case["steps"] if case["kind"] == "decode" else case["m"]) + 63) // 64 * 64


def _cached(case, seed):
    """The keys and values of the cached positions, [n_seq][layers][pos][kv_dim], as N(0, 1)."""
    g = _gen(seed + (1 << 40))
    shape = (case.get("n_seq", 1), case["layers"], case["pos"], case["kv_heads"] * case["head_dim"])
    return _randn(g, *shape), _randn(g, *shape)


def _tokens(case, seed):
    n = case["n_seq"] if case["kind"] == "decode" else case["m"]
    return np.random.default_rng(seed).integers(0, case["vocab"], n).astype(np.int32)


class _Handle:
    """A library decoder and the weights it reads; destroyed with the last tensor that looks at its caches."""

    def __init__(self, gpu, model, n_seq, max_seq, tensors):
        self.gpu, self.tensors, d = gpu, tensors, C.c_void_p()
        self.d = None
        gpu.check(gpu.lib.hako_gpu_decoder_create(C.byref(model), n_seq, max_seq, C.byref(d)), "decoder_create")
        self.d = d.value

    def __del__(self):
        if self.d:
            self.gpu.lib.hako_gpu_decoder_destroy(self.d)
            self.d = None


class _View:
    """A device array of a decoder's, for torch to look at in place."""

    def __init__(self, handle, ptr, shape):
        self.handle = handle
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


class _Decoder:
    """A decoder over weights in device memory, with its caches filled."""

    def __init__(self, case, seed):
        gpu, t = _lib(), _model_tensors(case, seed)
        self.gpu = gpu
        n_seq, max_seq = case.get("n_seq", 1), _max_seq(case)
        blocks = (Block * case["layers"])()
        for l, b in enumerate(blocks):
            for role in ("attn_norm", "ffn_norm", "wq", "wk", "wv", "wo", "bq", "bk", "bv", "gate", "up", "down"):
                setattr(b, role, t["%d.%s" % (l, role)].data_ptr())
            b.t_q = b.t_k = b.t_v = b.t_o = b.t_gate = b.t_up = TYPE_Q4_K
            b.t_down = TYPE_Q6_K
        m = Model(n_layers=case["layers"], d_model=case["heads"] * case["head_dim"], n_heads=case["heads"],
                  n_kv_heads=case["kv_heads"], head_dim=case["head_dim"], ffn_dim=case["ffn"], vocab=case["vocab"],
                  rope_theta=1e6, rms_eps=1e-6, blocks=blocks, tok_embd=t["tok_embd"].data_ptr(),
                  t_embd=TYPE_Q6_K if case["tied"] else TYPE_Q4_K, out_norm=t["out_norm"].data_ptr(),
                  out_weight=t["tok_embd" if case["tied"] else "output"].data_ptr(), t_out=TYPE_Q6_K)
        torch.cuda.synchronize()
        self.handle = _Handle(gpu, m, n_seq, max_seq, t)
        self.d = self.handle.d
        kp, vp = C.c_void_p(), C.c_void_p()
        gpu.check(gpu.lib.hako_gpu_decoder_kv(self.d, C.byref(kp), C.byref(vp)), "decoder_kv")
        shape = (n_seq, case["layers"], max_seq, case["kv_heads"] * case["head_dim"])
        self.k, self.v = (torch.as_tensor(_View(self.handle, p.value, shape), device="cuda") for p in (kp, vp))
        if case["pos"]:
            k, v = _cached(case, seed)
            self.k[:, :, :case["pos"]] = k
            self.v[:, :, :case["pos"]] = v
        self.pos = np.full(n_seq, case["pos"], np.int32)
        self.tokens = _tokens(case, seed)
        self.logits = np.empty((n_seq, case["vocab"]), np.float32)
        self.next = np.zeros(n_seq, np.int32)
        self.out = np.zeros((max(1, case.get("steps", 1) - 1), n_seq), np.int32)
        torch.cuda.synchronize()

    def decode(self, steps, pos):
        lib, check = self.gpu.lib, self.gpu.check
        check(lib.hako_gpu_decoder_set_pos(self.d, self.pos.ctypes.data), "set_pos")
        check(lib.hako_gpu_decoder_step(self.d, self.tokens.ctypes.data, self.logits.ctypes.data, self.next.ctypes.data),
              "step")
        check(lib.hako_gpu_decoder_generate(self.d, self.next.ctypes.data, steps - 1, self.out.ctypes.data), "generate")
        return dict(self.written(pos, steps), logits=self.logits, next=self.next, tokens=self.out)

    def prompt(self, m, pos):
        lib, check = self.gpu.lib, self.gpu.check
        check(lib.hako_gpu_decoder_set_pos(self.d, self.pos.ctypes.data), "set_pos")
        check(lib.hako_gpu_decoder_prefill(self.d, 0, self.tokens.ctypes.data, m, self.logits.ctypes.data,
                                           self.next.ctypes.data), "prefill")
        return dict(self.written(pos, m), logits=self.logits, next=self.next)

    def written(self, pos, n):
        """The keys and values of n positions, the first block's apart from the others'."""
        both = {"k": self.k[:, :, pos:pos + n], "v": self.v[:, :, pos:pos + n]}
        return {name + str(i): c[:, part] for name, c in both.items()
                for i, part in ((0, slice(0, 1)), (1, slice(1, None))) if c[:, part].numel()}


def _matmul_inputs(case, seed):
    g = _gen(seed)
    w = _weight(g, case["type"], case["n_out"], case["n_in"])
    x = _activation(g, case["m"], case["n_in"], case["type"] == "q6_k")
    return w, x, 0.1 * _randn(g, case["n_out"]) if case["bias"] else None


def _layer_inputs(case, seed):
    g = _gen(seed)
    acts = {"x": _activation(g, 1, case["d_model"], False), "att": _activation(g, 1, case["d_model"], False),
            "xf": _activation(g, 1, case["d_model"], False), "h": _activation(g, 1, case["ffn"], True)}
    return acts, [(n, t, o, i, a, _weight(g, t, o, i), 0.1 * _randn(g, o) if b else None)
                  for n, t, o, i, a, b in _layer_plan(case)]


def prepare(case, seed):
    if case["kind"] in ("decode", "prompt"):
        return case, _Decoder(case, seed)
    gpu = _lib()
    if case["kind"] == "layer":
        acts, mats = _layer_inputs(case, seed)
        calls = [(torch.zeros(o, device="cuda"), acts[a], TYPE_ID[t], w, b, o, i) for _, t, o, i, a, w, b in mats]
        args = [(y.data_ptr(), x.data_ptr(), t, w.data_ptr(), None if b is None else b.data_ptr(), o, i)
                for y, x, t, w, b, o, i in calls]
        return case, (gpu, args, [c[0] for c in calls], calls)
    w, x, bias = _matmul_inputs(case, seed)
    y = torch.zeros(case["m"], case["n_out"], device="cuda")
    return case, (gpu, y, x, w, bias)


def run(state):
    case, s = state
    if case["kind"] == "decode":
        return s.decode(case["steps"], case["pos"])
    if case["kind"] == "prompt":
        return s.prompt(case["m"], case["pos"])
    if case["kind"] == "layer":
        gpu, args, ys, _ = s
        for a in args:
            gpu.matmul(*a)
        return ys
    gpu, y, x, w, bias = s
    b = None if bias is None else bias.data_ptr()
    if case["m"] == 1:
        gpu.matmul(y.data_ptr(), x.data_ptr(), TYPE_ID[case["type"]], w.data_ptr(), b, case["n_out"], case["n_in"])
    else:
        gpu.matmul_batch(y.data_ptr(), x.data_ptr(), TYPE_ID[case["type"]], w.data_ptr(), b, case["m"], case["n_out"],
                         case["n_in"])
    return y


# ── what a pass cannot do without ──

def _mat(qtype, n_out, n_in):
    return n_out * (n_in // 256) * BLOCK_BYTES[qtype] if qtype != "f32" else 4 * n_in


def work(case):
    if case["kind"] == "matmul":
        m, o, i = case["m"], case["n_out"], case["n_in"]
        return {"bytes": _mat(case["type"], o, i) + 4 * m * (o + i) + (4 * o if case["bias"] else 0), "flops": 2 * m * o * i}
    if case["kind"] == "layer":
        plan = _layer_plan(case)
        acts = 4 * (3 * case["d_model"] + case["ffn"])
        return {"bytes": acts + sum(_mat(t, o, i) + 4 * o + (4 * o if b else 0) for _, t, o, i, _, b in plan),
                "flops": sum(2 * o * i for _, _, o, i, _, _ in plan)}
    plan = _model_plan(case)
    head = "tok_embd" if case["tied"] else "output"
    blocks = [v for k, v in plan.items() if k not in ("tok_embd", "output")]
    weights = sum(_mat(*v) for v in blocks) + _mat(*plan[head])
    dots = sum(o * i for t, o, i in blocks if t != "f32")
    out = case["vocab"] * plan[head][2]
    kv, D = case["kv_heads"] * case["head_dim"], case["heads"] * case["head_dim"]
    if case["kind"] == "decode":
        n, steps = case["n_seq"], case["steps"]
        seen = sum(case["pos"] + s + 1 for s in range(steps))   # positions attended over, per sequence and layer
        return {"bytes": steps * weights + 8 * n * case["layers"] * kv * seen + 4 * n * case["vocab"],
                "flops": 2 * n * steps * (dots + out) + 4 * n * case["layers"] * D * seen}
    m, pos = case["m"], case["pos"]
    seen = m * pos + m * (m + 1) // 2
    return {"bytes": weights + 8 * case["layers"] * kv * (pos + m) + 4 * case["vocab"],
            "flops": 2 * m * dots + 2 * out + 4 * case["layers"] * D * seen}


def tolerance(case):
    """About four times the distance from exact() at the start: 2.0e-7 (Q4_K) and 6.3e-7 (Q6_K) for the matmuls. In a
    decoder every block rounds its activations to 8 bits, where a value next to an edge falls on either side and the
    blocks after it differ: 1.2e-4 of the keys over four blocks, 1.9e-4 over 36."""
    if case["kind"] in ("decode", "prompt"):
        return {"rel": 5e-4 if case["layers"] <= 4 else 8e-4, "differ": 0.01}
    return {"rel": 1e-6 if case.get("type") == "q4_k" else 2.5e-6}


# ── the same in 64 bits, with plain torch ──

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(b, qtype, n_out, n_in):
    """The weights of random blocks in float64, [n_out][n_in]."""
    if qtype == "q4_k":
        d, dmin = _f16(b[:, 0:2]), _f16(b[:, 2:4])
        p = b[:, 4:16].int()
        s = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1)
        m = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1)
        q = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        w = (d * s).unsqueeze(2) * q - (dmin * m).unsqueeze(2)
    else:
        lo = b[:, :128].reshape(-1, 2, 1, 64)
        lo = torch.cat([lo & 15, lo >> 4], 2).reshape(-1, 2, 4, 32)
        hi = b[:, 128:192].reshape(-1, 2, 1, 32)
        hi = torch.cat([(hi >> (2 * k)) & 3 for k in range(4)], 2)
        q = (lo | (hi << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b[:, 208:210])
        w = q.reshape(-1, 16, 16) * sc.unsqueeze(2)
    return w.reshape(n_out, n_in)


def _q8(x):
    """x rounded to the 8-bit blocks of 32 that a Q4_K matrix meets (the call's own rounding, in 32 bits), in float64."""
    v = x.float().cpu().numpy().reshape(-1, 32)
    amax = np.abs(v).max(1, keepdims=True)
    scale = amax * np.float32(1 / 127)
    inv = np.divide(np.float32(127), amax, out=np.zeros_like(amax), where=scale > 0)
    q = np.clip(np.rint(v * inv), -127, 127).astype(np.float64) * scale
    return torch.from_numpy(q.reshape(x.shape)).cuda()


def _product(x, w, qtype, n_out, n_in, bias=None):
    """[rows of x][n_out] in float64, the weights taken 16384 rows at a time."""
    x = _q8(x) if qtype == "q4_k" else x.double()
    rows = w.reshape(n_out, -1)
    y = [x @ _dequant(rows[r:r + 16384].reshape(-1, BLOCK_BYTES[qtype]), qtype, len(rows[r:r + 16384]), n_in).t()
         for r in range(0, n_out, 16384)]
    return torch.cat(y, 1) + (0 if bias is None else bias.double())


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.float32(1e-6))) * w.double()


def _rope(x, p, head_dim):
    """Rotates [rows][heads * head_dim] for positions p; the angles are float32, as the path defines them."""
    f = np.power(1e6, -np.arange(0, head_dim, 2) / head_dim).astype(np.float32)
    a = torch.from_numpy((p.astype(np.float32)[:, None] * f).astype(np.float64)).cuda().unsqueeze(1)
    x = x.reshape(len(p), -1, head_dim)
    u, v = x[..., :head_dim // 2], x[..., head_dim // 2:]
    return torch.cat([u * a.cos() - v * a.sin(), u * a.sin() + v * a.cos()], 2).reshape(len(p), -1)


def _forward(case, t, tokens, p, cache):
    """The blocks over a prompt of `tokens` at positions p. `cache`: per layer [k, v], [positions][kv_dim] in float64,
    appended to here; the last block's values past its keys and values are not needed."""
    D, F, hd, kvh = case["heads"] * case["head_dim"], case["ffn"], case["head_dim"], case["kv_heads"]
    KV, G = kvh * hd, case["heads"] // kvh
    qt = "q6_k" if case["tied"] else "q4_k"
    rb = t["tok_embd"].reshape(case["vocab"], -1)[torch.from_numpy(tokens.astype(np.int64)).cuda()]
    x = _dequant(rb.reshape(-1, BLOCK_BYTES[qt]), qt, len(tokens), D)
    mask = torch.arange(int(p[-1]) + 1, device="cuda")[None, :] > torch.from_numpy(p.astype(np.int64)).cuda()[:, None]
    for l in range(case["layers"]):
        def mul(name, v, qtype, n_out, n_in, bias=None):
            return _product(v, t["%d.%s" % (l, name)], qtype, n_out, n_in, t["%d.%s" % (l, bias)] if bias else None)

        xn = _rms(x, t["%d.attn_norm" % l])
        cache[l][0] = torch.cat([cache[l][0], _rope(mul("wk", xn, "q4_k", KV, D, "bk"), p, hd)])
        cache[l][1] = torch.cat([cache[l][1], mul("wv", xn, "q4_k", KV, D, "bv")])
        if l + 1 == case["layers"]:
            return
        q = _rope(mul("wq", xn, "q4_k", D, D, "bq"), p, hd)
        k, v = (c.reshape(-1, kvh, hd) for c in cache[l])
        heads = []
        for h in range(case["heads"]):
            sc = q[:, h * hd:(h + 1) * hd] @ k[:, h // G].t() / math.sqrt(hd)
            heads.append(torch.softmax(sc.masked_fill(mask, -math.inf), 1) @ v[:, h // G])
        x = x + mul("wo", torch.cat(heads, 1), "q4_k", D, D)
        xn = _rms(x, t["%d.ffn_norm" % l])
        g, u = mul("gate", xn, "q4_k", F, D), mul("up", xn, "q4_k", F, D)
        x = x + mul("down", g * torch.sigmoid(g) * u, "q6_k", D, F)


def exact(case, seed):
    if case["kind"] == "matmul":
        w, x, bias = _matmul_inputs(case, seed)
        return _product(x, w, case["type"], case["n_out"], case["n_in"], bias)
    if case["kind"] == "layer":
        acts, mats = _layer_inputs(case, seed)
        return [_product(acts[a], w, t, o, i, b).reshape(-1) for _, t, o, i, a, w, b in mats]
    # Past the first 8-bit rounding a decoder's outputs have no 64-bit value that 32-bit sums come near: a value next to
    # an edge falls on either side, and the outputs of a few rows jump with it (the distance of decode_3b's keys from
    # this was 6e-5 to 1.9e-4 from seed to seed). Over the rows of a prompt that evens out (9.2e-6 to 1.1e-5).
    if case["kind"] == "decode":
        return None
    t, pos = _model_tensors(case, seed), case["pos"]
    kv = case["kv_heads"] * case["head_dim"]
    k, v = _cached(case, seed)
    cache = [[c[0, l].double().reshape(-1, kv) for c in (k, v)] for l in range(case["layers"])]
    _forward(case, t, _tokens(case, seed), pos + np.arange(case["m"]), cache)
    out = {"logits": None, "next": None}
    for i, name in enumerate("kv"):
        new = torch.stack([c[i][pos:] for c in cache]).unsqueeze(0)
        out[name + "0"] = new[:, :1]
        if case["layers"] > 1:
            out[name + "1"] = new[:, 1:] if case["m"] >= 128 else None
    return out
