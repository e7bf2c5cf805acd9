"""The work that users of this library give it, as measurable cases.

gpt.c's programs train a GPT-2 (train_gpt.c) and sample from one (infer_gpt.c); this library serves them through
gpt.c's own layer objects and device entry points (include/*.h), driven here through gptc.py.  Each case is one call
or one step of such a program:

  attention_forward   causal self-attention of a (B, T, 3C) qkv tensor, forward only (sampling, validation)
  attention_step      the same forward and its backward (training)
  linear_step         one Linear layer's forward and backward
  block_forward       one transformer block's forward (a layer of the prefill)
  block_step          one transformer block's forward and backward, its parameter gradients included
  head_step           the vocabulary projection with the cross-entropy loss, forward and backward
  decode              one token of a whole GPT-2 over its K/V caches
  train_step          a whole GPT-2 training step: forward, loss, backward, AdamW

All values are 32-bit floats, the library's only data type.
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gpt.c_amd"))
import gptc  # noqa: E402

V_GPT2 = 50257


def listed():
    return [
        # A short batch through one attention layer: the smallest call that GPT-2 small's sampling makes at B = 8.
        {"name": "attention_forward_b8_t128", "kind": "attention_forward", "B": 8, "T": 128, "H": 12, "D": 64},
        # A training batch of short ragged sequences on a small model.
        {"name": "attention_step_b2_t100", "kind": "attention_step", "B": 2, "T": 100, "H": 4, "D": 64},
        # GPT-2 small's attention layer in training.
        {"name": "attention_step_b8_t1024", "kind": "attention_step", "B": 8, "T": 1024, "H": 12, "D": 64},
        # GPT-2 XL's: 25 heads, so neither heads nor channels are a power of two.
        {"name": "attention_step_b4_t1024_h25", "kind": "attention_step", "B": 4, "T": 1024, "H": 25, "D": 64},
        # A ragged middle length: T is no multiple of any tile.
        {"name": "attention_step_b3_t333_h5", "kind": "attention_step", "B": 3, "T": 333, "H": 5, "D": 64},
        # Heads of 128 at full length.
        {"name": "attention_step_b2_t1024_d128", "kind": "attention_step", "B": 2, "T": 1024, "H": 8, "D": 128},
        # The MLP's first Linear on a small batch.
        {"name": "linear_step_1024x768x3072", "kind": "linear_step", "rows": 1024, "in": 768, "out": 3072},
        # A layer of the prefill that infer_gpt.c runs for every token: one window of 1024 tokens.
        {"name": "block_forward_b1_t1024", "kind": "block_forward", "B": 1, "T": 1024, "H": 12, "D": 64},
        # A GPT-2 small layer in training.
        {"name": "block_step_b8_t1024", "kind": "block_step", "B": 8, "T": 1024, "H": 12, "D": 64},
        # GPT-2's tied vocabulary projection with its loss, on a small batch.
        {"name": "head_step_1024", "kind": "head_step", "B": 2, "T": 512, "C": 768, "V": V_GPT2},
        # GPT-2 124M generating: one token at the middle of a 512-token context.
        {"name": "decode_gpt2_b1", "kind": "decode", "B": 1, "pos": 300, "L": 512, "layers": 12, "H": 12, "C": 768,
         "V": V_GPT2},
        # GPT-2 124M in training.
        {"name": "train_step_gpt2_b8", "kind": "train_step", "B": 8, "T": 1024, "layers": 12, "H": 12, "C": 768,
         "V": V_GPT2},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng):
    """Heads and their size: GPT-2's 64 in most programs."""
    D = 64 if rng.random() < 0.7 else rng.choice([16, 24, 32, 48, 80, 96, 128])
    return rng.choice([1, 2, 4, 5, 6, 8, 12, 16, 20, 25]), D


def draw(rng):
    kind = rng.choice(["attention_forward", "attention_step", "attention_step", "linear_step", "block_forward",
                       "block_step", "head_step", "decode", "train_step"])
    if kind in ("attention_forward", "attention_step"):
        while True:
            H, D = _heads(rng)
            B, T = _spread(rng, 1, 8), _spread(rng, 1, 2048)
            if B * H * T * T * D <= 8 * 12 * 1024 * 1024 * 64:
                return {"kind": kind, "B": B, "T": T, "H": H, "D": D}
    if kind == "linear_step":
        while True:
            rows, fin, fout = _spread(rng, 1, 8192), _spread(rng, 24, 4096), _spread(rng, 24, 4096)
            if rng.random() < 0.5:  # most layers' widths are multiples of 64
                fin, fout = max(64, fin // 64 * 64), max(64, fout // 64 * 64)
            if rows * fin * fout <= 8192 * 768 * 3072:
                return {"kind": kind, "rows": rows, "in": fin, "out": fout}
    if kind in ("block_forward", "block_step"):
        while True:
            H, D = _heads(rng)
            B, T = _spread(rng, 1, 8), _spread(rng, 1, 1024)
            if B * T * (H * D) ** 2 <= 8192 * 768 * 768:
                return {"kind": kind, "B": B, "T": T, "H": H, "D": D}
    if kind == "head_step":
        return {"kind": kind, "B": _spread(rng, 1, 4), "T": _spread(rng, 8, 512), "C": 64 * _spread(rng, 1, 16),
                "V": rng.choice([V_GPT2, _spread(rng, 97, V_GPT2)])}
    H = rng.choice([2, 4, 6, 8, 12])
    C = H * rng.choice([64, 64, 64, 32])
    if kind == "decode":
        L = rng.choice([256, 512, 1024])
        return {"kind": kind, "B": _spread(rng, 1, 8), "pos": rng.randrange(min(L, 600)), "L": L,
                "layers": rng.randint(1, 12), "H": H, "C": C, "V": rng.choice([V_GPT2, _spread(rng, 97, V_GPT2)])}
    return {"kind": kind, "B": _spread(rng, 1, 4), "T": _spread(rng, 16, 512), "layers": rng.randint(1, 3), "H": H,
            "C": C, "V": rng.choice([V_GPT2, _spread(rng, 97, V_GPT2)])}


# ---- inputs ----

_runtime = None


def _rt():
    global _runtime
    if _runtime is None:
        torch.cuda.init()
        _runtime = gptc.Runtime()
        _runtime.init()
    return _runtime


class _Draws:
    """Torch tensors on the GPU from one seed, in the order they are asked for."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.empty(shape, device="cuda").normal_(0.0, std, generator=self.gen)

    def ids(self, high, *shape):
        """Token ids as the library takes them: whole numbers held in floats."""
        return torch.randint(0, high, shape, device="cuda", generator=self.gen).float()


def _wrap(x):
    """A tensor_t over a torch tensor's memory (the torch tensor stays the owner)."""
    t = gptc.Tensor()
    t.t = ctypes.cast(x.data_ptr(), ctypes.POINTER(ctypes.c_float))
    t.ndims, t.length, t.device = x.dim(), x.numel(), gptc.CUDA
    for i, n in enumerate(x.shape):
        t.shape[i] = n
    return t


class _Memory:
    def __init__(self, t):
        c = t.contents
        self.__cuda_array_interface__ = {
            "shape": tuple(c.shape[:c.ndims]), "typestr": "<f4", "version": 3, "strides": None,
            "data": (ctypes.cast(c.t, ctypes.c_void_p).value, False)}


def _view(t):
    """A torch tensor over the memory of one of the library's tensors."""
    return torch.as_tensor(_Memory(t), device="cuda")


def _attention_inputs(case, seed):
    B, T, C = case["B"], case["T"], case["H"] * case["D"]
    d = _Draws(seed)
    return d.normal(B, T, 3 * C), d.normal(B, T, C)


def _linear_inputs(case, seed):
    rows, fin, fout = case["rows"], case["in"], case["out"]
    d = _Draws(seed)
    return d.normal(rows, fin), d.normal(fout, fin, std=0.02), d.normal(fout, std=0.02), d.normal(rows, fout)


def _head_inputs(case, seed):
    B, T, C, V = case["B"], case["T"], case["C"], case["V"]
    d = _Draws(seed)
    return d.normal(B, T, C), d.normal(V, C, std=0.02), d.ids(V, B, T)


def _block_shapes(C):
    return [(C,), (C,), (3 * C, C), (3 * C,), (C, C), (C,), (C,), (C,), (4 * C, C), (4 * C,), (C, 4 * C), (C,)]


def _block_params(d, C):
    """A block in the middle of its training: GPT-2's init with biases and LayerNorms that have moved."""
    out = [d.normal(*s, std=0.02) for s in _block_shapes(C)]
    out[0] += 1.0
    out[6] += 1.0
    return out


def _block_inputs(case, seed):
    B, T, C = case["B"], case["T"], case["H"] * case["D"]
    d = _Draws(seed)
    return d.normal(B, T, C), d.normal(B, T, C), _block_params(d, C)


def _model_params(d, case, block_size):
    C = case["C"]
    out = [d.normal(case["V"], C, std=0.02), d.normal(block_size, C, std=0.02)]
    for _ in range(case["layers"]):
        out += _block_params(d, C)
    return out + [1.0 + d.normal(C, std=0.02), d.normal(C, std=0.02)]


def _decode_inputs(case, seed):
    return _Draws(seed).ids(case["V"], case["B"], case["pos"] + 1)


def _train_inputs(case, seed):
    d = _Draws(seed)
    params = _model_params(d, case, case["T"])
    return params, d.ids(case["V"], case["B"], case["T"]), d.ids(case["V"], case["B"], case["T"])


_MODEL_SEED = 20240415  # the weights of the model that decode serves


# ---- the states a program keeps, and one pass of each kind ----

class _Attention:
    """One attention layer's buffers, allocated once: the compact cache layout of include/gpu_kernels.h."""

    def __init__(self, case, seed):
        self.rt = rt = _rt()
        lib = rt.lib
        B, T, H, D = case["B"], case["T"], case["H"], case["D"]
        C = H * D
        self.qkv, self.dy = _attention_inputs(case, seed)
        self.y = torch.empty(B, T, C, device="cuda")
        self.lse = torch.empty(B, H, T, device="cuda")
        self.dqkv = torch.empty(B, T, 3 * C, device="cuda")
        self.mask = torch.ones(T, T, device="cuda").tril_()
        torch.cuda.synchronize()
        self.t = [_wrap(x) for x in (self.qkv, self.mask, self.y, self.lse, self.dy, self.dqkv)]
        qkv, mask, y, lse, dy, dqkv = [ctypes.pointer(t) for t in self.t]
        # The library remembers checked masks only in its own memory.
        self.own_mask = rt.empty((T, T))
        lib.tensor_copy(self.own_mask, mask)
        self.state = rt.empty((int(lib.gptc_attention_state_floats(B, T, C, H)),))
        self.cache = (gptc.TensorP * 4)(qkv, y, lse, self.state)
        self.fwd = (qkv, self.own_mask, H, self.cache, y)
        self.bwd = (dy, self.cache, H, dqkv)
        self.step = case["kind"] == "attention_step"
        rt.sync()

    def run(self):
        self.rt.lib.attention_forward_cuda_kernel(*self.fwd)
        if not self.step:
            return self.y
        self.rt.lib.attention_backward_cuda_kernel(*self.bwd)
        return self.y, self.dqkv

    def __del__(self):
        self.rt.free(self.own_mask)
        self.rt.free(self.state)


class _Linear:
    def __init__(self, case, seed):
        self.rt = _rt()
        x, W, b, g = self.inputs = _linear_inputs(case, seed)
        self.y, self.dx = torch.empty_like(g), torch.empty_like(x)
        self.dW, self.db = torch.zeros_like(W), torch.zeros_like(b)
        torch.cuda.synchronize()
        self.t = [_wrap(v) for v in (x, W, b, g, self.y, self.dx, self.dW, self.db)]
        x, W, b, g, y, dx, dW, db = [ctypes.pointer(t) for t in self.t]
        self.grads = (gptc.TensorP * 2)(dW, db)
        self.fwd = (W, b, x, y)
        self.bwd = (g, x, W, dW, db, dx)

    def run(self):
        lib = self.rt.lib
        lib.zero_grad_adamW_cuda_kernel(self.grads, 2)
        lib.linear_forward_cuda_kernel(*self.fwd)
        lib.linear_backward_cuda_kernel(*self.bwd)
        return self.y, self.dx, self.dW, self.db


class _Head:
    def __init__(self, case, seed):
        self.rt = _rt()
        x, W, ids = self.inputs = _head_inputs(case, seed)
        B, T, V = case["B"], case["T"], case["V"]
        self.logits = torch.empty(B, T, V, device="cuda")
        self.lsm, self.dlogits = torch.empty_like(self.logits), torch.empty_like(self.logits)
        self.loss, self.dx, self.dW = torch.zeros(1, device="cuda"), torch.empty_like(x), torch.zeros_like(W)
        self.ones = torch.ones(B, T, device="cuda")
        torch.cuda.synchronize()
        self.t = [_wrap(v) for v in (x, W, ids, self.logits, self.lsm, self.dlogits, self.loss, self.dx, self.dW,
                                     self.ones)]
        x, W, ids, logits, lsm, dlogits, loss, dx, dW, ones = [ctypes.pointer(t) for t in self.t]
        cache = (gptc.TensorP * 2)(lsm, ids)
        self.grads = (gptc.TensorP * 1)(dW)
        self.calls = ((W, None, x, logits), (logits, ids, cache, loss), (ones, cache, dlogits),
                      (dlogits, x, W, dW, None, dx))

    def run(self):
        lib = self.rt.lib
        lib.zero_grad_adamW_cuda_kernel(self.grads, 1)
        lib.linear_forward_cuda_kernel(*self.calls[0])
        lib.cross_entropy_forward_cuda_kernel(*self.calls[1])
        lib.cross_entropy_backward_cuda_kernel(*self.calls[2])
        lib.linear_backward_cuda_kernel(*self.calls[3])
        return self.logits, self.loss, self.dx, self.dW


class _BlockT(ctypes.Structure):
    """block_t (include/blocks.h)."""
    _fields_ = ([(n, ctypes.c_int) for n in ("n_embd", "n_heads", "use_bias", "block_size", "_num_param_tensors")] +
                [("_pad", ctypes.c_byte * 4)] +
                [(n, ctypes.c_void_p) for n in ["ln1", "ln2", "mlp", "attn"] + gptc._MODEL_FNS])


def _load(rt, layer, params):
    """Writes torch tensors into a layer's parameters (both on the GPU)."""
    torch.cuda.synchronize()
    for t, x in zip(layer.parameters(), params):
        rt.lib.tensor_copy(t, ctypes.byref(_wrap(x)))
    rt.sync()


class _Block:
    """Block objects consume their input and the gradient they are given, so each pass hands them fresh tensors."""

    def __init__(self, case, seed):
        self.rt = rt = _rt()
        C = case["H"] * case["D"]
        self.x, self.dy, params = _block_inputs(case, seed)
        self.block = gptc._Layer(rt, rt.lib.Block(C, case["H"], case["T"], 1), _BlockT)
        self.block.to(gptc.CUDA)
        _load(rt, self.block, params)
        self.step = case["kind"] == "block_step"
        grads = self.block.gradients()
        self.grads = (gptc.TensorP * len(grads))(*grads)
        self.views = [_view(g) for g in grads]
        self.tx, self.tdy = _wrap(self.x), _wrap(self.dy)
        self.shape = tuple(self.x.shape)
        self.held = []

    def fresh(self, src):
        t = self.rt.empty(self.shape)
        self.rt.lib.tensor_copy(t, ctypes.byref(src))
        return t

    def drop(self):
        for t in self.held:
            self.rt.free(t)
        self.held = []

    def run(self):
        self.drop()
        if self.step:
            self.rt.lib.zero_grad_adamW_cuda_kernel(self.grads, len(self.grads))
        y = self.block.forward(self.fresh(self.tx))
        self.held.append(y)
        if not self.step:
            self.block.free_cache()
            return _view(y)
        dx = self.block.backward(self.fresh(self.tdy))
        self.held.append(dx)
        return [_view(y), _view(dx)] + self.views

    def __del__(self):
        self.drop()
        self.block.free()


_served = {}  # the one model that decode cases share, by its sizes


def _served_model(case):
    key = tuple(case[k] for k in ("layers", "H", "C", "V"))
    if key not in _served:
        for m in _served.values():
            m.free()
        _served.clear()
        rt = _rt()
        model = gptc.GPT2Model(rt, 1024, case["V"], case["layers"], case["H"], case["C"])
        model.to(gptc.CUDA)
        _load(rt, model, _model_params(_Draws(_MODEL_SEED), case, 1024))
        _served[key] = model
    return _served[key]


class _Decode:
    """A generation at position pos: the K/V caches hold the tokens before it."""

    def __init__(self, case, seed):
        self.rt = rt = _rt()
        self.model = _served_model(case)
        self.ids = _decode_inputs(case, seed).t().contiguous()  # (pos + 1, B)
        self.kv = gptc.KVCache(rt, self.model, case["B"], case["L"])
        torch.cuda.synchronize()
        self.t = [_wrap(row.view(-1, 1)) for row in self.ids]
        self.pos = case["pos"]
        self.logits = None
        for p in range(self.pos):
            rt.free(self.kv.decode(ctypes.byref(self.t[p]), p))
        rt.sync()

    def run(self):
        if self.logits:
            self.rt.free(self.logits)
        self.logits = self.kv.decode(ctypes.byref(self.t[self.pos]), self.pos)
        return _view(self.logits)

    def __del__(self):
        if self.logits:
            self.rt.free(self.logits)
        self.kv.free()


class _Train:
    """train_gpt.c's loop body: zero_grad, forward, loss, backward, AdamW step."""

    LR, BETA1, BETA2, EPS = 3e-4, 0.9, 0.99, 1e-8

    def __init__(self, case, seed):
        self.rt = rt = _rt()
        params, ids, targets = _train_inputs(case, seed)
        self.model = gptc.GPT2Model(rt, case["T"], case["V"], case["layers"], case["H"], case["C"])
        self.model.to(gptc.CUDA)
        _load(rt, self.model, params)
        self.opt = gptc.AdamWOptimizer(rt, self.model, lr=self.LR, beta1=self.BETA1, beta2=self.BETA2, eps=self.EPS)
        self.loss = gptc.CrossEntropy(rt)
        self.src = (ids, targets, torch.ones_like(ids))
        torch.cuda.synchronize()
        self.t = [_wrap(x) for x in self.src]
        # The matrices' gradients (1-D parameters are left out: an answer holds at most 64 outputs), and the
        # embedding tables that the step updates.
        self.views = [_view(g) for g in self.model.gradients() if g.contents.ndims == 2]
        self.views += [_view(p) for p in self.model.parameters()[:2]]
        self.held = []

    def fresh(self, i):
        t = self.rt.empty(tuple(self.src[i].shape))
        self.rt.lib.tensor_copy(t, ctypes.byref(self.t[i]))
        return t

    def drop(self):
        for t in self.held:
            self.rt.free(t)
        self.held = []

    def run(self):
        self.drop()
        self.opt.zero_grad()
        logits = self.model.forward(self.fresh(0))
        loss = self.loss.forward(logits, self.fresh(1))
        self.held += [logits, loss]
        g = self.model.backward(self.loss.backward(self.fresh(2)))
        if g:
            self.rt.free(g)
        self.opt.step()
        return [_view(logits), _view(loss)] + self.views

    def __del__(self):
        self.drop()
        self.loss.free()
        self.opt.free()
        self.model.free()


_STATES = {"attention_forward": _Attention, "attention_step": _Attention, "linear_step": _Linear,
           "block_forward": _Block, "block_step": _Block, "head_step": _Head, "decode": _Decode, "train_step": _Train}


def prepare(case, seed):
    return _STATES[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without ----

def _attention_flops(case, C, contractions):
    """One causal contraction: T (T + 1) / 2 pairs of C multiply-adds for each sequence."""
    return contractions * case["B"] * case["T"] * (case["T"] + 1) * C


def work(case):
    kind = case["kind"]
    if kind in ("attention_forward", "attention_step"):
        btc = case["B"] * case["T"] * case["H"] * case["D"]
        step = kind == "attention_step"
        # forward: qkv in, y out; backward: dy in, dqkv out
        return {"bytes": 4 * btc * (8 if step else 4),
                "flops": _attention_flops(case, case["H"] * case["D"], 6 if step else 2)}
    if kind == "linear_step":
        r, i, o = case["rows"], case["in"], case["out"]
        return {"bytes": 4 * (2 * r * i + 2 * r * o + 2 * i * o + 2 * o), "flops": 6 * r * i * o}
    if kind == "head_step":
        r, C, V = case["B"] * case["T"], case["C"], case["V"]
        return {"bytes": 4 * (2 * r * C + 2 * C * V + r * V), "flops": 6 * r * C * V}
    if kind in ("block_forward", "block_step"):
        C, step = case["H"] * case["D"], kind == "block_step"
        r = case["B"] * case["T"]
        return {"bytes": 4 * ((4 if step else 2) * r * C + (2 if step else 1) * 12 * C * C),
                "flops": (6 if step else 2) * r * 12 * C * C + _attention_flops(case, C, 6 if step else 2)}
    C, V, n = case["C"], case["V"], case["layers"]
    weights = n * 12 * C * C + V * C
    if kind == "decode":
        B, keys = case["B"], case["pos"] + 1
        return {"bytes": 4 * (weights + n * B * keys * 2 * C + B * V),
                "flops": 2 * B * weights + n * B * keys * 4 * C}
    r = case["B"] * case["T"]
    # AdamW reads weights, gradients and both moments and writes weights and moments; the logits come out.
    return {"bytes": 4 * (7 * (weights + case["T"] * C) + r * V),
            "flops": 6 * r * weights + n * _attention_flops(case, C, 6)}


def tolerance(case):
    """About four times the error against 64 bits that 32-bit sums show (measured on the MI355X over these ranges)."""
    return {"attention_forward": {"rel": 2e-6, "max": 4e-5},
            "attention_step": {"rel": 3e-6, "max": 1e-4},
            "linear_step": {"rel": 7e-6, "max": 4e-5},
            "block_forward": {"rel": 2e-6, "max": 2e-5},
            "block_step": {"rel": 8e-6, "max": 6e-5},
            "head_step": {"rel": 8e-6, "max": 6e-5},
            "decode": {"rel": 2e-6, "max": 1e-5},
            "train_step": {"rel": 2e-5, "max": 4e-3}}[case["kind"]]


# ---- the same in 64 bits ----

def _attention64(qkv, H):
    B, T, C3 = qkv.shape
    D = C3 // 3 // H
    q, k, v = (x.reshape(B, T, H, D).transpose(1, 2).contiguous() for x in qkv.split(C3 // 3, dim=2))
    hidden = torch.ones(T, T, dtype=torch.bool, device=qkv.device).triu(1)
    out = []
    for b in range(B):  # a sequence at a time: the scores of all would be large
        s = (q[b] @ k[b].transpose(1, 2).contiguous()) / math.sqrt(D)
        out.append(torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[b])
    return torch.stack(out).transpose(1, 2).reshape(B, T, C3 // 3)


def _block64(x, p, H):
    C = x.shape[-1]
    F = torch.nn.functional
    h = F.linear(F.layer_norm(x, (C,), p[0], p[1], 1e-5), p[2], p[3])
    x = x + F.linear(_attention64(h, H), p[4], p[5])
    h = F.gelu(F.linear(F.layer_norm(x, (C,), p[6], p[7], 1e-5), p[8], p[9]), approximate="tanh")
    return x + F.linear(h, p[10], p[11])


def _model64(ids, p, H, last_row):
    T = ids.shape[1]
    x = p[0][ids.long()] + p[1][:T]
    for i in range(2, len(p) - 2, 12):
        x = _block64(x, p[i:i + 12], H)
    x = torch.nn.functional.layer_norm(x[:, -1:] if last_row else x, (x.shape[-1],), p[-2], p[-1], 1e-5)
    return x @ p[0].t()


def _double(*xs):
    return [x.double() for x in xs]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("attention_forward", "attention_step"):
        qkv, dy = _double(*_attention_inputs(case, seed))
        if kind == "attention_forward":
            return _attention64(qkv, case["H"])
        qkv.requires_grad_()
        y = _attention64(qkv, case["H"])
        return y.detach(), torch.autograd.grad(y, qkv, dy)[0]
    if kind == "linear_step":
        x, W, b, g = _double(*_linear_inputs(case, seed))
        return x @ W.t() + b, g @ W, g.t() @ x, g.sum(0)
    if kind == "head_step":
        x, W, ids = _head_inputs(case, seed)
        x, W = x.double().requires_grad_(), W.double().requires_grad_()
        logits = x @ W.t()
        loss = torch.nn.functional.cross_entropy(logits.reshape(-1, case["V"]), ids.long().reshape(-1))
        dx, dW = torch.autograd.grad(loss, (x, W))
        return logits.detach(), loss.detach().reshape(1), dx, dW
    if kind in ("block_forward", "block_step"):
        x, dy, p = _block_inputs(case, seed)
        x, dy, p = x.double(), dy.double(), _double(*p)
        if kind == "block_forward":
            return _block64(x, p, case["H"])
        leaves = [v.requires_grad_() for v in [x] + p]
        y = _block64(x, p, case["H"])
        return [y.detach()] + list(torch.autograd.grad(y, leaves, dy))
    if kind == "decode":
        p = _double(*_model_params(_Draws(_MODEL_SEED), case, 1024))
        with torch.no_grad():
            return _model64(_decode_inputs(case, seed), p, case["H"], last_row=True)
    params, ids, targets = _train_inputs(case, seed)
    p = [v.requires_grad_() for v in _double(*params)]
    logits = _model64(ids, p, case["H"], last_row=False)
    loss = torch.nn.functional.cross_entropy(logits.reshape(-1, case["V"]), targets.long().reshape(-1))
    grads = torch.autograd.grad(loss, p)
    # The first AdamW step without weight decay, its moments corrected for their zero start.
    new = [w.detach() - _Train.LR * g / (g.abs() + _Train.EPS) for w, g in zip(p[:2], grads[:2])]
    return [logits.detach(), loss.detach().reshape(1)] + [g for g in grads if g.dim() == 2] + new
