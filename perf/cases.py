"""Performance cases: the calls that programs built on this library spend their time in.

Four kinds of call, all through the C ABI as turkce-llm_amd/trlm.py binds it:

  gemm    trlm_gemm on device buffers: C = op(A) @ op(B) (+ bias) (+ residual).  NN is a layer's forward
          product, NT the tied LM head (or a layer's dX), TN a weight gradient.  Leading dimensions are the
          trainer's (rows padded to 16 bytes) or tight, which for odd sizes leaves the rows unaligned.
  model   the trainer: a forward to logits on the host, the evaluation loss, or a training step
          (forward, cross-entropy, backward, gradient norm, AdamW).
  decode  the KV-cache decoder: a prefill, then given tokens step by step or greedy generation, and the
          logits of the last position.
  node    node_matmul2d_gpu: the autograd node on host tensors, forward and backward.

Sizes come from the repository's model (V 31769, D 384, 6 heads, 12 layers, F 1024; B8 T1024, B1 T128 and
64 sequences of decode) and its tests' small models; draw() spreads over what lies between.
"""
import ctypes as C
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
REAL = {"V": 31769, "D": 384, "H": 6, "L": 12, "F": 1024}
EPS = 1e-5
LR, BETA1, BETA2, ADAM_EPS, DECAY = 3e-4, 0.9, 0.95, 1e-8, 0.1


def _trlm():
    """The binding, loaded by path (its folder's name is no identifier)."""
    if "trlm_amd" not in sys.modules:
        path = os.path.join(ROOT, "turkce-llm_amd", "trlm.py")
        spec = importlib.util.spec_from_file_location("trlm_amd", path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["trlm_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["trlm_amd"]


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one decode step's QKV projection: 64 rows, the smallest call, where latency counts
        _gemm("gemm nn 64 rows", "nn", 64, 1152, 384, bias=True),
        # a layer's QKV projection over a training batch (B8 T1024)
        _gemm("gemm nn qkv", "nn", 8192, 1152, 384, bias=True),
        # the gate/up weight gradient: few outputs, a long sum over the batch's rows
        _gemm("gemm tn gate_up dW", "tn", 384, 2048, 8192),
        # the tied LM head over a training batch: the largest product of the model
        _gemm("gemm nt lm head", "nt", 8192, 31769, 384),
        # odd sizes with tight rows, so nothing is 16-byte aligned
        _gemm("gemm nn ragged", "nn", 1000, 701, 333, pad=False, resid=True),
        # one short prompt through the real model, every logit to the host
        dict(REAL, name="logits B1 T128", kind="model", op="logits", B=1, T=128),
        # validation loss of a full batch
        dict(REAL, name="eval B8 T1024", kind="model", op="eval", B=8, T=1024),
        # a full training step of the real model
        dict(REAL, name="train B8 T1024", kind="model", op="train", B=8, T=1024),
        # a training step of a small model with ragged sizes (F no multiple of 32, T of no tile)
        dict(name="train small", kind="model", op="train", V=1001, D=96, H=3, L=2, F=200, B=3, T=100),
        # 64 sequences: prefill of 128 tokens each, then 32 tokens step by step
        dict(REAL, name="decode B64", kind="decode", op="steps", B=64, P=128, S=32),
        # one user: a prompt of 100 tokens, 48 tokens generated greedily
        dict(REAL, name="generate B1", kind="decode", op="greedy", B=1, P=100, S=48),
        # the hybrid path: a 128-token sequence through one projection, forward and backward, host to host
        dict(name="node 128x384x1024", kind="node", M=128, K=384, N=1024),
    ]


def _gemm(name, layout, M, N, K, pad=True, bias=False, resid=False):
    c = dict(kind="gemm", layout=layout, M=M, N=N, K=K, pad=pad, bias=bias, resid=resid)
    return dict(c, name=name) if name else c


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _small_model(rng):
    hd = rng.choice([16, 32, 64])
    H = rng.randint(1, min(6, 384 // hd))
    return {"V": _logint(rng, 50, 8000), "D": hd * H, "H": H, "L": rng.randint(1, 4), "F": _logint(rng, 32, 1024)}


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "model", "decode", "node"])
    if kind == "gemm":
        layout = rng.choice(["nn", "nt", "tn"])
        while True:
            M, N, K = _logint(rng, 1, 8192), _logint(rng, 8, 31769), _logint(rng, 16, 8192)
            if 1e5 <= 2.0 * M * N * K <= 1.5e11 and M * K + K * N + M * N <= 3e8:
                break
        return _gemm(None, layout, M, N, K, pad=rng.random() < 0.75, bias=rng.random() < 0.5,
                     resid=rng.random() < 0.25)
    if kind == "model":
        T = _logint(rng, 12, 1024)
        return dict(_small_model(rng), kind="model", op=rng.choice(["train", "train", "eval", "logits"]),
                    B=rng.randint(1, max(1, min(8, 8192 // T))), T=T)
    if kind == "decode":
        # greedy picks of one sequence only: a pick between two logits that rounding cannot tell apart
        # changes everything after it
        op = rng.choice(["steps", "steps", "greedy"])
        P, m = _logint(rng, 1, 512), _small_model(rng)
        m["F"] = (m["F"] + 3) // 4 * 4     # the decoder takes d_ff in fours
        return dict(m, kind="decode", op=op, P=P, S=_logint(rng, 4, 48),
                    B=1 if op == "greedy" else _logint(rng, 1, min(64, max(1, 16384 // P))))
    return dict(kind="node", M=_logint(rng, 1, 512), K=_logint(rng, 16, 1024), N=_logint(rng, 16, 2048))


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)


def _normal(gen, shape, std=1.0):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std


def _shapes(c):
    V, D, F = c["V"], c["D"], c["F"]
    s = [(V, D)]
    for _ in range(c["L"]):
        s += [(D,), (D, 3 * D), (3 * D,), (D, D), (D,), (D,), (D, 2 * F), (2 * F,), (F, D), (D,)]
    return s + [(D,)]


def _params(c, gen):
    """Parameters as lm_model.c initialises them, N(0, 0.02), with norm weights near one."""
    shapes = _shapes(c)
    out = []
    for i, s in enumerate(shapes):
        norm = i == len(shapes) - 1 or (i and (i - 1) % 10 in (0, 5))
        out.append(_normal(gen, s, 0.02) + (1.0 if norm else 0.0))
    return out


def _flat(params):
    return torch.cat([p.reshape(-1) for p in params])


def _tokens(gen, shape, V):
    return torch.randint(0, V, shape, generator=gen, device="cuda").cpu().numpy().astype(np.uint32)


def _operands(c, seed):
    """op(A) [M, K], op(B) [K, N] as stored rows (with their padding), bias and residual."""
    gen, (M, N, K) = _gen(seed), (c["M"], c["N"], c["K"])
    ta, tb = c["layout"][0] == "t", c["layout"][1] == "t"

    def stored(rows, cols, std):
        ld = (cols + 3) // 4 * 4 if c["pad"] else cols
        return _normal(gen, (rows, ld), std)

    # activations N(0,1) against weights N(0,0.02); in a weight gradient, against a batch mean's gradients
    A = stored(K, M, 1.0) if ta else stored(M, K, 1.0)
    B = stored(N, K, 0.02) if tb else stored(K, N, 1e-4 if ta else 0.02)
    bias = _normal(gen, (N,), 0.02) if c["bias"] else None
    ldc = (N + 3) // 4 * 4 if c["pad"] else N
    resid = _normal(gen, (M, ldc)) if c["resid"] else None
    return A, B, bias, resid, ldc, ta, tb


_device = None


def _gemm_device():
    """One context and GEMM engine for the process, as a program that multiplies matrices keeps."""
    global _device
    if _device is None:
        _device = _trlm().Device()
    return _device


class _Model:
    """A model resident on the GPU, its optimizer and, for decode cases, its decoder."""

    def __init__(self, c, seed):
        trlm = _trlm()
        gen = _gen(seed)
        self.params = _flat(_params(c, gen)).cpu().numpy()
        self.hm = trlm.HostModel(c["V"], c["D"], c["H"], c["L"], c["F"], self.params, eps=EPS)
        self.dec = self.adam = None
        if c["kind"] == "decode":
            self.tr = trlm.Trainer(self.hm, 1, 8)
            self.dec = trlm.Decoder(self.tr, c["B"], c["P"] + c["S"])
            self.prompt = _tokens(gen, (c["B"], c["P"]), c["V"])
            self.given = _tokens(gen, (c["S"], c["B"]), c["V"])
        else:
            self.tr = trlm.Trainer(self.hm, c["B"], c["T"])
            self.ids = _tokens(gen, (c["B"] * c["T"],), c["V"])
            self.targets = _tokens(gen, (c["B"] * c["T"],), c["V"])
            if c["op"] == "train":
                self.adam = trlm.Adam(self.hm, lr=LR, b1=BETA1, b2=BETA2, eps=ADAM_EPS)
                self.tr.upload(self.adam)

    def __del__(self):
        if getattr(self, "dec", None) is not None:
            self.dec.destroy()
        if getattr(self, "tr", None) is not None:
            self.tr.destroy()
        if getattr(self, "hm", None) is not None:
            self.hm.close()


class _Resident:
    """Device memory of a model as an array (it keeps the model alive)."""

    def __init__(self, model, ptr, n):
        self.model = model
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False), "version": 2,
                                         "strides": None}


def _resident(model):
    """(parameters, gradients) where the trainer holds them: GpuTrainer's total_scalars field and the
    pointers after it (gpu_train.h: params, grads, adam_m, adam_v)."""
    raw = list(model.tr.g.raw)
    n = model.hm.total
    at = next(i for i in range(len(raw) - 4)
              if raw[i] == n and all(0 <= raw[i + k + 1] - raw[i + k] - 4 * n < 256 for k in (1, 2, 3)))
    return [torch.as_tensor(_Resident(model, raw[at + k], n), device="cuda") for k in (1, 2)]


class _HostNode:
    """Leaves A [M, K], B [K, N] in a host arena and the gradient that arrives at the product."""

    def __init__(self, c, seed):
        trlm = _trlm()
        host, hip = trlm.libs()
        global _ops_ready
        if not _ops_ready:
            self.scratch = host.allocator_create(1 << 24)
            hip.gpu_ops_init(C.byref(self.scratch), trlm.KERNELS.encode())
            _ops_ready = True
        M, K, N = c["M"], c["K"], c["N"]
        gen = _gen(seed)
        A, B, self.dC = [_normal(gen, s, std).cpu().numpy()
                         for s, std in (((M, K), 1.0), ((K, N), 0.02), ((M, N), 1e-3))]
        self.arena = host.allocator_create(16 * (M * K + K * N) + (1 << 20))
        self.a, self.b = [self._leaf(x) for x in (A, B)]
        self.bytes = 32 * (M * K + K * N + M * N) + (1 << 20)   # what one pass allocates, and to spare

    def _leaf(self, x):
        trlm = _trlm()
        host, _ = trlm.libs()
        t = host.tensor_create(C.byref(self.arena), (C.c_uint64 * 2)(*x.shape), 2)
        trlm.tensor_np(t)[:] = x.ravel()
        return host.node_leaf(C.byref(self.arena), t, 1)

    def __del__(self):
        if getattr(self, "arena", None) is not None:
            _trlm().libs()[0].allocator_destroy(C.byref(self.arena))


_ops_ready = False


def prepare(case, seed):
    if case["kind"] == "gemm":
        A, B, bias, resid, ldc, ta, tb = _operands(case, seed)
        out = torch.zeros((case["M"], ldc), device="cuda", dtype=torch.float32)
        return {"case": case, "dev": _gemm_device(), "A": A, "B": B, "bias": bias, "resid": resid, "C": out,
                "ta": int(ta), "tb": int(tb)}
    if case["kind"] == "node":
        return {"case": case, "node": _HostNode(case, seed)}
    model = _Model(case, seed)
    state = {"case": case, "model": model}
    if case["kind"] == "model" and case["op"] == "train":
        state["params"], state["grads"] = _resident(model)
    return state


# ---------------------------------------------------------------- one pass

def run(state):
    c = state["case"]
    return {"gemm": _run_gemm, "model": _run_model, "decode": _run_decode, "node": _run_node}[c["kind"]](c, state)


def _run_gemm(c, s):
    dev, A, B, out = s["dev"], s["A"], s["B"], s["C"]
    dev.current()
    dev.matmul(s["ta"], s["tb"], A.data_ptr(), B.data_ptr(), out.data_ptr(), c["M"], c["N"], c["K"], A.shape[1],
               B.shape[1], out.shape[1], bias=s["bias"].data_ptr() if s["bias"] is not None else None,
               resid=s["resid"].data_ptr() if s["resid"] is not None else None)
    return out[:, :c["N"]]


def _run_model(c, s):
    m = s["model"]
    if c["op"] == "logits":
        return m.tr.forward_logits(m.ids)
    if c["op"] == "eval":
        return float(m.tr.eval_loss(m.ids, m.targets))
    loss = float(m.tr.forward_backward(m.ids, m.targets))
    norm = float(m.tr.grad_norm())
    m.tr.adamw_step(m.adam, DECAY)
    return {"loss": loss, "norm": norm, "grads": s["grads"], "params": s["params"]}


def _run_decode(c, s):
    m = s["model"]
    if c["op"] == "greedy":
        tokens = m.dec.generate_greedy(m.prompt, c["S"])
        return {"tokens": tokens.astype(np.int64), "logits": m.dec.logits()}
    m.dec.prefill(m.prompt)
    for ids in m.given:
        m.dec.step(ids)
    return m.dec.logits()


def _run_node(c, s):
    trlm, n = _trlm(), s["node"]
    host, hip = trlm.libs()
    arena = host.allocator_create(n.bytes)     # a step's arena, as the training loop makes one
    ga, gb = [trlm.tensor_np(x.contents.grad) for x in (n.a, n.b)]
    ga[:] = 0
    gb[:] = 0
    out = hip.node_matmul2d_gpu(C.byref(arena), n.a, n.b)
    value = trlm.tensor_np(out.contents.value).copy()
    trlm.tensor_np(out.contents.grad)[:] = n.dC.ravel()
    C.CFUNCTYPE(None, trlm.NodeP, C.POINTER(trlm.Allocator))(out.contents.backward_fn)(out, C.byref(arena))
    host.allocator_destroy(C.byref(arena))
    M, K, N = c["M"], c["K"], c["N"]
    return {"C": value.reshape(M, N), "dA": ga.copy().reshape(M, K), "dB": gb.copy().reshape(K, N)}


# ---------------------------------------------------------------- what a pass cannot do without

def _forward_flops(c, B, T, head_rows):
    """Causal forward of B sequences of T tokens, with logits of head_rows rows."""
    N, D, F = B * T, c["D"], c["F"]
    layer = 2.0 * N * (4 * D * D + 3 * D * F) + 4.0 * B * D * T * (T + 1) / 2
    return c["L"] * layer + 2.0 * head_rows * D * c["V"]


def work(case):
    c = case
    if c["kind"] == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        n = M * K + K * N + M * N + (N if c["bias"] else 0) + (M * N if c["resid"] else 0)
        return {"bytes": 4.0 * n, "flops": 2.0 * M * N * K}
    if c["kind"] == "node":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4.0 * 2 * (M * K + K * N + M * N), "flops": 6.0 * M * N * K}
    P = float(sum(int(np.prod(s)) for s in _shapes(c)))
    if c["kind"] == "model":
        N = c["B"] * c["T"]
        f = _forward_flops(c, c["B"], c["T"], N)
        if c["op"] == "train":     # parameters, both moments: read and written; gradients written
            return {"bytes": 4.0 * (7 * P + 2 * N), "flops": 3.0 * f}
        return {"bytes": 4.0 * (P + 2 * N + (N * c["V"] if c["op"] == "logits" else 0)), "flops": f}
    # decode: a step reads the parameters once and the keys and values of all positions
    flops, nbytes = _forward_flops(c, c["B"], c["P"], c["B"]), P
    for s in range(c["S"] if c["op"] == "steps" else c["S"] - 1):
        ctx = c["P"] + s + 1
        flops += 2.0 * c["B"] * (c["L"] * (4 * c["D"] ** 2 + 3 * c["D"] * c["F"] + 2 * c["D"] * ctx)
                                 + c["D"] * c["V"])
        nbytes += P + 2.0 * c["L"] * c["B"] * c["D"] * ctx
    return {"bytes": 4.0 * (nbytes + c["B"] * c["V"]), "flops": flops}


def tolerance(case):
    """About four times what the fp32 path was seen to be off from 64 bits."""
    c = case
    if c["kind"] == "gemm":
        return {"rel": 4e-6}       # 8e-7 at K = 8192, 3.5e-7 at K = 384
    if c["kind"] == "node":
        return {"rel": 2e-6}       # 2e-7 at K = 128 to 1024
    if c["op"] == "train":
        # 1.7e-6 (12 layers).  max: AdamW's first step moves a weight by lr times the sign of its gradient,
        # so a gradient that is rounding noise moves it either way (2 lr = 6e-4, against weights of 0.02)
        return {"rel": 8e-6, "max": 0.1}
    return {"rel": 4e-6}           # 7e-7 (12 layers)


# ---------------------------------------------------------------- the same in 64 bits

def _rope(T, hd):
    """cos and sin of fp32 angles, position times base ** (-2k / hd), as model/rope.c:4-18 defines them."""
    k = np.arange(hd // 2, dtype=np.float32)
    freq = np.power(10000.0, (-(2.0 * k) / np.float32(hd)).astype(np.float64)).astype(np.float32)
    ang = (np.arange(T, dtype=np.float32)[:, None] * freq[None, :]).astype(np.float64)
    return [torch.from_numpy(f(ang)).cuda() for f in (np.cos, np.sin)]


def _rotate(x, cos, sin):
    """Pairs (2k, 2k+1) of [B, H, T, hd] rotated by their position's angles."""
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * cos - b * sin, a * sin + b * cos), dim=-1).reshape(x.shape)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w


def _hidden64(c, p, ids):
    """Final-norm output [B, T, D] of token ids [B, T]."""
    B, T = ids.shape
    D, H, F = c["D"], c["H"], c["F"]
    hd = D // H
    cos, sin = _rope(T, hd)
    future = torch.ones((T, T), dtype=torch.bool, device="cuda").triu(1)
    x = p[0][ids]
    for l in range(c["L"]):
        n1, wqkv, bqkv, wo, bo, n2, wgu, bgu, wd, bd = p[1 + 10 * l:11 + 10 * l]
        q, k, v = [t.reshape(B, T, H, hd).transpose(1, 2).contiguous()
                   for t in (_rms(x, n1) @ wqkv + bqkv).split(D, dim=-1)]
        q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
        score = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(hd)
        att = torch.matmul(torch.softmax(score.masked_fill(future, -math.inf), dim=-1), v)
        x = x + (att.transpose(1, 2).reshape(B, T, D) @ wo + bo)
        gate, up = (_rms(x, n2) @ wgu + bgu).split(F, dim=-1)
        x = x + ((torch.nn.functional.silu(gate) * up) @ wd + bd)
    return _rms(x, p[-1])


def exact(case, seed):
    c = case
    if c["kind"] == "gemm":
        A, B, bias, resid, _, ta, tb = _operands(c, seed)
        A = A.double()[:, :c["M"] if ta else c["K"]]
        B = B.double()[:, :c["K"] if tb else c["N"]]
        r = (A.t() if ta else A) @ (B.t() if tb else B)
        if bias is not None:
            r += bias.double()
        if resid is not None:
            r += resid.double()[:, :c["N"]]
        return r
    gen = _gen(seed)
    if c["kind"] == "node":
        M, K, N = c["M"], c["K"], c["N"]
        A, B, dC = [_normal(gen, s, std).double() for s, std in (((M, K), 1.0), ((K, N), 0.02), ((M, N), 1e-3))]
        return {"C": A @ B, "dA": dC @ B.t(), "dB": A.t() @ dC}
    p = [t.double() for t in _params(c, gen)]
    if c["kind"] == "decode":
        ids = torch.from_numpy(_tokens(gen, (c["B"], c["P"]), c["V"]).astype(np.int64)).cuda()
        given = torch.from_numpy(_tokens(gen, (c["S"], c["B"]), c["V"]).astype(np.int64)).cuda()
        if c["op"] == "steps":
            return _hidden64(c, p, torch.cat([ids, given.t()], dim=1))[:, -1] @ p[0].t()
        picks = []
        for s in range(c["S"]):
            if s:
                ids = torch.cat([ids, picks[-1][:, None]], dim=1)
            logits = _hidden64(c, p, ids)[:, -1] @ p[0].t()
            picks.append(logits.argmax(dim=-1))
        return {"tokens": torch.stack(picks, dim=1), "logits": logits}
    B, T = c["B"], c["T"]
    ids, targets = [torch.from_numpy(_tokens(gen, (B * T,), c["V"]).astype(np.int64)).cuda() for _ in range(2)]
    if c["op"] == "logits":
        return _hidden64(c, p, ids.reshape(B, T)).reshape(B * T, -1) @ p[0].t()
    if c["op"] == "eval":
        rows = _hidden64(c, p, ids.reshape(B, T)).reshape(B * T, -1) @ p[0].t()
        return float(torch.nn.functional.cross_entropy(rows, targets))
    p = [t.requires_grad_(True) for t in p]
    rows = _hidden64(c, p, ids.reshape(B, T)).reshape(B * T, -1) @ p[0].t()
    loss = torch.nn.functional.cross_entropy(rows, targets)
    grads = torch.autograd.grad(loss, p)
    g, w = _flat(grads), _flat([t.detach() for t in p])
    m, v = (1 - BETA1) * g / (1 - BETA1), (1 - BETA2) * g * g / (1 - BETA2)
    w = w - LR * m / (torch.sqrt(v) + ADAM_EPS) - LR * DECAY * w
    return {"loss": float(loss.detach()), "norm": float(torch.sqrt((g * g).sum())), "grads": g, "params": w}
