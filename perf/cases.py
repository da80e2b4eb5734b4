"""The calls a program makes of this package, with the sizes it makes them at.

A case is a dict of plain values.  ``listed()`` are the cases that are always
looked at, ``draw(rng)`` gives one more of the same ranges, ``prepare(case,
seed)`` makes what the program has in hand before the call (weights stored in a
manager, activations, buffers), ``run(state)`` makes the call once through the
public entry points and returns what the program gets, ``work(case)`` is what a
pass cannot do without and ``tolerance(case)`` how far two correct
implementations may be apart.

Kinds
  read      ``Manager.read``: one stored weight back as a dense tensor
  encode    ``nz_encode`` of the C ABI: one weight into a container and a packed
            stream that the caller owns
  rewrite   an optimizer step's end and the next pass's beginning:
            ``Manager.write_many`` of a block's weights under their handles, then
            ``Manager.read`` of each
  block     the seven Linears of a gated decoder block converted by
            ``Manager.convert``, for one to a few activation rows (a token, a
            small batch, a speculative step) or for many (a prompt)
  train     one step on the four Linears of a GPT-2-shaped block: forward,
            backward, and the update hook that decompresses, updates and
            re-compresses every weight
  gather    a compressed ``Embedding`` looked up for some tokens
"""
from __future__ import annotations

import ctypes
import math
from functools import partial

import torch
import torch.nn.functional as F

import neuzip_amd
from neuzip_amd import _lib

# entropy of the exponents in bytes per element: N(0, 0.02) at any precision, and
# Student-t(3) x 0.02 with a few large columns, zeros and subnormals
_EXP_BYTES = {"normal": 0.3184, "heavy": 0.349}


def listed():
    return [
        # the attention output projection of a GPT-2-medium block, read on its own: the
        # smallest weight that models of the configured shapes hold, bound by latency
        {"name": "read_1024x1024", "kind": "read", "rows": 1024, "cols": 1024, "precision": 7, "normalizer": 0,
         "values": "normal"},
        # a ragged weight (no dimension a multiple of anything) at the lossy setting with
        # block normalizers, the reference's options for inference memory
        {"name": "read_5003x3001_p3_n64", "kind": "read", "rows": 5003, "cols": 3001, "precision": 3,
         "normalizer": 64, "values": "normal"},
        # the benchmark's own weight, lossless
        {"name": "read_16384x4096", "kind": "read", "rows": 16384, "cols": 4096, "precision": 7, "normalizer": 0,
         "values": "normal"},
        # the benchmark's stress weight: heavy tails, outlier columns, zeros, subnormals;
        # larger than the last-level cache
        {"name": "read_8192x28672_heavy", "kind": "read", "rows": 8192, "cols": 28672, "precision": 7,
         "normalizer": 0, "values": "heavy"},
        # compression of the benchmark's weight, the codec's other direction
        {"name": "encode_16384x4096", "kind": "encode", "rows": 16384, "cols": 4096, "precision": 7,
         "normalizer": 0, "values": "normal"},
        # compression of a small ragged weight at a lossy setting: few workgroups
        {"name": "encode_3071x1021_p3", "kind": "encode", "rows": 3071, "cols": 1021, "precision": 3,
         "normalizer": 0, "values": "normal"},
        # the weights of a GPT-2-medium block after an optimizer step: stored again in one
        # call, then read by the next forward pass
        {"name": "rewrite_gpt2m_block", "kind": "rewrite", "width": 1024, "precision": 7, "normalizer": 0,
         "values": "normal"},
        # single-token inference through the Linears of an 8B-shaped decoder block
        {"name": "block_8b_token", "kind": "block", "width": 4096, "kv": 1024, "ffn": 14336, "tokens": 1,
         "precision": 7, "normalizer": 0, "values": "normal"},
        # the same block for a small batch (a speculative step), the most rows the fused
        # product takes
        {"name": "block_8b_tokens8", "kind": "block", "width": 4096, "kv": 1024, "ffn": 14336, "tokens": 8,
         "precision": 7, "normalizer": 0, "values": "normal"},
        # the same block for the benchmark's prompt of 512 tokens
        {"name": "block_8b_prompt512", "kind": "block", "width": 4096, "kv": 1024, "ffn": 14336, "tokens": 512,
         "precision": 7, "normalizer": 0, "values": "normal"},
        # a training step of the GPT-2-medium-shaped block at the benchmark's batch of
        # 8 x 1024 tokens
        {"name": "train_gpt2m_block", "kind": "train", "width": 1024, "tokens": 8192, "precision": 7,
         "normalizer": 0, "values": "normal"},
        # one token looked up in the 8B-shaped model's embedding table
        {"name": "gather_128256x4096_token", "kind": "gather", "rows": 128256, "cols": 4096, "tokens": 1,
         "precision": 7, "normalizer": 0, "values": "normal"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["read", "read", "encode", "encode", "rewrite", "block", "block", "train", "gather"])
    # lossless is what the package is used for most; the lossy settings and the
    # block normalizers are options
    precision = rng.choice([7, 7, 7, 3, 1, 0])
    normalizer = rng.choice([0, 0, 0, 8, 64, 512])
    case = {"kind": kind, "precision": precision, "normalizer": normalizer,
            "values": rng.choice(["normal", "normal", "heavy"])}
    if kind in ("read", "encode"):
        n = _log_uniform(rng, 1 << 18, 1 << 27)
        cols = min(_log_uniform(rng, 256, 16384), n // 64)
        if rng.random() < 0.5:
            cols = max(64, cols // 64 * 64)
        case.update(rows=max(1, n // cols), cols=cols)
    elif kind == "rewrite":
        case.update(width=64 * _log_uniform(rng, 8, 40))
    elif kind == "block":
        width = 128 * _log_uniform(rng, 8, 40)
        kv = rng.choice([width, width // 2, width // 4])
        ffn = 64 * ((int(width * rng.uniform(2.5, 4.0))) // 64)
        case.update(width=width, kv=kv, ffn=ffn, tokens=_log_uniform(rng, 1, 512), normalizer=0)
    elif kind == "train":
        case.update(width=64 * _log_uniform(rng, 8, 32), tokens=_log_uniform(rng, 128, 8192), normalizer=0)
    else:
        cols = 128 * _log_uniform(rng, 4, 32)
        case.update(rows=_log_uniform(rng, 8000, 128000), cols=cols, tokens=_log_uniform(rng, 1, 1024))
    return case


def _values(kind, rows, cols, gen):
    """A bf16 weight: N(0, 0.02), or Student-t(3) x 0.02 with 16 columns x 50, 1 % zeros and
    0.1 % subnormals."""
    z = torch.randn(rows, cols, device="cuda", generator=gen)
    if kind == "heavy":
        chi = torch.randn(rows, cols, device="cuda", generator=gen).square_()
        for _ in range(2):
            chi += torch.randn(rows, cols, device="cuda", generator=gen).square_()
        z /= (chi / 3.0).sqrt_()
        del chi
        z[:, torch.randperm(cols, device="cuda", generator=gen)[:16]] *= 50.0
    w = z.mul_(0.02).to(torch.bfloat16)
    if kind == "heavy":
        r = torch.rand(rows, cols, device="cuda", generator=gen)
        w.masked_fill_(r < 0.01, 0.0)
        w.masked_fill_((r >= 0.01) & (r < 0.011), 1e-39)
    return w


def _manager(case):
    return neuzip_amd.Manager(precision=case["precision"], normalizer_size=case["normalizer"])


def _linear(out_features, in_features, bias, case, gen):
    lin = torch.nn.Linear(in_features, out_features, bias=bias, device="meta")
    lin.weight = torch.nn.Parameter(_values(case["values"], out_features, in_features, gen))
    if bias:
        lin.bias = torch.nn.Parameter((torch.randn(out_features, device="cuda", generator=gen) * 0.02)
                                      .to(torch.bfloat16))
    return lin


def _rows(n, width, gen):
    return torch.randn(n, width, device="cuda", generator=gen).to(torch.bfloat16)


class _Gated(torch.nn.Module):
    """The Linears of a gated decoder block in the order of the block; what stands
    between them (attention over a cache) is replaced by a slice of what it reads."""

    def __init__(self, case, gen):
        super().__init__()
        d, kv, ffn = case["width"], case["kv"], case["ffn"]
        self.q_proj = _linear(d, d, False, case, gen)
        self.k_proj = _linear(kv, d, False, case, gen)
        self.v_proj = _linear(kv, d, False, case, gen)
        self.o_proj = _linear(d, d, False, case, gen)
        self.gate_proj = _linear(ffn, d, False, case, gen)
        self.up_proj = _linear(ffn, d, False, case, gen)
        self.down_proj = _linear(d, ffn, False, case, gen)

    def forward(self, h, a, m):
        q, k, v = self.q_proj(h), self.k_proj(h), self.v_proj(h)
        o = self.o_proj(a)
        y = self.down_proj(F.silu(self.gate_proj(m)) * self.up_proj(m))
        return q, k, v, o, y


class _Gpt2(torch.nn.Module):
    """The four Linears of a GPT-2 block with its norms; attention is replaced by the values."""

    def __init__(self, case, gen):
        super().__init__()
        d = case["width"]
        self.ln1 = torch.nn.LayerNorm(d, device="cuda", dtype=torch.bfloat16)
        self.qkv = _linear(3 * d, d, True, case, gen)
        self.proj = _linear(d, d, True, case, gen)
        self.ln2 = torch.nn.LayerNorm(d, device="cuda", dtype=torch.bfloat16)
        self.fc = _linear(4 * d, d, True, case, gen)
        self.fc2 = _linear(d, 4 * d, True, case, gen)

    def forward(self, x):
        q, k, v = self.qkv(self.ln1(x)).chunk(3, dim=-1)
        x = x + self.proj(torch.sigmoid(q) * v + k)
        return x + self.fc2(F.gelu(self.fc(self.ln2(x))))


class _Rate:
    """The learning rate of a fine-tuning run, where the update hook asks for it."""

    def get_last_lr(self):
        return [1e-6]


def _rewrite_shapes(case):
    d = case["width"]
    return [(3 * d, d), (d, d), (4 * d, d), (d, 4 * d)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "read":
        st["manager"] = _manager(case)
        st["handle"] = st["manager"].write(_values(case["values"], case["rows"], case["cols"], gen))
        st["manager"].flush()
    elif kind == "encode":
        L = _lib.load()
        n = case["rows"] * case["cols"]
        chunk, lane, s = _lib.DEFAULT_CHUNK, _lib.DEFAULT_LANE_SYMS, case["precision"]
        byte = partial(torch.zeros, dtype=torch.uint8, device="cuda")
        st["dense"] = _values(case["values"], case["rows"], case["cols"], gen)
        st["packed"] = byte(max(8, L.nz_packed_stored_bytes(n, s, chunk, lane)))
        st["comp"] = byte(L.nz_exp_bound_bytes(n, chunk, lane))
        st["scratch"] = byte(L.nz_encode_workspace_bytes(n, chunk, lane))
        st["norm"] = byte(L.nz_norm_bytes(n, case["normalizer"]) + 8)
        st["total"] = torch.zeros(1, dtype=torch.int64, device="cuda")
        st["status"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "rewrite":
        st["manager"] = _manager(case)
        shapes = _rewrite_shapes(case)
        old = [_values(case["values"], r, c, gen) for r, c in shapes]
        st["handles"] = [st["manager"].write(w) for w in old]
        st["manager"].flush()
        # the step moves a weight by a thousandth of its size
        st["new"] = [(w.float() + 2e-5 * torch.randn(w.shape, device="cuda", generator=gen)).to(torch.bfloat16)
                     for w in old]
    elif kind == "block":
        st["manager"] = _manager(case)
        st["model"] = st["manager"].convert(_Gated(case, gen))
        d = case["width"]
        st["x"] = [_rows(case["tokens"], d, gen) for _ in range(3)]
    elif kind == "train":
        st["manager"] = _manager(case)
        model = st["model"] = st["manager"].convert(_Gpt2(case, gen))
        st["x"] = _rows(case["tokens"], case["width"], gen).requires_grad_(True)
        st["gy"] = _rows(case["tokens"], case["width"], gen) * 1e-3
        st["grads"] = []

        def update(p):
            st["grads"].append(p._gradient)
            neuzip_amd.compressed_lomo_hook(_Rate(), p)

        for p in model.parameters():
            if isinstance(p, neuzip_amd.nn.Parameter):
                p.register_post_accumulate_grad_hook(update)
    else:
        st["manager"] = _manager(case)
        table = torch.nn.Embedding(case["rows"], case["cols"], device="meta")
        table.weight = torch.nn.Parameter(_values(case["values"], case["rows"], case["cols"], gen))
        st["embedding"] = neuzip_amd.nn.Embedding(st["manager"], table)
        st["manager"].flush()
        st["manager"].trim()
        st["ids"] = torch.randint(0, case["rows"], (1, case["tokens"]), device="cuda", generator=gen)
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "read":
        return state["manager"].read(state["handle"])
    if kind == "encode":
        d = state["dense"]
        rc = _lib.load().nz_encode(
            d.data_ptr(), d.numel(), case["precision"], _lib.DEFAULT_CHUNK, _lib.DEFAULT_LANE_SYMS,
            state["packed"].data_ptr(), state["comp"].data_ptr(), state["comp"].numel(),
            state["scratch"].data_ptr(), state["scratch"].numel(), state["total"].data_ptr(),
            state["status"].data_ptr(), None, case["normalizer"], state["norm"].data_ptr(),
            torch.cuda.current_stream().cuda_stream)
        _lib.raise_for(rc)
        return {k: state[k] for k in ("comp", "packed", "norm", "total", "status")}
    if kind == "rewrite":
        m = state["manager"]
        m.write_many(state["new"], state["handles"])
        return [m.read(h) for h in state["handles"]]
    if kind == "block":
        with torch.no_grad():
            return state["model"](*state["x"])
    if kind == "train":
        model, x = state["model"], state["x"]
        x.grad = None
        for p in model.parameters():
            p.grad = None
        state["grads"].clear()
        y = model(x)
        y.backward(state["gy"])
        dense = [p.grad for p in model.parameters() if not isinstance(p, neuzip_amd.nn.Parameter)]
        return [y.detach(), x.grad, *dense, *state["grads"]]
    return state["embedding"](state["ids"])


def _stored(n, case):
    """Bytes of a stored weight: exponents at their entropy, sign and mantissa bits, normalizer bytes."""
    b = n * (_EXP_BYTES[case["values"]] + (case["precision"] + 1) / 8)
    return b + (n / case["normalizer"] if case["normalizer"] else 0)


def work(case):
    kind = case["kind"]
    if kind in ("read", "encode"):
        n = case["rows"] * case["cols"]
        return {"bytes": int(2 * n + _stored(n, case)), "flops": 0}
    if kind == "rewrite":
        n = sum(r * c for r, c in _rewrite_shapes(case))
        return {"bytes": int(2 * (2 * n + _stored(n, case))), "flops": 0}
    t = case["tokens"]
    if kind == "block":
        d, kv, ffn = case["width"], case["kv"], case["ffn"]
        n = 2 * d * d + 2 * kv * d + 3 * ffn * d
        return {"bytes": int(_stored(n, case) + 2 * t * (3 * d + 3 * d + 2 * kv)), "flops": 2 * n * t}
    if kind == "train":
        d = case["width"]
        n = 12 * d * d
        # weights once each way (stored bytes read and written), gradients out, activations in and out
        return {"bytes": int(2 * _stored(n, case) + 2 * n + 2 * t * 4 * d), "flops": 6 * n * t}
    n = t * case["cols"]
    return {"bytes": int(_stored(n, case) + 2 * n + 8 * t), "flops": 0}


def tolerance(case):
    if case["kind"] == "block":
        # bf16 outputs of fp32 sums in another order, measured against the product in float64:
        # 1.7e-3 of the result (2-norm) for the plain products, 3.9e-3 for the one behind the gate
        return {"rel": 1.0e-2}
    if case["kind"] == "train":
        # bf16 activations and gradients through four layers, measured against the same step
        # with float32 arithmetic: up to 4.5e-3 (the weight gradients)
        return {"rel": 1.5e-2}
    return "exact"


def _stored_values(w, precision):
    """What a bf16 weight reads back as after it was stored with `precision` mantissa bits (half-up
    rounding of the magnitude, the carry running into the exponent)."""
    if precision == 7:
        return w
    bits = w.view(torch.int16).to(torch.int32) & 0xFFFF
    mag = ((bits & 0x7FFF) + (1 << (6 - precision))) & 0x7FFF & ~((1 << (7 - precision)) - 1)
    bits = (bits & 0x8000) | mag
    return torch.where(bits >= 0x8000, bits - 0x10000, bits).to(torch.int16).view(torch.bfloat16)


def exact(case, seed):
    """The outputs of `run` on the inputs of `prepare(case, seed)` in float64; None for the kinds
    whose outputs are stored values and bytes."""
    kind = case["kind"]
    if kind not in ("block", "train"):
        return None
    gen = torch.Generator(device="cuda").manual_seed(seed)
    model = (_Gated if kind == "block" else _Gpt2)(case, gen)
    for m in model.modules():
        if isinstance(m, torch.nn.Linear):
            m.weight.data = _stored_values(m.weight.data, case["precision"])
    model = model.double()
    if kind == "block":
        x = [_rows(case["tokens"], case["width"], gen).double() for _ in range(3)]
        with torch.no_grad():
            return model(*x)
    x = _rows(case["tokens"], case["width"], gen).double().requires_grad_(True)
    gy = (_rows(case["tokens"], case["width"], gen) * 1e-3).double()
    y = model(x)
    y.backward(gy)
    weights = [model.qkv.weight, model.proj.weight, model.fc.weight, model.fc2.weight]
    dense = [p.grad for p in model.parameters() if not any(p is w for w in weights)]
    # the compressed weights' gradients come in the order of the backward pass
    return [y.detach(), x.grad, *dense, *[w.grad for w in reversed(weights)]]
