"""The workloads this framework's speed is judged by, as data and plain functions.

Three families, each through public entry points:

  product    one weight matrix times 1..64 activation vectors (aotk_matvec /
             aotk_matmul over device pointers, include/aotk.h): the projections
             of a layer, one vector per decode step and up to 64 per prompt
             chunk, in every weight format that models are stored in;
  attention  aotk_attention: one decode row or up to 64 prompt rows against the
             KV cache, grouped heads, with and without a sliding window;
  model      Model / State: a prompt evaluated in 64-token chunks and / or
             tokens generated, from position 0 or behind a filled KV cache,
             logits and tokens returned.

The library's contract is that its results are the bits of one sequential
float32 definition (the order of every sum is part of it), and its own tests
compare bits. So every tolerance is "exact".
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "aot-llm_amd")  # run from the repository's root
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import aotk  # noqa: E402
from aotk import abi, configs  # noqa: E402

CHUNK = 64  # prompt tokens per forward_batch call, State.prompt's default


# ------------------------------------------------------------------- cases
def _product(name, kind, rows, cols, m):
    return {"name": name, "family": "product", "kind": kind, "rows": rows, "cols": cols, "m": m}


def _attention(name, n_head, n_kv_head, head_dim, pos0, m, window):
    return {"name": name, "family": "attention", "n_head": n_head, "n_kv_head": n_kv_head, "head_dim": head_dim,
            "pos0": pos0, "m": m, "window": window}


def _model(name, config, past, prompt, gen):
    return {"name": name, "family": "model", "config": config, "past": past, "prompt": prompt, "gen": gen}


def listed():
    return [
        # A short chat turn on the smallest model: 6 prompt tokens, 32 greedy
        # tokens. Launch- and latency-bound.
        _model("tinyllama_6_prompt_32_greedy", "tinyllama-1.1b-q4km", 0, 6, 32),
        # Decoding an 8B model behind a 512-token prompt: 16 steps of the token loop.
        _model("llama3_8b_decode_at_512", "llama3-8b-q4km", 512, 1, 17),
        # Reading a 512-token prompt with the 8B model.
        _model("llama3_8b_prompt_512", "llama3-8b-q4km", 0, 512, 0),
        # The FFN up / gate projection of one decode step, the most common format.
        _product("matvec_q4_k_14336x4096", "q4_k", 14336, 4096, 1),
        # The FFN down projection of one decode step of an 8-bit model.
        _product("matvec_q8_0_4096x12288", "q8_0", 4096, 12288, 1),
        # The FFN down projection over a full prompt chunk, K-quants.
        _product("matmul_q6_k_4096x14336_m64", "q6_k", 4096, 14336, 64),
        # The FFN up projection over a full prompt chunk, 8-bit.
        _product("matmul_q8_0_12288x4096_m64", "q8_0", 12288, 4096, 64),
        # A projection of an unquantized model over a ragged last chunk.
        _product("matmul_f16_4096x4096_m37", "f16", 4096, 4096, 37),
        # A small model's FFN over a 6-token prompt.
        _product("matmul_q5_0_5632x2048_m6", "q5_0", 5632, 2048, 6),
        # One decode row over a long history (32 query heads on 8 kv heads).
        _attention("attention_decode_at_4100", 32, 8, 128, 4100, 1, 0),
        # The last chunk of a 4096-token prompt.
        _attention("attention_prompt_64_at_4032", 32, 8, 128, 4032, 64, 0),
        # A ragged chunk through a local layer: 1024-position window, head_dim 256.
        _attention("attention_window_1024_50_at_3001", 8, 4, 256, 3001, 50, 1024),
    ]


_KINDS = ("q4_k", "q5_k", "q6_k", "q8_0", "q4_0", "q5_0", "f16", "bf16")
# (query heads, kv heads, head_dim, window of local layers) of the configurations
_HEADS = ((32, 4, 64, 0), (32, 8, 128, 0), (8, 4, 256, 0), (8, 4, 256, 1024))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng):
    """Rows of a call: a decode step, a short or ragged chunk, a full chunk."""
    u = rng.random()
    return 1 if u < 0.35 else CHUNK if u < 0.6 else _log(rng, 2, CHUNK)


def draw(rng):
    """One more case of the listed ranges. Rows are any number (odd ones
    included), columns whole 256-value blocks as every model here has them."""
    u = rng.random()
    if u < 0.55:
        kind = rng.choice(_KINDS)
        cols = 256 * _log(rng, 4, 56)
        rows = _log(rng, 512, 16384)
        while rows * cols > 14336 * 4096:
            rows //= 2
        return {k: v for k, v in _product("", kind, rows, cols, _batch(rng)).items() if k != "name"}
    if u < 0.85:
        nh, nkv, hd, window = rng.choice(_HEADS)
        return {k: v for k, v in _attention("", nh, nkv, hd, _log(rng, 16, 8000), _batch(rng), window).items()
                if k != "name"}
    config = rng.choice(sorted(configs.CONFIGS))
    past = rng.choice((0, _log(rng, 32, 2048)))
    prompt, gen = (_log(rng, 2, 128), 0) if rng.random() < 0.5 else (_log(rng, 1, 48), _log(rng, 2, 8))
    return {k: v for k, v in _model("", config, past, prompt, gen).items() if k != "name"}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _put_f16(raw, at, value):
    raw[:, at:at + 2] = value.to(torch.float16).view(torch.uint8).view(-1, 2)


def _weight_bytes(kind, rows, cols, g):
    """A matrix in the stored format: weights of about N(0, 0.02)'s size."""
    if kind in (abi.F16, abi.BF16):
        w = torch.randn(rows, cols, generator=g, device="cuda") * 0.02
        return w.to(torch.float16 if kind == abi.F16 else torch.bfloat16).view(torch.uint8).reshape(-1)
    nb = rows * cols // abi.BLOCK[kind]
    raw = torch.randint(0, 256, (nb, abi.TYPE_SIZE[kind]), generator=g, device="cuda", dtype=torch.uint8)
    s = 0.75 + 0.5 * torch.rand(nb, generator=g, device="cuda")  # block scales differ
    if kind == abi.Q8_0:
        _put_f16(raw, 0, s * 2.7e-4)
    elif kind == abi.Q4_0:
        _put_f16(raw, 0, s * 4.3e-3)
    elif kind == abi.Q5_0:
        _put_f16(raw, 0, s * 2.2e-3)
    elif kind in (abi.Q4_K, abi.Q5_K):
        levels = 15 if kind == abi.Q4_K else 31
        _put_f16(raw, 0, s * (0.06 / 31.5 / levels * 2))
        _put_f16(raw, 2, s * (0.06 / 31.5))
    else:
        _put_f16(raw, 208, s * 1.5e-5)
    return raw.reshape(-1)


def _act_blocks(kind, m, cols, g):
    """m activation vectors as the kernels' input blocks (f32 for float
    matrices): the values of a normed hidden state."""
    x = torch.randn(m, cols, generator=g, device="cuda")
    a = abi.activation(kind)
    if a == 0:
        return x
    n = 32 if a == 1 else 256
    b = x.view(-1, n)
    d = (b.abs().amax(1, keepdim=True) / 127).clamp_min(1e-12)
    q = torch.round(b / d).to(torch.int8)
    parts = [d.view(torch.uint8), q.view(torch.uint8)]
    if a == 2:
        sums = q.view(-1, 16, 16).sum(2, dtype=torch.int32).to(torch.int16)
        parts.append(sums.view(torch.uint8).view(-1, 32))
    return torch.cat(parts, 1).contiguous()


def _product_inputs(case, seed):
    g = _gen(seed)
    kind = abi.KIND_BY_NAME[case["kind"]]
    raw = _weight_bytes(kind, case["rows"], case["cols"], g)
    return kind, raw, _act_blocks(kind, case["m"], case["cols"], g)


def _attention_inputs(case, seed):
    g = _gen(seed)
    nh, nkv, hd = case["n_head"], case["n_kv_head"], case["head_dim"]
    ctx = case["pos0"] + case["m"]
    # queries somewhat larger than the keys, so that the softmax has peaks
    q = torch.randn(case["m"], nh, hd, generator=g, device="cuda") * 1.5
    k = torch.randn(ctx, nkv, hd, generator=g, device="cuda")
    v = torch.randn(ctx, nkv, hd, generator=g, device="cuda")
    return ctx, q, k, v


def prepare(case, seed):
    aotk.init(0)
    lib = abi.load()
    if case["family"] == "product":
        kind, raw, x = _product_inputs(case, seed)
        torch.cuda.synchronize()
        w = abi.check_ptr(lib.aotk_weight_from_dev(kind, raw.data_ptr(), case["rows"], case["cols"]))
        out = torch.empty(case["m"], case["rows"], device="cuda")
        torch.cuda.synchronize()
        return _Product(lib, w, x, case["m"], out)
    if case["family"] == "attention":
        ctx, q, k, v = _attention_inputs(case, seed)
        out = torch.empty_like(q)
        torch.cuda.synchronize()
        return _Attention(lib, case, ctx, q, k, v, out)
    return _ModelRun(case, seed)


class _Product:
    """A weight handle, the input blocks and the output buffer."""

    def __init__(self, lib, w, x, m, out):
        self.lib, self.w, self.x, self.m, self.out = lib, w, x, m, out

    def run(self):
        if self.m == 1:
            abi.check(self.lib.aotk_matvec(self.w, self.x.data_ptr(), self.out.data_ptr()))
        else:
            abi.check(self.lib.aotk_matmul(self.w, self.x.data_ptr(), self.m, self.out.data_ptr()))
        return self.out

    def __del__(self):
        self.lib.aotk_weight_free(self.w)


class _Attention:
    def __init__(self, lib, case, ctx, q, k, v, out):
        self.lib, self.q, self.k, self.v, self.out = lib, q, k, v, out
        self.dims = (case["n_head"], case["n_kv_head"], case["head_dim"], ctx, 0, case["pos0"], case["m"], case["window"])

    def run(self):
        abi.check(self.lib.aotk_attention(self.out.data_ptr(), self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(),
                                          *self.dims))
        return self.out


class _ModelRun:
    """A model and one sequence's state: `past` positions already in the KV
    cache, then the prompt, then greedy tokens."""

    def __init__(self, case, seed):
        spec = configs.build(case["config"])
        d = spec.d
        self.past, self.gen = case["past"], case["gen"]
        self.tokens = configs.prompt_tokens(seed, case["prompt"], d["vocab"])
        self.model = aotk.Model(spec, seed=int(seed) & 0x7FFFFFFFFFFFFFFF)
        ctx = 64 * ((self.past + case["prompt"] + self.gen + 63) // 64)
        self.state = aotk.State(self.model, ctx, CHUNK)
        if self.past:
            g = _gen(seed)
            n = d["n_layer"] * self.past * d["n_kv_head"] * d["head_dim"]
            k = torch.randn(n, generator=g, device="cuda").cpu().numpy()
            v = torch.randn(n, generator=g, device="cuda").mul_(0.5).cpu().numpy()
            self.state.kv_upload(self.past, k, v)
        torch.cuda.synchronize()

    def run(self):
        st, n = self.state, len(self.tokens)
        if self.past == 0:
            st.prompt(self.tokens, batch=CHUNK)
        else:
            for i in range(0, n, CHUNK):
                part, last = self.tokens[i:i + CHUNK], i + CHUNK >= n
                if len(part) == 1:
                    st.forward(part[0], self.past + i, last)
                else:
                    st.forward_batch(part, self.past + i, last)
        out = {}
        if self.gen:
            out["tokens"] = np.asarray(st.generate(self.past + n, self.gen), np.uint32)
        out["logits"] = st.logits()
        return out

    def __del__(self):
        self.state.free()
        self.model.free()


def run(state):
    return state.run()


# -------------------------------------------------------------------- work
def _span_rows(pos0, m, window):
    """Attended positions summed over the rows, and the first one of all."""
    total = sum(min(p + 1, window) if window else p + 1 for p in range(pos0, pos0 + m))
    first = max(0, pos0 + 1 - window) if window else 0
    return total, first


def work(case):
    if case["family"] == "product":
        kind = abi.KIND_BY_NAME[case["kind"]]
        rows, cols, m = case["rows"], case["cols"], case["m"]
        return {"bytes": rows * abi.row_bytes(kind, cols) + m * abi.act_bytes(kind, cols) + 4 * m * rows,
                "flops": 2 * m * rows * cols}
    if case["family"] == "attention":
        nh, nkv, hd, m = case["n_head"], case["n_kv_head"], case["head_dim"], case["m"]
        total, first = _span_rows(case["pos0"], m, case["window"])
        return {"bytes": 8 * (case["pos0"] + m - first) * nkv * hd + 8 * m * nh * hd, "flops": 4 * total * nh * hd}
    spec = configs.build(case["config"])
    d = spec.d
    steps = max(0, case["gen"] - 1)
    head = spec.out_tensor.len
    layers = spec.decode_weight_bytes() - head
    per_token = 0
    for li in range(d["n_layer"]):
        L = spec.layers[li]
        per_token += 2 * sum(getattr(L, s).rows * getattr(L, s).cols for s in ("wq", "wk", "wv", "wo", "gate", "up", "down"))
    flops = (case["prompt"] + steps) * per_token + (1 + steps) * 2 * d["vocab"] * d["dim"]
    # the prompt's weights once, each later token's again: it needs the one before
    bytes_ = (1 + steps) * (layers + head) + 4 * d["vocab"]
    for li in range(d["n_layer"]):
        w = spec.cfg.get("swa_window", 0) if spec.layers[li].local_attn else 0
        total, first = _span_rows(case["past"], case["prompt"] + steps, w)
        flops += 4 * total * d["n_head"] * d["head_dim"]
        kv = 8 * d["n_kv_head"] * d["head_dim"]
        bytes_ += kv * (case["past"] + case["prompt"] - first)
        for s in range(steps):
            bytes_ += kv * _span_rows(case["past"] + case["prompt"] + s, 1, w)[0]
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------- exact
def _f16_at(raw, at):
    return raw[:, at:at + 2].contiguous().view(torch.float16).double()


def _low_high(b):
    return torch.cat([b & 15, b >> 4], -1).double()


def _decode(kind, raw, rows, cols):
    """The stored format's weights in 64 bits."""
    if kind in (abi.F16, abi.BF16):
        return raw.view(torch.float16 if kind == abi.F16 else torch.bfloat16).view(rows, cols).double()
    raw = raw.view(-1, abi.TYPE_SIZE[kind])
    if kind == abi.Q8_0:
        w = _f16_at(raw, 0) * raw[:, 2:].view(torch.int8).double()
    elif kind == abi.Q4_0:
        w = _f16_at(raw, 0) * (_low_high(raw[:, 2:]) - 8)
    elif kind == abi.Q5_0:
        bits = torch.arange(8, device=raw.device, dtype=torch.uint8)
        hi = ((raw[:, 2:6, None] >> bits) & 1).reshape(-1, 32).double()
        w = _f16_at(raw, 0) * (_low_high(raw[:, 6:]) + 16 * hi - 16)
    elif kind in (abi.Q4_K, abi.Q5_K):
        d, dmin, s = _f16_at(raw, 0), _f16_at(raw, 2), raw[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = raw[:, 16:] if kind == abi.Q4_K else raw[:, 48:]
        q = _low_high(qs.reshape(-1, 4, 32)).view(-1, 8, 32)
        if kind == abi.Q5_K:
            bits = torch.arange(8, device=raw.device, dtype=torch.uint8)[None, :, None]
            q = q + 16 * ((raw[:, None, 16:48] >> bits) & 1).double()
        w = (d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]
    else:  # Q6_K: per half of 128 values, 64 bytes of low and 32 bytes of high bits
        d = _f16_at(raw, 208)
        lo, hi = raw[:, :128].view(-1, 2, 64), raw[:, 128:192].view(-1, 2, 32)
        low = torch.cat([lo & 15, lo >> 4], 2).view(-1, 2, 4, 32)
        high = torch.stack([(hi >> (2 * i)) & 3 for i in range(4)], 2)
        q = (low + 16 * high).double().view(-1, 16, 16) - 32
        w = d[:, :, None] * raw[:, 192:208].view(torch.int8).double()[:, :, None] * q
    return w.reshape(rows, cols)


def _decode_act(kind, x, m, cols):
    a = abi.activation(kind)
    if a == 0:
        return x.double()
    n = 32 if a == 1 else 256
    d = x[:, :4].contiguous().view(torch.float32).double()
    return (d * x[:, 4:4 + n].contiguous().view(torch.int8).double()).view(m, cols)


def exact(case, seed):
    if case["family"] == "product":
        kind, raw, x = _product_inputs(case, seed)
        xs = _decode_act(kind, x, case["m"], case["cols"])
        return xs @ _decode(kind, raw, case["rows"], case["cols"]).t().contiguous()
    if case["family"] == "attention":
        ctx, q, k, v = _attention_inputs(case, seed)
        m, group = case["m"], case["n_head"] // case["n_kv_head"]
        row = torch.arange(case["pos0"], case["pos0"] + m, device="cuda")[:, None]
        col = torch.arange(ctx, device="cuda")[None, :]
        hidden = col > row
        if case["window"]:
            hidden |= col + case["window"] <= row
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        for h in range(case["n_head"]):
            kh, vh = k[:, h // group].double(), v[:, h // group].double()
            s = (q[:, h].double() @ kh.t().contiguous()) / math.sqrt(case["head_dim"])
            out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), 1) @ vh
        return out
    return None  # a whole model in 64 bits takes minutes
