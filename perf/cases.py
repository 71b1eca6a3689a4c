"""The work that programs have this framework do, as cases that can be timed and compared.

One case is one call (or the two or three calls that always go together) through the
public Python entry points:

    step      AttentionBlock.step: one decode token per sequence from the wire (rotate,
              append, attend); the state is a cache that already holds `ctx - 1` tokens
    attend    CompressedAttention.attend: one query per sequence over a batch of caches of
              ragged lengths, the attend of a batched decode
    prefill   AttentionBlock.prefill: a prompt into an empty cache (rotate, append, attend
              every query causally)
    extend    CompressedAttention.attend_prefill: the queries of the last `n` of `ctx`
              cached tokens (a prompt that continues a cached conversation)
    append    CompressedCache.append_wire: a prompt's k/v rows into the next sequence of a
              batch (rotate, encode, pack, write), with no attend
    block     AttentionBlock.forward: hidden states in, hidden states out, behind `ctx`
              cached tokens (fp16 projections, RoPE, the cast, the seam, W_o')
    project   HostHalf.project_qkv and HostHalf.output: the block's projections alone

The shapes are the repository's: 32 query heads of 64 over 8 KV heads (4-bit keys and
2-bit values), the same over 4 KV heads with 3-bit keys (QuantConfig's default), and 32 heads
of 128 over 8 KV heads with 3-bit keys and values. Inputs are N(0, 1) in Q8.16 with outlier
channels, as insitu_amd.workload draws them; `scaled` cases multiply the queries by
1/sqrt(d) as the seam of a model does (a flat softmax: most cached tokens carry weight),
the others leave them as the benchmark configurations do (a peaked softmax).
"""

import ctypes
import math

import numpy as np
import torch

from insitu_amd import AttentionBlock, CompressedAttention, CompressedCache, ModelConfig, QuantConfig, Weights, _lib
from insitu_amd.runtime import default_context

N_Q = 32                     # query heads of every shape
WINDOW = 64                  # decode tokens a step or block state holds before it rewinds its cache
SLOTS = 8                    # sequences an append state fills before it empties its cache

# (head_dim, KV heads, key bits, value bits) that the repository's configurations and tests run
SHAPES = [(64, 8, 4, 2), (64, 4, 3, 2), (128, 8, 3, 3), (64, 8, 3, 2), (128, 8, 4, 2)]


def _case(kind, shape=(64, 8, 4, 2), *, ctx=0, n=1, batch=1, mode="online", scaled=True, name=None):
    d, n_kv, kb, vb = shape
    c = {"kind": kind, "d": d, "n_kv": n_kv, "key_bits": kb, "value_bits": vb, "ctx": ctx, "n": n,
         "batch": batch, "mode": mode, "scaled": scaled}
    return {"name": name, **c} if name else c


def listed():
    small, tiny, wide = SHAPES[0], SHAPES[1], SHAPES[2]
    return [
        # the first tokens of an answer to a short question: latency and launches
        _case("step", small, ctx=100, name="step_ctx100"),
        # the benchmark's headline step: one long sequence, peaked softmax
        _case("step", small, ctx=32768, scaled=False, name="step_ctx32768"),
        # a decode token as the model adapter runs it by default (two-pass softmax)
        _case("step", small, ctx=4097, mode="two_pass", name="step_two_pass_ctx4097"),
        # 8 query heads to a KV head with the default 3-bit keys
        _case("step", tiny, ctx=2047, name="step_group8_ctx2047"),
        # a serving batch of 64 ragged sequences, one launch
        _case("attend", small, ctx=8192, batch=64, scaled=False, name="attend_batch64_ragged"),
        # the larger heads at the longest context, one layer of a batch of 16
        _case("attend", wide, ctx=131072, batch=16, scaled=False, name="attend_d128_batch16_ctx131072"),
        # a long prompt into an empty cache
        _case("prefill", small, n=4096, name="prefill_4096"),
        # an ordinary prompt, the larger heads, two-pass softmax
        _case("prefill", wide, n=1000, mode="two_pass", name="prefill_d128_two_pass_1000"),
        # a prompt's rows alone (a cache filled for later use)
        _case("append", small, n=32767, name="append_32767"),
        # one decode token through a whole block at a long context
        _case("block", small, ctx=32768, name="block_token_ctx32768"),
        # the next turn of a conversation through a whole block
        _case("block", small, ctx=2000, n=333, name="block_turn_333"),
        # the projections of an ordinary prompt
        _case("project", small, n=512, name="project_512"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "attend", "attend", "prefill", "prefill", "extend", "append",
                       "block", "project"])
    shape = rng.choice(SHAPES)
    mode = rng.choice(["online", "online", "two_pass"])
    scaled = rng.random() < 0.6
    if kind == "step":
        return _case(kind, shape, ctx=_log(rng, 1, 65536), batch=rng.choice([1, 1, 1, 2, 5]), mode=mode, scaled=scaled)
    if kind == "attend":
        ctx = _log(rng, 64, 131072)
        return _case(kind, shape, ctx=ctx, batch=_log(rng, 1, min(64, (1 << 20) // ctx)), mode=mode, scaled=scaled)
    # a prompt's work grows with its square: the wider heads stop earlier
    if kind == "prefill":
        return _case(kind, shape, n=_log(rng, 2, 4096 if shape[0] == 64 else 2048), mode=mode, scaled=scaled)
    if kind == "extend":
        n = _log(rng, 1, 512)
        return _case(kind, shape, ctx=n + _log(rng, 1, 12288 if shape[0] == 64 else 6144), n=n, mode=mode, scaled=scaled)
    if kind == "append":
        return _case(kind, shape, n=_log(rng, 1, 32767))
    if kind == "block":
        n = rng.choice([1, 1, _log(rng, 2, 512)])
        return _case(kind, shape, ctx=_log(rng, 1, 32768 if n == 1 else 8192) + n, n=n, mode=mode)
    return _case(kind, shape, n=_log(rng, 1, 2048))


def _lengths(case):
    """The lengths of an attend case's sequences: ctx / 8 to ctx, the longest in full; one
    sequence, or a batch at the longest context of all, is not ragged."""
    b, ctx = case["batch"], case["ctx"]
    if b == 1 or ctx >= 131072:
        return [ctx] * b
    lens = np.random.default_rng(3).integers(max(1, ctx // 8), ctx + 1, size=b)
    lens[b // 2] = ctx
    return [int(x) for x in lens]


class _Draw:
    """Wire rows of the seam: N(0, 1) with outlier channels, in Q8.16 (24 bits), made on the GPU."""

    def __init__(self, case, seed):
        self.case = case
        self.dev = default_context(0).torch_device
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        host = torch.Generator().manual_seed(seed)
        self.k_scale, self.v_scale, self.q_scale = (self._outliers(h, host) for h in (case["n_kv"], case["n_kv"], N_Q))
        if case["scaled"]:
            self.q_scale = self.q_scale / math.sqrt(case["d"])

    def _outliers(self, heads, host):
        d = self.case["d"]
        s = torch.ones(heads, d)
        if d == 64:            # four channels of each head, x8
            at = torch.stack([torch.randperm(d, generator=host)[:4] for _ in range(heads)])
            s.scatter_(1, at, 8.0)
        else:                  # one channel in a hundred, x16
            s[torch.rand(heads, d, generator=host) < 0.01] = 16.0
        return s.to(self.dev)

    def _rows(self, n, scale):
        x = torch.randn((n, *scale.shape), generator=self.gen, device=self.dev) * scale
        return torch.round(x * 65536.0).clamp_(-(1 << 23), (1 << 23) - 1).to(torch.int32)

    def kv(self, n):
        return self._rows(n, self.k_scale), self._rows(n, self.v_scale)

    def q(self, n):
        return self._rows(n, self.q_scale)

    def fill(self, cache, seq, n):
        """n tokens of k/v into sequence seq."""
        for t0 in range(0, n, 16384):
            k, v = self.kv(min(16384, n - t0))
            cache.append_wire(k, v, seq=seq)


def _model(case):
    return ModelConfig(hidden_size=N_Q * case["d"], num_heads=N_Q, num_kv_heads=case["n_kv"], head_dim=case["d"],
                       rope_theta=500000.0, max_position=65536)


def _quant(case):
    return QuantConfig(key_bits=case["key_bits"], value_bits=case["value_bits"])


class _Planes:
    """A cache's device memory as an array: the rows that a call leaves behind."""

    def __init__(self, cache):
        lay = _lib.Layout()
        _lib.check(cache.ctx.lib.insitu_cache_layout(cache.handle, ctypes.byref(lay)))
        self.cache = cache
        self.__cuda_array_interface__ = {"shape": (int(lay.total_bytes),), "typestr": "|u1", "version": 3,
                                         "data": (int(lay.device_base), False)}

    @staticmethod
    def of(cache):
        return torch.as_tensor(_Planes(cache), device=cache.ctx.torch_device)


def prepare(case, seed):
    kind, n, ctx, batch = case["kind"], case["n"], case["ctx"], case["batch"]
    make = _Draw(case, seed)
    s = {"kind": kind, "case": case, "at": 0}
    if kind in ("step", "prefill", "block"):
        room = {"step": ctx + WINDOW, "prefill": n, "block": ctx + (WINDOW if n == 1 else 0)}[kind]
        s["block"] = blk = AttentionBlock(_model(case), _quant(case), capacity=room, batch=batch, softmax=case["mode"])
        s["base"] = base = {"step": ctx - 1, "prefill": 0, "block": ctx - n}[kind]
        for b in range(batch):
            make.fill(blk.cache, b, base)
    if kind == "step":
        s["q"] = make.q(batch * WINDOW).reshape(WINDOW, batch, N_Q, case["d"])
        k, v = make.kv(batch * WINDOW)
        s["k"], s["v"] = (x.reshape(WINDOW, batch, case["n_kv"], case["d"]) for x in (k, v))
        s["planes"] = _Planes.of(blk.cache)
    elif kind == "prefill":
        s["q"], (s["k"], s["v"]) = make.q(n), make.kv(n)
        s["planes"] = _Planes.of(blk.cache)
    elif kind == "block":
        blk.weights = Weights.random(blk.model, blk.rotation, seed=seed)
        blk.host                            # the projections' weights and the RoPE tables on the device
        s["planes"] = _Planes.of(blk.cache)
        s["x"] = torch.randn((WINDOW if n == 1 else n, blk.model.hidden_size), generator=make.gen, device=make.dev)
    elif kind in ("attend", "extend"):
        lens = _lengths(case) if kind == "attend" else [ctx]
        s["cache"] = cache = CompressedCache(case["n_kv"], case["d"], max(lens), _quant(case), batch=len(lens), n_q_heads=N_Q)
        for b, length in enumerate(lens):
            make.fill(cache, b, length)
        s["attn"] = CompressedAttention(cache)
        s["q"] = cache.rotation.apply(make.q(batch if kind == "attend" else n))
    elif kind == "append":
        s["cache"] = CompressedCache(case["n_kv"], case["d"], n, _quant(case), batch=SLOTS, n_q_heads=N_Q)
        s["k"], s["v"] = make.kv(n)
        s["planes"] = _Planes.of(s["cache"])
    else:
        blk = AttentionBlock(_model(case), _quant(case), capacity=16)
        blk.weights = Weights.random(blk.model, blk.rotation, seed=seed)
        s["host"] = blk.host
        s["x"] = torch.randn((n, blk.model.hidden_size), generator=make.gen, device=make.dev)
        # attention outputs: averages of unit values, smaller than the values themselves
        s["out"] = torch.round(torch.randn((n, N_Q * case["d"]), generator=make.gen, device=make.dev)
                               * (0.1 * 65536)).to(torch.int32)
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "step" or kind == "block" and case["n"] == 1:
        blk, t = s["block"], s["at"]
        if t == WINDOW:                     # the state's tokens are used up: back to where it began
            for b in range(case["batch"]):
                blk.cache.set_length(s["base"], b)
            t = 0
        s["at"] = t + 1
        if kind == "step":
            return {"out": blk.step(s["q"][t], s["k"][t], s["v"][t], stats=False), "cache": s["planes"]}
        return {"y": blk.forward(s["x"][t], stats=False)[0], "cache": s["planes"]}
    if kind == "block":
        if s["at"]:
            s["block"].cache.set_length(s["base"])
        s["at"] = 1
        # with its report, as the model adapter calls it
        return {"y": s["block"].forward(s["x"])[0], "cache": s["planes"]}
    if kind == "prefill":
        if s["at"]:
            s["block"].reset()
        s["at"] = 1
        return {"out": s["block"].prefill(s["q"], s["k"], s["v"], stats=False), "cache": s["planes"]}
    if kind == "attend":
        return {"out": s["attn"].attend(s["q"], case["mode"], stats=False)[0]}
    if kind == "extend":
        return {"out": s["attn"].attend_prefill(s["q"], case["ctx"] - case["n"], case["mode"], stats=False)[0]}
    if kind == "append":
        if s["at"] == SLOTS:
            s["cache"].reset()
            s["at"] = 0
        s["cache"].append_wire(s["k"], s["v"], seq=s["at"])
        s["at"] += 1
        return {"cache": s["planes"]}
    return {"qkv": s["host"].project_qkv(s["x"]), "y": s["host"].output(s["out"])}


def work(case):
    """The rows and weights read once, the inputs in and the outputs out; 2 operations for each
    (query, row, channel) of the scores and of the values, and for each weight a token meets."""
    kind, d, n, ctx, batch, n_kv = (case[k] for k in ("kind", "d", "n", "ctx", "batch", "n_kv"))
    row = n_kv * (d * (case["key_bits"] + case["value_bits"]) // 8 + 4)      # one token, every KV head
    wire = 4 * d * (N_Q + 2 * n_kv)
    out = 4 * d * N_Q
    attend = 4 * d * N_Q                                                    # per (token, query)
    hidden = N_Q * d
    weights = 2 * hidden * (N_Q * d + 2 * n_kv * d) + 2 * hidden * N_Q * d
    if kind == "step":
        return {"bytes": batch * (row * ctx + wire + out), "flops": batch * attend * ctx}
    if kind == "attend":
        t = sum(_lengths(case))
        return {"bytes": row * t + batch * 2 * out, "flops": attend * t}
    if kind == "prefill":
        return {"bytes": n * (row + wire + out), "flops": attend * n * (n + 1) // 2}
    if kind == "extend":
        return {"bytes": row * ctx + 2 * n * out, "flops": attend * (n * (ctx - n) + n * (n + 1) // 2)}
    if kind == "append":
        return {"bytes": n * (8 * d * n_kv + row), "flops": 2 * n * n_kv * d * 6}
    if kind == "block":
        return {"bytes": weights + row * ctx + 8 * hidden * n,
                "flops": weights * n + attend * (n * (ctx - n) + n * (n + 1) // 2)}
    return {"bytes": weights + n * (4 * hidden + 4 * d * (N_Q + 2 * n_kv) + out + 4 * hidden), "flops": weights * n}


def tolerance(case):
    """Below the seam every output is an integer or a byte that the reference's recurrence fixes.
    The projections are fp32 sums of fp16 products. A block's wire rows are those sums rounded to
    Q8.16, so that another order of them moves a wire value by one or two of its last places, and
    now and then a code or a probability with it. Four times what was measured: the projections
    are 2.9e-7 from their 64-bit values; a block whose projections are summed in 64 bits is
    1.4e-4 from one that sums them in fp32 (largest 2.9e-3), with few of its rows' bytes."""
    if case["kind"] == "project":
        return {"rel": 1.2e-6, "max": 2e-5}
    if case["kind"] == "block":
        return {"rel": 6e-4, "max": 0.012, "differ": 0.002}
    return "exact"


def exact(case, seed):
    """The projections in 64 bits (fp16 inputs and weights, as the block holds them). The other
    outputs are integers, or (a block's y) follow from rounded integers: they have no 64-bit value."""
    if case["kind"] != "project":
        return None
    s = prepare(case, seed)
    w = s["host"].weights

    def product(x, weight):
        half = weight.view(torch.float16).to(torch.float64)
        return x.to(torch.float32).to(torch.float16).to(torch.float64) @ half.T

    return {"qkv": product(s["x"], w.qkv), "y": product(s["out"].to(torch.float64) / 65536.0, w.o)}
