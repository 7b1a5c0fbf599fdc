"""Performance cases: the linear layers a Tomoul model runs through this backend.

A case is a dict of plain values; `kind` says which public entry point it
takes:

  linear   one product on resident operands, _abi.gemm_ex_dev (any weight format,
           bias, activation, residual): a GEMM past 8 rows, the [K,N] GEMV below
  layer    the four linears of one encoder layer on resident operands: fused QKV,
           out-projection + residual, FFN up + GELU, FFN down + residual (the
           FFN's second product reads the first one's output)
  decode   one decoder step's product on a prepared weight, _abi.gemm_prepared_ex
  vocab    the tied vocabulary projection on the stored embedding
           (_abi.prepare_rows_dev, then _abi.gemm_prepared)
  host     dispatch.matmulWithWeightBias on host tensors with a registered
           weight, as a drop-in caller uses the library

Sizes are the encoder, decoder and sentence-embedding shapes of bench.py and the
tests (Whisper tiny and large-v3-turbo, XLM-RoBERTa-large, the 384-wide
sentence transformer) and generic ones in between; drawn cases spread M, N, K,
format and epilogue over the same ranges, ragged sizes among them.
"""
import math

import numpy as np
import torch

from tomoul_amd import _abi, dispatch
from tomoul_amd.tensor import Tensor

FMT = {"f32": _abi.FMT_F32, "q8": _abi.FMT_Q8_0, "q4": _abi.FMT_Q4_0, "q8k": _abi.FMT_Q8_K, "f16": _abi.FMT_F16,
       "q8pc": _abi.FMT_Q8_0_PC}
ACT = {"none": _abi.ACT_NONE, "gelu_erf": _abi.ACT_GELU_ERF, "gelu_tanh": _abi.ACT_GELU_TANH}
FLOPS_MOST = 60.0e9  # a drawn case's work stays below the largest listed one's


def listed():
    return [
        # One decoder step of one linear, int8 weight: the smallest call, latency alone.
        dict(name="decode_q8_m1", kind="decode", fmt="q8", m=1, n=4096, k=1024, act="none", bias=False, res=False),
        # The turbo decoder's FFN down-projection, four beams, int4 weight, with its residual connection.
        dict(name="decode_q4_m4", kind="decode", fmt="q4", m=4, n=1280, k=5120, act="none", bias=True, res=True),
        # The same decoder's FFN up-projection for eight beams on a weight that was not prepared.
        dict(name="decode_kn_q4_m8", kind="linear", fmt="q4", m=8, n=5120, k=1280, act="gelu_erf", bias=True, res=False),
        # The vocabulary projection of one decode step on the stored fp32 embedding.
        dict(name="vocab_f32_m1", kind="vocab", fmt="f32", m=1, n=51866, k=1280, act="none", bias=False, res=False),
        # Whisper-tiny encoder MLP, 30 s of audio, fp32.
        dict(name="tiny_mlp_f32", kind="linear", fmt="f32", m=1500, n=1536, k=384, act="gelu_erf", bias=True, res=False),
        # XLM-RoBERTa-large encoder layer at 512 tokens, fp32.
        dict(name="xlmr_layer_f32", kind="layer", fmt="f32", m=512, d=1024, ff=4096, act="gelu_tanh"),
        # Whisper large-v3-turbo encoder layer at 1500 frames, fp32.
        dict(name="turbo_layer_f32", kind="layer", fmt="f32", m=1500, d=1280, ff=5120, act="gelu_erf"),
        # The same layer with int8 weights.
        dict(name="turbo_layer_q8", kind="layer", fmt="q8", m=1500, d=1280, ff=5120, act="gelu_erf"),
        # A 128-token prompt through an int8 FFN up-projection.
        dict(name="prompt_q8_m128", kind="linear", fmt="q8", m=128, n=4096, k=1024, act="none", bias=True, res=False),
        # Sentence-transformer layer with f16 weights on a batch whose tokens fill no whole tile.
        dict(name="sentence_layer_f16", kind="layer", fmt="f16", m=391, d=384, ff=1536, act="gelu_tanh"),
        # The same encoder with 32-block int8 weights (Q8_K), 512 tokens.
        dict(name="sentence_layer_q8k", kind="layer", fmt="q8k", m=512, d=384, ff=1536, act="gelu_tanh"),
        # A drop-in caller: host tensors in and out, the weight registered once.
        dict(name="host_mlp_f32", kind="host", fmt="f32", m=1500, n=1536, k=384, act="none", bias=True, res=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["linear", "layer", "decode", "kn", "vocab", "host"], [36, 24, 18, 8, 7, 7])[0]
    if kind == "layer":
        while True:
            d = 64 * _log_int(rng, 6, 24)
            c = dict(kind="layer", fmt=rng.choice(["f32", "f32", "q8", "q4", "f16", "q8k"]), m=_log_int(rng, 40, 3000),
                     d=d, ff=4 * d, act=rng.choice(["gelu_erf", "gelu_tanh"]))
            if work(c)["flops"] <= FLOPS_MOST:
                return c
    if kind in ("decode", "kn"):
        fmt = rng.choice(["q8", "q4", "f32", "f16"] if kind == "decode" else ["q8", "q4", "f32", "q8k"])
        return dict(kind="decode" if kind == "decode" else "linear", fmt=fmt, m=rng.randint(1, 8),
                    n=32 * _log_int(rng, 12, 200), k=32 * _log_int(rng, 12, 200), act="none", bias=rng.random() < 0.7,
                    res=rng.random() < 0.3)
    if kind == "vocab":
        return dict(kind="vocab", fmt=rng.choice(["f32", "f16", "q8", "q4"]), m=rng.randint(1, 8),
                    n=_log_int(rng, 20000, 52000), k=64 * _log_int(rng, 6, 24), act="none", bias=False, res=False)
    while True:
        fmt = rng.choice(["f32", "f32", "f32", "q8", "q4", "q8k", "f16", "q8pc"]) if kind == "linear" else "f32"
        # most widths are whole vectors; one in six is odd, which every format takes on its general path
        step = 1 if rng.random() < 1 / 6 and kind == "linear" and fmt not in ("q8k", "q4") else 32
        c = dict(kind=kind, fmt=fmt, m=_log_int(rng, 9, 3000), n=step * _log_int(rng, 384 // step, 5632 // step),
                 k=step * _log_int(rng, 384 // step, 5632 // step), act="none", bias=True, res=False)
        if kind == "linear":
            c["act"] = rng.choice(["none", "none", "gelu_erf", "gelu_tanh"])
            c["res"] = c["act"] == "none" and rng.random() < 0.5
        if work(c)["flops"] <= (FLOPS_MOST if kind == "linear" else 8e9):
            return c


# ------------------------------------------------------------------ inputs
def _linears(case):
    """(K, N, activation, bias, residual) of each product of a pass."""
    if case["kind"] != "layer":
        return [(case["k"], case["n"], case["act"], case["bias"], case["res"])]
    d, ff = case["d"], case["ff"]
    return [(d, 3 * d, "none", True, False), (d, d, "none", True, True), (d, ff, case["act"], True, False),
            (ff, d, "none", True, True)]


def _activations(gen, m, k, dev):
    """What a normalisation layer hands to a linear: N(0, 1) rows whose channels
    carry a gain, one channel in 256 an outlier's."""
    gain = torch.exp(0.3 * torch.randn(k, generator=gen, device=dev))
    gain[::256] *= 8.0
    return torch.randn(m, k, generator=gen, device=dev) * gain


def _quantize(fmt, w):
    """(weight bytes on the device, scales or None, per-tensor scale) of w [K,N]."""
    if fmt == "f32":
        return w, None, 1.0
    if fmt == "f16":
        return w.half(), None, 1.0
    if fmt == "q8pc":
        s = w.abs().amax(0) / 127.0
        return torch.round(w / s).to(torch.int8), s.contiguous(), 1.0
    if fmt == "q8k":  # one scale per 32 elements of the flattened matrix
        flat = torch.nn.functional.pad(w.reshape(-1), (0, -w.numel() % 32)).reshape(-1, 32)
        s = flat.abs().amax(1) / 127.0
        return torch.round(flat / s[:, None]).to(torch.int8).reshape(-1)[: w.numel()].contiguous(), s.contiguous(), 1.0
    top = 127.0 if fmt == "q8" else 7.0
    s = float(w.abs().max()) / top
    q = torch.round(w / s).to(torch.int8)
    if fmt == "q4":  # two to a byte, the even element in the low nibble
        flat = torch.nn.functional.pad(q.reshape(-1), (0, q.numel() % 2)).reshape(-1, 2)
        q = ((flat[:, 0] & 15) | (flat[:, 1] << 4)).to(torch.uint8).contiguous()
    return q, None, float(np.float32(s))


def _dequantize(fmt, q, scales, scale, k, n):
    """The weight's values [K,N] in 64 bits."""
    if fmt == "q4":
        b = q.to(torch.int16)
        q = torch.stack([((b & 15) ^ 8) - 8, ((b >> 4) ^ 8) - 8], 1).reshape(-1)[: k * n]
    v = q.double().reshape(k, n) if fmt != "q8k" else q.double()
    if fmt == "q8k":
        return (v * scales.double().repeat_interleave(32)[: k * n]).reshape(k, n)
    return v * (scales.double() if fmt == "q8pc" else scale)


def _inputs(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(1_000_003 * seed + 17)
    ops = []
    for i, (k, n, _, bias, res) in enumerate(_linears(case)):
        w = 0.02 * torch.randn(k, n, generator=gen, device=dev)
        q, scales, scale = _quantize(case["fmt"], w)
        if case["kind"] == "vocab":  # the embedding is stored [n_vocab, d]
            q, scales, scale = _quantize(case["fmt"], w.t().contiguous())
        # the FFN's second product reads the first one's output
        x = None if case["kind"] == "layer" and i == 3 else _activations(gen, case["m"], k, dev)
        ops.append(dict(x=x, q=q, scales=scales, scale=scale,
                        bias=0.02 * torch.randn(n, generator=gen, device=dev) if bias else None,
                        res=torch.randn(case["m"], n, generator=gen, device=dev) if res else None))
    return ops


class _Prepared:
    """A prepared weight for as long as the state that holds it."""

    def __init__(self, handle):
        self.handle = handle

    def __del__(self):
        _abi.prepared_free(self.handle)


def _ptr(t):
    return None if t is None else t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


class _Host:
    """Host tensors and the registered weight of a drop-in caller."""

    def __init__(self, op, m, n, k):
        self.x = Tensor(op["x"].cpu().numpy(), (m, k))
        self.w = Tensor(op["q"].cpu().numpy(), (k, n))
        self.bias = Tensor(op["bias"].cpu().numpy(), (n,))
        _abi.weight_register(self.w.data)

    def __del__(self):
        _abi.weight_release(self.w.data)


def prepare(case, seed):
    ops = _inputs(case, seed)
    state = dict(case=case, ops=ops, lin=_linears(case))
    kind, m = case["kind"], case["m"]
    if kind == "host":
        state["host"] = _Host(ops[0], m, case["n"], case["k"])
        return state
    state["out"] = [torch.empty(m, n, device="cuda") for _, n, *_ in state["lin"]]
    if kind == "decode":
        o = ops[0]
        state["w"] = _Prepared(_abi.prepare_dev(FMT[case["fmt"]], case["k"], case["n"], _ptr(o["q"]), o["scale"],
                                                _stream()))
    elif kind == "vocab":
        o = ops[0]
        row = _abi.weight_bytes(FMT[case["fmt"]], 1, case["k"])
        state["w"] = _Prepared(_abi.prepare_rows_dev(FMT[case["fmt"]], case["k"], case["n"], _ptr(o["q"]), row,
                                                     o["scale"], _stream()))
    return state


def run(state):
    case, ops, out = state["case"], state["ops"], state.get("out")
    kind, m, st = case["kind"], case["m"], _stream()
    if kind == "host":
        h = state["host"]
        return dispatch.matmulWithWeightBias(h.x, h.w, h.bias).numpy()
    if kind in ("decode", "vocab"):
        o = ops[0]
        if kind == "vocab":
            _abi.gemm_prepared(state["w"].handle, m, _ptr(o["x"]), _ptr(out[0]), stream=st)
        else:
            _abi.gemm_prepared_ex(state["w"].handle, m, _ptr(o["x"]), _ptr(out[0]), act=ACT[case["act"]],
                                  residual_ptr=_ptr(o["res"]), bias_ptr=_ptr(o["bias"]), stream=st)
        return out[0]
    fmt = FMT[case["fmt"]]
    for i, (o, (k, n, act, _, _)) in enumerate(zip(ops, state["lin"])):
        x = o["x"] if o["x"] is not None else out[i - 1]
        _abi.gemm_ex_dev(fmt, m, n, k, _ptr(x), _ptr(o["q"]), _ptr(out[i]), act=ACT[act], residual_ptr=_ptr(o["res"]),
                         scale=o["scale"], scales_ptr=_ptr(o["scales"]), bias_ptr=_ptr(o["bias"]), stream=st)
    return out if len(out) > 1 else out[0]


# ------------------------------------------------------------ bounds, checks
def work(case):
    m, size, flops = case["m"], 0, 0
    fmt = FMT[case["fmt"]]
    for i, (k, n, _, bias, res) in enumerate(_linears(case)):
        scales = 4 * _abi.scale_count(fmt, k, n) if case["fmt"] in ("q8k", "q8pc") else 0
        size += _abi.weight_bytes(fmt, k, n) + scales + 4 * m * k + 4 * m * n * (2 if res else 1) + (4 * n if bias else 0)
        flops += 2 * m * n * k
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # Measured against exact() over the listed and 36 drawn cases, times about
    # four: products of fp32 activations show 2-norm errors up to 1.1e-6 and single
    # values up to 1.2e-5, the int8 / int4 ones, whose activations are split into
    # two 16-bit terms, up to 2.6e-6 and 2.8e-5.
    if case["fmt"] in ("q8", "q4", "q8pc"):
        return {"rel": 1e-5, "max": 1.2e-4}
    return {"rel": 4e-6, "max": 5e-5}


def _activate(v, act):
    """The reference's two GELU forms in 64 bits: erf by its five-term
    polynomial, and tanh by its rational form with real tanh on the last
    (M*N) % 8 values (src/core/ops.zig:1947-2057)."""
    if act == "gelu_erf":
        a = (0.254829592, -0.284496736, 1.421413741, -1.453152027, 1.061405429)
        x = v * 0.7071067811865476
        t = 1.0 / (1.0 + 0.3275911 * x.abs())
        p = t * (a[0] + t * (a[1] + t * (a[2] + t * (a[3] + t * a[4]))))
        return v * 0.5 * (1.0 + torch.sign(x) * (1.0 - p * torch.exp(-x * x)))
    if act == "gelu_tanh":
        inner = 0.7978845608 * (v + 0.044715 * v ** 3)
        x2 = inner * inner
        th = (inner * (27.0 + x2) / (27.0 + 9.0 * x2)).clamp(-1.0, 1.0)
        flat, tail = th.reshape(-1), v.numel() % 8
        if tail:
            flat[-tail:] = torch.tanh(inner.reshape(-1)[-tail:])
        return 0.5 * v * (1.0 + flat.reshape(v.shape))
    return v


def exact(case, seed):
    outs = []
    for o, (k, n, act, _, _) in zip(_inputs(case, seed), _linears(case)):
        if case["kind"] == "vocab":
            w = _dequantize(case["fmt"], o["q"], o["scales"], o["scale"], n, k).t()
        else:
            w = _dequantize(case["fmt"], o["q"], o["scales"], o["scale"], k, n)
        v = (outs[-1] if o["x"] is None else o["x"].double()) @ w
        if o["bias"] is not None:
            v = v + o["bias"].double()
        if o["res"] is not None:
            v = v + o["res"].double()
        outs.append(_activate(v, act))
    return outs if len(outs) > 1 else outs[0].cpu().numpy() if case["kind"] == "host" else outs[0]
