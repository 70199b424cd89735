"""Timed cases of the quantized-weight path, as a program that uses the library meets it.

Three kinds, each through the C ABI of include/yvex_rocm.h:

  moe    a phase of `layers` MoE layers over a batch of rows: `execute_rows` with deferred
         completion, layer after layer on one stream as a decoder calls it (router, top-k, routed and
         shared experts, combine and, with `streams`, the residual-stream envelope around them), and
         one `complete_rows`
  dense  one projection of a batch of F32 rows by a packed matrix: `encoded_matvec`, which
         quantizes the rows to Q8_K, multiplies and reports completion
  head   the end of a decode step: the packed output head over the batch's rows and
         `select_greedy_rows` on its logits

Weights are random packed bytes with small positive block scales, resident before the call, as
are the rows; every pass reads all of them again.
"""
import ctypes
import math

import numpy as np
import torch

from yvex_amd import abi
from yvex_amd.host import Backend, RowBatchLayer

Q8_0, Q2_K, Q4_K, IQ2_XXS = 8, 10, 12, 16
# values and bytes a block, byte offset of its fp16 scales, number of them, their lowest value and range
_BLOCK = {Q8_0: (32, 34, 0, 1, 1e-4, 1e-3), Q2_K: (256, 84, 80, 2, 1e-4, 1e-3),
          Q4_K: (256, 144, 0, 2, 2e-5, 1e-4), IQ2_XXS: (256, 66, 0, 1, 1e-4, 3.5e-4)}
_DENSE = {"q8_0": Q8_0, "q4_k": Q4_K, "iq2_xxs": IQ2_XXS}
# formats of a layer's matrices: routed gate and up, routed down, shared expert; and whether the
# IQ2_XXS ones are resident as the backend's own image of them
_LAYERS = {"iq2_xxs": (IQ2_XXS, IQ2_XXS, IQ2_XXS, True), "q4_k": (Q4_K, Q4_K, Q4_K, False),
           "model_file": (IQ2_XXS, Q2_K, Q8_0, True)}
# the benchmark's layer, and the geometry of the reference's model file
_WIDE = dict(hidden=7168, intermediate=2048, experts=256, topk=8)
_MODEL = dict(hidden=4096, intermediate=2048, experts=256, topk=6)
VOCABULARY = 129280


def _moe(name, geometry, formats, rows, streams=0, skew=0.0):
    # decoding runs through several layers a phase, a prompt's long launches are measured a layer at a time
    layers = 3 if rows <= 128 else 1
    case = dict(geometry, kind="moe", formats=formats, layers=layers, rows=rows, streams=streams, skew=skew)
    return dict(case, name=name) if name else case


def _dense(name, qtype, rows, width, inputs):
    case = dict(kind="dense", qtype=qtype, weight_rows=rows, width=width, rows=inputs)
    return dict(case, name=name) if name else case


def _head(name, width, inputs):
    case = dict(kind="head", qtype="q8_0", weight_rows=VOCABULARY, width=width, rows=inputs)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one token of one session, the model file's formats and its four residual streams
        _moe("decode_1_model_file", _MODEL, "model_file", 1, streams=4),
        # a handful of sessions, or one that verifies a few drafted tokens
        _moe("decode_5_iq2_xxs", _WIDE, "iq2_xxs", 5),
        # a server's batch: the benchmark's decode step, the same with 4-bit experts and a ragged
        # batch, and a batch that is large for decoding
        _moe("decode_32_iq2_xxs", _WIDE, "iq2_xxs", 32),
        _moe("decode_23_q4_k", _WIDE, "q4_k", 23),
        _moe("decode_96_model_file", _MODEL, "model_file", 96, streams=4),
        # prompts: a short one, the benchmark's batch with its uneven experts, a ragged long one
        _moe("prefill_333_model_file", _MODEL, "model_file", 333, streams=4),
        _moe("prefill_2048_iq2_xxs", _WIDE, "iq2_xxs", 2048, skew=1.1),
        _moe("prefill_1111_q4_k", _WIDE, "q4_k", 1111, skew=1.1),
        # projections around the experts: one token, a ragged decode batch, a prompt
        _dense("dense_1_q8_0", "q8_0", 4096, 4096, 1),
        _dense("dense_19_q4_k", "q4_k", 2048, 7168, 19),
        _dense("dense_2048_q8_0", "q8_0", 4096, 4096, 2048),
        # the next tokens of a few sessions
        _head("head_3_q8_0", 7168, 3),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "dense", "dense", "head"])
    if kind == "dense":
        qtype = rng.choice(["q8_0", "q8_0", "q4_k", "iq2_xxs"])
        rows, width = rng.choice([(4096, 4096), (2048, 7168), (7168, 2048), (1024, 4096), (7168, 7168)])
        return _dense(None, qtype, rows, width, _log_uniform(rng, 1, 2048))
    if kind == "head":
        return _head(None, rng.choice([4096, 7168]), _log_uniform(rng, 1, 48))
    geometry, formats = rng.choice([(_WIDE, "iq2_xxs"), (_WIDE, "q4_k"), (_MODEL, "model_file"),
                                    (_MODEL, "iq2_xxs"), (_MODEL, "model_file")])
    streams = rng.choice([0, 4]) if formats == "model_file" else 0
    if kind == "decode":
        return _moe(None, geometry, formats, _log_uniform(rng, 1, 128), streams)
    return _moe(None, geometry, formats, _log_uniform(rng, 192, 2048), streams, rng.choice([0.0, 1.1]))


# ---- inputs ---------------------------------------------------------------------------------

def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _packed(qtype, values, gen):
    """`values` random weights as packed blocks: uniform codes, positive fp16 block scales."""
    block, nbytes, at, scales, low, span = _BLOCK[qtype]
    raw = torch.empty((values // block, nbytes), dtype=torch.uint8, device="cuda").random_(generator=gen)
    d = torch.rand((values // block, scales), device="cuda", generator=gen).mul_(span).add_(low).to(torch.float16)
    raw[:, at:at + 2 * scales] = d.view(torch.uint8)
    return raw.reshape(-1)


class _Owned:
    """Closes a backend when the last that uses its memory is gone: a state, or an output of one
    that outlives it."""

    def __init__(self, closed):
        self.closed = closed

    def __del__(self):
        for each in self.closed:
            each.close()


class _DeviceRows:
    """A backend tensor's F32 rows for torch, without a copy; torch keeps this object, and with it
    the owner, as long as the memory is in use."""

    def __init__(self, owner, tensor, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(tensor.contents.data), False), "shape": tuple(shape),
                                         "typestr": "<f4", "version": 2}


def _as_torch(owner, tensor, shape):
    return torch.as_tensor(_DeviceRows(owner, tensor, shape), device="cuda")


def _layer(case, gen, x):
    """A layer's random weights behind the library's layer object."""
    hidden, width, experts, streams = (case[k] for k in ("hidden", "intermediate", "experts", "streams"))
    gate_up, down, shared, image = _LAYERS[case["formats"]]
    routed = tuple(_packed(q, experts * width * hidden, gen) for q in (gate_up, gate_up, down))
    common = tuple(_packed(shared, width * hidden, gen) for _ in range(3))
    # the rows share a direction, on which the router's rows lean by the experts' popularity (Zipf
    # with exponent `skew`) and by nothing else
    lean = _lean(hidden)
    rank = torch.randperm(experts, device="cuda", generator=gen).float().add_(1.0)
    router = torch.randn((experts, hidden), device="cuda", generator=gen) / hidden ** 0.5
    router -= ((router @ lean + 2.0 * case["skew"] * torch.log(rank)) / hidden)[:, None] * lean
    envelope = None
    if streams:
        mixing = (streams + 2) * streams
        envelope = dict(
            streams=streams, iterations=20, scale=torch.tensor([0.5, -0.25, 0.75], device="cuda"),
            function=torch.randn((mixing, streams * hidden), device="cuda", generator=gen) / (streams * hidden) ** 0.5,
            base=torch.randn(mixing, device="cuda", generator=gen) * 0.5,
            norm=(1.0 + 0.2 * torch.randn(hidden, device="cuda", generator=gen)).to(torch.bfloat16))
    torch.cuda.synchronize()
    return RowBatchLayer(torch, routed, common, router.contiguous(), x, case["rows"], hidden=hidden, intermediate=width,
                         experts=experts, topk=case["topk"], qtype=gate_up, down_qtype=down, shared_qtype=shared,
                         sweep_image=image, envelope=envelope)


def _lean(hidden):
    return torch.randint(0, 2, (hidden,), device="cuda", generator=_generator(hidden)).float().mul_(2.0).sub_(1.0)


class _Stack:
    """Layers one after another on one backend: its stream, its workspace, its rows."""

    def __init__(self, case, seed):
        gen = _generator(seed)
        rows, hidden = case["rows"], case["hidden"]
        x = torch.randn((rows, max(case["streams"], 1), hidden), device="cuda", generator=gen) + 0.5 * _lean(hidden)
        x = x.reshape(rows, -1).cpu().numpy()
        self.layers = [_layer(case, gen, x) for _ in range(case["layers"])]
        self.first = self.layers[0]
        self.owner = _Owned(self.layers)
        self.calls, self.out = [], []
        for layer in self.layers:
            target = self.first.b.empty_f32(rows * self.first.width)
            batch = abi.RowBatch.from_buffer_copy(self.first.batch)
            batch.device_rows, batch.device_outputs = self.first.rows_in, target
            layer.job.eager_execution, layer.job.device_completion = 0, ctypes.pointer(layer.deferred)
            self.calls.append((layer, batch))
            self.out.append(_as_torch(self.owner, target, (rows, self.first.width)))

    def run(self):
        first = self.first
        ops, handle, err = first.ops, first.b.handle, ctypes.byref(first.err)
        for layer, batch in self.calls:
            if ops.execute_rows(handle, ctypes.byref(layer.job), ctypes.byref(batch), ctypes.byref(layer.out),
                                ctypes.byref(layer.result), err) != 0:
                raise RuntimeError(first.err.message.decode())
        first.complete()
        return self.out


class _Projection:
    def __init__(self, case, seed):
        gen = _generator(seed)
        self.qtype = _DENSE[case["qtype"]]
        self.count, self.width, self.rows = case["weight_rows"], case["width"], case["rows"]
        weights = _packed(self.qtype, self.count * self.width, gen).cpu().numpy()
        x = torch.randn((self.rows, self.width), device="cuda", generator=gen).cpu().numpy()
        self.backend = Backend()
        if not self.backend.ok:
            raise RuntimeError(self.backend.err.message.decode())
        self.owner = _Owned([self.backend])
        self.encoded, (_, self.base) = weights.nbytes, self.backend.resident(weights)
        self.input, self.output = self.backend.f32(x), self.backend.empty_f32(self.rows * self.count)
        self.backend.workspace(self.rows * (self.width // 256) * 292 + self.rows * 1024 + (1 << 20))
        self.out = _as_torch(self.owner, self.output, (self.rows, self.count))
        self.facts, self.err = abi.OperationFacts(), abi.Error()
        self.greedy = case["kind"] == "head"
        if self.greedy:
            self.tokens, self.values, self.ties = (np.zeros(self.rows, t) for t in (np.uint32, np.float32, np.uint64))

    def run(self):
        b, facts, err = self.backend, ctypes.byref(self.facts), ctypes.byref(self.err)
        if b.lib.yvex_rocm_encoded_matvec(b.handle, self.base, self.encoded, self.qtype, self.count, self.width,
                                          self.encoded // self.count, self.rows, self.input, None, 0, None,
                                          self.output, 1, facts, err) != 0:
            raise RuntimeError(self.err.message.decode())
        if not self.greedy:
            return self.out
        if b.lib.yvex_rocm_select_greedy_rows(b.handle, self.output, self.rows, self.count, self.tokens.ctypes.data,
                                              self.values.ctypes.data, self.ties.ctypes.data, facts, err) != 0:
            raise RuntimeError(self.err.message.decode())
        return {"logits": self.out, "tokens": self.tokens.astype(np.int64), "values": self.values,
                "ties": self.ties.astype(np.int64)}


def prepare(case, seed):
    return _Stack(case, seed) if case["kind"] == "moe" else _Projection(case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without --------------------------------------------------------------

def _row_bytes(qtype, width):
    return width // _BLOCK[qtype][0] * _BLOCK[qtype][1]


def _distinct(case):
    """Routed experts that a batch is expected to reach."""
    popularity = [rank ** -case["skew"] for rank in range(1, case["experts"] + 1)]
    total = sum(popularity)
    return sum(1.0 - (1.0 - p / total) ** (case["topk"] * case["rows"]) for p in popularity)


def work(case):
    rows = case["rows"]
    if case["kind"] != "moe":
        count, width = case["weight_rows"], case["width"]
        return {"bytes": count * _row_bytes(_DENSE[case["qtype"]], width) + 4 * rows * (width + count),
                "flops": 2 * rows * count * width}
    hidden, width, experts = case["hidden"], case["intermediate"], case["experts"]
    gate_up, down, shared, _ = _LAYERS[case["formats"]]

    def expert_bytes(up, low):
        return 2 * width * _row_bytes(up, hidden) + hidden * _row_bytes(low, width)
    expanded, mixing = max(case["streams"], 1) * hidden, (case["streams"] + 2) * case["streams"]
    read = (_distinct(case) * expert_bytes(gate_up, down) + expert_bytes(shared, shared)
            + 4 * (experts * hidden + mixing * expanded + 2 * rows * expanded))
    flops = 2 * rows * ((case["topk"] + 1) * 3 * width * hidden + experts * hidden + mixing * expanded)
    return {"bytes": case["layers"] * read, "flops": case["layers"] * flops}


def tolerance(case):
    if case["kind"] == "moe":
        return {"rel": 1e-2}     # bf16 results of bf16 stages with int8 activations between them
    return {"rel": 1e-5}         # exact integer block sums, added in 32 bits or more
