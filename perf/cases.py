"""The work a program built on this package has the GPU do, as timed cases.

``listed()`` names representative cases, ``draw(rng)`` gives one more of the same ranges.  A case is a dict of plain
values whose ``kind`` picks one of the paths:

  moe        the routed-expert MXFP8 FFN forward (``MoKSession.forward`` / ``forward_static``) on resident inputs
  quantize   the MXFP8 block quantiser on activations (``mxfp8_quantize_device``)
  weights    loading expert weights: quantise, then the two layouts the forward streams
  attention  flash-attention prefill, causal or with a sliding window (``host.attention``)
  decode     one token of the decode megakernel (``host.megakernel``)
  gemm       bf16 GEMM with the scale + bias epilogue over one accumulator home (``host.one_epilogue``), or with the
             bias + GELU epilogue (``host.gemm_split``)

``prepare`` makes what a program holds before the call (inputs in HBM, a session or a loaded pipeline), ``run`` is one
pass through the public entry point."""
from __future__ import annotations

import math
import weakref

import numpy as np
import torch

from pipelink_amd.host import attention as fa_host
from pipelink_amd.host import gemm_split as gs_host
from pipelink_amd.host import megakernel as mk_host
from pipelink_amd.host import one_epilogue as oe_host
from pipelink_amd.host import mok_inputs
from pipelink_amd.host.backend import HipBackend
from pipelink_amd.host.mok import (MoKSession, code_pitch, mxfp8_quantize_device, scale_pitch, weight_codes_to_k64_tiled,
                                   weight_scales_to_slot_major)
from pipelink_amd.stages.attention import build as fa_build
from pipelink_amd.stages.gemm_split import build as gs_build
from pipelink_amd.stages.megakernel import build as mk_build
from pipelink_amd.stages.megakernel import params as mk_params
from pipelink_amd.stages.mok import build as mok_build
from pipelink_amd.stages.one_epilogue import build as oe_build

# the expert layer the benchmark runs, and the one the tests' larger cases run
LARGE = dict(hidden=2880, intermediate=2880, experts=32, top_k=4)
SMALL = dict(hidden=448, intermediate=704, experts=8, top_k=2)
# the model of the decode megakernel's stated configuration
LLAMA_1B = dict(layers=16, d=2048, hq=32, hkv=8, dff=8192, vocab=128256)


def listed() -> list[dict]:
    moe = dict(kind="moe", padded=True, static=False)
    return [
        # one sequence decoding: four experts of one row each; latency and the weights of four experts
        dict(name="moe_decode_1", tokens=1, **LARGE, **moe),
        # a serving batch decoding, through the entry point graph-captured loops use: almost every expert, a few rows each
        dict(name="moe_decode_27", tokens=27, **LARGE, **dict(moe, static=True)),
        # a large serving batch: every expert's weights for about sixteen rows
        dict(name="moe_decode_128", tokens=128, **LARGE, **moe),
        # a prefill chunk of ragged size: experts of about 125 rows, none a whole row tile
        dict(name="moe_chunk_1003", tokens=1003, **LARGE, **moe),
        # the benchmark's shape: a whole batch's prefill
        dict(name="moe_prefill_8192", tokens=8192, **LARGE, **moe),
        # a small expert layer whose hidden rows are not whole cache lines
        dict(name="moe_small_509", tokens=509, **SMALL, **dict(moe, padded=False)),
        # the activations of a batch, quantised on the way into the expert layer
        dict(name="quantize_activations", kind="quantize", rows=8191, k=2880, dtype="bf16", padded=True),
        # one projection of all experts, from the checkpoint's values to what the forward streams
        dict(name="load_expert_weights", kind="weights", experts=32, n=2880, k=2880, dtype="fp32"),
        # the stated prefill: four sequences of 4096
        dict(name="attention_4096", kind="attention", batch=4, hq=32, hkv=8, seq=4096, window=0),
        # one sequence of 1152 with a sliding window: few long tiles
        dict(name="attention_window_1152", kind="attention", batch=1, hq=32, hkv=8, seq=1152, window=700),
        # the stated decode step, 4096 cached positions
        dict(name="decode_1b_4096", kind="decode", pos=4096, attn="plain", **LLAMA_1B),
        # the stated GEMM, through the largest tile
        dict(name="gemm_8192", kind="gemm", home="full", m=8192, n=8192, k=8192),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["moe"] * 6 + ["quantize", "weights", "attention", "attention", "decode", "gemm"])
    if kind == "moe":
        layer = rng.choice([LARGE, LARGE, LARGE, SMALL, dict(hidden=64 * _log_int(rng, 4, 45), intermediate=64 * _log_int(rng, 4, 45),
                                                              experts=rng.choice([4, 8, 16, 32]), top_k=rng.choice([1, 2, 4]))])
        return dict(kind=kind, tokens=_log_int(rng, 1, 8192), **layer, padded=rng.random() < 0.8, static=rng.random() < 0.3)
    if kind == "quantize":
        return dict(kind=kind, rows=_log_int(rng, 1, 32768), k=32 * _log_int(rng, 8, 90), dtype=rng.choice(["bf16", "fp32"]),
                    padded=rng.random() < 0.5)
    if kind == "weights":
        return dict(kind=kind, experts=rng.choice([1, 3, 8, 32]), n=64 * _log_int(rng, 4, 45), k=64 * _log_int(rng, 4, 45),
                    dtype=rng.choice(["bf16", "fp32"]))
    if kind == "attention":
        hq, hkv = rng.choice([(32, 8), (8, 2), (16, 16), (32, 4)])
        seq = 128 * _log_int(rng, 1, 32)
        return dict(kind=kind, batch=rng.randint(1, 4), hq=hq, hkv=hkv, seq=seq, window=rng.choice([0, 0, _log_int(rng, 1, 4096)]))
    if kind == "decode":
        hq = rng.choice([8, 16, 32])
        return dict(kind=kind, pos=_log_int(rng, 1, 4096), attn=rng.choice(["plain", "wide"]), layers=_log_int(rng, 1, 16), d=64 * hq,
                    hq=hq, hkv=hq // 4, dff=256 * hq, vocab=_log_int(rng, 1000, 128256))
    home = rng.choice(["agpr", "vgpr", "lds", "wide", "full", "full", "gelu"])
    tile_m, tile_n = {"wide": (256, 128), "full": (256, 256)}.get(home, (128, 128))
    return dict(kind=kind, home=home, m=tile_m * _log_int(rng, 1, 8192 // tile_m), n=tile_n * _log_int(rng, 1, 8192 // tile_n),
                k=64 * _log_int(rng, 4, 128))


# ---- what a program holds -----------------------------------------------------------------------------------
def _close(session) -> None:
    torch.cuda.synchronize()
    session.close()


class Opened:
    """A session, closed when nothing holds it any more: its state and the tensors that look into its buffers do."""

    def __init__(self, session):
        self.session = session
        weakref.finalize(self, _close, session)

    def view(self, name: str) -> torch.Tensor:
        """A buffer of a pipeline session as a tensor (no copy)."""
        address, _, (shape, dtype) = self.session.buffers[name]
        if np.dtype(dtype) == np.uint16:   # bf16 bit patterns
            return torch.as_tensor(_Buffer(self, address, shape, "<i2"), device="cuda").view(torch.bfloat16)
        return torch.as_tensor(_Buffer(self, address, shape, np.dtype(dtype).str), device="cuda")


class _Buffer:
    """What torch.as_tensor makes a tensor of; the tensor holds it, and it holds the session."""

    def __init__(self, owner: Opened, address: int, shape: tuple, typestr: str):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(address, False), shape=tuple(shape), typestr=typestr, version=3, strides=None)


class State:
    """One case's inputs and handles."""

    def __init__(self, case: dict):
        self.case = case

    def open(self, session) -> None:
        self.opened, self.session = Opened(session), session


def _bits(t: torch.Tensor) -> np.ndarray:
    return t.to(torch.bfloat16).view(torch.int16).cpu().numpy().view(np.uint16)


def _backend() -> HipBackend:
    return HipBackend(torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)


def _randn(shape, g: torch.Generator, scale: float = 1.0, dtype=torch.float32) -> torch.Tensor:
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _expert_weights(w: torch.Tensor, experts: int, n: int, k: int) -> tuple[torch.Tensor, torch.Tensor]:
    q, sc = mxfp8_quantize_device(w)
    return (weight_codes_to_k64_tiled(q.view(experts, n, k), k),
            weight_scales_to_slot_major(sc.view(experts, n, scale_pitch(k)), k))


def prepare(case: dict, seed: int) -> State:
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = State(case)
    kind = case["kind"]
    if kind == "moe":
        t, h, i, e = case["tokens"], case["hidden"], case["intermediate"], case["experts"]
        counts, row_token = mok_inputs.route(_randn((t, e), g), case["top_k"])   # softmax of N(0,1) logits, uneven counts
        x_q, x_sc = mxfp8_quantize_device(_randn((t, h), g), pitch=code_pitch(h) if case["padded"] else h)
        d = {}
        for name, n, k in (("w_gate", i, h), ("w_up", i, h), ("w_down", h, i)):
            d[name + "_q"], d[name + "_sc"] = _expert_weights(_randn((e * n, k), g, 0.02), e, n, k)
        rows = t * case["top_k"]
        s.y = torch.zeros((rows, h), dtype=torch.bfloat16, device="cuda")
        hidden_q = torch.zeros((rows, code_pitch(i) if case["padded"] else i), dtype=torch.uint8, device="cuda")
        hidden_sc = torch.zeros((rows, scale_pitch(i)), dtype=torch.uint8, device="cuda")
        paths = mok_build.images()
        s.open(MoKSession(paths["linked"].read_bytes(), str(paths["link_json"])))
        s.problem = s.session.problem(x_q=x_q, x_sc=x_sc, row_token=row_token, tokens_per_expert=counts, hidden_q=hidden_q,
                                      hidden_sc=hidden_sc, y=s.y, **d)
    elif kind == "quantize":
        # activations of different magnitude per token
        s.src = _randn((case["rows"], case["k"]), g) * torch.exp2(torch.randint(-3, 4, (case["rows"], 1), generator=g, device="cuda").float())
        s.src = s.src.to(torch.bfloat16 if case["dtype"] == "bf16" else torch.float32)
        s.pitch = code_pitch(case["k"]) if case["padded"] else None
    elif kind == "weights":
        s.src = _randn((case["experts"] * case["n"], case["k"]), g, 0.02, torch.bfloat16 if case["dtype"] == "bf16" else torch.float32)
    elif kind == "attention":
        b, hq, hkv, seq, window = case["batch"], case["hq"], case["hkv"], case["seq"], case["window"]
        q, k, v = (_bits(_randn((b, heads, seq, 128), g)) for heads in (hq, hkv, hkv))
        s.open(fa_host.open_session(fa_build.images()["window_link_json" if window else "link_json"], q, k, v, window=window or None,
                                    backend=_backend()))
        s.out = s.opened.view("o")
    elif kind == "decode":
        dims = {n: case[n] for n in ("layers", "d", "hq", "hkv", "dff", "vocab")}
        per_layer = mk_params.layer_elems(dims["d"], dims["hq"], dims["hkv"], dims["dff"])
        weights = _randn((dims["layers"] * per_layer + dims["d"] + dims["vocab"] * dims["d"],), g, 0.02, torch.bfloat16)
        # a layer is norm | qkv, o | norm | up, gate, down; the norms of an initialised model are ones
        d, attn = dims["d"], (2 * dims["hq"] + 2 * dims["hkv"]) * mk_params.HEAD_DIM * dims["d"]
        layers = weights[:dims["layers"] * per_layer].view(dims["layers"], per_layer)
        layers[:, :d] = 1
        layers[:, d + attn:2 * d + attn] = 1
        weights[dims["layers"] * per_layer:dims["layers"] * per_layer + d] = 1
        cache = _randn((dims["layers"], 2, case["pos"] + 1, dims["hkv"], mk_params.HEAD_DIM), g, 1.0, torch.bfloat16)
        s.embedding = _randn((d,), g)
        images = mk_build.images()
        s.open(mk_host.open_session(images["swap_link_json" if case["attn"] == "wide" else "link_json"], _bits(weights), _bits(cache),
                                    s.embedding.cpu().numpy(), pos=case["pos"], workgroups=256, backend=_backend(), **dims))
        s.x, s.logits, s.cache = (s.opened.view(n) for n in ("x", "logits", "kv_cache"))
    else:
        m, n, k, home = case["m"], case["n"], case["k"], case["home"]
        bias = _randn((n,), g, 0.1).cpu().numpy()
        if home == "gelu":
            s.open(gs_host.open_session(gs_build.images()["link_json"], _bits(_randn((m, k), g, 0.05)), _bits(_randn((n, k), g, 0.05)),
                                        bias, backend=_backend()))
        else:
            scale = 1 + _randn((n,), g, 0.1).cpu().numpy()
            s.open(oe_host.open_session(oe_build.images(home)["link_json"], home, _bits(_randn((m, k), g, 0.02)),
                                        _bits(_randn((n, k), g, 0.02)), bias, scale, backend=_backend()))
        s.out = s.opened.view("c")
    torch.cuda.synchronize()
    return s


def run(s: State):
    kind = s.case["kind"]
    if kind == "moe":
        (s.session.forward_static if s.case["static"] else s.session.forward)(s.problem)
        return s.y
    if kind == "quantize":
        return mxfp8_quantize_device(s.src, pitch=s.pitch)
    if kind == "weights":
        return _expert_weights(s.src, s.case["experts"], s.case["n"], s.case["k"])
    if kind == "decode":
        s.x.copy_(s.embedding)   # the token's embedding goes where the step reads and leaves its residual stream
        s.session.launch()
        return s.logits, s.x, s.cache
    s.session.launch()
    return s.out


# ---- what a pass cannot do without --------------------------------------------------------------------------
def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "moe":
        t, h, i, e, top = case["tokens"], case["hidden"], case["intermediate"], case["experts"], case["top_k"]
        rows = t * top
        active = e * (1 - (1 - top / e) ** t)   # experts that get a row, on average
        mx = 1 + 1 / 32
        return dict(bytes=int(active * 3 * h * i * mx + t * h * mx + rows * 4 + rows * h * 2), flops=6 * rows * h * i)
    if kind in ("quantize", "weights"):
        n = case["rows"] * case["k"] if kind == "quantize" else case["experts"] * case["n"] * case["k"]
        return dict(bytes=int(n * ((2 if case["dtype"] == "bf16" else 4) + 1 + 1 / 32)), flops=2 * n)
    if kind == "attention":
        b, hq, hkv, seq = case["batch"], case["hq"], case["hkv"], case["seq"]
        w = min(case["window"] or seq, seq)
        pairs = w * (w + 1) // 2 + (seq - w) * w
        return dict(bytes=2 * b * seq * 128 * (2 * hq + 2 * hkv), flops=4 * b * hq * 128 * pairs)
    if kind == "decode":
        d, hq, hkv, layers = case["d"], case["hq"], case["hkv"], case["layers"]
        params = layers * mk_params.layer_elems(d, hq, hkv, case["dff"]) + d + case["vocab"] * d
        cache = layers * 2 * case["pos"] * hkv * mk_params.HEAD_DIM
        return dict(bytes=2 * params + 2 * cache + 4 * case["vocab"] + 8 * d,
                    flops=2 * params + layers * 4 * hq * mk_params.HEAD_DIM * (case["pos"] + 1))
    m, n, k = case["m"], case["n"], case["k"]
    return dict(bytes=2 * (m * k + n * k + m * n) + 8 * n, flops=2 * m * n * k)


def tolerance(case: dict):
    """About four times what the path differs by from itself computed in 64 bits and rounded at the same places."""
    kind = case["kind"]
    if kind in ("quantize", "weights"):
        return "exact"
    if kind == "moe":          # seen: up to 1.6e-3 (bf16 results; a thousandth of the e4m3 codes between the products falls the other way)
        return dict(rel=6.5e-3)
    if kind == "attention":    # seen: 2.2e-3 (probabilities in bf16)
        return dict(rel=8e-3)
    if kind == "decode":       # seen: 7e-7 (fp32 activations, 114 sums one after the other)
        return dict(rel=5e-6)
    return dict(rel=1e-4)      # seen: 2.5e-5 (fp32 sums; one bf16 result in ten thousand falls the other way)
