"""Performance cases of the packed-TCQ framework.

Each case is one thing a program that serves (or makes) a packed model has
the framework do, called through the public entry points:

  linear  -- one eager ``PackedTCQLinear(mode="hip")`` call: a decode step
             (batch 1..8), a small batch of sequences or a chunk of a prompt
             (9..32), a whole prompt (33..2048 rows)
  layer   -- the seven projections of one decoder layer, one launch per
             shared input (``decode_step.layer_forward``), replayed from a HIP
             graph as a captured decode step replays them
  stack   -- the projections of several decoder layers as one prepared plan
             (``decode_step.LinearStack``), the bandwidth path
  tiled   -- ``PackedTCQLinear(mode="tiled")``: packed streams resident, row
             tiles decoded on every call
  load    -- building a ``PackedTCQLinear`` from a payload on the GPU: mode
             "cached" (fp16 weights folded back to the original basis), or
             mode "hip" and its first token
  encode  -- ``tcq_quantize_rows``: scales, trellis search, refit and a second
             search of a weight matrix on the GPU (compress time)

Shapes are the decoder projections that the package itself configures
(SmolLM2-135M, Qwen3-0.6B, Qwen3-4B) and, for ``draw``, sizes between and
around them; weights, scales, signs and activations have the distributions of
``turbopress_amd.synthetic``.
"""

from __future__ import annotations

import math

import torch

from turbopress_amd.codebooks import default_codebook
from turbopress_amd.decode_step import LinearStack, layer_forward
from turbopress_amd.encoder import tcq_quantize_rows
from turbopress_amd.runtime import PackedTCQLinear
from turbopress_amd.synthetic import QWEN3_0_6B_LAYER, QWEN3_4B_LAYER

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
LAYERS = {"qwen3-0.6b": QWEN3_0_6B_LAYER, "qwen3-4b": QWEN3_4B_LAYER}
# the input each projection of a decoder layer reads
INPUT_OF = {"q_proj": "attn", "k_proj": "attn", "v_proj": "attn", "o_proj": "o",
            "gate_proj": "mlp", "up_proj": "mlp", "down_proj": "down"}
ORDER = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")


def _linear(name, n, d, bits, batch, n_states=64, bias=False, dtype="fp16"):
    return {"name": name, "kind": "linear", "n": n, "d": d, "bits": bits, "n_states": n_states, "batch": batch,
            "bias": bias, "dtype": dtype}


def listed() -> list:
    return [
        # one small projection per token of a small model (SmolLM2-135M up_proj)
        _linear("linear_smollm_up_b1", 1536, 576, 2, 1),
        # a decoder layer of one captured decode step (Qwen3-0.6B, batch 1)
        {"name": "layer_qwen3_0p6b_b1", "kind": "layer", "model": "qwen3-0.6b", "bits": 3, "n_states": 64, "batch": 1},
        # an MLP projection at the highest rate, eight sequences decoding together
        _linear("linear_gate_k4_b8", 9728, 2560, 4, 8),
        # the long-K projection at batch 32 (a chunk of a prompt, or many sequences)
        _linear("linear_down_b32", 2560, 9728, 3, 32),
        # a prompt of an odd length through the projection with 4096-column Hadamard blocks
        _linear("prefill_o_b199", 2560, 4096, 3, 199),
        # a long prompt through the widest projection
        _linear("prefill_gate_b2048", 9728, 2560, 3, 2048),
        # every projection of nine Qwen3-4B layers as one plan: single-sequence decode ...
        {"name": "stack_qwen3_4b_b1", "kind": "stack", "model": "qwen3-4b", "layers": 9, "bits": 3, "n_states": 64, "batch": 1},
        # ... and 32 sequences decoding together
        {"name": "stack_qwen3_4b_b32", "kind": "stack", "model": "qwen3-4b", "layers": 9, "bits": 3, "n_states": 64, "batch": 32},
        # the mode that keeps the packed streams as stored and decodes row tiles per call
        {"name": "tiled_gate_b4", "kind": "tiled", "n": 3072, "d": 1024, "bits": 3, "n_states": 16, "batch": 4, "bias": False, "dtype": "fp16"},
        # load time: decompress a projection once into fp16 weights
        {"name": "load_cached_down", "kind": "load", "mode": "cached", "n": 2560, "d": 9728, "bits": 3, "n_states": 64, "batch": 1, "bias": False},
        # load time: lay a projection out for the packed path, then its first token
        {"name": "load_hip_gate", "kind": "load", "mode": "hip", "n": 9728, "d": 2560, "bits": 3, "n_states": 64, "batch": 1, "bias": False},
        # compress time: one MLP projection
        {"name": "encode_gate", "kind": "encode", "n": 9728, "d": 2560, "bits": 3, "n_states": 64},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """A case of the same ranges: row counts (odd ones too), input widths with
    Hadamard blocks from 8 to 4096 columns, rates 2..4, every trellis size."""
    kind = rng.choice(["linear", "linear", "linear", "prefill", "prefill", "layer", "stack", "tiled", "load", "encode"])
    bits = rng.choice([2, 3, 4])
    n_states = rng.choice([64, 64, 64, 16, 8, 4])
    if kind == "layer":
        return {"kind": kind, "model": rng.choice(sorted(LAYERS)), "bits": bits, "n_states": n_states,
                "batch": rng.randint(1, 8)}
    if kind == "stack":
        return {"kind": kind, "model": rng.choice(sorted(LAYERS)), "layers": rng.randint(2, 9), "bits": rng.choice([2, 3]),
                "n_states": n_states, "batch": rng.choice([1, 2, 4, 7, 16, 31])}
    n = _log_uniform(rng, 192, 9728)
    block = rng.choice([8, 16, 32, 64, 128, 256, 512, 1024, 2048, 4096])
    d = block * (2 * rng.randint(0, 9) + 1)
    while d > 9728 or d < 256:
        d = block * (2 * rng.randint(0, 300) + 1)
    if rng.random() < 0.6:
        n = (n + 15) // 16 * 16
    bias = rng.random() < 0.25
    dtype = rng.choice(["fp16", "fp16", "fp16", "bf16", "fp32"])
    if kind == "encode":
        return {"kind": kind, "n": min(n, 2560), "d": d, "bits": rng.choice([1, 2, 3, 4]), "n_states": n_states}
    if kind == "load":
        return {"kind": kind, "mode": rng.choice(["cached", "hip"]), "n": n, "d": d,
                "bits": bits, "n_states": n_states, "batch": rng.randint(1, 8), "bias": bias}
    batch = rng.randint(1, 8)
    if kind == "linear" and rng.random() < 0.4:
        batch = rng.randint(9, 32)
    if kind == "prefill":
        batch = _log_uniform(rng, 33, 2048)
    if kind == "tiled":
        return {"kind": kind, "n": min(n, 4096), "d": d, "bits": rng.choice([1, 2, 3, 4]), "n_states": n_states,
                "batch": batch, "bias": bias, "dtype": dtype}
    return {"kind": "linear", "n": n, "d": d, "bits": bits, "n_states": n_states, "batch": batch, "bias": bias, "dtype": dtype}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _block(d: int) -> int:
    return d & -d


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _payload(gen, n, d, bits, n_states, bias=False) -> dict:
    """A format-v2 payload drawn on the GPU (the distributions of
    ``turbopress_amd.synthetic.make_payload``): every byte string is a legal
    stream; bits past a row's last weight are zero."""
    def stream(nbits):
        p = torch.randint(0, 256, (n, (nbits + 7) // 8), generator=gen, dtype=torch.uint8, device="cuda")
        if nbits % 8:
            p[:, -1] &= (1 << (nbits % 8)) - 1
        return p

    path = stream(d)
    member = stream(d * (bits - 1)) if bits > 1 else None
    scales = (torch.randn(n, generator=gen, device="cuda").abs() * 0.02 + 1e-3).half()
    equil = torch.exp(torch.randn(d, generator=gen, device="cuda") * 0.25)
    inv_equil = (1.0 / equil.half().float()).half()
    signs = torch.randint(0, 256, (1, (d + 7) // 8), generator=gen, dtype=torch.uint8, device="cuda")
    b = (torch.randn(n, generator=gen, device="cuda") * 0.1).half() if bias else None
    return {"format": 2, "n": n, "d": d, "bits": bits, "n_states": n_states, "block": _block(d), "path_packed": path,
            "member_packed": member, "scales": scales, "signs_packed": signs, "inv_equil": inv_equil,
            "codebook": default_codebook(bits, n_states).cuda(), "bias": b, "seed": 0}


def _activation(gen, batch, d, dtype="fp16"):
    """N(0, 1) rows with 1 % of the channels scaled by 20."""
    x = torch.randn(batch, d, generator=gen, device="cuda")
    idx = torch.randperm(d, generator=gen, device="cuda")[:math.ceil(0.01 * d)]
    x[:, idx] *= 20.0
    return x.to(DTYPES[dtype])


def _layer_inputs(gen, shapes, batch):
    widths = {INPUT_OF[p]: shapes[p][0] for p in ORDER}
    return {k: _activation(gen, batch, widths[k]) for k in ("attn", "o", "mlp", "down")}


def _inputs(case: dict, seed: int) -> dict:
    """Payloads and activations of a case, from the seed alone."""
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "encode":
        w = torch.randn(case["n"], case["d"], generator=gen, device="cuda")
        rows = torch.exp(torch.randn(case["n"], 1, generator=gen, device="cuda") * 0.3) * 0.02
        return {"w": w * rows}
    if kind in ("layer", "stack"):
        shapes = LAYERS[case["model"]]
        layers = []
        for _ in range(case.get("layers", 1)):
            pay = {p: _payload(gen, shapes[p][1], shapes[p][0], case["bits"], case["n_states"]) for p in ORDER}
            layers.append((pay, _layer_inputs(gen, shapes, case["batch"])))
        return {"layers": layers}
    pay = _payload(gen, case["n"], case["d"], case["bits"], case["n_states"], case["bias"])
    return {"payload": pay, "x": _activation(gen, case["batch"], case["d"], case.get("dtype", "fp16"))}


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind in ("encode", "load"):
        return dict(inp, kind=kind, mode=case.get("mode"), bits=case["bits"], n_states=case["n_states"])
    if kind in ("linear", "tiled"):
        lin = PackedTCQLinear(inp["payload"], mode="hip" if kind == "linear" else "tiled")
        return {"kind": kind, "lin": lin, "x": inp["x"]}
    layers = [({p: PackedTCQLinear(pay[p], mode="hip") for p in ORDER}, xs) for pay, xs in inp["layers"]]
    if kind == "stack":
        entries = [(mods[p], xs[INPUT_OF[p]], 0) for mods, xs in layers for p in ORDER]
        return {"kind": kind, "stack": LinearStack(entries)}
    mods, xs = layers[0]
    # capture the layer's launches once, as a decode loop does (one side
    # stream for the warm-up and the capture)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            layer_forward(mods, xs)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = layer_forward(mods, xs)
    return {"kind": kind, "graph": graph, "out": [out[p] for p in ORDER], "mods": mods, "xs": xs}


def run(state: dict):
    kind = state["kind"]
    if kind in ("linear", "tiled"):
        return state["lin"](state["x"])
    if kind == "layer":
        state["graph"].replay()
        return state["out"]
    if kind == "stack":
        return state["stack"].run()
    if kind == "load":
        lin = PackedTCQLinear(state["payload"], mode=state["mode"])
        return lin._w_cache if state["mode"] == "cached" else lin(state["x"])
    q = tcq_quantize_rows(state["w"], bits=state["bits"], n_states=state["n_states"])
    return q.level_codes, q.path_bits, q.member_codes, q.scales


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _linear_work(n, d, bits, batch, itemsize=2):
    by = n * d * bits / 8 + 2 * n + 2 * d + 2 * (2 << bits) + itemsize * batch * (n + d)
    fl = 2.0 * n * d * batch + batch * d * max(1, int(math.log2(_block(d))))
    return by, fl


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("layer", "stack"):
        by = fl = 0.0
        for p in ORDER:
            d, n = LAYERS[case["model"]][p]
            b, f = _linear_work(n, d, case["bits"], case["batch"])
            by, fl = by + b, fl + f
        # (projections that share an input read it once)
        shapes = LAYERS[case["model"]]
        by -= 2 * case["batch"] * (2 * shapes["q_proj"][0] + shapes["gate_proj"][0])
        k = case.get("layers", 1)
        return {"bytes": k * by, "flops": k * fl}
    n, d, bits = case["n"], case["d"], case["bits"]
    if kind == "encode":
        # two searches: per weight and state two adds and a compare, per weight
        # and subset the nearest member's squared error
        per_weight = 3 * case["n_states"] + 4 * (2 + (1 << (bits - 1)))
        return {"bytes": 4.0 * n * d + 3.0 * n * d + 4 * n, "flops": 2.0 * n * d * per_weight}
    if kind == "load" and case["mode"] == "cached":
        return {"bytes": n * d * bits / 8 + 2.0 * n * d, "flops": n * d * max(1.0, math.log2(_block(d)))}
    size = {"fp16": 2, "bf16": 2, "fp32": 4}[case.get("dtype", "fp16")]
    by, fl = _linear_work(n, d, bits, case["batch"], size)
    if kind == "load":
        by += 2 * n * d * bits / 8  # the streams read and laid out, before the call reads them
    return {"bytes": by, "flops": fl}


def tolerance(case: dict):
    if case["kind"] == "encode":
        return "exact"
    if case["kind"] == "load" and case["mode"] == "cached":
        # each weight is rounded to fp16 twice (decoded, folded back)
        return {"rel": 1e-3}
    # fp16 rotated activations and outputs, fp32 sums
    return {"rel": 8e-3 if case.get("dtype") == "bf16" else 1e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
_GENERATORS = {4: (0o5, 0o7), 8: (0o15, 0o17), 16: (0o23, 0o35), 64: (0o133, 0o171)}


def _unpack(packed, count, width):
    """Little-endian fields of `width` bits: uint8 [n, count]."""
    shift = torch.arange(8, dtype=torch.uint8, device=packed.device)
    bits = ((packed[:, :, None] >> shift) & 1).reshape(packed.shape[0], -1)[:, :count * width]
    out = torch.zeros(packed.shape[0], count, dtype=torch.uint8, device=packed.device)
    for j in range(width):
        out |= bits[:, j::width] << j
    return out


def _weights64(p):
    """Rotated weights codebook[level] * scale in fp64."""
    n, d, s = p["n"], p["d"], p["n_states"]
    m = s.bit_length() - 1
    path = _unpack(p["path_packed"], d, 1)
    sub = torch.zeros_like(path)
    for bit, g in enumerate(_GENERATORS[s]):
        par = torch.zeros_like(path)
        for delay in range(m + 1):
            # the shift register holds the newest bit at position 0 of the
            # state, the incoming one at position m
            pos = m if delay == 0 else delay - 1
            if (g >> pos) & 1:
                par[:, delay:] ^= path[:, :d - delay]
        sub |= par << bit
    level = sub
    if p["bits"] > 1:
        level = sub + 4 * _unpack(p["member_packed"], d, p["bits"] - 1)
    w = p["codebook"].double()[level.long()]
    return w * p["scales"].double()[:, None]


def _fwht64(x, block):
    n, d = x.shape
    y = x.reshape(-1, block)
    h = 1
    while h < block:
        v = y.reshape(-1, block // (2 * h), 2, h)
        y = torch.stack((v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]), dim=2).reshape(-1, block)
        h *= 2
    return (y / math.sqrt(block)).reshape(n, d)


def _rot_scale64(p):
    signs = _unpack(p["signs_packed"], p["d"], 1)[0].double() * 2 - 1
    return signs * p["inv_equil"].double()


def _forward64(p, x):
    z = _fwht64(x.double() * _rot_scale64(p), p["block"])
    y = z @ _weights64(p).T
    return y if p["bias"] is None else y + p["bias"].double()


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "encode":
        return None  # decisions of an fp32 search, compared bit for bit
    inp = _inputs(case, seed)
    if kind in ("layer", "stack"):
        return [_forward64(pay[p], xs[INPUT_OF[p]]) for pay, xs in inp["layers"] for p in ORDER]
    p = inp["payload"]
    if kind == "load" and case["mode"] == "cached":
        return _fwht64(_weights64(p), p["block"]) * _rot_scale64(p)[None, :]
    return _forward64(p, inp["x"])
