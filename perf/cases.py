"""What a user of this framework has it do, as cases to measure.

Every case goes through the public surface: an ``IqkSwitchLinear`` called with
``(x, indices)`` (decode up to 63 token-expert pairs, prefill above or with
``sorted_indices``), its multi-token verify forms, its dequantization and its
wire ingest.  The geometry is the routed layer of the repository's benchmark and
tests: stacks of up to 256 experts, gate/up ``[2048 x 4096]``, down
``[4096 x 2048]``, top-6 routing (top-1 to top-8 in the drawn cases), uniform
or Zipf(1.1), in the three members.

Weights are N(0, 0.02) rows quantized by the package codec under a
Uniform(0.1, 1) imatrix: a pool of 256 rows per projection, from which every
row of every expert is drawn, so each expert owns its bytes at its own address.
Activations are fp16 N(0, 1).  Expert ids are int64 as ``torch.topk`` gives them,
or int32 where a program keeps them so.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "mlx-iqk_amd"))

from mlx_iqk_amd import codec  # noqa: E402
from mlx_iqk_amd import format as fmt  # noqa: E402
from mlx_iqk_amd.iq1grid import grid_values  # noqa: E402
from mlx_iqk_amd.nn import DECODE_MAT_LIMIT, IqkSwitchLinear  # noqa: E402

MEMBERS = ("iq2_ks", "iq2_k", "iq1_s_r4")
GEOMETRY = {"gate": (2048, 4096), "down": (4096, 2048)}  # out, in (up is gate's)
POOL_ROWS = 256
DEVICE = "cuda"
_SIGNED = {torch.uint32: torch.int32, torch.uint16: torch.int16}


def listed() -> list[dict]:
    def call(name, member, proj, tokens, **over):
        case = {"name": name, "kind": "forward", "member": member, "proj": proj, "tokens": tokens, "experts": 256,
                "top_k": 6, "zipf": 0.0, "sorted": False, "ids": "int64"}
        case.update(over)
        return case

    return [
        # one token of one sequence, eagerly, one projection: the smallest call there is
        call("decode_ks_gate_t1", "iq2_ks", "gate", 1, ids="int32"),
        # the same in the 1.5-bit member, its down projection (one row a pair), ids from topk
        call("decode_iq1_down_t1", "iq1_s_r4", "down", 1),
        # one token through a layer's experts (gate, up, silu * up, down) as the graph a serving loop replays
        {"name": "layer_graph_t1", "kind": "layer", "member": "iq2_ks", "tokens": 1, "experts": 256, "top_k": 6,
         "zipf": 0.0},
        # eight sequences decoded together: 48 pairs, the small-batch decode
        call("decode_k_gate_t8", "iq2_k", "gate", 8, ids="int32"),
        # eight draft tokens verified together, whose experts come from few: the union form
        {"name": "verify_k_gate_t8", "kind": "verify", "form": "union", "member": "iq2_k", "proj": "gate",
         "tokens": 8, "experts": 256, "top_k": 6, "pool": 9},
        # 24 sequences decoded together: 144 pairs, a few to an expert, past the decode limit
        call("batch_ks_gate_t24", "iq2_ks", "gate", 24),
        # a short prompt of odd length
        call("prefill_iq1_gate_t149", "iq1_s_r4", "gate", 149),
        # a prompt of middle length, pairs sorted by expert by the caller, down projection
        call("prefill_k_down_t512", "iq2_k", "down", 512, zipf=1.1, sorted=True, ids="int32"),
        # the benchmark's prompt: 2048 tokens, Zipf(1.1)
        call("prefill_ks_gate_t2048", "iq2_ks", "gate", 2048, zipf=1.1),
        # a batch of long prompts: the largest call
        call("prefill_k_gate_t8192", "iq2_k", "gate", 8192, zipf=1.1),
        # fp16 weights of a row range of a stack, for a caller's own matmul
        {"name": "dequant_ks_gate_e64", "kind": "dequant", "member": "iq2_ks", "proj": "gate", "experts": 64,
         "start": 512, "rows": 1024},
        # a checkpoint's wire rows laid out on the GPU at load time
        {"name": "load_k_down_e64", "kind": "load", "member": "iq2_k", "proj": "down", "experts": 64},
    ]


def draw(rng) -> dict:
    kind = rng.choice(("decode", "decode", "verify", "prefill", "prefill", "prefill", "prefill", "layer", "dequant",
                       "load"))
    member, proj = rng.choice(MEMBERS), rng.choice(tuple(GEOMETRY))
    experts = rng.choice((32, 64, 96, 128, 160, 256))
    zipf = rng.choice((0.0, 1.1))

    def spread(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    if kind == "layer":
        return {"kind": kind, "member": member, "tokens": rng.randint(1, 5), "experts": experts,
                "top_k": rng.choice((2, 4, 6)), "zipf": zipf}
    if kind == "verify":
        top_k = rng.choice((2, 4, 6, 8))
        return {"kind": kind, "form": rng.choice(("union", "union", "sorted")), "member": rng.choice(MEMBERS[:2]),
                "proj": proj, "tokens": spread(2, 24), "experts": experts, "top_k": top_k,
                "pool": rng.randint(top_k, 32)}
    if kind == "dequant":
        rows = rng.choice((256, 512, 1024))
        return {"kind": kind, "member": member, "proj": proj, "experts": rng.randint(4, 64),
                "start": rng.randint(0, GEOMETRY[proj][0] - rows), "rows": rows}
    if kind == "load":
        return {"kind": kind, "member": member, "proj": proj, "experts": spread(2, 64)}
    top_k = rng.choice((1, 2, 4, 6, 8))
    if kind == "decode":
        tokens = rng.randint(1, max(1, min(16, DECODE_MAT_LIMIT // top_k)))
    else:
        tokens = spread(64 // top_k + 1, 49152 // top_k)
        tokens = min(tokens, 8192)
    return {"kind": "forward", "member": member, "proj": proj, "tokens": tokens, "experts": experts, "top_k": top_k,
            "zipf": zipf, "sorted": kind == "prefill" and rng.random() < 0.3, "ids": rng.choice(("int32", "int64"))}


# ------------------------------------------------------------------ inputs ---


def _rng(seed: int, *parts) -> np.random.Generator:
    return np.random.default_rng([int(seed), *(sum(ord(c) << (i % 16) for i, c in enumerate(str(p))) for p in parts)])


def _pool_wire(member: str, n: int, seed: int, label: str) -> np.ndarray:
    """Quantized wire of POOL_ROWS rows."""
    rng = _rng(seed, "rows", label, member, n)
    w = (rng.standard_normal((POOL_ROWS, n), dtype=np.float32) * np.float32(0.02))
    return codec.quantize(member, w, rng.uniform(0.1, 1.0, n).astype(np.float32))


def _signed(t: torch.Tensor) -> torch.Tensor:
    return t.view(_SIGNED.get(t.dtype, t.dtype))


def _generator(seed: int, label: str) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(_rng(seed, "device", label).integers(1 << 62)))
    return g


def _streams(member: str, experts: int, proj: str, seed: int, label: str = "") -> dict:
    """Stacked relayout streams on the device, each row one of the pool's."""
    out, n = GEOMETRY[proj]
    pool = fmt.pack(member, _pool_wire(member, n, seed, label + proj), n)
    shapes = fmt.component_shapes(member, experts, out, n)
    pick = torch.randint(POOL_ROWS, (experts * out,), generator=_generator(seed, label + proj), device=DEVICE)
    streams = {}
    for k, rows in pool.items():
        t = torch.from_numpy(np.ascontiguousarray(rows)).to(DEVICE)
        t = t.reshape(POOL_ROWS, *shapes[k][2:])
        streams[k] = _signed(t)[pick].view(t.dtype).reshape(shapes[k])
    return streams


def _module(member: str, experts: int, proj: str, streams: dict) -> IqkSwitchLinear:
    out, n = GEOMETRY[proj]
    module = IqkSwitchLinear(member, experts, out, n, device=DEVICE)
    module.load_streams(streams)
    return module


def _routing(case: dict, seed: int) -> np.ndarray:
    """``[tokens, top_k]`` expert ids, a token's ids distinct: uniform, Zipf
    over a random order of the experts, or (verify) uniform over a few."""
    rng = _rng(seed, "routing")
    experts, tokens, k = case["experts"], case["tokens"], case["top_k"]
    pool = rng.permutation(experts)[:case.get("pool", experts)]
    weight = np.arange(1, pool.size + 1, dtype=np.float64) ** -case.get("zipf", 0.0)
    # the k largest of log weight + Gumbel noise: k draws without replacement
    key = np.log(weight) + rng.gumbel(size=(tokens, pool.size))
    return pool[np.argsort(-key, axis=1)[:, :k]].astype(np.int64)


def _normal(shape, seed: int, label: str) -> torch.Tensor:
    return torch.randn(shape, generator=_generator(seed, label), device=DEVICE).to(torch.float16)


def _forward_inputs(case: dict, seed: int):
    """x and ids as the call takes them."""
    n = GEOMETRY[case["proj"]][1]
    ids = torch.from_numpy(_routing(case, seed)).to(DEVICE)
    T, k = ids.shape
    x = _normal((T, 1, 1, n) if case["proj"] == "gate" else (T, k, 1, n), seed, "x")
    if case["sorted"]:  # pairs in expert order, one activation row each
        order = torch.argsort(ids.reshape(-1), stable=True)
        x = x.expand(T, k, 1, n).reshape(T * k, 1, n)[order].contiguous()
        ids = ids.reshape(-1)[order]
    return x, ids.to(getattr(torch, case["ids"]))


def _verify_inputs(case: dict, seed: int):
    n = GEOMETRY[case["proj"]][1]
    ids = torch.from_numpy(_routing(case, seed)).to(DEVICE).reshape(-1)
    order = torch.argsort(ids, stable=True)
    x = _normal((case["tokens"], n), seed, "x")
    return x, ids[order].to(torch.int32), (order // case["top_k"]).to(torch.int32)


def _load_inputs(case: dict, seed: int) -> torch.Tensor:
    member, (out, n) = case["member"], GEOMETRY[case["proj"]]
    wire = torch.from_numpy(_pool_wire(member, n, seed, case["proj"])).to(DEVICE)
    group = 4 if member == "iq1_s_r4" else 1  # rows the wire interleaves
    units = wire.view(POOL_ROWS // group, group * wire.shape[1])
    pick = torch.randint(units.shape[0], (case["experts"] * out // group,), generator=_generator(seed, "wire"),
                         device=DEVICE)
    return units[pick].view(case["experts"] * out, wire.shape[1])


LAYER = (("gate", "gate"), ("up", "gate"), ("down", "down"))


def prepare(case: dict, seed: int) -> dict:
    kind, member = case["kind"], case["member"]
    if kind == "layer":
        modules = {label: _module(member, case["experts"], proj, _streams(member, case["experts"], proj, seed, label))
                   for label, proj in LAYER}
        x = _normal((case["tokens"], 1, 1, GEOMETRY["gate"][1]), seed, "x")
        ids = torch.from_numpy(_routing(case, seed)).to(DEVICE, torch.int32)

        def step():
            h = torch.nn.functional.silu(modules["gate"](x, ids)) * modules["up"](x, ids)
            return modules["down"](h, ids)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = step()
        return {"kind": kind, "graph": graph, "y": y, "keep": (modules, x, ids)}
    if kind == "load":
        out, n = GEOMETRY[case["proj"]]
        return {"kind": kind, "module": IqkSwitchLinear(member, case["experts"], out, n, device=DEVICE),
                "wire": _load_inputs(case, seed)}
    module = _module(member, case["experts"], case["proj"], _streams(member, case["experts"], case["proj"], seed))
    state = {"kind": kind, "module": module}
    if kind == "dequant":
        state.update(start=case["start"], rows=case["rows"])
    elif kind == "verify":
        x, ids, toks = _verify_inputs(case, seed)
        state.update(x=x, ids=ids, toks=toks, form=case["form"])
    else:
        x, ids = _forward_inputs(case, seed)
        state.update(x=x, ids=ids, sorted=case["sorted"])
    return state


def run(state: dict):
    kind = state["kind"]
    if kind == "forward":
        return state["module"](state["x"], state["ids"], sorted_indices=state["sorted"])
    if kind == "verify":
        module = state["module"]
        form = module.gemv_union if state["form"] == "union" else module.gemv_sorted
        return form(state["x"], state["ids"], state["toks"])
    if kind == "layer":
        state["graph"].replay()
        return state["y"]
    module = state["module"]
    if kind == "dequant":
        return module.dequantized_range(state["start"], state["rows"])
    module.load_wire(state["wire"])
    return {name: _signed(getattr(module, name)) for name in module.stream_names()}


# ---------------------------------------------------------- what it is held to ---


def work(case: dict) -> dict:
    kind, member = case["kind"], case["member"]
    if kind == "layer":
        parts = [work({**case, "kind": "forward", "proj": proj, "sorted": False, "ids": "int32"}) for _, proj in LAYER]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    out, n = GEOMETRY[case["proj"]]
    row = fmt.ik_row_bytes(member, n)
    if kind == "load":
        return {"bytes": 2 * case["experts"] * out * row, "flops": 0}
    if kind == "dequant":
        rows = case["experts"] * case["rows"]
        return {"bytes": rows * (row + 2 * n), "flops": rows * n}
    ids = _routing(case, 0)
    pairs = ids.size
    per_pair = kind == "forward" and (case["sorted"] or case["proj"] == "down")
    x_rows = pairs if per_pair else case["tokens"]
    distinct = int(np.unique(ids).size)
    return {"bytes": distinct * out * row + 2 * (x_rows * n + pairs * out) + 4 * pairs,
            "flops": 2 * pairs * out * n}


def tolerance(case: dict):
    if case["kind"] in ("dequant", "load"):
        return "exact"  # the format's own fp16 weights and bytes
    if case["kind"] == "layer":
        return {"rel": 2e-3, "max": 2e-2}  # three projections with fp16 values between them
    # f32 sums of fp16 operands, rounded to fp16 once: 2e-4 from 64 bits
    return {"rel": 8e-4, "max": 4e-3}


# ----------------------------------------------------------------- in 64 bits ---


def _bits(words: torch.Tensor, width: int, per: int) -> torch.Tensor:
    """The ``per`` fields of ``width`` bits of each word, lowest first, along the last axis."""
    words = words.view(_SIGNED.get(words.dtype, words.dtype)).to(torch.int64)
    shift = torch.arange(per, device=words.device, dtype=torch.int64) * width
    fields = (words[..., None] >> shift) & ((1 << width) - 1)
    return fields.reshape(*words.shape[:-1], -1)


_ALPHABET = ((-31.0, -13.0, 1.0, 17.0), (-26.0, -8.0, 6.0, 22.0))


def _weights(member: str, streams: dict) -> torch.Tensor:
    """Relayout rows ``[..., rows, *]`` -> their weights in float64."""
    dv = streams["dv"].to(torch.float64)
    if member == "iq1_s_r4":
        grid = torch.from_numpy(grid_values().astype(np.float64)).to(DEVICE)
        qh = _bits(streams["qh"], 16, 1)
        low = _bits(streams["qs"], 8, 4).reshape(*qh.shape, 4)
        high = _bits(qh, 3, 4).reshape(*qh.shape, 4)
        values = grid[low | (high << 8)].reshape(*qh.shape, 32)
        shift = torch.where(qh >= 32768, -0.125, 0.125).to(torch.float64)
        scale = dv[..., None] * (2 * ((qh >> 12) & 7) + 1)
        return ((values + shift[..., None]) * scale[..., None]).flatten(-2)
    codes = _bits(streams["qs"], 2, 16)
    alpha = _bits(streams["sex"], 1, 8)
    nibble = _bits(streams["scl"], 4, 2)
    if member == "iq2_ks":
        index, scale = nibble + 16 * _bits(streams["sch"], 1, 8) - 16, dv[..., None]
    else:
        index, scale = nibble - 8, dv.repeat_interleave(16, dim=-1)
    sub = codes.reshape(*index.shape, codes.shape[-1] // index.shape[-1])
    table = torch.tensor(_ALPHABET, dtype=torch.float64, device=DEVICE)
    return (table[alpha[..., None], sub] * (scale * index)[..., None]).flatten(-2)


def _project(member: str, streams: dict, x: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
    """Row p: float64 x[p] through expert ids[p]."""
    out = streams["dv"].shape[1]
    y = torch.empty((ids.numel(), out), dtype=torch.float64, device=DEVICE)
    for e in torch.unique(ids).tolist():
        rows = torch.nonzero(ids == e).reshape(-1)
        w = _weights(member, {k: v[e] for k, v in streams.items()})
        y[rows] = x[rows].to(torch.float64) @ w.T.contiguous()
    return y


def exact(case: dict, seed: int):
    kind, member, experts = case["kind"], case["member"], case["experts"]
    if kind in ("dequant", "load"):
        return None  # held to the bit by the tolerance
    if kind == "layer":
        ids = torch.from_numpy(_routing(case, seed)).to(DEVICE)
        T, k = ids.shape
        x = _normal((T, 1, 1, GEOMETRY["gate"][1]), seed, "x")
        x = x.expand(T, k, 1, x.shape[-1]).reshape(T * k, -1)
        s = {label: _streams(member, experts, proj, seed, label) for label, proj in LAYER}
        gate = _project(member, s["gate"], x, ids.reshape(-1))
        h = gate * torch.sigmoid(gate) * _project(member, s["up"], x, ids.reshape(-1))
        return _project(member, s["down"], h, ids.reshape(-1)).reshape(T, k, 1, -1)
    streams = _streams(member, experts, case["proj"], seed)
    if kind == "verify":
        x, ids, toks = _verify_inputs(case, seed)
        return _project(member, streams, x[toks.long()], ids)
    x, ids = _forward_inputs(case, seed)
    rows = x.expand(*ids.shape, 1, x.shape[-1]).reshape(ids.numel(), -1)
    return _project(member, streams, rows, ids.reshape(-1)).reshape(*ids.shape, 1, -1)
