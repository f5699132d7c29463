"""Workloads of the EXL3 linear and routed-MoE paths, through the calls a serving program makes.

Three kinds of work:

* ``linear``: ``LinearEXL3.forward`` on the matrices of ``layers`` successive layers (an attention or
  shared-expert projection), from one decoded token to a prefill chunk of 2048 rows.
* ``fan``: ``ops.gemm_group`` on the matrices that read one attention layer's hidden state.
* ``moe``: ``apply_exl3_experts`` on ``layers`` successive routed-expert layers, the decode kernels up to
  32 rows and the grouped GEMMs above.

A serving engine captures its decode step once and replays it, and runs prefill chunks as they come; a case
with ``graph`` does the first (the calls are captured in ``prepare`` and ``run`` replays them), the others
call the entry points in ``run``.  Weights are laid out, and the pointer tables and scratch prepared, once.
Weights are uniform random trellis bits with +-1 input signs and per-column output scales in
[0.5, 2] / sqrt(in), inputs are standard normal, routing is the top-k of a router's logits, softmax weights
over the k."""

from __future__ import annotations

import math
import types

import torch

from dsv4_carve_amd import ops, vllm_exl3

DTYPE = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
SWIGLU_LIMIT = 10.0
MULTIPLIER = {"mcg": 0xCBAC1FED, "mul1": 0x83DCD12D}
H_FAN = "1024,512,1024,1024,256,256"       # wq_a, wkv, compressor wkv/wgate, indexer compressor wkv/wgate


def _linear(name, rows, k, n, bits, *, out="fp16", codebook="mcg", layers=1, graph=False):
    return {"name": name, "kind": "linear", "rows": rows, "k": k, "n": n, "bits": bits, "out": out,
            "codebook": codebook, "layers": layers, "graph": graph}


def _moe(name, rows, *, hidden=4096, inter=2048, experts=256, topk=8, hi=3, lo=2, shared=0, dtype="bf16",
         zipf=0.0, layers=1, graph=False):
    return {"name": name, "kind": "moe", "rows": rows, "hidden": hidden, "inter": inter, "experts": experts,
            "topk": topk, "hi": hi, "lo": lo, "shared": shared, "dtype": dtype, "zipf": zipf, "layers": layers,
            "graph": graph}


def listed():
    return [
        # one sequence decoding: the square 6-bit projections of sixteen layers, one captured step
        _linear("linear decode 1 row", 1, 4096, 4096, 6, layers=16, graph=True),
        # a small ragged batch called one by one, outside any captured step: host and launch latency count
        _linear("linear eager 13 rows", 13, 1536, 4096, 3, out="fp32"),
        # a batch of four decoding: the six matrices that read one attention layer's hidden state, eight layers
        {"name": "fan decode 4 rows", "kind": "fan", "rows": 4, "k": 4096, "ns": H_FAN, "bits": 6, "layers": 8,
         "graph": True},
        # a large or speculative decode batch in a captured step
        _linear("linear batch 72 rows", 72, 4096, 4096, 4, layers=4, graph=True),
        # a prefill chunk of 512 tokens on the widest projection
        _linear("linear prefill 512 rows", 512, 4096, 12288, 6, out="bf16"),
        # a long prefill chunk, ragged
        _linear("linear prefill 2000 rows", 2000, 4096, 4096, 3),
        # one sequence decoding through four routed layers of the 256-expert model
        _moe("moe decode 1 row", 1, layers=4, graph=True),
        # a full decode batch on the 256-expert layer
        _moe("moe decode 16 rows", 16, dtype="fp16", graph=True),
        # a batch past 16 rows with the 6-bit shared expert as one more slot
        _moe("moe decode 24 rows shared", 24, shared=6, graph=True),
        # one GPU's share of the layer under 8-way tensor parallelism, eight layers
        _moe("moe slice decode 4 rows", 4, inter=256, topk=6, hi=2, layers=8, graph=True),
        # a prefill chunk of 512 tokens, a few experts hot
        _moe("moe prefill 512 tokens", 512, dtype="fp16", zipf=1.1),
        # a long ragged prefill chunk with the shared expert
        _moe("moe prefill 1999 tokens", 1999, shared=6, zipf=0.8),
    ]


def _spread(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, step * round(v / step))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "fan", "moe", "moe"))
    if kind == "linear":
        rows = _spread(rng, 1, 2048)
        graph = rows <= 256
        c = _linear("", rows, _spread(rng, 512, 8192, 128), _spread(rng, 256, 12288, 128),
                    rng.choice((2, 3, 4, 5, 6)), out=rng.choice(("fp16", "bf16", "fp32")),
                    codebook=rng.choice(("mcg", "mcg", "mcg", "mcg", "mul1")),
                    layers=rng.randint(2, 8) if graph else 1, graph=graph)
    elif kind == "fan":
        ns = [_spread(rng, 256, 4096, 128) for _ in range(rng.randint(2, 6))]
        c = {"kind": "fan", "rows": rng.randint(1, 16), "k": _spread(rng, 512, 4096, 128),
             "ns": ",".join(str(n) for n in ns), "bits": rng.choice((2, 3, 4, 6)), "layers": rng.randint(2, 8),
             "graph": True}
    else:
        decode = rng.random() < 0.5
        hi = rng.choice((2, 3, 3, 4))
        c = _moe("", _spread(rng, 1, 32) if decode else _spread(rng, 33, 1999),
                 hidden=_spread(rng, 1024, 4096, 256), inter=_spread(rng, 256, 2048, 256),
                 experts=_spread(rng, 32, 256), topk=rng.randint(4, 8), hi=hi, lo=rng.choice((2, hi)),
                 shared=rng.choice((0, 0, 6)), dtype=rng.choice(("bf16", "fp16")),
                 zipf=rng.choice((0.0, 0.8, 1.1)), layers=rng.randint(1, 3) if decode else 1, graph=decode)
    c.pop("name", None)
    return c


# ---------------------------------------------------------------- weights and inputs


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _signs(gen, *shape):
    return (torch.randint(0, 2, shape, generator=gen, device=gen.device, dtype=torch.int8) * 2 - 1).half()


def _packed(gen, count, k, n, bits):
    """`count` EXL3 matrices: trellis int16 [count, k/16, n/16, 16 bits], suh [count, k], svh [count, n]."""
    dev = gen.device
    trellis = torch.randint(-32768, 32768, (count, k // 16, n // 16, 16 * bits), generator=gen, device=dev,
                            dtype=torch.int16)
    suh = _signs(gen, count, k)
    scale = (torch.rand((count, n), generator=gen, device=dev) * 1.5 + 0.5) / math.sqrt(k)
    return trellis, suh, (_signs(gen, count, n).float() * scale).half()


def _normal(gen, rows, k, dtype):
    return torch.randn((rows, k), generator=gen, device=gen.device).to(dtype)


def _marker(device):
    return torch.tensor([vllm_exl3.MCG_MARKER_SIGNED_INT32], dtype=torch.int32, device=device)


def _tensors(case, seed):
    """What the case's seed makes, apart from any object of the framework."""
    gen = _generator(seed)
    if case["kind"] == "linear":
        return [(_normal(gen, case["rows"], case["k"], torch.float16),
                 _packed(gen, 1, case["k"], case["n"], case["bits"])) for _ in range(case["layers"])]
    if case["kind"] == "fan":
        ns = [int(n) for n in case["ns"].split(",")]
        return [(_normal(gen, case["rows"], case["k"], torch.float16),
                 [_packed(gen, 1, case["k"], n, case["bits"]) for n in ns]) for _ in range(case["layers"])]
    return [_moe_tensors(case, gen) for _ in range(case["layers"])]


def _expert_groups(case):
    """(expert count, bits) of the layer's runs of experts: the first half of the routed experts at `hi` bits,
    the rest at `lo`, then the shared expert."""
    e = case["experts"]
    groups = [(e // 2, case["hi"]), (e - e // 2, case["lo"])]
    return groups + ([(1, case["shared"])] if case["shared"] else [])


def _moe_tensors(case, gen):
    rows, experts, topk = case["rows"], case["experts"], case["topk"]
    h, i = case["hidden"], case["inter"]
    groups = [(count, bits, [_packed(gen, count, *kn, bits) for kn in ((h, i), (h, i), (i, h))])
              for count, bits in _expert_groups(case)]
    x = _normal(gen, rows, h, DTYPE[case["dtype"]])
    logits = torch.randn((rows, experts), generator=gen, device=gen.device)
    if case["zipf"]:
        # top-k of log p + Gumbel noise: drawn without replacement, expert of rank j with p ~ j ** -zipf
        rank = torch.randperm(experts, generator=gen, device=gen.device).float() + 1.0
        u = torch.rand((rows, experts), generator=gen, device=gen.device).clamp(1e-7, 1 - 1e-6)
        ids = (-case["zipf"] * rank.log() - (-u.log()).log()).topk(topk, dim=1).indices
    else:
        ids = logits.topk(topk, dim=1).indices
    weights = torch.softmax(logits.gather(1, ids), dim=1)
    if case["shared"]:
        ids = torch.cat([ids, torch.full((rows, 1), experts, dtype=ids.dtype, device=ids.device)], dim=1)
        weights = torch.cat([weights, torch.ones((rows, 1), device=ids.device)], dim=1)
    return groups, x, ids.contiguous(), weights.contiguous()


# ---------------------------------------------------------------- prepare and run


def _linear_call(case, x, packed):
    trellis, suh, svh = (t[0] for t in packed)
    mark = {"mcg": _marker(x.device)} if case["codebook"] == "mcg" else \
        {"mul1": torch.tensor([vllm_exl3.MUL1_MARKER_SIGNED_INT32], dtype=torch.int32, device=x.device)}
    lin = vllm_exl3.LinearEXL3(None, case["k"], case["n"], trellis=trellis, suh=suh, svh=svh, **mark)
    return lambda: lin.forward(x, {}, out_dtype=DTYPE[case["out"]])


def _fan_call(x, members):
    members = [tuple(t[0] for t in packed) for packed in members]
    return lambda: ops.gemm_group(x, members, ops.CB_MCG, torch.float32)


def _moe_call(case, groups, x, ids, weights):
    mark = _marker(x.device)
    inners = []
    for count, _, packs in groups:
        for e in range(count):
            inners.append({w: vllm_exl3.make_linear_exl3(*(t[e] for t in p), mark)
                           for w, p in zip(("gate", "up", "down"), packs)})
    layer = types.SimpleNamespace(prefix="model.layers.0.mlp.experts", expert_map=None, _exl3_inners=inners,
                                  _exl3_hidden_size=case["hidden"], _exl3_intermediate_local=case["inter"])
    vllm_exl3.build_exl3_fused_state(layer, inners)
    return lambda: vllm_exl3.apply_exl3_experts(x, ids, weights, layer, limit=SWIGLU_LIMIT)


def _calls(case, seed):
    made = _tensors(case, seed)
    if case["kind"] == "linear":
        return [_linear_call(case, *t) for t in made]
    if case["kind"] == "fan":
        return [_fan_call(*t) for t in made]
    return [_moe_call(case, *t) for t in made]


def prepare(case, seed):
    calls = _calls(case, seed)
    if not case["graph"]:
        return {"calls": calls}
    for call in calls:            # the shared scratch grows outside a capture
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [call() for call in calls]
    return {"calls": calls, "graph": graph, "outs": outs}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    return [call() for call in state["calls"]]


# ---------------------------------------------------------------- work


def _matrix_bytes(k, n, bits):
    return k * n * bits / 8 + 2 * (k + n)


def _distinct(case):
    """Expected number of distinct routed experts of a layer, and of those at `hi` bits."""
    e, k, rows = case["experts"], case["topk"], case["rows"]
    if not case["zipf"]:
        hit = [1.0 - (1.0 - k / e) ** rows] * e
    else:
        # k successive draws approximated by inclusion probabilities min(1, c p_j) with sum k
        p = [j ** -case["zipf"] for j in range(1, e + 1)]
        lo, hi = 0.0, 1e6
        for _ in range(200):
            c = (lo + hi) / 2
            lo, hi = (c, hi) if sum(min(1.0, c * q) for q in p) < k else (lo, c)
        hit = [1.0 - (1.0 - min(1.0, c * q)) ** rows for q in p]
    total = sum(hit)
    return total, total * (e // 2) / e


def work(case):
    rows, layers = case["rows"], case["layers"]
    if case["kind"] == "linear":
        k, n = case["k"], case["n"]
        b = _matrix_bytes(k, n, case["bits"]) + rows * (2 * k + (4 if case["out"] == "fp32" else 2) * n)
        return {"bytes": layers * b, "flops": layers * 2.0 * rows * k * n}
    if case["kind"] == "fan":
        k, ns = case["k"], [int(n) for n in case["ns"].split(",")]
        b = sum(_matrix_bytes(k, n, case["bits"]) + 4 * rows * n for n in ns) + 2 * rows * k
        return {"bytes": layers * b, "flops": layers * 2.0 * rows * k * sum(ns)}
    h, i = case["hidden"], case["inter"]
    expert = lambda bits: 2 * _matrix_bytes(h, i, bits) + _matrix_bytes(i, h, bits)  # noqa: E731
    total, high = _distinct(case)
    slots = case["topk"] + (1 if case["shared"] else 0)
    b = high * expert(case["hi"]) + (total - high) * expert(case["lo"])
    b += (expert(case["shared"]) if case["shared"] else 0) + 4 * rows * h + 12 * rows * slots
    return {"bytes": layers * b, "flops": layers * 6.0 * rows * slots * h * i}


# ---------------------------------------------------------------- tolerance and the 64-bit result


def tolerance(case):
    # About four times the distance from exact(): 2.1e-4 to 3.1e-4 for an fp32 output (the rotated input is
    # fp16, and so is the weight of the many-row path), 2.9e-4 to 4.7e-4 for fp16 (the routed layer's fp16
    # activation and the output's rounding on top), 1.7e-3 for bf16 (the output's rounding alone).
    out = case.get("out") or case.get("dtype") or "fp32"
    return {"rel": {"fp32": 1.3e-3, "fp16": 2e-3, "bf16": 7e-3}[out]}


_PERM = {}


def _windows(trellis, bits):
    """The 16-bit window of every weight: int64 [k, n] of one matrix's trellis [k/16, n/16, 16 bits]."""
    dev = trellis.device
    if (bits, dev) not in _PERM:
        k, n = torch.meshgrid(torch.arange(16), torch.arange(16), indexing="ij")
        t = 8 * (4 * (n & 7) + ((k & 7) >> 1)) + 4 * (n >> 3) + 2 * (k >> 3) + (k & 1)
        start = ((t + 1) * bits - 16) % (256 * bits)           # first of the window's 16 stream bits
        _PERM[bits, dev] = (start // 16).reshape(-1).to(dev), (16 - start % 16).reshape(-1).to(dev)
    first, shift = _PERM[bits, dev]
    k16, n16, words = trellis.shape
    # the stream runs through each 32-bit word from its top bit: the high half first
    s = (trellis.reshape(k16, n16, words // 2, 2).flip(-1).reshape(k16, n16, words).to(torch.int64)) & 0xFFFF
    w = (((s[..., first] << 16) | s[..., (first + 1) % words]) >> shift) & 0xFFFF
    return w.reshape(k16, n16, 16, 16).permute(0, 2, 1, 3).reshape(k16 * 16, n16 * 16)


def _weights64(trellis, bits, codebook):
    """The codebook's values in 64 bits (the two halves' sum of the MCG codebook is not rounded)."""
    x = (_windows(trellis, bits) * MULTIPLIER[codebook]) & 0xFFFFFFFF
    if codebook == "mul1":
        total = sum((x >> s) & 0xFF for s in (0, 8, 16, 24)) + 1024
        scale, shift = (float(torch.tensor([v], dtype=torch.int16).view(torch.float16)) for v in (0x1EEE, 0xC931 - 65536))
        return total.double() * scale + shift
    x = (x & 0x8FFF8FFF) ^ 0x3B603B60
    half = lambda v: torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.float16).double()  # noqa: E731
    return half(x & 0xFFFF) + half(x >> 16)


def _rotate(x):
    """Each 128-block of the last dimension times the natural-order Hadamard matrix / sqrt(128)."""
    h = torch.ones((1, 1), dtype=torch.float64, device=x.device)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ h).reshape(x.shape) / math.sqrt(128.0)


def _linear64(x, trellis, suh, svh, bits, codebook="mcg"):
    return _rotate(_rotate(x * suh.double()) @ _weights64(trellis, bits, codebook)) * svh.double()


def _moe64(case, groups, x, ids, weights):
    x, out, e = x.double(), torch.zeros(x.shape, dtype=torch.float64, device=x.device), 0
    for count, bits, packs in groups:
        for j in range(count):
            rows, slots = (ids == e + j).nonzero(as_tuple=True)
            if rows.numel():
                gate, up = (_linear64(x[rows], *(t[j] for t in p), bits) for p in packs[:2])
                gate, up = gate.clamp(max=SWIGLU_LIMIT), up.clamp(-SWIGLU_LIMIT, SWIGLU_LIMIT)
                down = _linear64(gate * torch.sigmoid(gate) * up, *(t[j] for t in packs[2]), bits)
                out.index_add_(0, rows, down * weights[rows, slots].double().unsqueeze(1))
        e += count
    return out


def exact(case, seed):
    made = _tensors(case, seed)
    if case["kind"] == "linear":
        return [_linear64(x.double(), *(t[0] for t in p), case["bits"], case["codebook"]) for x, p in made]
    if case["kind"] == "fan":
        return [[_linear64(x.double(), *(t[0] for t in p), case["bits"]) for p in ps] for x, ps in made]
    return [_moe64(case, *t) for t in made]
