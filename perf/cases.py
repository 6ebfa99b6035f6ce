"""Performance cases of the ternary expert-linear path: single linears, grouped decode launches and routed-expert layers.

A case is a dict of plain values. ``kind`` is the public entry point that the case goes through:

* ``linear``: ``TernaryLinear.__call__`` - a dense projection (attention, shared expert) of a decode step or a prompt;
* ``grouped``: ``grouped_ternary_gemm`` with device offsets - one launch over many experts with a few token rows each;
* ``moe``: ``TernaryMoE.__call__`` (``pattern`` "standard") or ``TernaryMoE.routed`` ("v4") - one routed-expert layer
  from the router's logits (or its output) to the layer's bf16 rows.

Matrix sizes are those of this repository's benchmark and tests; weights are iid trits with |N(0, 1)| scales, activations
N(0, 1), router logits N(0, 1.5) (skewed expert loads).
"""

import math

import torch

from deepseekternarized_amd import PackedTerm, TernaryLinear, grouped_ternary_gemm
from deepseekternarized_amd.moe import TernaryMoE

GROUP = 128

#: (K, N) of dense projections and of one expert's matrix in a grouped launch.
MATRICES = [(7168, 2048), (2048, 7168), (4096, 2048), (4096, 4096), (2048, 4096), (2048, 6144), (2048, 2048), (1024, 2048)]

#: hidden, intermediate size, experts, experts per token of the routed layers.
LAYERS = [(4096, 2048, 64, 6), (2048, 1024, 64, 8), (4096, 2048, 384, 6)]


def listed():
    return [
        # One token of one request through one projection: launch and host latency.
        {"name": "linear_tq1_bf16_1", "kind": "linear", "fmt": "tq1", "terms": 1, "act": "bf16", "T": 1, "K": 7168, "N": 2048},
        # The stacked q | k | v projection of a decode step of 64 sequences, activations quantised to int8 (the default).
        {"name": "linear_tq2_int8_64", "kind": "linear", "fmt": "tq2", "terms": 1, "act": "int8", "T": 64, "K": 2048, "N": 6144},
        # A shared expert's projection in the two-term format over one prompt of an odd length.
        {"name": "linear_tq1_2term_bf16_777", "kind": "linear", "fmt": "tq1", "terms": 2, "act": "bf16", "T": 777, "K": 4096, "N": 2048},
        # The same q | k | v projection over the prompts of 64 sequences of 128 tokens.
        {"name": "linear_tq2_int8_8192", "kind": "linear", "fmt": "tq2", "terms": 1, "act": "int8", "T": 8192, "K": 2048, "N": 6144},
        # One row per expert over 128 matrices: the decode launch whose weights do not fit any cache.
        {"name": "grouped_tq1_bf16_1", "kind": "grouped", "fmt": "tq1", "terms": 1, "act": "bf16", "E": 128, "rows": 1, "ragged": False, "K": 7168, "N": 2048},
        # A decode batch spread over 128 experts: 0 to 4 rows each, int8 activations quantised by the caller.
        {"name": "grouped_tq2_int8_0to4", "kind": "grouped", "fmt": "tq2", "terms": 1, "act": "int8", "E": 128, "rows": 4, "ragged": True, "K": 2048, "N": 7168},
        # Routed layer, one token: a decode step of a single request.
        {"name": "moe_tq1_bf16_1", "kind": "moe", "pattern": "standard", "fmt": "tq1", "terms": 1, "act": "bf16", "T": 1, "layer": 0},
        # Routed layer, a decode batch of 32 sequences.
        {"name": "moe_tq1_bf16_32", "kind": "moe", "pattern": "standard", "fmt": "tq1", "terms": 1, "act": "bf16", "T": 32, "layer": 0},
        # Routed layer of the smaller decoder, a decode batch of 64 sequences, int8 activations.
        {"name": "moe_tq2_int8_64", "kind": "moe", "pattern": "standard", "fmt": "tq2", "terms": 1, "act": "int8", "T": 64, "layer": 1},
        # Routed layer in the call pattern with float32 weights and clamps, one short prompt of an odd length.
        {"name": "moe_v4_tq1_bf16_251", "kind": "moe", "pattern": "v4", "fmt": "tq1", "terms": 1, "act": "bf16", "T": 251, "layer": 0},
        # Routed layer with 384 experts in two terms, a prompt of 2048 tokens: the grouped prefill GEMM.
        {"name": "moe_tq2_2term_bf16_2048", "kind": "moe", "pattern": "standard", "fmt": "tq2", "terms": 2, "act": "bf16", "T": 2048, "layer": 2},
        # Routed layer of the smaller decoder over the prompts of 64 sequences of 128 tokens.
        {"name": "moe_tq2_int8_8192", "kind": "moe", "pattern": "standard", "fmt": "tq2", "terms": 1, "act": "int8", "T": 8192, "layer": 1},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """A case of the listed ranges: 1 to 8192 tokens per linear or layer, 1 to 4 rows per expert in grouped launches, both
    formats, one or two terms, both activation types, every matrix and layer above."""
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["linear", "linear", "grouped", "moe", "moe", "moe"])
        c = {"kind": kind, "fmt": rng.choice(["tq1", "tq2"]), "terms": rng.choice([1, 1, 2]), "act": rng.choice(["bf16", "int8"])}
        if kind == "moe":
            layer = rng.choice([0, 0, 1, 1, 2])
            c.update(pattern=rng.choice(["standard", "standard", "v4"]), T=_log_int(rng, 1, 8192), layer=layer)
        else:
            K, N = rng.choice(MATRICES)
            if kind == "linear":
                c.update(T=_log_int(rng, 1, 8192), K=K, N=N)
            else:
                c.update(E=_log_int(rng, 8, 128), rows=rng.randint(1, 4), ragged=rng.random() < 0.5, K=K, N=N)
        if _cost(c) <= most:
            return c


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 1e15)


def _packed(fmt, E, N, K, gen):
    """Packed rows of iid trits, a third each, as pack() writes them: TQ1 five base-3 digits per byte, TQ2 four 2-bit codes;
    the digits past K are 1 (trit 0)."""
    per = 5 if fmt == "tq1" else 4
    Kp = -(-K // per)
    out = torch.empty(E, N, Kp, dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 28) // (N * Kp))
    for e in range(0, E, step):
        n = min(step, E - e)
        v = torch.randint(0, 3**per, (n, N, Kp), dtype=torch.uint8, device="cuda", generator=gen)
        if fmt == "tq2":
            d = [v % 3, (v // 3) % 3, (v // 9) % 3, v // 27]
            v = d[0] | d[1] << 2 | d[2] << 4 | d[3] << 6
        elif K % per:
            left = K % per
            v[:, :, -1] = v[:, :, -1] % 3**left + sum(3**i for i in range(left, per))
        out[e : e + n] = v
    return out


def _terms(fmt, terms, E, N, K, gen):
    """``terms`` stacked (packed, scale) pairs; the second term is a residual a quarter of the first one's size."""
    return [(_packed(fmt, E, N, K, gen),
             (0.02 * 0.25**i * torch.randn(E, N, K // GROUP, device="cuda", generator=gen).abs()).half()) for i in range(terms)]


def _rows_per_expert(case, seed):
    E, rows = case["E"], case["rows"]
    if not case["ragged"]:
        return torch.full((E,), rows, dtype=torch.int64)
    gen = torch.Generator().manual_seed(seed)
    return (torch.arange(E) % (rows + 1))[torch.randperm(E, generator=gen)]


def _inputs(case, seed):
    """The tensors that a case's inputs and weights are made of, as its program reads them from its files and its caller."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    normal = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)  # noqa: E731
    fmt, terms, act, kind = case["fmt"], case["terms"], case["act"], case["kind"]
    if kind == "linear":
        K, N, T = case["K"], case["N"], case["T"]
        return {"terms": _terms(fmt, terms, 1, N, K, gen), "x": normal(T, K).bfloat16()}
    if kind == "grouped":
        K, N, E = case["K"], case["N"], case["E"]
        stack = _terms(fmt, terms, E, N, K, gen)
        counts = _rows_per_expert(case, seed)
        T = int(counts.sum())
        if act == "int8":
            x = torch.randint(-127, 128, (T, K), dtype=torch.int8, device="cuda", generator=gen)
            x_scale = 0.01 + 0.02 * torch.rand(T, device="cuda", generator=gen)
        else:
            x, x_scale = normal(T, K).bfloat16(), None
        return {"terms": stack, "counts": counts, "x": x, "x_scale": x_scale}
    H, I, E, k = LAYERS[case["layer"]]
    gate, up = _terms(fmt, terms, E, I, H, gen), _terms(fmt, terms, E, I, H, gen)
    down = _terms(fmt, terms, E, H, I, gen)
    x = normal(case["T"], H).bfloat16()
    logits = 1.5 * normal(case["T"], E)
    raw = {"gate": gate, "up": up, "down": down, "x": x, "logits": logits}
    if case["pattern"] == "v4":  # this pattern's router is the caller's: normalised float32 weights of the chosen experts
        scores, raw["experts"] = torch.topk(torch.softmax(logits, -1), k)
        raw["weights"] = scores / scores.sum(-1, keepdim=True)
    return raw


def prepare(case, seed):
    fmt, act, kind, raw = case["fmt"], case["act"], case["kind"], _inputs(case, seed)
    state = {"case": case, "x": raw["x"]}
    if kind == "linear":
        state["linear"] = TernaryLinear([PackedTerm(p[0], s[0]) for p, s in raw["terms"]], case["K"], fmt, GROUP, act=act)
    elif kind == "grouped":
        state["packed"], state["scale"] = [p for p, _ in raw["terms"]], [s for _, s in raw["terms"]]
        state["offsets"] = torch.cat([torch.zeros(1, dtype=torch.int64), raw["counts"].cumsum(0)]).cuda()
        state["x_scale"] = raw["x_scale"]
    else:
        H, I, _, k = LAYERS[case["layer"]]
        v4 = case["pattern"] == "v4"
        state["moe"] = TernaryMoE(raw["gate"], raw["up"], raw["down"], H, I, k, fmt, GROUP, act=act, pattern=case["pattern"],
                                  swiglu_limit=10.0 if v4 else 0.0)
        state.update({name: raw[name] for name in (("experts", "weights") if v4 else ("logits",))})
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "linear":
        return state["linear"](state["x"])
    if case["kind"] == "grouped":
        return grouped_ternary_gemm(state["x"], state["x_scale"], state["offsets"], state["packed"], state["scale"], case["K"], GROUP,
                                    case["fmt"], max_rows=case["rows"])
    if case["pattern"] == "v4":
        return state["moe"].routed(state["x"], state["weights"], state["experts"])
    return state["moe"](state["x"], state["logits"])


def _weight_bytes(case, N, K):
    per = 5 if case["fmt"] == "tq1" else 4
    return case["terms"] * N * (-(-K // per) + 2 * (K // GROUP))


def work(case):
    """Weights of the experts that have rows (their expected number for a routed layer), activations in, results out."""
    if case["kind"] == "linear":
        T, K, N = case["T"], case["K"], case["N"]
        return {"bytes": _weight_bytes(case, N, K) + 2 * T * K + 2 * T * N, "flops": 2 * T * N * K * case["terms"]}
    if case["kind"] == "grouped":
        K, N, E = case["K"], case["N"], case["E"]
        counts = _rows_per_expert(case, 0)
        T, active = int(counts.sum()), int((counts > 0).sum())
        row = K + 4 if case["act"] == "int8" else 2 * K
        return {"bytes": active * _weight_bytes(case, N, K) + T * row + 8 * (E + 1) + 4 * T * N, "flops": 2 * T * N * K * case["terms"]}
    H, I, E, k = LAYERS[case["layer"]]
    T = case["T"]
    active = E * (1 - (1 - k / E) ** T)
    router = T * k * 12 if case["pattern"] == "v4" else 4 * T * E
    out = 4 if case["pattern"] == "v4" else 2
    return {"bytes": round(active * (_weight_bytes(case, 2 * I, H) + _weight_bytes(case, H, I))) + (2 + out) * T * H + router,
            "flops": 6 * T * k * H * I * case["terms"]}


def tolerance(case):
    """Four times what separates the path from the same rounding points over float64 sums: float32 results of a grouped
    launch differ by 2e-6, a linear's bf16 results by the values that fall on the other side of a rounding step (8e-5, one
    step of 2^-8 at most), a layer's by such steps of gate, up, hidden and expert rows (1.1e-3, at most 0.03)."""
    if case["kind"] == "grouped":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "linear":
        return {"rel": 4e-4, "max": 0.032}
    return {"rel": 4e-3, "max": 0.12}


def _dense(terms, e, K, fmt):
    """The float64 [N, K] matrix of expert ``e``: the sum of its terms' trits times scales."""
    total = 0
    for packed, scale in terms:
        v = packed[e].int()
        digits = [v // 3**i % 3 for i in range(5)] if fmt == "tq1" else [v >> 2 * i & 3 for i in range(4)]
        trits = torch.stack(digits, -1).flatten(1)[:, :K].double() - 1
        total = total + trits * scale[e].double().repeat_interleave(GROUP, -1)
    return total


def _int8(x):
    """Rows as whole numbers -127 .. 127 and float32 scales: absmax / 127, halves to even."""
    scale = (x.float().abs().amax(-1, keepdim=True) / 127).clamp(min=1e-8)
    return (x.float() / scale).round().clamp(-127, 127).double(), scale.double()


def exact(case, seed):
    """The same products and sums in 64 bits, with the places where the path rounds to bf16 or quantises to int8: a linear's
    activations, gate, up, hidden and expert rows of a layer. A linear's and a layer's own result are not rounded."""
    raw, fmt = _inputs(case, seed), case["fmt"]
    rows = lambda x: _int8(x) if case["act"] == "int8" else (x.double(), 1.0)  # noqa: E731
    if case["kind"] == "linear":
        q, scale = rows(raw["x"])
        return q @ _dense(raw["terms"], 0, case["K"], fmt).T * scale
    if case["kind"] == "grouped":
        parts = [x.double() @ _dense(raw["terms"], e, case["K"], fmt).T for e, x in enumerate(raw["x"].split(raw["counts"].tolist())) if len(x)]
        out = torch.cat(parts)
        return out if raw["x_scale"] is None else out * raw["x_scale"].double()[:, None]
    H, I, E, k = LAYERS[case["layer"]]
    v4 = case["pattern"] == "v4"
    if v4:
        weights, experts = raw["weights"], raw["experts"]
    else:
        weights, experts = torch.topk(torch.softmax(raw["logits"].double(), -1), k)
        weights = weights.bfloat16()
    out = torch.zeros(case["T"], H, dtype=torch.float64, device="cuda")
    for e in range(E):
        token, slot = (experts == e).nonzero(as_tuple=True)
        if not len(token):
            continue
        w = weights[token, slot].double()[:, None]
        q, scale = rows(raw["x"][token])
        gate, up = ((q @ _dense(raw[n], e, H, fmt).T * scale).bfloat16().double() for n in ("gate", "up"))
        if v4:
            gate, up = gate.clamp(max=10.0), up.clamp(-10.0, 10.0)
            h = (w * (gate * torch.sigmoid(gate) * up)).bfloat16()
        else:
            h = ((gate * torch.sigmoid(gate)).bfloat16().double() * up).bfloat16()
        q, scale = rows(h)
        y = (q @ _dense(raw["down"], e, I, fmt).T * scale).bfloat16().double()
        out[token] += y if v4 else (y * w).bfloat16().double()
    return out
