"""Performance cases of the PlaceMoE expert layer on one GPU.

Three kinds of work, each through the entry points a training or serving
program calls:

* ``layer``: ``fused_moe_forward`` on one batch, without gradients (serving)
  or with the whole backward (training), with a registered placement (the
  expert-parallel arithmetic over the physical copies) or without one (one
  slot per expert, router weights on the fc2 input), merged or split fc1
  weights, bf16 or fp16; optionally followed by the replica-gradient fold;
* ``payload``: the two halves of one rank's expert-parallel exchange, the
  rank-deduplicated dispatch payload and the combine's aggregation.

The layer shapes are those of ``placemoe_amd/workloads.py`` (and, in drawn
cases, others between them); weights are scaled so that gate and up
activations are about N(0, 0.9), as there.
"""

import math

import numpy as np
import torch

import placemoe_amd
from placemoe_amd import ep_payload
from placemoe_amd.placement import PLACEMENTS, LayerPlacement

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _layer(name, T, H, I, E, C, K, S, routing, placed, grad, split=False, dtype="bf16", fold=False):
    """T tokens, hidden H, intermediate I, E experts in C physical copies, K
    experts per token, S token sources."""
    case = dict(kind="layer", T=T, H=H, I=I, E=E, C=C, K=K, S=S, routing=routing, placed=placed, grad=grad, split=split,
                dtype=dtype, fold=fold)
    return dict(case, name=name) if name else case


def _payload(name, T, H, K, R, C, dtype="bf16"):
    """T tokens of one rank, K slots each out of C slots over R ranks."""
    case = dict(kind="payload", T=T, H=H, K=K, R=R, C=C, dtype=dtype)
    return dict(case, name=name) if name else case


def listed():
    return [
        # One decode step of a small serving batch: a few rows per expert, most experts idle.
        _layer("decode-8", 8, 2048, 768, 128, 128, 8, 1, "router", placed=False, grad=False),
        # One decode step of a loaded server with replicated hot experts: 4-5 rows per copy.
        _layer("decode-96-placed", 96, 2048, 768, 128, 160, 8, 8, "router", placed=True, grad=False),
        # Decode on one expert-parallel rank of a large model: received rows (already mapped, top-1) over 16 big copies.
        _layer("decode-ep-rank-200", 200, 7168, 2048, 16, 16, 1, 1, "zipf1.0", placed=True, grad=False),
        # Prefill of one prompt of odd length, fp16 weights, no placement.
        _layer("prefill-1531-fp16", 1531, 2048, 768, 128, 128, 8, 1, "router", placed=False, grad=False, dtype="fp16"),
        # The forward-only toy configuration: few experts with wide intermediates, 4096 tokens.
        _layer("forward-toy-4096", 4096, 1024, 2816, 8, 12, 2, 4, "router", placed=True, grad=False),
        # Training on a short micro-batch (short sequences, fine-tuning): ~25 rows per copy.
        _layer("train-512-placed", 512, 2048, 768, 128, 160, 8, 8, "router", placed=True, grad=True),
        # Training without expert parallelism, split fc1 weights, odd token count.
        _layer("train-4099-split", 4099, 2048, 768, 128, 128, 8, 1, "router", placed=False, grad=True, split=True),
        # The 128-expert training configuration: 16384 tokens, the 32 hottest experts replicated.
        _layer("train-16384-placed", 16384, 2048, 768, 128, 160, 8, 8, "router", placed=True, grad=True),
        # The same shape with 1-4 copies of every expert and the replica-gradient fold after the backward.
        _layer("train-16384-fold", 16384, 2048, 768, 128, 256, 8, 8, "zipf1.0", placed=True, grad=True, fold=True),
        # Skewed routing: a few very hot experts, some nearly idle.
        _layer("train-32768-skew", 32768, 4096, 1536, 64, 96, 4, 16, "zipf1.4", placed=True, grad=True),
        # One expert-parallel rank of a large model: 65536 received rows over 16 copies (the benchmark's default).
        _layer("train-ep-rank-65536", 65536, 7168, 2048, 16, 16, 1, 1, "zipf1.0", placed=True, grad=True),
        # One rank's halves of the expert-parallel exchange around the all-to-all.
        _payload("ep-payload-16384", 16384, 2048, 8, 8, 160),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: forward and training steps over token
    counts, layer widths, expert counts and options, and EP payloads."""
    kind = rng.choice(["forward", "forward", "forward", "train", "train", "train", "payload"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind == "payload":
        R = rng.choice([2, 4, 8, 16])
        return _payload("", _log_int(rng, 256, 24576), rng.choice([1024, 2048, 2880, 4096]), rng.choice([2, 4, 6, 8]), R,
                        R * rng.randint(6, 20), dtype)
    while True:
        E = rng.choice([8, 16, 32, 64, 128])
        K = rng.choice([1, 2, 4, 6, 8])
        H = 64 * _log_int(rng, 16, 112)
        I = 64 * _log_int(rng, 10, 44)
        if rng.random() < 0.15:
            I -= 24  # a multiple of 8 only
        placed = rng.random() < 0.6
        C = E + rng.randint(0, E) if placed else E
        S = rng.choice([1, 4, 8, 16]) if placed else 1
        T = _log_int(rng, 1, 8192) if kind == "forward" else _log_int(rng, 64, 32768)
        fold = kind == "train" and placed and C > E and rng.random() < 0.3
        if K <= E // 2 and 6 * C * I * H <= 6e9 and T * K * H * I <= 3e11 and T * K * max(H, 2 * I) * 2 <= 2e9:
            break
    return _layer("", T, H, I, E, C, K, S, rng.choice(["router", "router", "zipf1.0", "zipf1.4"]), placed, kind == "train",
                  split=rng.random() < 0.3, dtype=dtype, fold=fold)


# ---------------------------------------------------------------------------


def _normal(gen, shape, std, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype).mul_(std)


def _expert_demand(case, rng):
    """Relative demand of the experts (its logarithm is the router's bias)."""
    E = case["E"]
    if case["routing"] == "router":
        return np.exp(rng.normal(0.0, 0.5, E))
    return np.arange(1, E + 1, dtype=np.float64) ** -float(case["routing"][4:])


def _copies(demand, E, C):
    """slot -> expert: one slot per expert, then the extra copies one by one
    to the expert with the most demand per copy (at most 4 copies each)."""
    copies = np.ones(E)
    slots = list(range(E))
    for _ in range(C - E):
        e = int(np.argmax(np.where(copies < 4, demand / copies, -1.0)))
        copies[e] += 1
        slots.append(e)
    return np.array(slots, dtype=np.int64)


def _route(case, gen, demand):
    """(router weights [T, K], expert ids [T, K]): top-K of the router's logits, softmax weights renormalised."""
    bias = torch.as_tensor(np.log(demand), dtype=torch.float32, device="cuda")
    u = torch.rand((case["T"], case["E"]), generator=gen, device="cuda").clamp_(1e-7, 1 - 1e-7)
    top, sel = torch.topk(bias - torch.log(-torch.log(u)), case["K"], dim=-1)
    if case["K"] == 1:  # received rows carry one weight of their token's softmax each
        w = 0.05 + 0.95 * torch.rand((case["T"], 1), generator=gen, device="cuda")
    else:
        w = torch.softmax(top, dim=-1)
    return w.to(DTYPES[case["dtype"]]), sel


def _layer_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    T, H, I, E, C, S = (case[k] for k in ("T", "H", "I", "E", "C", "S"))
    dt = DTYPES[case["dtype"]]
    demand = _expert_demand(case, rng)
    w, sel = _route(case, gen, demand)
    s = {"x": _normal(gen, (T, H), 1.0, dt), "w": w, "sel": sel}
    s["fc1"] = _normal(gen, (C, 2 * I, H), 0.9 / math.sqrt(H), dt)
    s["fc2"] = _normal(gen, (C, H, I), 0.9 / math.sqrt(H), dt)
    slots = _copies(demand, E, C)
    # every copy of an expert holds the expert's weights
    for c in range(E, C):
        s["fc1"][c].copy_(s["fc1"][int(slots[c])])
        s["fc2"][c].copy_(s["fc2"][int(slots[c])])
    s["slots"] = slots
    by_expert = [np.nonzero(slots == e)[0] for e in range(E)]
    s["M"] = np.array([[c[k % len(c)] for c in by_expert] for k in range(S)], dtype=np.int64)
    s["src"] = torch.randint(0, S, (T,), generator=gen, device="cuda") if S > 1 else None
    s["dout"] = _normal(gen, (T, H), 1.0, dt) if case["grad"] else None
    return s


def _distinct_ranks(case):
    """Ranks that a token reaches: what K slots drawn at random hit on average."""
    R, K = case["R"], case["K"]
    return max(1, min(R, K, round(R * (1 - (1 - 1 / R) ** K))))


def _payload_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T, H, K, R, C = (case[k] for k in ("T", "H", "K", "R", "C"))
    dt = DTYPES[case["dtype"]]
    d, per_rank = _distinct_ranks(case), C // R
    s = {"x": _normal(gen, (T, H), 1.0, dt)}
    # K distinct slots per token on d ranks, in random order
    ranks = torch.rand((T, R), generator=gen, device="cuda").argsort(1)[:, :d]
    slots = torch.rand((T, per_rank), generator=gen, device="cuda").argsort(1)
    k = torch.arange(K, device="cuda")
    phys = ranks[:, k % d] * per_rank + slots[:, k // d]
    s["phys"] = phys.gather(1, torch.rand((T, K), generator=gen, device="cuda").argsort(1))
    s["w"] = torch.softmax(torch.randn((T, K), generator=gen, device="cuda"), -1).to(dt)
    # the assignments received back: T * d (source rank, token) pairs with K / d assignments each on average,
    # by source rank and within a rank by token
    N, runs = T * K, T * d
    rank = torch.sort(torch.randint(0, R, (runs,), generator=gen, device="cuda")).values
    token = torch.cumsum(torch.randint(1, 3, (runs,), generator=gen, device="cuda"), 0)
    first = torch.zeros(N, dtype=torch.int64, device="cuda")
    first[1 + torch.randperm(N - 1, generator=gen, device="cuda")[:runs - 1]] = 1
    run = torch.cumsum(first, 0)
    s["run"], s["src_rank"], s["src_token"] = run, rank[run], token[run]
    s["pos"] = torch.randperm(N, generator=gen, device="cuda")
    s["recv_w"] = torch.rand((N,), generator=gen, device="cuda").to(dt)
    s["y"] = _normal(gen, (N, H), 1.0, dt)
    return s


def prepare(case, seed):
    if case["kind"] == "payload":
        return {"case": case, **_payload_inputs(case, seed)}
    placemoe_amd.apply_veomni_fused_moe_patch("hip")
    s = _layer_inputs(case, seed)
    I = case["I"]
    state = {"case": case, "x": s["x"], "w": s["w"], "sel": s["sel"], "dout": s["dout"], "fc2": s["fc2"], "key": None}
    if case["split"]:
        state["gate"], state["up"], state["fc1"] = s["fc1"][:, :I].contiguous(), s["fc1"][:, I:].contiguous(), None
    else:
        state["gate"] = state["up"] = None
        state["fc1"] = s["fc1"]
    if case["placed"]:
        state["key"] = "perf.%d" % seed
        state["placement"] = LayerPlacement(
            key=state["key"], num_experts=case["E"], slot_to_logical=s["slots"], source_logical_to_physical=s["M"],
            owner_slots=np.arange(case["E"]), token_sources=s["src"])
        state["placement"].mapping_for_device(s["x"].device)
        if case["fold"]:
            state["placement"].copy_tables_for_device(s["x"].device)
    state["params"] = [state[k] for k in ("x", "w", "fc1", "gate", "up", "fc2") if state[k] is not None]
    if case["grad"]:
        for p in state["params"]:
            p.requires_grad_(True)
    return state


def _run_payload(s):
    c = s["case"]
    hidden, meta, weights, tokens, unique_splits, assign_splits, ranks = ep_payload.build_local_payload(
        s["x"], s["phys"], s["w"], c["C"], c["R"])
    sums, splits = ep_payload.combine_aggregate(s["y"], s["pos"], s["recv_w"], s["src_rank"], s["src_token"], c["R"])
    return {"hidden": hidden, "meta": meta, "weights": weights, "tokens": tokens, "ranks": ranks, "sums": sums,
            "splits": np.array([unique_splits, assign_splits, splits])}


def run(state):
    c = state["case"]
    if c["kind"] == "payload":
        return _run_payload(state)
    if state["key"] is not None:
        PLACEMENTS.register(state["placement"])

    def forward():
        return placemoe_amd.fused_moe_forward(c["E"], state["w"], state["sel"], state["x"], state["gate"], state["up"],
                                              state["fc2"], state["fc1"], layer_key=state["key"])

    if not c["grad"]:
        with torch.no_grad():
            return {"out": forward()}
    out = forward()
    grads = torch.autograd.grad(out, state["params"], state["dout"])
    result = {"out": out.detach(), "grads": list(grads)}
    if c["fold"]:
        result["logical"] = [placemoe_amd.fold_replica_gradients(state["placement"], g) for g in grads[2:]]
    if state["key"] is not None:
        state["placement"].clear_slot_tokens()
    return result


# ---------------------------------------------------------------------------


def work(case):
    T, H, K = case["T"], case["H"], case["K"]
    A = T * K
    if case["kind"] == "payload":
        distinct = _distinct_ranks(case)
        runs = T * distinct
        sent = T * H * 2 + T * distinct * H * 2 + A * (8 + 2 + 12 + 2 + 8) + T * distinct * 8
        received = A * H * 2 + runs * H * 2 + A * (8 + 2 + 8 + 8)
        return {"bytes": sent + received, "flops": 2 * A * H}
    I, C = case["I"], case["C"]
    active = C * (1 - (1 - 1 / C) ** A)  # copies with rows, if they were equally likely
    weights = 3 * I * H * 2
    io = 2 * T * H * 2 + A * 10
    if not case["grad"]:
        return {"bytes": active * weights + io, "flops": 6 * A * H * I}
    bytes_ = active * weights + C * weights + 2 * io
    if case["fold"]:  # the copies' gradients read, the sums written in fp32 and back to the copies
        bytes_ += 2 * C * weights + 2 * case["E"] * weights
    return {"bytes": bytes_, "flops": 18 * A * H * I}


def tolerance(case):
    # Every stage of the layer rounds its output to the 16-bit type: the
    # results measure 4.1e-3 to 4.8e-3 (bf16) and 5.7e-4 (fp16) off the 64-bit
    # values.  Two correct implementations, each with such an error of its own,
    # differ by up to sqrt(2) of it; about twice that is allowed.
    # The payload's sums round twice (2.1e-3, bf16).
    rel = 7e-3 if case["kind"] == "payload" else 1.2e-2
    return {"rel": rel if case["dtype"] == "bf16" else rel / 8}


def exact(case, seed):
    if case["kind"] == "payload":
        s = _payload_inputs(case, seed)
        rows = s["y"][s["pos"]].double() * s["recv_w"].double()[:, None]
        sums = torch.zeros((case["T"] * _distinct_ranks(case), case["H"]), dtype=torch.float64, device="cuda")
        sums.index_add_(0, s["run"], rows)
        return {"hidden": None, "meta": None, "weights": None, "tokens": None, "ranks": None, "sums": sums, "splits": None}
    s = _layer_inputs(case, seed)
    T, H, I, E, C, K = (case[k] for k in ("T", "H", "I", "E", "C", "K"))
    M = torch.as_tensor(s["M"], device="cuda")
    src = s["src"] if s["src"] is not None else torch.zeros(T, dtype=torch.int64, device="cuda")
    phys = M[src[:, None], s["sel"]].reshape(-1)
    x, w = s["x"], s["w"].double().reshape(-1)
    out = torch.zeros((T, H), dtype=torch.float64, device="cuda")
    if case["grad"]:
        dx = torch.zeros_like(out)
        dw = torch.zeros(T * K, dtype=torch.float64, device="cuda")
        d1 = torch.zeros((C, 2 * I, H), dtype=torch.float64, device="cuda")
        d2 = torch.zeros((C, H, I), dtype=torch.float64, device="cuda")
    order = torch.argsort(phys)
    ends = torch.cumsum(torch.bincount(phys, minlength=C), 0).tolist()
    for c in range(C):
        a = order[(ends[c - 1] if c else 0):ends[c]]
        if not a.numel():
            continue
        t, wa = a // K, w[a][:, None]
        xr, w1, w2 = x[t].double(), s["fc1"][c].double(), s["fc2"][c].double()
        g, u = (xr @ w1.t()).split(I, dim=1)
        sig = torch.sigmoid(g)
        act = g * sig * u
        y = act @ w2.t()
        out.index_add_(0, t, y * wa)
        if case["grad"]:
            d = s["dout"][t].double()
            dw[a] = (d * y).sum(1)
            dy = d * wa
            d2[c] = dy.t() @ act
            da = dy @ w2
            dg = torch.cat([da * u * sig * (1 + g * (1 - sig)), da * g * sig], 1)
            d1[c] = dg.t() @ xr
            dx.index_add_(0, t, dg @ w1)
    if not case["grad"]:
        return {"out": out}
    per_copy = [d1[:, :I], d1[:, I:], d2] if case["split"] else [d1, d2]
    result = {"out": out, "grads": [dx, dw.reshape(T, K)] + per_copy}
    if case["fold"]:
        slots = torch.as_tensor(s["slots"], device="cuda")
        result["logical"] = [torch.zeros((E, *g.shape[1:]), dtype=torch.float64, device="cuda").index_add_(0, slots, g)
                             for g in per_copy]
        result["grads"][2:] = [g[slots] for g in result["logical"]]
    return result
