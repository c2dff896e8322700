"""The measured work: fused MoE layers, the shared MLP and the W8A8 linears, each through its public entry point.

A case is a dict of plain values with a ``kind``:

* ``moe``: one MoE layer forward. ``dtype`` picks the weights (``w8a8``, ``w8a16``, ``bf16``),
  ``shared`` the routed+shared entry point, ``zipf`` a skewed routing, ``router`` the top-k
  softmax router in front of the layer, ``ids32`` int32 expert ids.
* ``shared_mlp``: the dense gate/up/down MLP.
* ``i8gemm``: one dynamic-per-row W8A8 linear; ``pair``: two that share the row quantisation.
"""

from __future__ import annotations

import math

import torch

from fused_cpp_amd import i8gemm, moe, router

# The DeepSeek-V3 layer that the repository's benchmark runs, its 384-expert form, the
# reference's tensor-parallel rank, and the plumbing layer of the benchmark.
_DSV3 = {"H": 7168, "F": 2048, "E": 256, "k": 8, "shared": True, "scale": 2.5}
_DSV3_384 = {**_DSV3, "E": 384}
_TP_RANK = {"H": 4096, "F": 512, "E": 20, "k": 6, "shared": True, "scale": 2.5}
_PLUMB = {"H": 1024, "F": 512, "E": 8, "k": 2, "shared": False, "scale": 1.0}

# DeepSeek-V4 attention projections: wq_b with the indexer's projection, and wo_b.
_PAIR_Q = {"K": 1536, "N": 24576, "N2": 8192}
_WO_B = {"K": 16384, "N": 7168}


def _moe(dtype, T, shape, *, act="silu", zipf=0.0, router=False, ids32=False, bias=False):
    return {"kind": "moe", "dtype": dtype, "T": T, **shape, "act": act, "zipf": zipf, "router": router,
            "ids32": ids32, "bias": bias}


def listed():
    return [
        # Bring-up and unit-sized layers: a call that is all launches and host work.
        {"name": "bf16_small_t32", **_moe("bf16", 32, _PLUMB)},
        # Single-stream decode: one token through a DeepSeek-V3 layer, latency bound.
        {"name": "w8a8_decode_t1", **_moe("w8a8", 1, _DSV3)},
        # The benchmark's headline: a decode batch of 64 sequences.
        {"name": "w8a8_decode_t64", **_moe("w8a8", 64, _DSV3)},
        # A serving step that mixes decodes with a chunk of a prompt, from the router's logits on.
        {"name": "w8a8_router_t333", **_moe("w8a8", 333, _DSV3, router=True, ids32=True)},
        # Prefill of a long prompt with skewed expert popularity.
        {"name": "w8a8_prefill_zipf_t4096", **_moe("w8a8", 4096, _DSV3, zipf=1.2)},
        # The largest step: 8192 prompt tokens over 384 experts.
        {"name": "w8a8_prefill_e384_t8192", **_moe("w8a8", 8192, _DSV3_384)},
        # Decode with unquantised experts.
        {"name": "bf16_decode_t32", **_moe("bf16", 32, _DSV3)},
        # One tensor-parallel rank's prompt chunk, clamped SwiGLU, an odd number of tokens.
        {"name": "bf16_tp_clamp_t2047", **_moe("bf16", 2047, _TP_RANK, act="clamp")},
        # Prefill with int8 checkpoint weights and bf16 activations.
        {"name": "w8a16_prefill_t4096", **_moe("w8a16", 4096, _DSV3)},
        # The shared expert run by itself in a decode step.
        {"name": "shared_mlp_t64", "kind": "shared_mlp", "T": 64, "H": 7168, "F": 2048, "act": "silu"},
        # Attention projections of a decode step that share one quantisation of the rows.
        {"name": "i8gemm_pair_t64", "kind": "pair", "T": 64, **_PAIR_Q},
        # The attention output projection of a prompt.
        {"name": "i8gemm_wo_b_t4096", "kind": "i8gemm", "T": 4096, **_WO_B, "x32": False, "out32": False,
         "bias": False},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_once(rng):
    kind = rng.choice(["w8a8", "w8a8", "w8a8", "bf16", "bf16", "w8a16", "w8a16", "shared_mlp", "i8gemm", "i8gemm",
                       "pair"])
    if kind == "shared_mlp":
        shape = rng.choice([(7168, 2048), (4096, 2048), (4096, 512), (rng.randrange(128, 4096), rng.randrange(64, 2048))])
        return {"kind": kind, "T": _log_int(rng, 1, 4096), "H": shape[0], "F": shape[1],
                "act": rng.choice(["silu", "clamp"])}
    if kind == "i8gemm":
        shape = rng.choice([_WO_B, {"K": 1536, "N": 24576}, {"K": 4096, "N": 7168},
                            {"K": rng.randrange(64, 8192), "N": rng.randrange(64, 8192)}])
        return {"kind": kind, "T": _log_int(rng, 1, 8192), **shape, "x32": rng.random() < 0.25,
                "out32": rng.random() < 0.25, "bias": rng.random() < 0.25}
    if kind == "pair":
        shape = rng.choice([_PAIR_Q, {"K": 7168, "N": 1536, "N2": 512},
                            {"K": rng.randrange(64, 8192), "N": rng.randrange(64, 8192), "N2": rng.randrange(64, 4096)}])
        return {"kind": kind, "T": _log_int(rng, 1, 8192), **shape}
    E = rng.choice([4, 16, 60, 128])
    odd = {"H": rng.randrange(128, 4096), "F": rng.randrange(64, 1536), "E": E, "k": rng.randint(1, min(8, E)),
           "shared": rng.random() < 0.5, "scale": 1.5}
    if kind != "bf16":  # int8 experts come in whole 16-channel tiles
        odd["H"], odd["F"] = odd["H"] // 16 * 16, odd["F"] // 16 * 16
    shape = rng.choice([_DSV3, _DSV3, _DSV3_384, {**_DSV3, "F": 256}, _TP_RANK, _PLUMB, odd])
    act = "silu"
    if kind != "w8a8":
        act = rng.choice(["silu", "clamp"] if shape["shared"] else ["silu", "clamp", "gelu"])
        if kind == "bf16" and not shape["shared"] and rng.random() < 0.3:
            act = "swigluoai"
    return _moe(kind, _log_int(rng, 1, 8192), shape, act=act, zipf=rng.choice([0.0, 0.0, 1.2]),
                router=rng.random() < 0.2, ids32=rng.random() < 0.5,
                bias=kind == "bf16" and not shape["shared"] and act != "clamp" and rng.random() < 0.5)


def _price(case):
    """Seconds of a pass at rates that the large listed cases come near to; only to bound what is drawn."""
    w = work(case)
    int8 = case["kind"] in ("i8gemm", "pair") or case.get("dtype") == "w8a8"
    return w["bytes"] / 6e12 + w["flops"] / (2e15 if int8 else 0.8e15)


def draw(rng):
    # By what the drawn sizes cost, none above the largest listed case.
    limit = max(_price(c) for c in listed())
    while True:
        case = _draw_once(rng)
        if _price(case) <= limit:
            return case


# ------------------------------------------------------------------ inputs --

def _gen(seed, stream, device):
    return torch.Generator(device=device).manual_seed((int(seed) * 1000003 + 7919 * stream + 17) % (2 ** 62))


def _int8_weight(seed, stream, n, k):
    """[n, k] int8 weights as per-channel quantisation of Gaussian weights leaves them, and their fp32 scales."""
    g = _gen(seed, stream, "cuda")
    q = torch.randn((n, k), generator=g, device="cuda", dtype=torch.bfloat16).mul_(30).round_().clamp_(-127, 127)
    scale = (torch.rand(n, generator=g, device="cuda") * 0.6 + 0.7) * (1.7 / math.sqrt(k) / 30)
    return q.to(torch.int8), scale


def _bf16_weight(seed, stream, n, k):
    return torch.randn((n, k), generator=_gen(seed, stream, "cuda"), device="cuda",
                       dtype=torch.bfloat16).mul_(1.7 / math.sqrt(k))


def _expert_bias(case, seed):
    if not case.get("bias"):
        return None, None
    g = _gen(seed, 3, "cuda")
    return (torch.randn((case["E"], 2 * case["F"]), generator=g, device="cuda") * 0.2,
            torch.randn((case["E"], case["H"]), generator=g, device="cuda") * 0.2)


def _rows(seed, rows, cols, dtype=torch.bfloat16):
    return torch.randn((rows, cols), generator=_gen(seed, 0, "cuda"), device="cuda").to(dtype)


def _logits(case, seed, device):
    """Router logits [T, E]: independent, or over a Zipf popularity of a random expert order."""
    g = _gen(seed, 1, device)
    T, E = case["T"], case["E"]
    if not case["zipf"]:
        return torch.randn((T, E), generator=g, device=device)
    rank = torch.randperm(E, generator=g, device=device).float() + 1
    uniform = torch.rand((T, E), generator=g, device=device).clamp_(1e-7, 1 - 1e-7)
    return -case["zipf"] * torch.log(rank)[None, :] - torch.log(-torch.log(uniform))


def _route(logits, k):
    """Top-k ids (the lower id first among equals) and the renormalised softmax weights, in the logits' own type."""
    top, ids = torch.sort(logits, dim=1, descending=True, stable=True)
    return ids[:, :k].contiguous(), torch.softmax(top[:, :k], dim=1).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "moe":
        return _prepare_moe(case, seed)
    if kind == "shared_mlp":
        w = moe.prepare_shared_mlp_bf16_tiled_weights(_bf16_weight(seed, 10, 2 * case["F"], case["H"]),
                                                      _bf16_weight(seed, 11, case["H"], case["F"]))
        return {"case": case, "x": _rows(seed, case["T"], case["H"]), "weights": w}
    first = i8gemm.prepare(*_int8_weight(seed, 10, case["N"], case["K"]))
    x = _rows(seed, case["T"], case["K"], torch.float32 if case.get("x32") else torch.bfloat16)
    if kind == "pair":
        return {"case": case, "x": x, "first": first,
                "second": i8gemm.prepare(*_int8_weight(seed, 11, case["N2"], case["K"]))}
    bias = torch.randn(case["N"], generator=_gen(seed, 3, "cuda"), device="cuda") if case["bias"] else None
    return {"case": case, "x": x, "first": first, "bias": bias}


def _prepare_moe(case, seed):
    E, H, F = case["E"], case["H"], case["F"]
    total = E + int(case["shared"])
    if case["dtype"] == "bf16":
        w13 = torch.empty((total, 2 * F, H), dtype=torch.bfloat16, device="cuda")
        w2 = torch.empty((total, H, F), dtype=torch.bfloat16, device="cuda")
        for e in range(total):
            w13[e] = _bf16_weight(seed, 10 + 2 * e, 2 * F, H)
            w2[e] = _bf16_weight(seed, 11 + 2 * e, H, F)
        if case["shared"]:
            weights = moe.prepare_routed_shared_moe_bf16_tiled_weights(w13[:E], w2[:E], w13[E], w2[E])
        else:
            weights = moe.prepare_fused_moe_bf16_tiled_weights(w13, w2, fuse_silu=case["act"] in ("silu", "clamp"))
    else:
        q13 = torch.empty((total, 2 * F, H), dtype=torch.int8, device="cuda")
        q2 = torch.empty((total, H, F), dtype=torch.int8, device="cuda")
        s13 = torch.empty((total, 2 * F), device="cuda")
        s2 = torch.empty((total, H), device="cuda")
        for e in range(total):
            q13[e], s13[e] = _int8_weight(seed, 10 + 2 * e, 2 * F, H)
            q2[e], s2[e] = _int8_weight(seed, 11 + 2 * e, H, F)
        name = case["dtype"]
        if case["shared"]:
            weights = getattr(moe, f"prepare_routed_shared_moe_{name}_tiled_quantized_weights")(
                q13[:E], s13[:E], q2[:E], s2[:E], q13[E], s13[E], q2[E], s2[E])
        else:
            weights = getattr(moe, f"prepare_fused_moe_{name}_tiled_quantized_weights")(q13, s13, q2, s2)
    state = {"case": case, "x": _rows(seed, case["T"], H), "weights": weights}
    logits = _logits(case, seed, "cuda")
    state["ids_dtype"] = torch.int32 if case["ids32"] else torch.int64
    if case["router"]:
        state["logits"] = logits
    else:
        ids, state["topk_weights"] = _route(logits, case["k"])
        state["topk_ids"] = ids.to(state["ids_dtype"])
    state["bias"] = _expert_bias(case, seed)
    return state


# --------------------------------------------------------------------- run --

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "moe":
        return _run_moe(case, state)
    if kind == "shared_mlp":
        return moe.shared_mlp_bf16_tiled(state["x"], state["weights"],
                                         swiglu_limit=10.0 if case["act"] == "clamp" else None)
    if kind == "pair":
        return i8gemm.dynamic_scaled_mm_pair(state["x"], state["first"], state["second"])
    return i8gemm.dynamic_scaled_mm(state["x"], state["first"], bias=state["bias"],
                                    out_dtype=torch.float32 if case["out32"] else torch.bfloat16)


def _run_moe(case, state):
    if case["router"]:
        ids, weights = router.topk_softmax(state["logits"], case["k"], ids_dtype=state["ids_dtype"])
    else:
        ids, weights = state["topk_ids"], state["topk_weights"]
    options = {}
    if case["dtype"] == "w8a8" or case["act"] == "clamp":
        options["swiglu_limit"] = 10.0
    elif case["act"] != "silu":
        options["activation"] = case["act"]
    if case["shared"]:
        call = getattr(moe, f"fused_moe_{case['dtype']}_tiled_with_shared")
        out = call(state["x"], state["weights"], weights, ids, routed_scaling_factor=case["scale"], **options)
    else:
        if case["bias"]:
            options["w13_bias"], options["w2_bias"] = state["bias"]
        out = moe.fused_moe_tiled(state["x"], state["weights"], weights, ids, **options)
    return (out, ids, weights) if case["router"] else out


# -------------------------------------------------------------------- work --

def work(case):
    kind, T = case["kind"], case["T"]
    if kind == "shared_mlp":
        H, F = case["H"], case["F"]
        return {"bytes": 6 * H * F + 4 * T * H, "flops": 6 * T * H * F}
    if kind in ("i8gemm", "pair"):
        K = case["K"]
        N = case["N"] + case.get("N2", 0)
        x, out = (4 if case.get("x32") else 2), (4 if case.get("out32") else 2)
        return {"bytes": N * K + 4 * N + T * (x * K + out * N), "flops": 2 * T * N * K}
    H, F, E, k = case["H"], case["F"], case["E"], case["k"]
    # One routing of the same distribution says how many experts' weights have to be read.
    ids, _ = _route(_logits(case, 0, "cpu"), k)
    active = int(torch.unique(ids).numel()) + int(case["shared"])
    size = 2 if case["dtype"] == "bf16" else 1
    expert = 3 * H * F * size + (4 * (2 * F + H) if size == 1 or case["bias"] else 0)
    routing = T * k * ((4 if case["ids32"] else 8) + 4)
    if case["router"]:
        routing += 4 * T * E
    return {"bytes": active * expert + 4 * T * H + routing, "flops": 6 * T * (k + int(case["shared"])) * H * F}


def tolerance(case):
    # About four times the distance from 64-bit arithmetic that was measured over listed and drawn
    # cases: fp32 results 4.1e-8 (largest 2.6e-7); bf16 results whose integers are exact 1.7e-3, which
    # is their rounding alone (largest 3.9e-3; 1.2e-2 where a requantised integer falls the other
    # way); with a bf16 intermediate of 32-bit sums 2.4e-3 (1.3e-2). Ids are ordered by the logits.
    if case["kind"] in ("i8gemm", "pair"):
        return {"rel": 2e-7, "max": 1.1e-6} if case.get("out32") else {"rel": 7e-3, "max": 1.6e-2}
    return {"rel": 7e-3 if case.get("dtype") == "w8a8" else 1e-2, "max": 5e-2, "differ": 0.0}


# ------------------------------------------------------------------- exact --

def _quantise(v, to_even=False):
    """Dynamic per-row int8: the integers and the row scales, as 64-bit values.

    The integers are defined by a binary32 scale and product (a quotient, rounded to even, for the
    linears); bf16 rows meet many exact ties, so that definition is kept here.
    """
    v = v.float()
    top = v.abs().amax(dim=1, keepdim=True)
    scale = torch.where(top > 0, top / torch.full_like(top, 127.0), torch.ones_like(top))
    if to_even:
        return torch.round(v / scale).clamp_(-128, 127).double(), scale.double()
    q = (v * (1.0 / scale)).clamp_(-127, 127).double()
    return torch.sign(q) * torch.floor(q.abs() + 0.5), scale.double()


def _activate(gu, act, f):
    if act == "swigluoai":
        gate, up = gu[:, 0::2].clamp(max=7.0), gu[:, 1::2].clamp(-7.0, 7.0)
        return (up + 1) * gate * torch.sigmoid(1.702 * gate)
    gate, up = gu[:, :f], gu[:, f:]
    if act == "gelu":
        return 0.5 * gate * (1 + torch.erf(gate / math.sqrt(2.0))) * up
    if act == "clamp":
        gate, up = gate.clamp(max=10.0), up.clamp(-10.0, 10.0)
    return gate * torch.sigmoid(gate) * up


def _expert_rows(case, seed, e, rows, scale, bias):
    """One expert's W2 rows in 64 bits; rows are the token rows, with the integers' scale for W8A8."""
    H, F = case["H"], case["F"]
    if case.get("dtype", "bf16") == "bf16":
        first = 10 if case["kind"] == "shared_mlp" else 10 + 2 * e
        w13, w2 = _bf16_weight(seed, first, 2 * F, H).double(), _bf16_weight(seed, first + 1, H, F).double()
        gu = rows @ w13.t()
        if bias[0] is not None:
            gu += bias[0][e].double()
        out = _activate(gu, case["act"], F) @ w2.t()
        return out if bias[1] is None else out + bias[1][e].double()
    q13, s13 = _int8_weight(seed, 10 + 2 * e, 2 * F, H)
    q2, s2 = _int8_weight(seed, 11 + 2 * e, H, F)
    gu = (rows @ q13.double().t()) * s13.double()
    if case["dtype"] == "w8a16":
        return (_activate(gu, case["act"], F) @ q2.double().t()) * s2.double()
    # The W8A8 layer is defined on a bf16 intermediate that is quantised again.
    y, y_scale = _quantise(_activate(gu * scale, "clamp", F).to(torch.bfloat16))
    return (y @ q2.double().t()) * (y_scale * s2.double())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("i8gemm", "pair"):
        x = _rows(seed, case["T"], case["K"], torch.float32 if case.get("x32") else torch.bfloat16)
        q, scale = _quantise(x.double(), to_even=True)
        outs = []
        for stream, n in ((10, case["N"]), (11, case.get("N2"))):
            if n is not None:
                w, s = _int8_weight(seed, stream, n, case["K"])
                outs.append((q @ w.double().t()) * (scale * s.double()))
        if case.get("bias"):
            outs[0] += torch.randn(case["N"], generator=_gen(seed, 3, "cuda"), device="cuda").double()
        return tuple(outs) if kind == "pair" else outs[0]
    x = _rows(seed, case["T"], case["H"]).double()
    if kind == "shared_mlp":
        return _expert_rows(case, seed, 0, x, None, (None, None))
    logits = _logits(case, seed, "cuda")
    ids, weights = _route(logits.double() if case["router"] else logits, case["k"])
    routed = weights.double() * (case["scale"] if case["shared"] else 1.0)
    rows, scale = _quantise(x) if case["dtype"] == "w8a8" else (x, torch.ones((case["T"], 1), device="cuda"))
    bias = _expert_bias(case, seed)
    out = torch.zeros((case["T"], case["H"]), dtype=torch.float64, device="cuda")
    for e in range(case["E"]):
        token, slot = torch.nonzero(ids == e, as_tuple=True)
        if token.numel():
            out.index_add_(0, token, _expert_rows(case, seed, e, rows[token], scale[token], bias)
                           * routed[token, slot][:, None])
    if case["shared"]:
        out += _expert_rows(case, seed, case["E"], rows, scale, bias)
    return (out, None, weights) if case["router"] else out
