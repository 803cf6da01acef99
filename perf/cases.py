"""The work that programs have this library do, as measurable cases.

Every case goes through the C ABI entry points of include/q38m.h by way of
the package's ctypes binding, as the binding's users do.  One model geometry
(hidden 2048, 512 experts of intermediate 512, top-10), the weight formats
the library serves, and token counts from one to a 32,768-token chunk:

  decode   one token through the MoE block of several layers, each layer
           with its own weights and its own hidden row (attention lies
           between two MoE blocks, so a row does not depend on the block
           before it); with the router and the shared expert (block) or
           from given logits (not block)
  slab     q38m_moe_prefill_v1, 2 to 512 tokens
  chunk    q38m_moe_prefill_wide_v1, 513 to 32,768 tokens
  dense    the router GEMM, its top-10 and the shared expert
  hyper    the hyper-connection prepare and finish around the block
  weights  the load of a piece of an artifact: bf16 -> quantised -> layout

Weight policies (gate/up, down): "mixed" W4 groups of 32 / W8 per channel,
"w4" W4 groups of 32 in both, "interior" W4 groups of 128 with bf16 scales
in both and "edge" W8 groups of 128 with bf16 scales in both (the formats of
an artifact's inner and outer layers).
"""
import ctypes
import importlib.util
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "qwen3.8-flash-next-dual-gpu_amd")

H, I, E, K = 2048, 512, 512, 10
STREAMS = 4

# (bits, group, bf16 scales, scale sigma); group 0 is one scale per channel
W4 = (4, 32, False, 0.02)
W8 = (8, 0, False, 0.002)
W4_128 = (4, 128, True, 0.02)
W8_128 = (8, 128, True, 0.002)
POLICIES = {"mixed": (W4, W8), "w4": (W4, W4), "interior": (W4_128, W4_128), "edge": (W8_128, W8_128)}


def _q38m():
    name = "q38m_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(PACKAGE, "__init__.py"), submodule_search_locations=[PACKAGE])
        module = importlib.util.module_from_spec(spec)
        sys.modules[name] = module
        spec.loader.exec_module(module)
    return sys.modules[name]


# ---- the cases --------------------------------------------------------------

def listed():
    return [
        # one generated token: the smallest call and the one a server makes
        # most often; twelve layers, so that no layer's experts are cached
        {"name": "decode_block", "kind": "decode", "block": True, "policy": "mixed", "layers": 12},
        # a handful of sequences decoded together, or a draft being verified
        {"name": "slab_5_interior", "kind": "slab", "tokens": 5, "policy": "interior", "zipf": 0.0, "shared": True},
        # a short prompt: the 64-token all-W4 layer of the benchmark
        {"name": "slab_64_w4", "kind": "slab", "tokens": 64, "policy": "w4", "zipf": 0.0, "shared": False},
        # a full prefill slab: the benchmark's headline layer
        {"name": "slab_512_mixed", "kind": "slab", "tokens": 512, "policy": "mixed", "zipf": 0.0, "shared": False},
        # a ragged mid-size prompt through an edge layer
        {"name": "chunk_1500_edge", "kind": "chunk", "tokens": 1500, "policy": "edge", "zipf": 0.8, "shared": True},
        # a long prompt with skewed routing: the benchmark's 4,096-token chunk
        {"name": "chunk_4096_mixed", "kind": "chunk", "tokens": 4096, "policy": "mixed", "zipf": 1.1, "shared": False},
        # a long ragged prompt through an inner layer of an artifact
        {"name": "chunk_6001_interior", "kind": "chunk", "tokens": 6001, "policy": "interior", "zipf": 0.8, "shared": True},
        # the largest chunk, a layer of the benchmark's 48-layer stack
        {"name": "chunk_32768_mixed", "kind": "chunk", "tokens": 32768, "policy": "mixed", "zipf": 0.8, "shared": False},
        # router and shared expert of a prefill slab
        {"name": "dense_512", "kind": "dense", "tokens": 512},
        # and of a ragged chunk
        {"name": "dense_4099", "kind": "dense", "tokens": 4099},
        # hyper-connection prepare and finish of a chunk
        {"name": "hyper_2000", "kind": "hyper", "tokens": 2000, "hidden": 2048, "rank": 320},
        # a piece of an artifact on its way into the kernels' layout
        {"name": "weights_64", "kind": "weights", "experts": 64, "policy": "mixed"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["decode", "slab", "slab", "chunk", "chunk", "dense", "hyper", "weights"])
    policy = rng.choice(sorted(POLICIES))
    if kind == "decode":
        return {"kind": kind, "block": rng.random() < 0.5, "policy": policy, "layers": rng.randint(2, 12)}
    if kind == "slab":
        return {"kind": kind, "tokens": _log_int(rng, 2, 512), "policy": policy,
                "zipf": rng.choice([0.0, 0.8, 1.1]), "shared": rng.random() < 0.5}
    if kind == "chunk":
        return {"kind": kind, "tokens": _log_int(rng, 513, 16384), "policy": policy,
                "zipf": rng.choice([0.0, 0.8, 1.1]), "shared": rng.random() < 0.5}
    if kind == "dense":
        return {"kind": kind, "tokens": _log_int(rng, 2, 32768)}
    if kind == "hyper":
        return {"kind": kind, "tokens": _log_int(rng, 2, 8192), "hidden": rng.choice([2048, 2560]),
                "rank": 32 * rng.randint(2, 10)}
    return {"kind": kind, "experts": _log_int(rng, 4, 64), "policy": policy}


# ---- inputs -----------------------------------------------------------------

def _generator(seed, part):
    return torch.Generator(device="cuda").manual_seed((seed * 1000 + part) & 0x7FFFFFFFFFFFFFFF)


def _normal(g, *shape, sigma=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=g, device="cuda") * sigma).to(dtype)


def _raw_weights(fmt, rows, columns, g):
    """Row-major integers and scales: (data bytes, scales)."""
    bits, group, bf16, sigma = fmt
    if bits == 4:
        data = torch.randint(0, 256, (E, rows, columns // 2), generator=g, device="cuda", dtype=torch.uint8)
    else:
        data = torch.randint(-127, 128, (E, rows, columns), generator=g, device="cuda", dtype=torch.int8)
    shape = (E, rows, columns // group) if group else (E, rows, 1)
    scales = torch.randn(*shape, generator=g, device="cuda").abs_().mul_(sigma)
    return data, scales.to(torch.bfloat16 if bf16 else torch.float16)


def _raw_layer(policy, seed, layer):
    gate_up, down = POLICIES[policy]
    g = _generator(seed, 10 + layer)
    return _raw_weights(gate_up, 2 * I, H, g), _raw_weights(down, H, I, g)


def _device_weights(q, fmt, raw, rows, columns, paired):
    """The weights as the kernels read them, and their descriptor."""
    bits, group, bf16, _ = fmt
    row_major = q.DeviceWeights(raw[0], raw[1], q.FORMAT_W4_SYM if bits == 4 else q.FORMAT_W8_SYM, group,
                                q.LAYOUT_ROW_MAJOR, E, rows, columns, q.SCALE_BF16 if bf16 else q.SCALE_F16)
    return q.repack(row_major, paired=paired)


def _device_layer(q, policy, seed, layer):
    gate_up, down = POLICIES[policy]
    raw = _raw_layer(policy, seed, layer)
    return (_device_weights(q, gate_up, raw[0], 2 * I, H, True), _device_weights(q, down, raw[1], H, I, False))


def _logits(g, tokens, zipf):
    logits = torch.randn(tokens, E, generator=g, device="cuda")
    if zipf:
        p = torch.arange(1, E + 1, device="cuda", dtype=torch.float64) ** -zipf
        popularity = torch.log(p / p.sum())[torch.randperm(E, generator=g, device="cuda")]
        logits += popularity.float()
    return logits


def _tokens_in(case, seed):
    """Hidden rows, router logits and the shared expert's outputs of a slab or chunk."""
    g, t = _generator(seed, 1), case["tokens"]
    x = {"hidden": _normal(g, t, H), "logits": _logits(g, t, case["zipf"]), "shared": None, "gate": None}
    if case["shared"]:
        x["shared"], x["gate"] = _normal(g, t, H, sigma=0.5), _normal(g, t)
    return x


def _dense_weights(g):
    return {"router": _normal(g, E, H, sigma=H ** -0.5), "w_gate": _normal(g, I, H, sigma=0.02),
            "w_up": _normal(g, I, H, sigma=0.02), "w_down": _normal(g, H, I, sigma=0.04),
            "w_out": _normal(g, 1, H, sigma=0.02)}


def _decode_in(case, seed, layer):
    g = _generator(seed, 500 + layer)
    x = {"hidden": _normal(g, 1, H), "residual": _normal(g, 1, H), "logits": _logits(g, 1, 0.0)}
    x.update(_dense_weights(g))
    return x


def _dense_in(case, seed):
    g = _generator(seed, 2)
    x = _dense_weights(g)
    x["hidden"] = _normal(g, case["tokens"], H)
    return x


def _hyper_in(case, seed):
    g, t, h, r = _generator(seed, 3), case["tokens"], case["hidden"], case["rank"]
    wide = STREAMS * h
    return {"hyper": _normal(g, t, wide), "norm": _normal(g, wide, sigma=0.1),
            "down": _normal(g, r, wide, sigma=wide ** -0.5), "up": _normal(g, wide, r, sigma=2 * r ** -0.5),
            "inject": _normal(g, STREAMS, wide, sigma=wide ** -0.5), "block": _normal(g, t, h)}


# ---- prepare, run -----------------------------------------------------------

def _bytes(n):
    return torch.empty(n, dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    q = _q38m()
    kind = case["kind"]
    if kind == "decode":
        layers = []
        for layer in range(case["layers"]):
            x = _decode_in(case, seed, layer)
            x["weights"] = _device_layer(q, case["policy"], seed, layer)
            x["out"] = torch.empty(1, H, dtype=torch.bfloat16, device="cuda")
            layers.append(x)
        lib = q.lib()
        scratch = _bytes(max(lib.q38m_moe_decode_block_scratch_bytes(), lib.q38m_moe_decode_scratch_bytes()))
        return {"kind": kind, "block": case["block"], "layers": layers, "scratch": scratch}
    if kind in ("slab", "chunk"):
        x = _tokens_in(case, seed)
        x["kind"], x["tokens"] = kind, case["tokens"]
        x["weights"] = _device_layer(q, case["policy"], seed, 0)
        x["ws"] = (q.PrefillWorkspace_ if kind == "slab" else q.WideWorkspace_)(case["tokens"])
        x["out"] = torch.empty(case["tokens"], H, dtype=torch.bfloat16, device="cuda")
        return x
    if kind == "dense":
        x, t = _dense_in(case, seed), case["tokens"]
        x["kind"], x["tokens"] = kind, t
        x["logits"] = torch.empty(t, E, device="cuda")
        x["ids"] = torch.empty(t, K, dtype=torch.int32, device="cuda")
        x["weights"] = torch.empty(t, K, device="cuda")
        x["scratch"] = _bytes(q.lib().q38m_moe_shared_expert_scratch_bytes(t, I))
        x["shared"] = torch.empty(t, H, dtype=torch.bfloat16, device="cuda")
        x["gate"] = torch.empty(t, dtype=torch.bfloat16, device="cuda")
        return x
    if kind == "hyper":
        x, t, h = _hyper_in(case, seed), case["tokens"], case["hidden"]
        x.update(kind=kind, tokens=t, hidden=h, rank=case["rank"])
        x["scratch"] = _bytes(q.lib().q38m_hyper_prepare_scratch_bytes(t, h, case["rank"]))
        x["mixed"] = torch.empty(t, h, dtype=torch.bfloat16, device="cuda")
        x["injection"] = torch.empty(t, STREAMS, dtype=torch.bfloat16, device="cuda")
        x["out"] = torch.empty(t, STREAMS * h, dtype=torch.bfloat16, device="cuda")
        return x
    parts, g = [], _generator(seed, 4)
    for fmt, rows, columns, paired in zip(POLICIES[case["policy"]], (2 * I, H), (H, I), (True, False)):
        bits, group, bf16, _ = fmt
        source = _normal(g, case["experts"], rows, columns, sigma=0.02)
        buffers = []
        for layout in (q.LAYOUT_ROW_MAJOR, q.LAYOUT_MFMA16_PAIRED if paired else q.LAYOUT_MFMA16):
            data = _bytes(source.numel() * bits // 8)
            scales = torch.empty(source.numel() // (group or columns), device="cuda",
                                 dtype=torch.bfloat16 if bf16 else torch.float16)
            buffers.append(q.DeviceWeights(data, scales, q.FORMAT_W4_SYM if bits == 4 else q.FORMAT_W8_SYM, group,
                                           layout, case["experts"], rows, columns,
                                           q.SCALE_BF16 if bf16 else q.SCALE_F16))
        parts.append((source, *buffers))
    return {"kind": kind, "parts": parts}


def run(state):
    q = _q38m()
    kind, ptr, ref = state["kind"], q.ptr, ctypes.byref
    stream = q.stream_handle()
    if kind == "decode":
        scratch = ptr(state["scratch"])
        for x in state["layers"]:
            gate_up, down = (ref(w.desc) for w in x["weights"])
            if state["block"]:
                q.call("q38m_moe_decode_block_v1", gate_up, down, ptr(x["hidden"]), ptr(x["router"]),
                       ptr(x["w_gate"]), ptr(x["w_up"]), ptr(x["w_down"]), ptr(x["w_out"]), I, K,
                       ptr(x["residual"]), scratch, ptr(x["out"]), stream, 0)
            else:
                q.call("q38m_moe_decode_v1", gate_up, down, ptr(x["hidden"]), ptr(x["logits"]), K, None, None,
                       ptr(x["residual"]), scratch, ptr(x["out"]), stream, 0)
        return [x["out"] for x in state["layers"]]
    if kind in ("slab", "chunk"):
        gate_up, down = (ref(w.desc) for w in state["weights"])
        name, ws = (("q38m_moe_prefill_v1", state["ws"].ws) if kind == "slab"
                    else ("q38m_moe_prefill_wide_v1", state["ws"].wide))
        q.call(name, gate_up, down, ptr(state["hidden"]), ptr(state["logits"]), state["tokens"], ref(ws),
               ptr(state["shared"]), ptr(state["gate"]), ptr(state["out"]), stream, 0)
        return state["out"]
    if kind == "dense":
        x, t = state, state["tokens"]
        q.call("q38m_moe_router_v1", ptr(x["hidden"]), ptr(x["router"]), t, H, ptr(x["logits"]), stream, 0)
        q.call("q38m_topk_router_f32", ptr(x["logits"]), ptr(x["ids"]), ptr(x["weights"]), t, E, K, 1, stream, 0)
        q.call("q38m_moe_shared_expert_v1", ptr(x["hidden"]), ptr(x["w_gate"]), ptr(x["w_up"]), ptr(x["w_down"]),
               ptr(x["w_out"]), t, H, I, ptr(x["scratch"]), ptr(x["shared"]), ptr(x["gate"]), stream, 0)
        return {"logits": x["logits"], "ids": x["ids"], "weights": x["weights"], "shared": x["shared"],
                "gate": x["gate"]}
    if kind == "hyper":
        x, t, h = state, state["tokens"], state["hidden"]
        q.call("q38m_hyper_prepare_v1", ptr(x["hyper"]), ptr(x["norm"]), ptr(x["down"]), ptr(x["up"]),
               ptr(x["inject"]), t, h, x["rank"], ptr(x["scratch"]), ptr(x["mixed"]), ptr(x["injection"]),
               stream, 0)
        q.call("q38m_hyper_inject_bf16", ptr(x["hyper"]), ptr(x["block"]), ptr(x["injection"]), ptr(x["out"]), t, h,
               stream, 0)
        return {"mixed": x["mixed"], "injection": x["injection"], "out": x["out"]}
    out = []
    for source, row_major, laid_out in state["parts"]:
        q.call("q38m_quantize_expert_weights", ptr(source), ref(row_major.desc), stream, 0)
        q.call("q38m_repack_expert_weights", ref(row_major.desc), ref(laid_out.desc), stream, 0)
        out += [laid_out.data, laid_out.scales]
    return out


# ---- what a pass cannot do without ------------------------------------------

def _expert_bytes(fmt, rows, columns):
    bits, group, _, _ = fmt
    return rows * columns * bits // 8 + 2 * rows * (columns // group if group else 1)


def _active_experts(tokens, zipf):
    """Experts that get a token, expected: uniform routing exactly, skewed
    routing from the Zipf share of each expert (capped at one route a token)."""
    share = [1.0 / E] * E
    if zipf:
        share = [(r + 1) ** -zipf for r in range(E)]
        share = [s / sum(share) for s in share]
    return sum(1.0 - (1.0 - min(1.0, K * s)) ** tokens for s in share)


def work(case):
    kind = case["kind"]
    dense = 2 * (E * H + 3 * H * I + H)  # bytes of the router and the shared expert
    if kind == "weights":
        gate_up, down = POLICIES[case["policy"]]
        n = case["experts"]
        written = n * (_expert_bytes(gate_up, 2 * I, H) + _expert_bytes(down, H, I))
        return {"bytes": n * 3 * I * H * 2 + written, "flops": 0}
    if kind == "dense":
        t = case["tokens"]
        return {"bytes": dense + t * (2 * H + 4 * E + 8 * K + 2 * H + 2),
                "flops": 2 * t * (E * H + 3 * H * I + H)}
    if kind == "hyper":
        t, h, r = case["tokens"], case["hidden"], case["rank"]
        wide = STREAMS * h
        return {"bytes": 2 * (t * (2 * wide + 2 * h + STREAMS) + wide * (2 * r + STREAMS + 1)),
                "flops": 2 * t * wide * (2 * r + STREAMS)}
    gate_up, down = POLICIES[case["policy"]]
    expert = _expert_bytes(gate_up, 2 * I, H) + _expert_bytes(down, H, I)
    if kind == "decode":
        layer = K * expert + 2 * 3 * H + (dense if case["block"] else 4 * E)
        flops = 2 * K * 3 * H * I + (2 * (E * H + 3 * H * I + H) if case["block"] else 0)
        return {"bytes": case["layers"] * layer, "flops": case["layers"] * flops}
    t = case["tokens"]
    per_token = 2 * H + 4 * E + 2 * H + (2 * H + 2 if case["shared"] else 0)
    return {"bytes": round(_active_experts(t, case["zipf"])) * expert + t * per_token,
            "flops": 2 * t * K * 3 * H * I}


def tolerance(case):
    # Measured against exact() on the kernels' own rounding sequence (bf16
    # gate, up and mid values, int8 rows): four times what that shows.
    kind = case["kind"]
    if kind == "weights":
        return "exact"
    if kind == "hyper":
        return {"rel": 1.0e-2}
    if kind == "dense":
        return {"rel": 1.2e-2, "differ": 1e-3}
    return {"rel": 1.6e-2}


# ---- 64-bit results ---------------------------------------------------------

def _exact_weights(fmt, raw, expert, columns):
    bits, group, _, _ = fmt
    data, scales = raw[0][expert], raw[1][expert].double()
    if bits == 4:
        low, high = (data & 15).to(torch.int16), (data >> 4).to(torch.int16)
        values = torch.stack((low, high), dim=-1).reshape(data.shape[0], columns)
        values = values - 16 * (values > 7)
    else:
        values = data
    return values.double() * scales.repeat_interleave(group or columns, dim=1)


def _exact_int8(x):
    """Rows as the int8 activations represent them (absmax / 127 per row)."""
    s = x.abs().amax(dim=1, keepdim=True) / 127
    s = torch.where(s == 0, torch.ones_like(s), s)
    return (x / s).round().clamp(-127, 127) * s


def _exact_silu(g):
    return g / (1 + torch.exp(-g))


def _exact_routed(policy, raw, hidden, logits):
    gate_up, down = POLICIES[policy]
    x = _exact_int8(hidden.double())
    top, ids = logits.double().topk(K, dim=1)
    weights = torch.softmax(top, dim=1)
    out = torch.zeros_like(x)
    for e in ids.unique().tolist():
        token, rank = (ids == e).nonzero(as_tuple=True)
        y = x[token] @ _exact_weights(gate_up, raw[0], e, H).t()
        mid = _exact_silu(y[:, :I]) * y[:, I:] * weights[token, rank].unsqueeze(1)
        out.index_add_(0, token, _exact_int8(mid) @ _exact_weights(down, raw[1], e, I).t())
    return out


def _exact_shared(x):
    h = x["hidden"].double()
    mid = _exact_silu(h @ x["w_gate"].double().t()) * (h @ x["w_up"].double().t())
    return mid @ x["w_down"].double().t(), (h @ x["w_out"].double().t())


def exact(case, seed):
    kind = case["kind"]
    if kind == "weights":
        return None  # bytes
    if kind == "decode":
        out = []
        for layer in range(case["layers"]):
            x = _decode_in(case, seed, layer)
            logits = x["hidden"].double() @ x["router"].double().t() if case["block"] else x["logits"]
            y = _exact_routed(case["policy"], _raw_layer(case["policy"], seed, layer), x["hidden"], logits)
            if case["block"]:
                shared, gate = _exact_shared(x)
                y = y + shared * torch.sigmoid(gate)
            out.append(y + x["residual"].double())
        return out
    if kind in ("slab", "chunk"):
        x = _tokens_in(case, seed)
        y = _exact_routed(case["policy"], _raw_layer(case["policy"], seed, 0), x["hidden"], x["logits"])
        if case["shared"]:
            y = y + x["shared"].double() * torch.sigmoid(x["gate"].double()).unsqueeze(1)
        return y
    if kind == "dense":
        x = _dense_in(case, seed)
        logits = x["hidden"].double() @ x["router"].double().t()
        shared, gate = _exact_shared(x)
        return {"logits": logits, "ids": None, "weights": torch.softmax(logits.topk(K, dim=1)[0], dim=1),
                "shared": shared, "gate": gate.squeeze(1)}
    x, t, h = _hyper_in(case, seed), case["tokens"], case["hidden"]
    state = x["hyper"].double()
    streams = state.view(t, STREAMS, h)
    norm = streams / torch.sqrt((streams * streams).mean(dim=2, keepdim=True) + 1e-6)
    norm = norm.reshape(t, -1) * (1 + x["norm"].double())
    low = _exact_silu((norm @ x["down"].double().t()) / STREAMS)
    mix = torch.sigmoid(low @ x["up"].double().t())
    mixed = (norm * mix).view(t, STREAMS, h).sum(dim=1) / STREAMS
    injection = 2 * torch.sigmoid((norm @ x["inject"].double().t()) / STREAMS)
    out = streams + x["block"].double().unsqueeze(1) * injection.unsqueeze(2)
    return {"mixed": mixed, "injection": injection, "out": out.reshape(t, -1)}
