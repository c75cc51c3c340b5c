"""Work that users have this package do, as cases that can be measured.

A case is one pass through the public entry points: a single `MatGPTQLinear` call, the linears of a
decoder's blocks as a serving engine runs them (decode steps and small batches from a captured graph,
larger batches eagerly), a token and a prompt of the decoder, and the load-time packing of a block.
`listed()` names the typical ones, `draw(rng)` gives others out of the same ranges.

Sizes of a block: `hidden`, `ffn`, `heads` and `kv_heads` of head dimension 128, q/k/v and gate/up fused,
sharded over `tp` ranks the way a tensor-parallel engine does (one rank's share is what runs here).
"""
import math

import torch

from matgptq_amd.decoder import DecodeSession, DecoderConfig, random_mixnmatch_decoder
from matgptq_amd.ops import matryoshka_slice
from matgptq_cuda.matgptq_linear import MatGPTQLinear
from vllm_matgptq import MatGPTQConfig, MatGPTQLinearMethod

HEAD_DIM = 128
BITS = (2, 3, 4, 6, 8)
LLAMA_8B = {"hidden": 4096, "ffn": 14336, "heads": 32, "kv_heads": 8, "tp": 1}
LLAMA_70B = {"hidden": 8192, "ffn": 28672, "heads": 64, "kv_heads": 8, "tp": 1}
STACK_BYTES = 512e6  # weights of a stack: past what the caches of the GPU hold, as a whole model's are


def listed():
    return [
        # one layer called on its own from Python, batch 1: the call's latency
        {"name": "call m1", "kind": "call", "n": 4096, "k": 4096, "m": 1, "bits": 4, "group": 128,
         "dtype": "float16", "zeros": False},
        # single-sequence decoding: the linears of eight blocks out of a graph
        {"name": "decode m1", "kind": "stack", **LLAMA_8B, "blocks": 8, "m": 1, "bits": 4, "group": 128,
         "dtype": "float16", "zeros": True, "planes": False},
        # a few sequences at once, low bitwidth, bfloat16 as serving engines default to
        {"name": "decode m8", "kind": "stack", **LLAMA_8B, "blocks": 10, "m": 8, "bits": 3, "group": 128,
         "dtype": "bfloat16", "zeros": False, "planes": False},
        # one rank of a large model sharded over eight: small, thin layers
        {"name": "decode m16 shard", "kind": "stack", **{**LLAMA_70B, "tp": 8}, "blocks": 10, "m": 16, "bits": 4,
         "group": 128, "dtype": "float16", "zeros": True, "planes": False},
        # one copy of the master codes in memory, bitwidth chosen at run time
        {"name": "decode m2 planes", "kind": "stack", **LLAMA_8B, "blocks": 4, "m": 2, "bits": 4, "group": 128,
         "dtype": "float16", "zeros": True, "planes": True},
        # a serving batch of 64 sequences
        {"name": "batch m64", "kind": "stack", **LLAMA_8B, "blocks": 5, "m": 64, "bits": 4, "group": 128,
         "dtype": "float16", "zeros": True, "planes": False},
        # a chunk of a prompt, ragged, bfloat16, one scale per 32 columns
        {"name": "prefill m333", "kind": "eager", **LLAMA_8B, "m": 333, "bits": 8, "group": 32, "dtype": "bfloat16",
         "zeros": False, "planes": False},
        # a long prompt on a large model
        {"name": "prefill m2048", "kind": "eager", **LLAMA_70B, "m": 2048, "bits": 4, "group": 128,
         "dtype": "float16", "zeros": True, "planes": False},
        # a prompt on the master-resident codes
        {"name": "prefill m512 planes", "kind": "eager", **LLAMA_8B, "m": 512, "bits": 3, "group": 128,
         "dtype": "float16", "zeros": True, "planes": True},
        # one token of a decoder with a bitwidth per layer, half a thousand tokens of context
        {"name": "token", "kind": "token", "hidden": 4096, "ffn": 14336, "heads": 32, "kv_heads": 8, "layers": 32,
         "vocab": 128256, "m": 512},
        # the prompt in front of it
        {"name": "prompt", "kind": "prompt", "hidden": 4096, "ffn": 14336, "heads": 32, "kv_heads": 8, "layers": 32,
         "vocab": 128256, "m": 512},
        # loading: master codes in GPU memory -> sliced and packed layers of one block
        {"name": "load", "kind": "load", **LLAMA_8B, "bits": 4, "group": 128, "dtype": "float16", "zeros": True,
         "route": "plugin"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _format(rng):
    return {"bits": rng.choice(BITS), "group": rng.choice((128, 128, 128, 32, -1)),
            "dtype": rng.choice(("float16", "float16", "bfloat16")), "zeros": rng.random() < 0.5}


def _block(rng):
    """Sizes of a decoder block and a tensor-parallel degree that divides them."""
    heads = _log_int(rng, 8, 64)
    kv_heads = rng.choice([h for h in (heads, heads // 2, heads // 4, heads // 8) if h and heads % h == 0])
    tp = rng.choice([t for t in (1, 1, 2, 4, 8) if heads % t == 0 and kv_heads % t == 0])
    ffn = 128 * tp * round(heads * rng.uniform(2.0, 4.0) / tp)
    return {"hidden": heads * HEAD_DIM, "ffn": ffn, "heads": heads, "kv_heads": kv_heads, "tp": tp}


def _draw(rng):
    kind = rng.choice(("call", "stack", "stack", "stack", "stack", "eager", "eager", "eager", "token", "prompt", "load"))
    if kind == "call":
        case = {"kind": kind, "n": 16 * _log_int(rng, 32, 1024), "k": 128 * _log_int(rng, 4, 128),
                "m": _log_int(rng, 1, 16), **_format(rng)}
        if case["group"] != 128 and rng.random() < 0.3:
            case["k"] += 64
        return case
    if kind in ("token", "prompt"):
        heads, kv_heads = rng.choice(((16, 4), (16, 16), (20, 20), (24, 3), (32, 8), (40, 40), (64, 8)))
        return {"kind": kind, "hidden": heads * HEAD_DIM, "ffn": 128 * round(heads * rng.uniform(2.5, 4.0)), "heads": heads,
                "kv_heads": kv_heads, "layers": rng.randint(4, 32), "vocab": rng.choice((32000, 50304, 128256)),
                "m": _log_int(rng, 64, 4096) if kind == "token" else _log_int(rng, 32, 2048)}
    block, fmt = _block(rng), _format(rng)
    planes = rng.random() < 0.25
    if fmt["group"] != 128 and not planes and block["tp"] == 1 and rng.random() < 0.3:
        block["ffn"] += 64  # down: a number of input features that is not a multiple of 128
    if kind == "load":
        return {"kind": kind, **block, **fmt, "route": rng.choice(("plugin", "plugin", "module", "planes"))}
    if kind == "eager":
        return {"kind": kind, **block, "m": _log_int(rng, 257, 4096), **fmt, "planes": planes}
    case = {"kind": kind, **block, "blocks": 16, "m": _log_int(rng, 1, 256), **fmt, "planes": planes}
    one = sum(n * k for n, k in shapes(case).values()) * (8 if planes else fmt["bits"]) / 8
    case["blocks"] = max(2, min(16, math.ceil(STACK_BYTES / one)))
    return case


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 1e15)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= most:
            return case


def shapes(case):
    """name -> (output features, input features) of one rank's linears of a block."""
    hidden, ffn, heads, kv_heads, tp = (case[k] for k in ("hidden", "ffn", "heads", "kv_heads", "tp"))
    return {"qkv": ((heads + 2 * kv_heads) * HEAD_DIM // tp, hidden), "o": (hidden, heads * HEAD_DIM // tp),
            "gate_up": (2 * ffn // tp, hidden), "down": (hidden, ffn // tp)}


def _groups(case, k):
    return 1 if case["group"] == -1 else k // case["group"]


def _dtype(case):
    return torch.bfloat16 if case.get("dtype") == "bfloat16" else torch.float16


def _checkpoint(gen, case, n, k):
    """Master codes, scales and zero points of a layer as a quantiser leaves them: bell-shaped codes around
    the zero point, weights of about 1 / sqrt(k)."""
    def new():
        return torch.empty((n, _groups(case, k)), dtype=torch.float32, device="cuda")

    codes = torch.empty((n, k), dtype=torch.float16, device="cuda").normal_(128.0, 36.0, generator=gen)
    codes = codes.round_().clamp_(0.0, 255.0).to(torch.uint8)
    scale = (new().uniform_(0.5, 1.5, generator=gen) / (36.0 * math.sqrt(k))).to(_dtype(case))
    zero = new().normal_(128.0, 6.0, generator=gen).round_().to(_dtype(case)) if case["zeros"] else None
    return codes, scale, zero


def _plugin_layer(case, codes, scale, zero, planes):
    """What a serving engine's loader hands to the quantisation method of a layer."""
    n, k = codes.shape
    config = MatGPTQConfig(case["group"], 8, case["bits"], case["dtype"], resident_master_planes=planes)
    method = MatGPTQLinearMethod(config)
    method.n_out_features, method.n_in_features = n, k
    layer = torch.nn.Module()
    for name, t in (("qweight", codes), ("scales", scale), ("zeros", zero)):
        if t is not None:
            layer.register_parameter(name, torch.nn.Parameter(t, requires_grad=False))
    method.process_weights_after_loading(layer)
    return method, layer


def _linear(gen, case, n, k):
    """One layer, ready to be called on activations [m, k]."""
    codes, scale, zero = _checkpoint(gen, case, n, k)
    if case.get("planes"):
        method, layer = _plugin_layer(case, codes, scale, zero, True)
        return lambda x: method.apply(layer, x)
    return MatGPTQLinear(matryoshka_slice(codes, 8, case["bits"]), scale, case["bits"], case["group"], zeros=zero)


def _activations(gen, case, k):
    x = torch.empty((case["m"], k), dtype=torch.float32, device="cuda").normal_(generator=gen)
    return x.to(_dtype(case))


def _decoder(case, seed, new_tokens):
    cfg = DecoderConfig(hidden=case["hidden"], ffn=case["ffn"], layers=case["layers"], heads=case["heads"],
                        kv_heads=case["kv_heads"], vocab=case["vocab"])
    decoder, _, _ = random_mixnmatch_decoder(cfg, case["m"] + new_tokens, BITS, seed, via_plugin=True)
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    return DecodeSession(decoder), torch.randint(0, cfg.vocab, (case["m"],), device="cuda", generator=gen)


def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case}
    if kind == "call":
        state["linear"] = _linear(gen, case, case["n"], case["k"])
        state["x"] = _activations(gen, case, case["k"])
    elif kind in ("stack", "eager"):
        layers = [(_linear(gen, case, n, k), _activations(gen, case, k))
                  for _ in range(case.get("blocks", 1)) for n, k in shapes(case).values()]
        state["layers"] = layers
        if kind == "stack":
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                for linear, x in layers:
                    linear(x)
            stream.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"], stream=stream):
                state["outputs"] = [linear(x) for linear, x in layers]
    elif kind == "load":
        state["layers"] = [_checkpoint(gen, case, n, k) for n, k in shapes(case).values()]
    else:
        session, prompt = _decoder(case, seed, 72)
        state.update(session=session, prompt=prompt)
        if kind == "token":
            session.prefill(prompt)
            session.capture()
            state["at"] = (session.token.clone(), session.pos.clone())
    return state


def _load(case, codes, scale, zero):
    if case["route"] == "module":
        layer = MatGPTQLinear(matryoshka_slice(codes, 8, case["bits"]), scale, case["bits"], case["group"], zeros=zero)
        packed = layer.matgptq_qweight
    else:
        _, layer = _plugin_layer(case, codes, scale, zero, case["route"] == "planes")
        packed = layer.matgptq_planes if case["route"] == "planes" else layer.matgptq_weights
    outputs = {"packed": packed.data.view(torch.int32), "scales": layer.matgptq_scales.data}
    if zero is not None:
        outputs["zeros"] = layer.matgptq_zeros.data
    return outputs


def run(state):
    kind = state["case"]["kind"]
    if kind == "call":
        return state["linear"](state["x"])
    if kind == "stack":
        state["graph"].replay()
        return state["outputs"]
    if kind == "eager":
        return [linear(x) for linear, x in state["layers"]]
    if kind == "load":
        return [_load(state["case"], *layer) for layer in state["layers"]]
    session = state["session"]
    if kind == "prompt":
        session.prefill(state["prompt"])
    else:
        # the same position each time: a sequence that went on would run out of cache
        session.token.copy_(state["at"][0])
        session.pos.copy_(state["at"][1])
        session.replay()
    # (the token chosen from the logits is left out: which of two equal ones wins is not a property of the path)
    return {"logits": session.logits, "cache": session.cache}


def _linear_work(case, n, k):
    m, bits = case["m"], case["bits"]
    stored = bits if not case.get("planes") else bits + 1 if bits <= 4 else 8
    aux = 2 if case["zeros"] else 1
    return n * k * stored / 8 + 2 * n * _groups(case, k) * aux + 2 * m * (n + k), 2.0 * m * n * k


def work(case):
    kind = case["kind"]
    if kind == "call":
        nbytes, flops = _linear_work(case, case["n"], case["k"])
    elif kind in ("stack", "eager"):
        parts = [_linear_work(case, n, k) for n, k in shapes(case).values()]
        nbytes, flops = (sum(p[i] for p in parts) * case.get("blocks", 1) for i in (0, 1))
    elif kind == "load":
        stored = 8 if case["route"] == "planes" else case["bits"]
        aux = 2 if case["zeros"] else 1
        nbytes = sum(n * k * (1 + stored / 8) + 4 * n * _groups(case, k) * aux for n, k in shapes(case).values())
        flops = 0.0
    else:
        layers, hidden, m = case["layers"], case["hidden"], case["m"]
        weights = layers * sum(n * k for n, k in shapes({**case, "tp": 1}).values())
        bits = sum(BITS) / len(BITS) + 2 * 16 / 128  # codes, scales and zero points
        head = case["vocab"] * hidden
        cache = layers * 2 * case["kv_heads"] * HEAD_DIM * 2 * m
        rows = 1 if kind == "token" else m
        pairs = m if kind == "token" else m * (m + 1) / 2
        nbytes = weights * bits / 8 + 2 * head + cache + 4 * case["vocab"]
        flops = 2.0 * rows * weights + 2.0 * head + layers * 4.0 * case["heads"] * HEAD_DIM * pairs
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    """About four times what the path is off by against the same product in 64 bits (fp16 storage 3.0e-4 in the
    2-norm and 1.6e-3 at most, bf16 2.4e-3 and 1.4e-2), or a decoder with fused operators, or a prompt in two
    chunks, against the plain operators and the prompt in one (3.0e-3 and 1.2e-1)."""
    if case["kind"] == "load":
        return "exact"
    if case["kind"] in ("token", "prompt"):
        return {"rel": 1.2e-2, "max": 0.4}
    return {"rel": 9e-3, "max": 5e-2} if case["dtype"] == "bfloat16" else {"rel": 1.2e-3, "max": 7e-3}
