"""The work this framework's users have it do, as cases that can be timed.

Every case is the linear layers of one kind of use: the decode of one token or
of a small batch of sequences, the prefill of a prompt, one projection called
by itself, and the 4-bit weights expanded to fp16 for a dense GEMM.  Weights
are seeded random bytes of the serialised formats with scales of the usual
size; activations are N(0, 1) with a few channels an order of magnitude larger,
as the inputs of a transformer's linear layers are.

A decode step runs as a serving loop has it: captured once in a graph on the
engine's stream, then replayed.  A prefill calls ROCmEngine.matmul per
projection.  Weights are uploaded before the call.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ztensor_amd import _lib
from ztensor_amd import storage as st
from ztensor_amd.engine import ROCmEngine

_DIMS_8B = {"hidden": 4096, "kv": 1024, "ffn": 14336}
_DIMS_70B = {"hidden": 8192, "kv": 1024, "ffn": 28672}
_DIMS_QWEN2_7B = {"hidden": 3584, "kv": 512, "ffn": 18944}
_DIMS_BITNET_2B = {"hidden": 2560, "kv": 2560, "ffn": 6912}
_LARGEST = 2048 * 7 * 4096 * 14336  # tokens x weights that no drawn case exceeds
_GROUP = 128  # GPTQ / AWQ group

# the 16 values of the interleaved 4-bit format
_IQ4 = (-1.0, -0.6961928, -0.5250730, -0.3947555, -0.2831612, -0.1790887, -0.0805542, 0.0,
        0.0805542, 0.1790887, 0.2831612, 0.3947555, 0.5250730, 0.6961928, 1.0, 1.3312578)

# values and bytes of one serialised block
_BLOCK = {"q4_0": (32, 18), "iq4_nl": (32, 18), "q5_0": (32, 22), "q8_0": (32, 36), "q4_k": (256, 144),
          "q5_k": (256, 176), "q6_k": (256, 210), "gptq": (_GROUP, _GROUP // 2 + 4), "awq": (_GROUP, _GROUP // 2 + 4),
          "ternary": (4, 1), "ternary_i8": (4, 1)}


def listed():
    return [
        # one k or v projection of one token, by itself: what a single call costs
        {"name": "call_q4_0_kv", "use": "call", "format": "q4_0", "rows": 1024, "k": 4096, "tokens": 1},
        # one token through two layers of an 8B model, q/k/v and gate/up grouped into one launch each
        {"name": "decode_q4_0_8b", "use": "decode", "format": "q4_0", **_DIMS_8B, "tokens": 1, "layers": 2},
        # the same model in the usual Q4_K / Q6_K mix (v and down in Q6_K)
        {"name": "decode_q4_k_m_8b", "use": "decode", "format": "q4_k_m", **_DIMS_8B, "tokens": 1, "layers": 2},
        # one token through a layer of a 70B model in 4-bit GPTQ with fp16 activations
        {"name": "decode_gptq_70b", "use": "decode", "format": "gptq", **_DIMS_70B, "tokens": 1, "layers": 1},
        # one token through layers of a 2B ternary model with int8 activations: small matrices, many launches
        {"name": "decode_ternary_2b", "use": "decode", "format": "ternary_i8", **_DIMS_BITNET_2B, "tokens": 1,
         "layers": 6},
        # continuous batching: 16 sequences decode together on the 70B layer
        {"name": "batch16_gptq_70b", "use": "decode", "format": "gptq", **_DIMS_70B, "tokens": 16, "layers": 1},
        # 8 sequences on a 7B model in IQ4_NL
        {"name": "batch8_iq4_nl_7b", "use": "decode", "format": "iq4_nl", **_DIMS_QWEN2_7B, "tokens": 8, "layers": 1},
        # 32 sequences on an 8B model in Q8_0
        {"name": "batch32_q8_0_8b", "use": "decode", "format": "q8_0", **_DIMS_8B, "tokens": 32, "layers": 1},
        # a 512-token prompt through an 8B layer in Q4_0
        {"name": "prefill512_q4_0_8b", "use": "prefill", "format": "q4_0", **_DIMS_8B, "tokens": 512},
        # a prompt of an odd length in the Q4_K / Q6_K mix
        {"name": "prefill317_q4_k_m_8b", "use": "prefill", "format": "q4_k_m", **_DIMS_8B, "tokens": 317},
        # a long prompt in GPTQ with fp16 activations, the largest case
        {"name": "prefill2048_gptq_8b", "use": "prefill", "format": "gptq", **_DIMS_8B, "tokens": 2048},
        # a 4-bit matrix expanded to the fp16 operand of a dense GEMM
        {"name": "expand_gptq_ffn", "use": "expand", "format": "gptq", "rows": 14336, "k": 4096, "tokens": 1},
    ]


def draw(rng):
    use = rng.choice(["call", "decode", "decode", "batch", "batch", "prefill", "prefill", "prefill", "expand"])
    if use == "expand":
        fmt = rng.choice(["q4_0", "gptq", "awq"])
    elif use == "decode":
        fmt = rng.choice(["q4_0", "q8_0", "q4_k_m", "q5_k", "q5_0", "iq4_nl", "gptq", "awq", "ternary_i8"])
    else:
        fmt = rng.choice(["q4_0", "q8_0", "q4_k_m", "q5_k", "q5_0", "iq4_nl", "gptq", "awq"])
    if use in ("call", "expand"):
        case = {"use": use, "format": fmt, "rows": int(math.exp(rng.uniform(math.log(256), math.log(28672)))),
                "k": 256 * round(math.exp(rng.uniform(math.log(4), math.log(56)))),
                "tokens": rng.choice([1, 1, 2, 5, 16]) if use == "call" else 1}
        return case
    if rng.random() < 0.5:  # a model's own sizes
        dims = dict(_DIMS_BITNET_2B if fmt == "ternary_i8" else
                    rng.choice([_DIMS_8B, _DIMS_QWEN2_7B, _DIMS_8B if use == "prefill" else _DIMS_70B]))
    else:  # sizes of no model here; kv heads x head size is any multiple of 8
        hidden = 256 * rng.randint(4, 24)
        dims = {"hidden": hidden, "kv": 8 * rng.randint(16, hidden // 16),
                "ffn": 256 * rng.randint(hidden // 128, hidden // 64)}
    if use == "prefill":
        params = 2 * dims["hidden"] * (dims["hidden"] + dims["kv"]) + 3 * dims["hidden"] * dims["ffn"]
        most = min(2048, _LARGEST // (2 * params))
        tokens = round(math.exp(rng.uniform(math.log(33), math.log(max(64, most)))))
        tokens = min(tokens, most)
        return {"use": "prefill", "format": fmt, **dims, "tokens": tokens}
    tokens = 1 if use == "decode" else rng.choice([2, 3, 4, 6, 8, 12, 16, 24, 32])
    return {"use": "decode", "format": fmt, **dims, "tokens": tokens, "layers": 1}


# ------------------------------------------------------------------ inputs


def _format_of(case, proj):
    if case["format"] == "q4_k_m":
        return "q6_k" if proj in ("v", "down") else "q4_k"
    return case["format"]


def _projections(case):
    """(projection, rows, K, input) in the order a layer calls them."""
    if case["use"] in ("call", "expand"):
        return [("one", case["rows"], case["k"], "x")]
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [("q", h, h, "attn"), ("k", kv, h, "attn"), ("v", kv, h, "attn"), ("o", h, h, "mix"),
            ("gate", f, h, "mlp"), ("up", f, h, "mlp"), ("down", h, f, "act")]


def _bytes(g, *shape):
    return np.frombuffer(g.bytes(int(np.prod(shape))), np.uint8).reshape(shape).copy()


def _f16(g, n, size):
    return (np.abs(g.standard_normal(n, dtype=np.float32)) * np.float32(size)).astype(np.float16)


def _weights(fmt, rows, k, seed):
    """The serialised bytes of one matrix, and its scales where they are apart."""
    g = np.random.Generator(np.random.SFC64(seed))
    vals, size = _BLOCK[fmt]
    n = rows * k // vals
    if fmt in ("gptq", "awq"):
        zeros = np.full(n, 8.0) if fmt == "gptq" else g.integers(5, 12, n)
        return _bytes(g, rows * k // 2), _f16(g, n, 0.02), zeros.astype(np.float16)
    raw = _bytes(g, n, size)
    if fmt in ("q4_0", "iq4_nl", "q5_0"):
        raw[:, :2] = _f16(g, n, 0.02 if fmt != "iq4_nl" else 0.01).reshape(n, 1).view(np.uint8)
    elif fmt == "q8_0":
        raw[:, :4] = _f16(g, n, 0.002).astype(np.float32).reshape(n, 1).view(np.uint8)
    elif fmt in ("q4_k", "q5_k"):
        raw[:, :2] = _f16(g, n, 0.002).reshape(n, 1).view(np.uint8)
        raw[:, 2:4] = _f16(g, n, 0.001).reshape(n, 1).view(np.uint8)
    elif fmt == "q6_k":
        raw[:, 208:] = _f16(g, n, 0.0005).reshape(n, 1).view(np.uint8)
    else:  # 2-bit codes 0, 1, 2: code 3 becomes 1
        raw = raw.reshape(-1)
        raw ^= ((raw & 0x55) & ((raw >> 1) & 0x55)) << 1
    return raw.reshape(-1), None, None


def _storage(fmt, rows, k, w):
    raw, scales, zeros = w
    n = rows * k
    if fmt == "q8_0":
        return st.Q8Storage(raw, n)
    if fmt == "gptq":
        return st.GPTQStorage(raw, scales.view(np.uint16), zeros.view(np.uint16), n, _GROUP)
    if fmt == "awq":
        return st.AWQStorage(raw.view("<u4"), scales.view(np.uint16), zeros.view(np.uint16), n, _GROUP)
    kind = {"q4_0": st.Q4Storage, "iq4_nl": st.IQ4NLStorage, "q5_0": st.Q5_0Storage, "q4_k": st.Q4KStorage,
            "q5_k": st.Q5KStorage, "q6_k": st.Q6KStorage, "ternary": st.TernaryStorage,
            "ternary_i8": st.TernaryStorage}[fmt]
    return kind(raw, n)


def _seed_of(seed, layer, i):
    return [int(seed), layer, i]


def _inputs(case, seed):
    """{(layer, input name): activations [tokens, K] on the GPU}."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7 + 3)
    found = {}
    for layer in range(case.get("layers", 1)):
        for _, _, k, name in _projections(case):
            if (layer, name) in found:
                continue
            x = torch.randn((case["tokens"], k), generator=g, device="cuda")
            x[:, torch.randint(0, k, (max(1, k // 512),), generator=g, device="cuda")] *= 10.0
            if case["format"] in ("gptq", "awq", "iq4_nl"):
                x = x.half()
            elif case["format"] == "ternary_i8":
                x = torch.clamp(torch.round(x * 32.0), -127, 127).to(torch.int8)
            found[layer, name] = x
    return found


def _ternary_step(eng, weights, x, ys, scale):
    """Ternary GEMVs over int8 activations, the projections of one input in one launch."""
    for layer, projs in enumerate(weights):
        for names in (("q", "k", "v"), ("o",), ("gate", "up"), ("down",)):
            mats = [(projs[p][0].data_ptr(), scale.data_ptr() + 4, ys[layer][p].data_ptr(), projs[p][1]) for p in names]
            _, _, k, src = projs[names[0]]
            eng.ternary_gemv_i8_group(mats, x[layer, src].data_ptr(), scale.data_ptr(), k)
    return ys


def _step(eng, case, weights, x):
    """Every projection of the case's layers."""
    out = []
    for layer, projs in enumerate(weights):
        ys = {}
        if case["tokens"] == 1 and case["use"] == "decode" and case["format"] in ("q4_0", "gptq", "awq"):
            for names in (("q", "k", "v"), ("o",), ("gate", "up"), ("down",)):
                src = x[layer, projs[names[0]][3]].reshape(-1)
                ys.update(zip(names, eng.gemv_group([projs[p][0] for p in names], src)))
        else:
            for p, (w, rows, k, src) in projs.items():
                ys[p] = eng.matmul(x[layer, src], st.Tensor((k, rows), w.storage))
        out.append(ys)
    return out


def prepare(case, seed):
    stream = torch.cuda.Stream() if case["use"] == "decode" else None
    eng = ROCmEngine(stream=stream)
    x = _inputs(case, seed)
    weights = []
    for layer in range(case.get("layers", 1)):
        projs = {}
        for i, (p, rows, k, src) in enumerate(_projections(case)):
            fmt = _format_of(case, p)
            s = _storage(fmt, rows, k, _weights(fmt, rows, k, _seed_of(seed, layer, i)))
            if fmt == "ternary_i8":
                projs[p] = (torch.from_numpy(s.row_aligned(rows, k)).cuda(), rows, k, src)
            else:
                projs[p] = (st.Tensor((rows, k), s), rows, k, src)
        weights.append(projs)
    state = {"case": case, "engine": eng, "weights": weights, "x": x, "graph": None}
    torch.cuda.synchronize()
    if case["format"] != "ternary_i8":
        eng.upload_weights([w[0].storage for projs in weights for w in projs.values()])
    if case["use"] == "decode":
        if case["format"] == "ternary_i8":
            scale = torch.tensor([1.0 / 32.0, 0.02], device="cuda")  # of the activations, of the weights
            ys = [{p: torch.empty(w[1], device="cuda") for p, w in projs.items()} for projs in weights]
            state["keep"] = (scale, ys)
            step = lambda: _ternary_step(eng, weights, x, ys, scale)  # noqa: E731
        else:
            step = lambda: _step(eng, case, weights, x)  # noqa: E731
        torch.cuda.synchronize()
        step()  # lays the weights out and sizes the workspace, outside the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            state["out"] = step()
        state["graph"] = graph
    torch.cuda.synchronize()
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    if state["case"]["use"] == "expand":
        return state["engine"].dequant_w4_to_fp16(state["weights"][0]["one"][0])
    return _step(state["engine"], state["case"], state["weights"], state["x"])


# ------------------------------------------------------- what a pass needs


def work(case):
    total = flops = 0
    seen = set()
    act = 2 if case["format"] in ("gptq", "awq", "iq4_nl") else 1 if case["format"] == "ternary_i8" else 4
    layers, t = case.get("layers", 1), case["tokens"]
    for p, rows, k, src in _projections(case):
        vals, size = _BLOCK[_format_of(case, p)]
        total += rows * k // vals * size
        if case["use"] == "expand":
            total += 2 * rows * k
            flops += 2 * rows * k
            continue
        total += 4 * rows * t + (0 if src in seen else act * k * t)
        seen.add(src)
        flops += 2 * rows * k * t
    return {"bytes": layers * total, "flops": layers * flops}


def tolerance(case):
    # fp32 sums of exact or nearly exact products; a GEMM's sums are spread over its outputs' rms
    if case["use"] == "expand":
        return {"rel": 2e-4, "max": 2e-3}  # one rounding to fp16
    if case["format"] in ("q4_0", "iq4_nl"):
        return {"rel": 1.2e-5, "max": 1.2e-4}  # nibbles with an offset taken off the sums; a codebook in fp16 parts
    return {"rel": 4e-6, "max": 4e-5}


# -------------------------------------------------- the same in 64 bits


def _nibbles(b):
    return b & 15, b >> 4


def _dense(fmt, rows, k, w):
    """The matrix in 64 bits, from its serialised bytes."""
    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a)).cuda()

    raw, scales, zeros = w
    if fmt in ("gptq", "awq"):
        lo, hi = _nibbles(dev(raw).reshape(rows * k // _GROUP, _GROUP // 2))
        q = torch.stack([lo, hi], dim=2).reshape(-1, _GROUP).double()
        return ((q - dev(zeros).double()[:, None]) * dev(scales).double()[:, None]).reshape(rows, k)
    if fmt in ("ternary", "ternary_i8"):
        b = dev(raw)
        return (torch.stack([(b >> s) & 3 for s in (0, 2, 4, 6)], dim=1).reshape(rows, k).double() - 1.0)
    vals, size = _BLOCK[fmt]
    b = dev(raw.reshape(-1, size))

    def half(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if fmt == "q8_0":
        out = b[:, 4:].contiguous().view(torch.int8).double() * b[:, :4].contiguous().view(torch.float32).double()
    elif fmt == "q4_0":
        out = (torch.cat(_nibbles(b[:, 2:]), dim=1).double() - 8.0) * half(0)
    elif fmt == "iq4_nl":
        table = torch.tensor(np.array(_IQ4, np.float32), device="cuda").double()
        out = table[torch.stack(_nibbles(b[:, 2:]), dim=2).reshape(-1, 32).long()] * half(0)
    elif fmt == "q5_0":
        bits = (b[:, 2:6, None] >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1
        q = torch.cat(_nibbles(b[:, 6:]), dim=1) | (bits.reshape(-1, 32) << 4)
        out = (q.double() - 16.0) * half(0)
    elif fmt == "q6_k":
        ql, qh, sc = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32), b[:, 192:208]
        lo, hi = _nibbles(ql)
        parts = [lo[..., :32] | ((qh & 3) << 4), lo[..., 32:] | (((qh >> 2) & 3) << 4),
                 hi[..., :32] | (((qh >> 4) & 3) << 4), hi[..., 32:] | ((qh >> 6) << 4)]
        q = torch.stack(parts, dim=2).reshape(-1, 16, 16).double() - 32.0
        out = q * (sc.contiguous().view(torch.int8).double() * half(208))[:, :, None]
    else:  # q4_k, q5_k
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], dim=1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1).double()
        qs = b[:, 16:144].reshape(-1, 4, 32)
        q = torch.stack(_nibbles(qs), dim=2).reshape(-1, 8, 32)
        if fmt == "q5_k":
            bits = (b[:, 144:176, None] >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1
            q = q | (bits.permute(0, 2, 1) << 4)
        out = q.double() * (half(0) * sc)[:, :, None] - (half(2) * mn)[:, :, None]
    return out.reshape(rows, k)


def exact(case, seed):
    x = _inputs(case, seed)
    out = []
    for layer in range(case.get("layers", 1)):
        ys = {}
        for i, (p, rows, k, src) in enumerate(_projections(case)):
            fmt = _format_of(case, p)
            w = _dense(fmt, rows, k, _weights(fmt, rows, k, _seed_of(seed, layer, i)))
            if case["use"] == "expand":
                return w
            y = x[layer, src].double() @ w.t()
            if fmt == "ternary_i8":
                y = y * (torch.tensor(0.02, dtype=torch.float32).double().item() / 32.0)
            grouped = case["tokens"] == 1 and case["use"] == "decode" and fmt in ("q4_0", "gptq", "awq", "ternary_i8")
            ys[p] = y.reshape(-1) if grouped else y
            del w
        out.append(ys)
    return out
