"""The work a user of this library has it do: quantized-weight products through nntrainer_amd.capi.

Three kinds of case, each through the public entry points in the order a decoder makes the calls:

  fc     one fully connected layer: `rows` activation rows against an n x k weight. mem "device": tensors on the
         GPU; "host": page-locked host memory, the framework plug-in's case (the call is synchronous).
         each_row: the rows are batch entries of a decode step, each a product of its own.
  layers the FCs of `layers` decoder layers: Q, K, V against one activation, the output projection, the gated MLP;
         with `vocab` the lm_head on the last row. Attention and norms between them are the user's own, so
         every layer gets its own input rows.
  moe    a mixture-of-experts feed-forward block with Q4_K experts, from router logits or the router's weight.

Weights are N(0, 0.02) quantized on the GPU, activations N(0, 1).
"""
import ctypes
import math
import weakref

import numpy as np
import torch

from nntrainer_amd import capi

# bytes per weight of the packed formats
BYTES = {"q4_0": 18 / 32, "q4_K": 144 / 256, "q6_K": 210 / 256}


def listed():
    return [
        # one decode token against a 4096 x 4096 Q4_0 layer: the smallest call, launch and latency
        {"name": "fc_q4_0_decode", "kind": "fc", "dtype": "q4_0", "rows": 1, "n": 4096, "k": 4096, "mem": "device", "each_row": False},
        # one decode token through all FCs of the Qwen3-0.6B-shaped decoder and its lm_head
        {"name": "decoder_q4_0_token", "kind": "layers", "dtype": "q4_0", "layers": 28, "rows": 1, "hidden": 1024, "inter": 3072,
         "q": 2048, "kv": 1024, "vocab": 151936},
        # a prompt of 512 tokens through four layers of the same decoder
        {"name": "decoder_q4_0_prompt", "kind": "layers", "dtype": "q4_0", "layers": 4, "rows": 512, "hidden": 1024, "inter": 3072,
         "q": 2048, "kv": 1024, "vocab": 0},
        # one decode token through a Qwen3-8B-shaped Q4_K layer
        {"name": "layer_q4_K_token", "kind": "layers", "dtype": "q4_K", "layers": 1, "rows": 1, "hidden": 4096, "inter": 12288,
         "q": 4096, "kv": 1024, "vocab": 0},
        # a long prompt of odd length through the same layer
        {"name": "layer_q4_K_prompt_1777", "kind": "layers", "dtype": "q4_K", "layers": 1, "rows": 1777, "hidden": 4096, "inter": 12288,
         "q": 4096, "kv": 1024, "vocab": 0},
        # the headline: FFN up-projection of a 512-token prompt
        {"name": "fc_q4_K_prompt_512", "kind": "fc", "dtype": "q4_K", "rows": 512, "n": 12288, "k": 4096, "mem": "device", "each_row": False},
        # a batch of eight decode rows through host memory, as the framework's FC layer makes the call
        {"name": "fc_q4_K_batch8_host", "kind": "fc", "dtype": "q4_K", "rows": 8, "n": 12288, "k": 4096, "mem": "host", "each_row": True},
        # lm_head of a decode token
        {"name": "lm_head_q6_K", "kind": "fc", "dtype": "q6_K", "rows": 1, "n": 151936, "k": 4096, "mem": "device", "each_row": False},
        # a short prompt of odd length against a Q6_K down-projection
        {"name": "fc_q6_K_prompt_333", "kind": "fc", "dtype": "q6_K", "rows": 333, "n": 4096, "k": 12288, "mem": "device", "each_row": False},
        # the Qwen3-30B-A3B-shaped block: one decode token, a batch of 64 (router logits given), a long prompt
        {"name": "moe_token", "kind": "moe", "tokens": 1, "hidden": 2048, "inter": 768, "experts": 128, "topk": 8, "router": True},
        {"name": "moe_64", "kind": "moe", "tokens": 64, "hidden": 2048, "inter": 768, "experts": 128, "topk": 8, "router": False},
        {"name": "moe_prompt_1000", "kind": "moe", "tokens": 1000, "hidden": 2048, "inter": 768, "experts": 128, "topk": 8, "router": True},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _k(rng, dtype, lo, hi):
    """A row length: whole super-blocks of 256, for Q4_0 in one case of four only whole blocks of 32."""
    step = 32 if dtype == "q4_0" and rng.random() < 0.25 else 256
    return step * max(1, round(_log(rng, lo, hi) / step))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("fc", "fc", "layers", "moe"))
        if kind == "fc":
            dtype = rng.choice(("q4_0", "q4_K", "q6_K"))
            rows = 1 if rng.random() < 0.3 else _log(rng, 1, 2048)
            case = {"kind": "fc", "dtype": dtype, "rows": rows, "n": _log(rng, 512, 65536), "k": _k(rng, dtype, 512, 12288),
                    "mem": "host" if rng.random() < 0.2 else "device", "each_row": rows <= 16 and rng.random() < 0.3}
        elif kind == "layers":
            dtype = rng.choice(("q4_0", "q4_K"))
            hidden = 256 * _log(rng, 3, 16)
            case = {"kind": "layers", "dtype": dtype, "layers": rng.randint(1, 4), "rows": 1 if rng.random() < 0.4 else _log(rng, 1, 2048),
                    "hidden": hidden, "inter": 256 * round(hidden / 256 * rng.uniform(2.0, 4.0)), "q": hidden * rng.choice((1, 1, 2)),
                    "kv": 128 * rng.randint(1, 8), "vocab": rng.choice((0, 0, 32000, 151936))}
        else:
            experts = rng.choice((8, 32, 64, 128))
            case = {"kind": "moe", "tokens": 1 if rng.random() < 0.3 else _log(rng, 1, 1500), "hidden": 256 * rng.randint(4, 12),
                    "inter": 256 * rng.randint(2, 8), "experts": experts, "topk": rng.choice((2, 4, 8)), "router": rng.random() < 0.5}
            if experts * case["hidden"] * case["inter"] > 128 * 2048 * 768:
                continue
        if _cost(case) <= most:
            return case


class _State:
    pass


def _normal(gen, shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _weights(gen, dtype, count, n, k):
    """`count` weights of n x k in device memory."""
    dense = _normal(gen, (count * n, k)).mul_(0.02)
    size = capi.weight_nbytes(dtype, n, k)
    blocks = torch.empty(count * size, dtype=torch.uint8, device="cuda")
    capi.quantize_weights(dtype, dense, count * n, k, blocks, stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return [capi.Weight(dtype, n, k, blocks[i * size:(i + 1) * size], mem=capi.MEM_DEVICE) for i in range(count)]


def _page_locked(shape):
    """A page-locked fp32 array; the memory is given back with the last view of it."""
    buf = (ctypes.c_float * int(np.prod(shape))).from_address(capi.host_alloc(4 * int(np.prod(shape))))
    weakref.finalize(buf, capi.host_free, ctypes.addressof(buf))
    return np.ctypeslib.as_array(buf).reshape(shape)


def _empty(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.float32)


def prepare(case, seed):
    capi.init(0)
    s = _State()
    s.case = case
    s.stream = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["kind"] == "fc":
        s.w = _weights(gen, case["dtype"], 1, case["n"], case["k"])[0]
        s.a = _normal(gen, (case["rows"], case["k"]))
        s.call = capi.matmul_each_row if case["each_row"] else capi.matmul
        s.mem = capi.MEM_HOST if case["mem"] == "host" else capi.MEM_DEVICE
        if case["mem"] == "host":
            a = s.a.cpu().numpy()
            s.a = _page_locked(a.shape)
            s.a[:] = a
            s.c = _page_locked((case["rows"], case["n"]))
        else:
            s.c = _empty(case["rows"], case["n"])
    elif case["kind"] == "layers":
        num, rows, hid, inter, q, kv = (case[x] for x in ("layers", "rows", "hidden", "inter", "q", "kv"))
        wq, wk, wv, wo, up, gate, down = (_weights(gen, case["dtype"], num, n, k) for n, k in (
            (q, hid), (kv, hid), (kv, hid), (hid, q), (inter, hid), (inter, hid), (hid, inter)))
        x, heads, mid = (_normal(gen, (num, rows, k)) for k in (hid, q, hid))
        s.out = {"q": _empty(num, rows, q), "k": _empty(num, rows, kv), "v": _empty(num, rows, kv),
                 "o": _empty(num, rows, hid), "mlp": _empty(num, rows, hid)}
        o = s.out
        s.layers = [{"qkv": (wq[i], wk[i], wv[i]), "o": wo[i], "mlp": (up[i], gate[i], down[i]), "x": x[i], "heads": heads[i],
                     "mid": mid[i], "qkv_out": (o["q"][i], o["k"][i], o["v"][i]), "o_out": o["o"][i], "mlp_out": o["mlp"][i]}
                    for i in range(num)]
        if case["vocab"]:
            s.head = _weights(gen, case["dtype"], 1, case["vocab"], hid)[0]
            s.last = _normal(gen, (1, hid))
            s.out["logits"] = _empty(1, case["vocab"])
    else:
        t, hid, inter, e = (case[x] for x in ("tokens", "hidden", "inter", "experts"))
        gate, up, down = (_weights(gen, "q4_K", e, n, k) for n, k in ((inter, hid), (inter, hid), (hid, inter)))
        s.experts = capi.Experts(gate, up, down)
        s.x = _normal(gen, (t, hid))
        s.logits = None if case["router"] else _normal(gen, (t, e))
        s.router = _normal(gen, (hid, e)).mul_(hid ** -0.5) if case["router"] else None
        s.y = _empty(t, hid)
        s.idx = torch.empty((t, case["topk"]), dtype=torch.int32, device="cuda")
        s.weights = _empty(t, case["topk"])
    return s


def run(s):
    case = s.case
    if case["kind"] == "fc":
        s.call(s.w, s.a, case["rows"], s.c, mem=s.mem, stream=s.stream)
        return s.c
    if case["kind"] == "layers":
        rows = case["rows"]
        for layer in s.layers:
            capi.matmul_multi(layer["qkv"], layer["x"], rows, layer["qkv_out"], stream=s.stream)
            capi.matmul(layer["o"], layer["heads"], rows, layer["o_out"], stream=s.stream)
            capi.mlp_swiglu_down(*layer["mlp"], layer["mid"], rows, layer["mlp_out"], stream=s.stream)
        if case["vocab"]:
            capi.matmul(s.head, s.last, 1, s.out["logits"], stream=s.stream)
        return s.out
    capi.moe_forward(case["tokens"], case["hidden"], case["inter"], case["experts"], case["topk"], s.experts, None, None,
                     s.x, s.y, router_logits=s.logits, router_weight=s.router, topk_idx=s.idx, topk_w=s.weights, stream=s.stream)
    return {"y": s.y, "idx": s.idx, "weights": s.weights}


def work(case):
    if case["kind"] == "fc":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * k * BYTES[case["dtype"]] + 4 * m * (n + k), "flops": 2 * m * n * k}
    if case["kind"] == "layers":
        m, hid, inter, q, kv = (case[x] for x in ("rows", "hidden", "inter", "q", "kv"))
        each = hid * (q + 2 * kv) + hid * q + 3 * hid * inter
        head = case["vocab"] * hid
        per = BYTES[case["dtype"]]
        return {"bytes": case["layers"] * (each * per + 4 * m * (hid + q + 2 * kv + q + hid + 2 * hid)) + head * per + 4 * (case["vocab"] and case["vocab"] + hid),
                "flops": 2 * (case["layers"] * m * each + head)}
    t, hid, inter, e, k = (case[x] for x in ("tokens", "hidden", "inter", "experts", "topk"))
    active = e * (1 - (1 - k / e) ** t)  # experts that t tokens reach on average
    return {"bytes": active * 3 * hid * inter * BYTES["q4_K"] + 8 * t * hid + 4 * e * (hid if case["router"] else t) + 8 * t * k,
            "flops": 2 * t * k * 3 * hid * inter + (2 * t * hid * e if case["router"] else 0)}


def tolerance(case):
    """Single products: exact integer block sums under fp32 scales, added up in fp32. Where a product's rows are quantized
    to 8 bits again (the MLP's and the experts' hidden rows), a last-bit difference moves single roundings by 1/127 of a
    block's largest value."""
    return {"rel": 1e-5} if case["kind"] == "fc" else {"rel": 1e-3}
