"""The work a host has this library do, as timed cases.

A case is one pass of a transformer layer's weight products (q/k/v, the
attention output, gate/up, down: the calls the engine makes), or of its
decode attention, through the Python binding of the C ABI:

  decode     one activation row per sequence and step, device pointers, the
             layers captured once in a HIP graph that is replayed each step
  prompt     M prompt rows through one layer, device pointers, launched
             directly (prompt lengths vary, so a graph is not kept)
  host       the same products for one row through host pointers, which is
             what the engine's gemv slot calls
  attention  decode attention over an f16 KV cache, captured like decode

Weights are GGUF blocks with uniform quant and scale fields and the block
scale ranges of siphon_amd.synth. Activations are normal with uneven channel
sizes; the down projection's input is a product of two normals (gated).
"""
import math

import numpy as np
import torch

import siphon_amd as sa

# a layer's sizes: hidden, kv rows, ffn (listed by the model class they are of)
LAYER_05B = {"hidden": 896, "kv": 128, "ffn": 4864}
LAYER_1B = {"hidden": 2048, "kv": 256, "ffn": 5632}
LAYER_8B = {"hidden": 4096, "kv": 1024, "ffn": 14336}
LAYER_32B = {"hidden": 5120, "kv": 1024, "ffn": 27648}
HEADS_8B = {"heads": 32, "kv_heads": 8, "head_dim": 128}
# Q4_K_M: Q4_K with wv and ffn_down in Q6_K; every other mix is one type
MIXES = ["Q4_K_M", "Q4_0", "Q5_0", "Q8_0", "Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "F16"]
UNIT_MIXES = ["Q4_0", "Q5_0", "Q8_0", "F16"]  # rows need not be a multiple of 256
# the matrices of a layer in the groups that share one input
GROUPS = [("wq", "wk", "wv"), ("wo",), ("gate", "up"), ("down",)]


def listed():
    return [
        # one generated token of a small Q8_0 model: every launch is a few
        # megabytes, so launches and latency count
        {"name": "decode_0.5b_q8_0", "kind": "decode", **LAYER_05B, "mix": "Q8_0", "rows": 1, "layers": 6},
        # one generated token of an 8B Q4_K_M model: the common local setup
        {"name": "decode_8b_q4km", "kind": "decode", **LAYER_8B, "mix": "Q4_K_M", "rows": 1, "layers": 2},
        # the same products through the engine's synchronous gemv slot
        {"name": "host_8b_q4km", "kind": "host", **LAYER_8B, "mix": "Q4_K_M", "rows": 1, "layers": 1},
        # a decode step of 8 sequences served together
        {"name": "batch8_8b_q4km", "kind": "decode", **LAYER_8B, "mix": "Q4_K_M", "rows": 8, "layers": 2},
        # a short chat turn
        {"name": "prompt37_8b_q4km", "kind": "prompt", **LAYER_8B, "mix": "Q4_K_M", "rows": 37, "layers": 1},
        # a usual prompt chunk
        {"name": "prompt512_8b_q4km", "kind": "prompt", **LAYER_8B, "mix": "Q4_K_M", "rows": 512, "layers": 1},
        # a long document in one chunk, the largest case
        {"name": "prompt2048_8b_q4km", "kind": "prompt", **LAYER_8B, "mix": "Q4_K_M", "rows": 2048, "layers": 1},
        # a prompt of a small Q8_0 model, ragged in rows and in n_out tiles
        {"name": "prompt300_0.5b_q8_0", "kind": "prompt", **LAYER_05B, "mix": "Q8_0", "rows": 300, "layers": 1},
        # a prompt of a 32B model in a five-bit quantization
        {"name": "prompt130_32b_q5_k", "kind": "prompt", **LAYER_32B, "mix": "Q5_K", "rows": 130, "layers": 1},
        # a prompt of an unquantized small model
        {"name": "prompt200_1.1b_f16", "kind": "prompt", **LAYER_1B, "mix": "F16", "rows": 200, "layers": 1},
        # decode attention early in a conversation
        {"name": "attention_600_8b", "kind": "attention", **HEADS_8B, "rows": 600, "layers": 8},
        # decode attention far into a long context
        {"name": "attention_7000_8b", "kind": "attention", **HEADS_8B, "rows": 7000, "layers": 4},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "attention"])
    if kind == "attention":
        kv_heads = rng.choice([2, 4, 8])
        return {"kind": kind, "heads": kv_heads * rng.randint(1, 8), "kv_heads": kv_heads,
                "head_dim": rng.choice([64, 80, 96, 128]), "rows": _log_int(rng, 16, 16384),
                "layers": rng.randint(2, 4)}
    mix = rng.choice(MIXES)
    step = 64 if mix in UNIT_MIXES else 256  # rows of the K-quants are whole super-blocks
    hidden = step * _log_int(rng, 768 // step, 5120 // step)
    case = {"kind": kind, "hidden": hidden, "kv": 64 * rng.randint(2, 16),
            "ffn": step * int(round(hidden * rng.uniform(2.5, 5.4) / step)), "mix": mix}
    if kind == "decode":
        return {**case, "rows": rng.choice([1, _log_int(rng, 2, 16)]), "layers": rng.randint(1, 3)}
    weights = 2 * hidden * hidden + 2 * hidden * case["kv"] + 3 * hidden * case["ffn"]
    most = int(min(2048, 4.4e11 / weights))  # no more products than the largest listed case
    return {**case, "rows": _log_int(rng, 17, most), "layers": 1}


# ---- inputs -----------------------------------------------------------------


def _shapes(case):
    hid, kv, ffn = case["hidden"], case["kv"], case["ffn"]
    return {"wq": (hid, hid), "wk": (kv, hid), "wv": (kv, hid), "wo": (hid, hid),
            "gate": (ffn, hid), "up": (ffn, hid), "down": (hid, ffn)}


def _type(case, name):
    if case["mix"] == "Q4_K_M":
        return sa.Q6_K if name in ("wv", "down") else sa.Q4_K
    return sa.TYPES[case["mix"]]


_SCALE_AT = {sa.Q4_0: (0,), sa.Q5_0: (0,), sa.Q8_0: (0,), sa.Q2_K: (80, 82), sa.Q3_K: (108,),
             sa.Q4_K: (0, 2), sa.Q5_K: (0, 2), sa.Q6_K: (208,)}


def _blocks(wtype, n_out, n_in, g):
    """GGUF bytes of an n_out x n_in matrix, uint8 [blocks, block bytes] on
    the GPU (F16: the rows)."""
    if wtype == sa.F16:
        w = torch.rand(n_out, n_in, device="cuda", generator=g).mul_(0.1).sub_(0.05).half()
        return w.view(torch.uint8)
    be, bb = sa.GEOM[wtype]
    n = n_out * (n_in // be)
    b = torch.randint(0, 256, (n, bb), dtype=torch.uint8, device="cuda", generator=g)
    if wtype == sa.Q6_K:
        b[:, 192:208] = torch.randint(-32, 32, (n, 16), dtype=torch.int8, device="cuda",
                                      generator=g).view(torch.uint8)
    if wtype == sa.Q8_0:
        b[:, 2:34] = torch.randint(-127, 128, (n, 32), dtype=torch.int8, device="cuda",
                                   generator=g).view(torch.uint8)
    for at in _SCALE_AT[wtype]:
        d = torch.rand(n, 1, device="cuda", generator=g).mul_(3.9e-3).add_(1e-4)
        b[:, at:at + 2] = d.half().view(torch.uint8)
    return b


def _layer_weights(case, seed):
    """name -> blocks, layer by layer."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + 17)
    for _ in range(case["layers"]):
        yield {n: _blocks(_type(case, n), *s, g) for n, s in _shapes(case).items()}


def _activations(case, seed):
    """The input of each group of a layer, per layer: f32 [rows, n_in] on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + 29)
    hid, ffn = case["hidden"], case["ffn"]
    M, out = case["rows"], []
    for _ in range(case["layers"]):
        xs = []
        for n in (hid, hid, hid):
            size = torch.randn(1, n, device="cuda", generator=g).mul_(0.5).exp_()
            xs.append(torch.randn(M, n, device="cuda", generator=g) * size)
        a = torch.randn(M, ffn, device="cuda", generator=g)
        xs.append(a * torch.randn(M, ffn, device="cuda", generator=g))
        out.append(xs)
    return out


def _attention_inputs(case, seed):
    """(q, k, v) per layer; caches of n_ctx positions, n_ctx a multiple of 256."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + 41)
    nh, nkv, hd = case["heads"], case["kv_heads"], case["head_dim"]
    n_ctx = (case["rows"] + 255) // 256 * 256
    out = []
    for _ in range(case["layers"]):
        q = torch.randn(nh, hd, device="cuda", generator=g)
        k = torch.randn(nkv, n_ctx, hd, device="cuda", generator=g).half()
        v = torch.randn(nkv, hd, n_ctx, device="cuda", generator=g).half()
        out.append((q, k, v))
    return out


# ---- state and pass -----------------------------------------------------------

_shared = {}


def _device():
    """One context and one stream for the process, as a host keeps them."""
    if not _shared:
        torch.cuda.init()
        _shared["dev"] = sa.Device(0)
        _shared["stream"] = torch.cuda.Stream()
    return _shared["dev"], _shared["stream"]


class _State:
    def __init__(self):
        self.weights, self.graph, self.outs = [], None, None

    def __del__(self):
        self.graph = None
        for layer in self.weights:
            for w in layer.values():
                w.free()


def prepare(case, seed):
    dev, stream = _device()
    s = _State()
    s.case, s.dev, s.stream = case, dev, stream.cuda_stream
    if case["kind"] == "attention":
        s.inputs = _attention_inputs(case, seed)
        s.outs = [torch.empty_like(q) for q, _, _ in s.inputs]
        call = _attend
    else:
        for blocks in _layer_weights(case, seed):
            s.weights.append({n: dev.upload(_type(case, n), *_shapes(case)[n], b.cpu().numpy())
                              for n, b in blocks.items()})
        s.inputs = _activations(case, seed)
        if case["kind"] == "host":
            s.inputs = [[x[0].cpu().numpy() for x in xs] for xs in s.inputs]
            return s
        if case["rows"] > 1:
            for layer in s.weights:
                for w in layer.values():
                    w.prepare_gemm()
        s.outs = [{n: torch.empty(case["rows"], o, device="cuda")
                   for n, (o, _) in _shapes(case).items()} for _ in s.weights]
        call = _products
    torch.cuda.synchronize()
    if case["kind"] in ("decode", "attention"):
        call(s)  # workspaces exist before the capture
        torch.cuda.synchronize()
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph, stream=stream):
            call(s)
        torch.cuda.synchronize()
    return s


def _products(s):
    M = s.case["rows"]
    for layer, xs, out in zip(s.weights, s.inputs, s.outs):
        for names, x in zip(GROUPS, xs):
            ws, ys = [layer[n] for n in names], [out[n].data_ptr() for n in names]
            if M == 1:
                s.dev.gemv_multi_dev(ws, x.data_ptr(), ys, s.stream)
            else:
                s.dev.gemm_multi_dev(ws, x.data_ptr(), M, ys, s.stream)


def _attend(s):
    nh, nkv, hd = (s.case[k] for k in ("heads", "kv_heads", "head_dim"))
    n = s.case["rows"]
    for (q, k, v), out in zip(s.inputs, s.outs):
        s.dev.attn_decode_dev(q.data_ptr(), k.data_ptr(), v.data_ptr(), nh, nkv, hd, k.shape[1],
                              n - 1, 1.0 / math.sqrt(hd), out.data_ptr(), stream=s.stream)


def run(s):
    if s.graph is not None:
        s.graph.replay()
    elif s.case["kind"] == "host":
        return [{n: s.dev.gemv(layer[n], x) for names, x in zip(GROUPS, xs) for n in names}
                for layer, xs in zip(s.weights, s.inputs)]
    else:
        _products(s)
    return s.outs


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    M, L = case["rows"], case["layers"]
    if case["kind"] == "attention":
        nh, nkv, hd = case["heads"], case["kv_heads"], case["head_dim"]
        return {"bytes": L * (2 * nkv * M * hd * 2 + 2 * nh * hd * 4), "flops": L * 4 * nh * M * hd}
    size = flops = 0
    for n, (o, i) in _shapes(case).items():
        size += o * sa.row_bytes(_type(case, n), i) + 4 * M * o
        flops += 2 * M * o * i
    return {"bytes": L * (size + 4 * M * (3 * case["hidden"] + case["ffn"])), "flops": L * flops}


def tolerance(case):
    # f32 sums of exact or once-rounded terms, in another order (measured
    # against 64 bits: 0.5 to 3e-7)
    if case["kind"] != "attention":
        return {"rel": 1.2e-6, "max": 1.2e-5}
    # f16 probabilities that round the other way (measured: 1e-5)
    return {"rel": 4e-5, "max": 1e-3}


# ---- the same in 64 bits ----------------------------------------------------------


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(wtype, b, n_out, n_in):
    """GGUF blocks -> f64 [n_out, n_in]."""
    if wtype == sa.F16:
        return _f16(b).reshape(n_out, n_in)
    n = b.shape[0]

    def bits(t, *shifts):
        return torch.stack([(t >> s) for s in shifts], 1)

    if wtype in (sa.Q4_0, sa.Q5_0, sa.Q8_0):
        d = _f16(b[:, 0:2])
        if wtype == sa.Q8_0:
            q = b[:, 2:34].contiguous().view(torch.int8).double()
        else:
            qs = b[:, -16:]
            q = torch.cat([qs & 15, qs >> 4], 1).double()
            if wtype == sa.Q5_0:
                hi = bits(b[:, 2:6], *range(8)).transpose(1, 2).reshape(n, 32) & 1
                q = q + 16 * hi.double() - 16
            else:
                q = q - 8
        return (d * q).reshape(n_out, n_in)
    if wtype in (sa.Q4_K, sa.Q5_K):
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, -128:].reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32).double()
        if wtype == sa.Q5_K:
            q = q + 16 * (bits(b[:, 16:48], *range(8)) & 1).double()
        w = (_f16(b[:, 0:2]) * sc.double()).unsqueeze(2) * q
        return (w - (_f16(b[:, 2:4]) * mn.double()).unsqueeze(2)).reshape(n_out, n_in)
    if wtype == sa.Q2_K:
        q = bits(b[:, 16:80].reshape(n, 2, 32).transpose(0, 1).reshape(2 * n, 32), 0, 2, 4, 6) & 3
        q = q.reshape(2, n, 4, 32).transpose(0, 1).reshape(n, 16, 16).double()
        w = (_f16(b[:, 80:82]) * (b[:, 0:16] & 15).double()).unsqueeze(2) * q
        return (w - (_f16(b[:, 82:84]) * (b[:, 0:16] >> 4).double()).unsqueeze(2)).reshape(n_out, n_in)
    if wtype == sa.Q3_K:
        q = bits(b[:, 32:96].reshape(n, 2, 32).transpose(0, 1).reshape(2 * n, 32), 0, 2, 4, 6) & 3
        q = q.reshape(2, n, 4, 32).transpose(0, 1).reshape(n, 8, 32).double()
        q = q - 4 * (1 - (bits(b[:, 0:32], *range(8)) & 1).double())
        s = b[:, 96:108]
        lo = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        hi = (bits(s[:, 8:12], 0, 2, 4, 6) & 3).reshape(n, 16)
        sc = (lo | (hi << 4)).double() - 32
        return ((_f16(b[:, 108:110]) * sc).unsqueeze(2) * q.reshape(n, 16, 16)).reshape(n_out, n_in)
    # Q6_K
    ql = b[:, 0:128].reshape(n, 2, 2, 32)
    ql = torch.stack([ql & 15, ql >> 4], 2).reshape(n, 2, 4, 32)  # nibble, then the 32-byte half
    qh = b[:, 128:192].reshape(n, 2, 1, 32)
    qh = torch.cat([qh, qh >> 2, qh >> 4, qh >> 6], 2) & 3
    q = (ql | (qh << 4)).double() - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return ((_f16(b[:, 208:210]) * sc).unsqueeze(2) * q.reshape(n, 16, 16)).reshape(n_out, n_in)


def _pair(wtype, x):
    """The activation as the weight type's pair format holds it, in f64: f32
    steps on the host, one rounding each, then quant times scale."""
    x = x.cpu()
    if wtype == sa.F16:
        return x.half().double()
    M, n = x.shape
    if wtype in (sa.Q4_0, sa.Q5_0, sa.Q8_0):
        v = x.reshape(M, n // 32, 32)
        mx = v.abs().amax(2, keepdim=True)
        c = torch.full_like(mx, 127.0)  # tensor by tensor: one rounded division
        d = (mx / c).half().double()
        q = (v * (c / mx)).round()
    else:
        v = x.reshape(M, n // 256, 256)
        vmax = v.gather(2, v.abs().argmax(2, keepdim=True))
        inv = torch.full_like(vmax, -127.0) / vmax
        q = (v * inv).round().clamp(max=127)
        d = (torch.ones_like(inv) / inv).double()
    return (q.double() * d).reshape(M, n)


def exact(case, seed):
    if case["kind"] == "attention":
        nh, nkv, hd = case["heads"], case["kv_heads"], case["head_dim"]
        n, outs = case["rows"], []
        for q, k, v in _attention_inputs(case, seed):
            qh = q.half().double().reshape(nkv, nh // nkv, hd)
            s = torch.matmul(qh, k[:, :n].double().transpose(1, 2).contiguous()) / math.sqrt(hd)
            p = torch.softmax(s, 2).half().double()
            outs.append(torch.matmul(p, v[:, :, :n].double().transpose(1, 2).contiguous()).reshape(nh, hd))
        return outs
    outs = []
    for blocks, xs in zip(_layer_weights(case, seed), _activations(case, seed)):
        out = {}
        for names, x in zip(GROUPS, xs):
            pairs = {}
            for n in names:
                t = _type(case, n)
                if t not in pairs:
                    pairs[t] = _pair(t, x).cuda()
                y = torch.matmul(pairs[t], _dequant(t, blocks[n], *_shapes(case)[n]).t())
                out[n] = y[0].cpu().numpy() if case["kind"] == "host" else y
        outs.append(out)
    return outs
