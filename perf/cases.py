"""The work a user of the quantized compute path has it do, as timed cases.

Decode matvecs (one token, and batches of 2 to 8), the output head, the dense
FFN half of a layer for one token and for a short prompt, the MoE layer and
its routed part in both expert orientations, the prefill matmul in two modes,
and the host-slice trait call. Shapes are those of the benchmark (dense 4096 /
12288, head 151936, MoE 128 experts x 2048 x 768 top-8) and generic ones.

A decode pass visits the matrices of several layers, as a token does on its
way through a model, so weights come from device memory and not from a cache
that a single matrix would fit.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "strata-rs_amd"))
import strata_hip as H  # noqa: E402

Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS, F32 = (int(getattr(H.QuantType, n)) for n in
                                       ("Q8_0", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "F32"))
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), IQ4_XS: (256, 136), F32: (1, 4)}
# rms of a weight over its block scale d for uniformly drawn codes and scales
RMS = {Q8_0: 73.0, Q4_K: 320.0, Q5_K: 650.0, Q6_K: 680.0, IQ4_XS: 1200.0}
NAMES = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K, "iq4_xs": IQ4_XS}
EPS = 1e-6


def listed():
    return [
        # the drop-in trait call: one host-slice matvec of an attention
        # projection with resident weights (the smallest call a user makes)
        {"name": "host_proj_q8_0", "op": "host_gemv", "quant": "q8_0", "rows": 4096, "cols": 4096},
        # one-token decode: the FFN down projection of eight layers
        {"name": "decode_down_q4k", "op": "gemv", "quant": "q4_k", "rows": 4096, "cols": 12288, "batch": 1,
         "layers": 8},
        # one-token decode: the output head
        {"name": "decode_head_q6k", "op": "gemv", "quant": "q6_k", "rows": 151936, "cols": 4096, "batch": 1,
         "layers": 1},
        # eight sequences decoded together: the gate projection of eight layers
        {"name": "batch8_gate_q4k", "op": "gemv", "quant": "q4_k", "rows": 12288, "cols": 4096, "batch": 8,
         "layers": 8},
        # four sequences decoded together: the output head
        {"name": "batch4_head_q6k", "op": "gemv", "quant": "q6_k", "rows": 151936, "cols": 4096, "batch": 4,
         "layers": 1},
        # one-token decode: the dense FFN half of three layers
        {"name": "ffn_1tok_q4k", "op": "ffn", "gate": "q4_k", "down": "q4_k", "embd": 4096, "ff": 12288, "tok": 1,
         "layers": 3},
        # a short prompt of an odd length through the dense FFN half of one
        # layer, with the usual mix of types (gate and up Q4_K, down Q6_K)
        {"name": "ffn_77tok_q4k_q6k", "op": "ffn", "gate": "q4_k", "down": "q6_k", "embd": 4096, "ff": 12288,
         "tok": 77, "layers": 1},
        # one-token decode: the whole MoE layer, eight tokens one after another
        {"name": "moe_layer_1tok", "op": "moe_layer", "gate": "q4_k", "down": "q6_k", "experts": 128, "top_k": 8,
         "embd": 2048, "ff": 768, "ff_sh": 768, "tok": 1, "out_major": False, "calls": 8},
        # sixteen sequences decoded together through the routed experts
        {"name": "moe_16tok", "op": "moe_ffn", "gate": "q4_k", "down": "q6_k", "experts": 128, "top_k": 8,
         "embd": 2048, "ff": 768, "tok": 16, "out_major": False, "calls": 1},
        # a prompt's chunk through the whole MoE layer, expert stacks as
        # llama.cpp files store them
        {"name": "moe_layer_96tok_out_major", "op": "moe_layer", "gate": "q4_k", "down": "q6_k", "experts": 128,
         "top_k": 8, "embd": 2048, "ff": 768, "ff_sh": 768, "tok": 96, "out_major": True, "calls": 1},
        # prefill: the gate projection for a 512-token chunk, bf16 activations
        {"name": "prefill_bf16_512_q4k", "op": "matmul", "quant": "q4_k", "rows": 12288, "cols": 4096, "m": 512,
         "mode": "bf16"},
        # prefill: the down projection for a prompt of odd length, int8 activations
        {"name": "prefill_q8_333_q5k", "op": "matmul", "quant": "q5_k", "rows": 4096, "cols": 12288, "m": 333,
         "mode": "q8"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gemv", "gemv", "batch", "batch", "ffn", "ffn", "moe_ffn", "moe_layer", "matmul", "matmul",
                     "host_gemv"])
    quant = rng.choice(list(NAMES))
    if op in ("gemv", "batch", "host_gemv"):
        cols = 256 * _log(rng, 2, 56)
        rows = _log(rng, 512, min(152064, 300_000_000 // cols))
        if op == "host_gemv":
            return {"op": "host_gemv", "quant": quant, "rows": min(rows, 16384), "cols": cols}
        layers = max(1, min(8, 200_000_000 // (rows * cols)))
        return {"op": "gemv", "quant": quant, "rows": rows, "cols": cols,
                "batch": 1 if op == "gemv" else rng.randint(2, 8), "layers": layers}
    if op == "matmul":
        cols = 256 * _log(rng, 2, 48)
        return {"op": "matmul", "quant": quant, "rows": _log(rng, 512, 12288), "cols": cols, "m": _log(rng, 9, 512),
                "mode": rng.choice(["bf16", "bf16", "q8"])}
    down = rng.choice(["q4_k", "q5_k", "q6_k", "q8_0"])
    gate = rng.choice(["q4_k", "q4_k", "q5_k", "q8_0"])
    if op == "ffn":
        return {"op": "ffn", "gate": gate, "down": down, "embd": 256 * _log(rng, 4, 16), "ff": 256 * _log(rng, 8, 48),
                "tok": rng.choice([1, _log(rng, 2, 77), _log(rng, 2, 77)]), "layers": 1}
    c = {"op": op, "gate": gate, "down": down, "experts": rng.choice([32, 64, 128]), "top_k": rng.choice([2, 4, 8]),
         "embd": 256 * rng.randint(4, 8), "ff": 256 * rng.randint(2, 4),
         "tok": rng.choice([1, _log(rng, 2, 96), _log(rng, 2, 96)]), "out_major": rng.random() < 0.5, "calls": 1}
    if op == "moe_layer":
        c["ff_sh"] = c["ff"]
    return c


# ---- packed weights, made on the GPU ---------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _weights(g, quant, rows, cols):
    """rows x cols of packed blocks: uniform codes and sub-block scales, block
    scales |N(0, 1)| times what brings the weights to about 1 / sqrt(fan-in
    of 64-to-4096-wide layers), so that outputs are of order one."""
    bs, nb = BLOCK[quant]
    if quant == F32:
        return _normal(g, rows, cols) / math.sqrt(cols)
    n = rows * (cols // bs)
    b = torch.randint(0, 256, (n, nb), generator=g, device="cuda", dtype=torch.uint8)
    d = (_normal(g, n).abs_() / (RMS[quant] * 64.0)).to(torch.float16)
    if quant == Q6_K:
        b[:, 192:208] = torch.randint(-64, 64, (n, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        b[:, 208:210] = d.view(torch.uint8).reshape(n, 2)
    else:
        b[:, 0:2] = d.view(torch.uint8).reshape(n, 2)
    if quant in (Q4_K, Q5_K):
        d2 = (_normal(g, n).abs_() / (RMS[quant] * 64.0)).to(torch.float16)
        b[:, 2:4] = d2.view(torch.uint8).reshape(n, 2)
    return b


def _flags(quant):
    # the readings that llama.cpp's files need
    return H.FLAG_Q6K_SIGNED_SCALES if quant == Q6_K else H.FLAG_IQ4XS_GGML if quant == IQ4_XS else 0


def _empty(*shape):
    return torch.empty(*shape, device="cuda", dtype=torch.float32)


def _workspace(nbytes):
    return torch.empty(max(int(nbytes), 256), device="cuda", dtype=torch.uint8)


# ---- what a program has in hand --------------------------------------------


def prepare(case, seed):
    g = _gen(seed)
    op = case["op"]
    st = dict(case)
    if op in ("gemv", "host_gemv", "matmul"):
        q = NAMES[case["quant"]]
        rows, cols = case["rows"], case["cols"]
        st["q"], st["flags"] = q, _flags(q)
    if op == "host_gemv":
        w = _weights(g, q, rows, cols).cpu().numpy()
        st["x"] = _normal(g, cols).cpu().numpy()
        st["y"] = np.empty(rows, np.float32)
        st["be"] = H.HipBackend(0)
        st["w"] = H.QuantTensor("proj", q, rows, cols, w, flags=st["flags"])
        st["be"].upload("proj", q, 1, rows, cols, w)
    elif op == "gemv":
        b = case["batch"]
        st["w"] = [_weights(g, q, rows, cols) for _ in range(case["layers"])]
        st["x"] = [_normal(g, b, cols) for _ in range(case["layers"])]
        st["y"] = [_empty(b, rows) for _ in range(case["layers"])]
        st["ws"] = _workspace(H.gemv_workspace_bytes(q, rows, cols, b))
    elif op == "matmul":
        m = case["m"]
        st["mm"] = H.MATMUL_BF16 if case["mode"] == "bf16" else H.MATMUL_Q8
        st["w"] = _weights(g, q, rows, cols)
        st["x"] = _normal(g, m, cols)
        st["y"] = _empty(m, rows)
        st["ws"] = _workspace(H.matmul_workspace_bytes(q, rows, cols, m, st["mm"]))
    elif op == "ffn":
        qg, qd, e, f, t = NAMES[case["gate"]], NAMES[case["down"]], case["embd"], case["ff"], case["tok"]
        st["w"] = [(_weights(g, qg, f, e), _weights(g, qg, f, e), _weights(g, qd, e, f))
                   for _ in range(case["layers"])]
        st["norm"] = [1.0 + 0.1 * _normal(g, e) for _ in range(case["layers"])]
        st["x"] = [_normal(g, t, e) for _ in range(case["layers"])]
        st["y"] = [_empty(t, e) for _ in range(case["layers"])]
        st["ws"] = _workspace(H.ffn_workspace_bytes(t, e, f))
        st["tensors"] = [[(q, _flags(q), w.data_ptr()) for q, w in zip((qg, qg, qd), ws)] for ws in st["w"]]
    else:
        qg, qd, n, e, f, t = (NAMES[case["gate"]], NAMES[case["down"]], case["experts"], case["embd"], case["ff"],
                              case["tok"])
        om = H.FLAG_EXPERT_OUT_MAJOR if case["out_major"] else 0
        in_out = ((n * f, e), (n * e, f)) if case["out_major"] else ((n * e, f), (n * f, e))
        experts = [_weights(g, qg, *in_out[0]), _weights(g, qg, *in_out[0]), _weights(g, qd, *in_out[1])]
        tensors = [(q, _flags(q) | om, w.data_ptr()) for q, w in zip((qg, qg, qd), experts)]
        st["x"] = [_normal(g, t, e) for _ in range(case["calls"])]
        st["y"] = [_empty(t, e) for _ in range(case["calls"])]
        if op == "moe_ffn":
            st["w"], st["tensors"] = experts, tensors
            st["logits"] = [_normal(g, t, n) for _ in range(case["calls"])]
            st["ws"] = _workspace(H.moe_workspace_bytes(t, case["top_k"], n, e, f, qg, qd))
        else:
            fs = case["ff_sh"]
            router, inp = _weights(g, F32, n, e), _weights(g, F32, 1, e)
            shared = [_weights(g, qg, fs, e), _weights(g, qg, fs, e), _weights(g, qd, e, fs)]
            st["w"] = [router] + experts + shared + [inp]
            st["tensors"] = ([(F32, 0, router.data_ptr())] + tensors +
                             [(q, _flags(q), w.data_ptr()) for q, w in zip((qg, qg, qd), shared)] +
                             [(F32, 0, inp.data_ptr())])
            st["ws"] = _workspace(H.moe_layer_workspace_bytes(t, case["top_k"], n, e, f, fs,
                                                              [F32, qg, qg, qd, qg, qg, qd, F32]))
    return st


def run(st):
    op = st["op"]
    if op == "host_gemv":
        st["be"].gemv(st["w"], st["x"], st["y"])
        return st["y"]
    ws, nws = st["ws"].data_ptr(), st["ws"].numel()
    if op == "gemv":
        for w, x, y in zip(st["w"], st["x"], st["y"]):
            if st["batch"] == 1:
                H.gemv_dev(st["q"], w.data_ptr(), st["rows"], st["cols"], x.data_ptr(), y.data_ptr(), 1,
                           flags=st["flags"])
            else:
                H.gemv_dev_ws(st["q"], w.data_ptr(), st["rows"], st["cols"], x.data_ptr(), y.data_ptr(), st["batch"],
                              ws, nws, flags=st["flags"])
    elif op == "matmul":
        H.matmul_dev(st["q"], st["w"].data_ptr(), st["rows"], st["cols"], st["x"].data_ptr(), st["m"],
                     st["y"].data_ptr(), st["mm"], ws, nws, flags=st["flags"])
    elif op == "ffn":
        for t, n, x, y in zip(st["tensors"], st["norm"], st["x"], st["y"]):
            H.ffn_dev(t, st["embd"], st["ff"], st["tok"], x.data_ptr(), n.data_ptr(), EPS, y.data_ptr(), ws, nws)
    elif op == "moe_ffn":
        for lg, x, y in zip(st["logits"], st["x"], st["y"]):
            H.moe_ffn_dev(*st["tensors"], st["experts"], st["embd"], st["ff"], lg.data_ptr(), st["tok"], st["top_k"],
                          x.data_ptr(), y.data_ptr(), ws, nws)
    else:
        for x, y in zip(st["x"], st["y"]):
            H.moe_layer_dev(st["tensors"], st["experts"], st["embd"], st["ff"], st["ff_sh"], st["tok"], st["top_k"],
                            x.data_ptr(), y.data_ptr(), ws, nws)
    return st["y"]


# ---- what a pass cannot do without ------------------------------------------


def _nbytes(q, rows, cols):
    bs, nb = BLOCK[q]
    return rows * (cols // bs) * nb


def work(case):
    op = case["op"]
    if op in ("gemv", "host_gemv", "matmul"):
        rows, cols = case["rows"], case["cols"]
        b = case.get("batch", case.get("m", 1))
        n = case.get("layers", 1)
        return {"bytes": n * (_nbytes(NAMES[case["quant"]], rows, cols) + 4 * b * (rows + cols)),
                "flops": n * 2 * b * rows * cols}
    qg, qd, e, f, t = NAMES[case["gate"]], NAMES[case["down"]], case["embd"], case["ff"], case["tok"]
    if op == "ffn":
        n = case["layers"]
        return {"bytes": n * (2 * _nbytes(qg, f, e) + _nbytes(qd, e, f) + 4 * e * (2 * t + 1)),
                "flops": n * t * 6 * e * f}
    n, k, calls = case["experts"], case["top_k"], case["calls"]
    # the experts that t tokens with k picks each touch, on average
    seen = n * (1.0 - (1.0 - k / n) ** t)
    bytes_ = seen * (2 * _nbytes(qg, e, f) + _nbytes(qd, f, e)) + 4 * t * 2 * e
    flops = t * k * 6 * e * f
    if op == "moe_ffn":
        bytes_ += 4 * t * n
    else:
        fs = case["ff_sh"]
        bytes_ += 4 * (n + 1) * e + 2 * _nbytes(qg, fs, e) + _nbytes(qd, e, fs)
        flops += t * (6 * e * fs + 2 * (n + 1) * e)
    return {"bytes": calls * bytes_, "flops": calls * flops}


def tolerance(case):
    # about four times the distance from exact() that the path shows
    if case["op"] == "matmul":
        # bf16: operands rounded to 8 bits (2.4e-3); q8: activations rounded
        # to 1/127 of the largest of 32 (5.4e-3)
        return {"rel": 1e-2} if case["mode"] == "bf16" else {"rel": 2e-2}
    # 32-bit activations and sums (5e-7; chained matvecs 8e-7), with room for
    # the order of a sum over the widest rows
    return {"rel": 5e-6}


# ---- the same in 64 bits ------------------------------------------------------


def _f16(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _scale_min(s):
    """The eight 6-bit scales and mins of 12 packed bytes."""
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return sc.to(torch.float64), mn.to(torch.float64)


_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _dequant(q, b):
    """n packed blocks -> [n][block] in 64 bits (signed Q6_K scales, llama.cpp's IQ4_XS)."""
    n = b.shape[0]
    if q == Q8_0:
        return _f16(b[:, 0:2]) * b[:, 2:34].view(torch.int8).to(torch.float64)
    if q in (Q4_K, Q5_K):
        d, m = _f16(b[:, 0:2]), _f16(b[:, 2:4])
        sc, mn = _scale_min(b[:, 4:16])
        qs = b[:, 16:144] if q == Q4_K else b[:, 48:176]
        c = qs.reshape(n, 4, 1, 32)
        c = torch.cat([c & 15, c >> 4], 2).reshape(n, 8, 32)
        if q == Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).reshape(1, 8, 1)
            c = c + (((b[:, 16:48].reshape(n, 1, 32) >> bit) & 1) << 4)
        return ((d * sc).unsqueeze(2) * c.to(torch.float64) - (m * mn).unsqueeze(2)).reshape(n, 256)
    if q == Q6_K:
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # [n][half][4][32]
        shift = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8).reshape(1, 1, 4, 1)
        c = (lo | (((qh >> shift) & 3) << 4)).to(torch.float64) - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        return (c.reshape(n, 16, 16) * (sc * _f16(b[:, 208:210])).unsqueeze(2)).reshape(n, 256)
    d = _f16(b[:, 0:2])
    sh = b[:, 2].to(torch.int64) | (b[:, 3].to(torch.int64) << 8)
    i = torch.arange(8, device=b.device)
    sl = b[:, 4:8].to(torch.int64)
    ls = ((sl[:, i // 2] >> (4 * (i % 2))) & 15) | (((sh.unsqueeze(1) >> (2 * i)) & 3) << 4)
    qs = b[:, 8:136].reshape(n, 8, 16)
    code = torch.tensor(_IQ4, device=b.device, dtype=torch.float64)[torch.cat([qs & 15, qs >> 4], 2).to(torch.int64)]
    return ((d * (ls - 32).to(torch.float64)).unsqueeze(2) * code).reshape(n, 256)


def _apply(q, w, rows, cols, x):
    """x [b][cols] times the rows of packed w, in 64 bits: [b][rows]."""
    x = x.to(torch.float64)
    if q == F32:
        return x @ w.to(torch.float64).reshape(rows, cols).t()
    per = cols // BLOCK[q][0]
    step = max(1, (1 << 26) // cols)
    out = []
    for r in range(0, rows, step):
        k = min(step, rows - r)
        out.append(x @ _dequant(q, w[r * per:(r + k) * per]).reshape(k, cols).t())
    return torch.cat(out, 1)


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _expert(q, w, e, rows, cols, x, out_major):
    """One expert's product: rows x cols as stored, blocks along cols."""
    per = rows * (cols // BLOCK[q][0])
    m = _dequant(q, w[e * per:(e + 1) * per]).reshape(rows, cols)
    return x @ (m.t() if out_major else m)


def exact(case, seed):
    st = prepare(case, seed)
    op = case["op"]
    if op == "host_gemv":
        w = torch.from_numpy(st["w"]._buf).cuda().reshape(-1, BLOCK[st["q"]][1])
        x = torch.from_numpy(st["x"]).cuda().reshape(1, -1)
        return _apply(st["q"], w, case["rows"], case["cols"], x).reshape(-1).cpu().numpy()
    if op == "gemv":
        return [_apply(st["q"], w, case["rows"], case["cols"], x) for w, x in zip(st["w"], st["x"])]
    if op == "matmul":
        return _apply(st["q"], st["w"], case["rows"], case["cols"], st["x"])
    qg, qd, e, f = NAMES[case["gate"]], NAMES[case["down"]], case["embd"], case["ff"]
    out = []
    if op == "ffn":
        for (wg, wu, wd), n, x in zip(st["w"], st["norm"], st["x"]):
            x = x.to(torch.float64)
            mixed = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * n.to(torch.float64)
            h = _silu(_apply(qg, wg, f, e, mixed)) * _apply(qg, wu, f, e, mixed)
            out.append(x + _apply(qd, wd, e, f, h))
        return out
    n, k, om = case["experts"], case["top_k"], case["out_major"]
    ga, dn = ((f, e), (e, f)) if om else ((e, f), (f, e))
    wg, wu, wd = st["w"][1:4] if op == "moe_layer" else st["w"]
    for i, x in enumerate(st["x"]):
        logits = _apply(F32, st["w"][0], n, e, x.to(torch.bfloat16)) if op == "moe_layer" else st["logits"][i]
        x = x.to(torch.float64)
        p, ids = torch.softmax(logits.to(torch.float64), 1).topk(k, 1)
        p = p / p.sum(1, keepdim=True).clamp_min(2.0 ** -14)
        y = torch.zeros_like(x)
        for ex in ids.unique().tolist():
            t, slot = (ids == ex).nonzero(as_tuple=True)
            h = (_silu(_expert(qg, wg, ex, *ga, x[t], om)) * _expert(qg, wu, ex, *ga, x[t], om))
            y.index_add_(0, t, p[t, slot].unsqueeze(1) * _expert(qd, wd, ex, *dn, h, om))
        if op == "moe_layer":
            fs = case["ff_sh"]
            sg, su, sd, inp = st["w"][4:8]
            h = _silu(_apply(qg, sg, fs, e, x)) * _apply(qg, su, fs, e, x)
            y = y + torch.sigmoid(_apply(F32, inp, 1, e, x)) * _apply(qd, sd, e, fs, h)
        out.append(y)
    return out
