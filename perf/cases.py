"""The work whose speed matters: calls of the loom_hip kernels as programs make
them, over the range of sizes, types and options they are made with.

``listed()`` names twelve of them, ``draw()`` gives more of the same ranges;
``prepare`` makes what a program holds before a call, ``run`` makes the call,
``work`` counts the bytes and operations the call cannot do without,
``tolerance`` bounds what another correct implementation may differ by, and
``exact`` computes the same outputs in 64 bits without this library.

Every case is a dict of plain values; ``op`` is the entry point (``ssd`` is the
prologue followed by the chunk scan, ``prologue`` the former alone) and ``dtype`` the 16-bit element type.
Block sizes (``tile``, ``tile_k``, ``tile_s``) of 0 leave the choice to the
library, as a call without them does.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "loom-dataflow_amd"))

import loom_hip  # noqa: E402

_TYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # the reference's own matmul example: a small projection, where the
        # launch and the host path weigh as much as the arithmetic
        {"name": "mm_small_f16", "op": "matmul", "dtype": "f16", "M": 2048, "N": 256, "K": 256,
         "tile": 0},
        # one ordinary square product
        {"name": "mm_1024", "op": "matmul", "dtype": "bf16", "M": 1024, "N": 1024, "K": 1024,
         "tile": 0},
        # extents as data gives them: rows off 16-byte boundaries in A, B and C
        {"name": "mm_ragged", "op": "matmul", "dtype": "bf16", "M": 1003, "N": 1531, "K": 2051,
         "tile": 0},
        # a batch of large products (the benchmark's headline)
        {"name": "bmm_16x2048", "op": "batch_matmul", "dtype": "bf16", "B": 16, "M": 2048,
         "N": 2048, "K": 2048, "tile": 0},
        # a long contraction with a small output, its K slabs gathered in fp32
        {"name": "split_k_16384", "op": "split_k", "dtype": "bf16", "M": 512, "N": 512,
         "K": 16384, "tile_k": 1024},
        # prefill of a batch of long prompts
        {"name": "attn_prefill", "op": "attention", "dtype": "bf16", "BH": 128, "Sq": 4096,
         "Skv": 4096, "D": 128, "causal": True},
        # prefill of one prompt of a thousand tokens
        {"name": "attn_prompt", "op": "attention", "dtype": "bf16", "BH": 32, "Sq": 1000,
         "Skv": 1000, "D": 128, "causal": True},
        # attention over another sequence of odd length
        {"name": "attn_cross_f16", "op": "attention", "dtype": "f16", "BH": 32, "Sq": 333,
         "Skv": 1003, "D": 64, "causal": False},
        # one decoding step of a serving batch with long caches
        {"name": "decode_batch", "op": "decode", "dtype": "bf16", "B": 32, "H": 32, "D": 128,
         "S": 8192, "tile_s": 1024},
        # one decoding step of a single sequence whose cache has grown to an
        # odd length (seven of eight steps find one off 16-byte rows)
        {"name": "decode_one", "op": "decode", "dtype": "bf16", "B": 1, "H": 32, "D": 128,
         "S": 4097, "tile_s": 0},
        # the scan of a training-size batch of long sequences
        {"name": "scan_batch", "op": "scan", "dtype": "bf16", "b": 4, "nc": 16, "H": 32, "G": 1,
         "Q": 256, "P": 64, "N": 128},
        # the whole SSD layer (prologue, then scan) on one sequence
        {"name": "ssd_one", "op": "ssd", "dtype": "bf16", "b": 1, "nc": 16, "H": 32, "G": 1,
         "Q": 256, "P": 64, "N": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """An extent between lo and hi, spread over its logarithm: half of them a
    multiple of 64 (sizes a model is built with), a quarter a multiple of 8,
    a quarter as data gives them."""
    v = _log(rng, lo, hi)
    k = rng.random()
    step = 64 if k < 0.5 else 8 if k < 0.75 else 1
    return max(lo, min(hi, (v + step // 2) // step * step or step))


def _draw_once(rng):
    op = rng.choice(["matmul", "matmul", "batch_matmul", "split_k", "attention", "attention",
                     "decode", "decode", "scan", "ssd"])
    c = {"op": op, "dtype": "bf16" if rng.random() < 0.65 else "f16"}
    if op == "matmul":
        c.update(M=_size(rng, 16, 8192), N=_size(rng, 64, 8192), K=_size(rng, 64, 8192), tile=0)
    elif op == "batch_matmul":
        c.update(B=_log(rng, 2, 32), M=_size(rng, 64, 4096), N=_size(rng, 64, 4096),
                 K=_size(rng, 64, 4096), tile=0)
    elif op == "split_k":
        k = _size(rng, 2048, 32768)
        c.update(M=_size(rng, 64, 1024), N=_size(rng, 64, 1024), K=k,
                 tile_k=max(64, k // rng.choice([4, 8, 16, 32]) // 64 * 64))
    elif op == "attention":
        causal = rng.random() < 0.5
        sq = _size(rng, 64, 8192)
        c.update(BH=rng.choice([8, 12, 16, 32, 40, 64, 96, 128]), Sq=sq,
                 Skv=sq if causal else _size(rng, 64, 8192),
                 D=rng.choice([64, 64, 80, 96, 128, 128, 128, 256]), causal=causal)
    elif op == "decode":
        c.update(B=_log(rng, 1, 64), H=rng.choice([8, 16, 32, 32, 48, 64, 71]),
                 D=rng.choice([64, 128, 128, 256]), S=_size(rng, 128, 16384), tile_s=0)
        if rng.random() < 0.3:
            c["tile_s"] = min(c["S"], rng.choice([256, 512, 1024]))
    else:
        c.update(b=_log(rng, 1, 4), nc=_log(rng, 1, 32), H=rng.choice([8, 16, 24, 32, 64]),
                 G=rng.choice([1, 1, 2, 4]), Q=rng.choice([64, 128, 192, 256, 256]),
                 P=rng.choice([32, 64, 64, 128]), N=rng.choice([32, 64, 128, 128]))
        if op == "ssd" and c["dtype"] == "f16":     # the f16 scan takes its side tensors in f16
            c["op"] = "prologue"
    if op in ("matmul", "batch_matmul") and rng.random() < 0.2:
        t = rng.choice([64, 128, 256])
        if t <= min(c["M"], c["N"]):
            c["tile"] = t
    return c


def draw(rng):
    """One more case, no more costly than the largest listed one of its kind."""
    most = {}
    for c in listed():
        w = work(c)
        kind = {"batch_matmul": "matmul"}.get(c["op"], c["op"])
        have = most.get(kind, (0, 0))
        most[kind] = (max(have[0], w["bytes"]), max(have[1], w["flops"]))
    most["ssd"] = most["prologue"] = most["scan"]
    while True:
        c = _draw_once(rng)
        w = work(c)
        b, f = most[{"batch_matmul": "matmul"}.get(c["op"], c["op"])]
        if w["bytes"] <= b and w["flops"] <= f:
            return c


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _uniform(g, shape, dtype):
    return (torch.rand(shape, generator=g, device="cuda") * 2 - 1).to(dtype)


def _ssd_raw(case, g):
    """x, dt, A, B, C, D of an SSD layer: dt past its softplus, A below zero."""
    b, nc, H, G, Q, P, N = (case[k] for k in ("b", "nc", "H", "G", "Q", "P", "N"))
    e = _TYPES[case["dtype"]]
    L = nc * Q
    x = _normal(g, (b, H, L, P), e)
    dt = torch.nn.functional.softplus(torch.randn((b, H, L), generator=g, device="cuda"))
    A = -torch.exp(torch.rand((H,), generator=g, device="cuda"))
    B = _normal(g, (b, G, L, N), e)
    C = _normal(g, (b, G, L, N), e)
    D = torch.randn((H,), generator=g, device="cuda")
    return x, dt, A, B, C, D


def _ssd_stages(case, x, dt, A, B, C, wide):
    """dA_cumsum, cb and prev_states_T of the layer's inputs, in `wide`."""
    b, nc, H, G, Q, P, N = (case[k] for k in ("b", "nc", "H", "G", "Q", "P", "N"))
    dt = dt.to(wide).view(b, H, nc, Q)
    dA = torch.cumsum(dt * A.to(wide).view(1, H, 1, 1), dim=-1)
    Bc = B.to(wide).view(b, G, nc, Q, N)
    Cc = C.to(wide).view(b, G, nc, Q, N)
    cb = torch.matmul(Cc, Bc.transpose(-1, -2).contiguous()).tril_()
    cb = cb.permute(0, 2, 1, 3, 4).contiguous()
    w = torch.exp(dA[..., -1:] - dA) * dt
    # states[b, h, c, n, p] = sum_k B[k, n] w[k] x[k, p]
    wx = x.to(wide).view(b, H, nc, Q, P) * w.unsqueeze(-1)
    Bt = Bc.transpose(-1, -2).contiguous()
    states = torch.empty((b, H, nc, N, P), dtype=wide, device=x.device)
    for h in range(H):
        states[:, h] = torch.matmul(Bt[:, h // (H // G)], wx[:, h])
    prev = torch.zeros((b, nc, H, N, P), dtype=wide, device=x.device)
    for c in range(1, nc):
        prev[:, c] = prev[:, c - 1] * torch.exp(dA[:, :, c - 1, -1]).view(b, H, 1, 1) \
            + states[:, :, c - 1]
    return dA, cb, prev


def _side(case):
    """Type of the scan's side tensors: fp32 beside bf16, f16 beside f16."""
    return torch.float32 if case["dtype"] == "bf16" else torch.float16


def _inputs(case, seed):
    g = _gen(seed)
    e = _TYPES[case["dtype"]]
    op = case["op"]
    if op == "matmul":
        return _uniform(g, (case["M"], case["K"]), e), _uniform(g, (case["K"], case["N"]), e)
    if op == "batch_matmul":
        return (_normal(g, (case["B"], case["M"], case["K"]), e, 0.02),
                _normal(g, (case["B"], case["K"], case["N"]), e, 0.02))
    if op == "split_k":
        return _uniform(g, (case["M"], case["K"]), e), _uniform(g, (case["K"], case["N"]), e)
    if op == "attention":
        return (_normal(g, (case["BH"], case["D"], case["Skv"]), e),
                _normal(g, (case["BH"], case["Skv"], case["D"]), e),
                _normal(g, (case["BH"], case["Sq"], case["D"]), e))
    if op == "decode":
        return (_normal(g, (case["B"], case["D"], case["S"]), e),
                _normal(g, (case["B"], case["S"], case["D"]), e),
                _normal(g, (case["B"], case["H"], case["D"]), e))
    x, dt, A, B, C, D = _ssd_raw(case, g)
    if op != "scan":
        return x, dt, A, B, C, D
    # the scan alone: its inputs as a prologue leaves them
    dA, cb, prev = _ssd_stages(case, x, dt, A, B, C, torch.float32)
    s = _side(case)
    return (cb.to(e), x, dt.view(case["b"], case["H"], case["nc"], case["Q"]).to(s), dA.to(s), C,
            D.to(s), prev.to(s))


def prepare(case, seed):
    t = _inputs(case, seed)
    state = {"case": case, "in": t}
    # programs that gather partial results hold the buffer they go to
    if case["op"] == "split_k":
        slabs = -(-case["K"] // case["tile_k"])
        state["partials"] = torch.empty((slabs, case["M"], case["N"]), dtype=torch.float32,
                                        device="cuda")
    if case["op"] == "decode" and case["tile_s"]:
        state["workspace"] = loom_hip.flash_decode_workspace(
            case["B"], case["H"], case["D"], case["S"], case["tile_s"], t[0].device)
    return state


def run(state):
    case, t = state["case"], state["in"]
    op = case["op"]
    if op == "matmul":
        tile = case["tile"] or None
        return loom_hip.matmul(*t, tile_m=tile, tile_n=tile)
    if op == "batch_matmul":
        tile = case["tile"] or None
        return loom_hip.batch_matmul(*t, tile_m=tile, tile_n=tile)
    if op == "split_k":
        return loom_hip.split_k_matmul_gather(*t, partials=state["partials"],
                                              tile_k=case["tile_k"])
    if op == "attention":
        return loom_hip.attention(*t, causal=case["causal"])
    if op == "decode":
        return loom_hip.flash_decode(*t, workspace=state.get("workspace"),
                                     tile_s=case["tile_s"] or None)
    if op == "scan":
        return loom_hip.helion_mamba2_chunk_scan_kernel(*t)
    x, dt, A, B, C, D = t
    dt4, dA, cb, prev = loom_hip.ssd_prologue(x, dt, A, B, C, case["Q"])
    if op == "prologue":
        return dA, cb, prev
    return loom_hip.helion_mamba2_chunk_scan_kernel(cb, x, dt4, dA, C, D, prev), dA, cb, prev


def work(case):
    op = case["op"]
    if op in ("matmul", "batch_matmul", "split_k"):
        z, M, N, K = case.get("B", 1), case["M"], case["N"], case["K"]
        nbytes = 2 * z * (M * K + K * N + M * N)
        if op == "split_k":         # the gathered slabs are an output too
            nbytes += 4 * -(-K // case["tile_k"]) * M * N
        return {"bytes": nbytes, "flops": 2 * z * M * N * K}
    if op == "attention":
        BH, Sq, Skv, D = case["BH"], case["Sq"], case["Skv"], case["D"]
        pairs = Sq * (Sq + 1) // 2 if case["causal"] else Sq * Skv
        return {"bytes": 2 * BH * D * (2 * Skv + 2 * Sq), "flops": 4 * BH * D * pairs}
    if op == "decode":
        B, H, D, S = case["B"], case["H"], case["D"], case["S"]
        return {"bytes": 2 * B * D * (2 * S + 2 * H), "flops": 4 * B * H * S * D}
    b, nc, H, G, Q, P, N = (case[k] for k in ("b", "nc", "H", "G", "Q", "P", "N"))
    L, tri = nc * Q, Q * (Q + 1) // 2
    side = 4 if case["dtype"] == "bf16" else 2
    xo = 2 * b * H * L * P * (1 if op == "prologue" else 2)     # x read, out written
    scan = 2 * b * H * (L * N * P + nc * tri * P)
    if op == "scan":
        nbytes = xo + 2 * b * nc * G * tri + 2 * b * G * L * N + side * (2 * b * H * L + H
                                                                        + b * nc * H * N * P)
        return {"bytes": nbytes, "flops": scan}
    # dt, A, D and B, C read; dA_cumsum, cb and prev_states_T written
    nbytes = xo + 4 * (b * H * L + 2 * H) + 2 * 2 * b * G * L * N \
        + 4 * b * H * L + 2 * b * nc * G * Q * Q + 4 * b * nc * H * N * P
    return {"bytes": nbytes, "flops": (scan if op == "ssd" else 0) + 2 * b * nc * G * tri * N
            + 2 * b * H * L * N * P}


def tolerance(case):
    # about four times the distance from 64-bit results: the rounding of the
    # output (1.7e-3 in bf16, 2.1e-4 in f16), and in attention and decode that
    # of the probabilities and the scaled queries too (up to 2.9e-3, 3.6e-4)
    soft = case["op"] in ("attention", "decode", "ssd")
    if case["dtype"] == "bf16":
        return {"rel": 1.2e-2 if soft else 7e-3}
    return {"rel": 1.5e-3 if soft else 9e-4}


def _softmax_out(s, v, mask=None):
    if mask is not None:
        s = s.masked_fill(mask, float("-inf"))
    return torch.matmul(torch.softmax(s, dim=-1), v)


def _scan64(case, cb, x, dt, dA, C, D, prev):
    """The chunk scan in 64 bits, one head at a time."""
    b, nc, H, G, Q, P, N = (case[k] for k in ("b", "nc", "H", "G", "Q", "P", "N"))
    f = torch.float64
    x, dt, dA = x.to(f).view(b, H, nc, Q, P), dt.to(f), dA.to(f)
    C = C.to(f).view(b, G, nc, Q, N)
    above = torch.ones((Q, Q), dtype=torch.bool, device=x.device).triu_(1)
    out = torch.empty((b, H, nc, Q, P), dtype=f, device=x.device)
    for h in range(H):
        g = h // (H // G)
        d = dA[:, h]
        decay = torch.exp((d.unsqueeze(-1) - d.unsqueeze(-2)).masked_fill(above, float("-inf")))
        w = cb[:, :, g].to(f) * decay * dt[:, h].unsqueeze(-2)
        out[:, h] = torch.matmul(w, x[:, h]) + D[h].to(f) * x[:, h] \
            + torch.exp(d).unsqueeze(-1) * torch.matmul(C[:, g], prev[:, :, h].to(f))
    return out.view(b, H, nc * Q, P)


def exact(case, seed):
    op = case["op"]
    t = _inputs(case, seed)
    f = torch.float64
    if op == "matmul":
        return torch.matmul(t[0].to(f), t[1].to(f))
    if op == "batch_matmul":
        return torch.stack([torch.matmul(a.to(f), b.to(f)) for a, b in zip(*t)])
    if op == "split_k":
        a, b = t[0].to(f), t[1].to(f)
        k = case["tile_k"]
        parts = torch.stack([torch.matmul(a[:, i:i + k], b[i:i + k])
                             for i in range(0, case["K"], k)])
        return parts.sum(0), parts
    if op == "attention":
        k, v, q = t
        scale = 1.0 / math.sqrt(case["D"])
        mask = torch.ones((case["Sq"], case["Skv"]), dtype=torch.bool, device=k.device).triu_(1) \
            if case["causal"] else None
        return torch.stack([_softmax_out(torch.matmul(q[i].to(f), k[i].to(f)) * scale, v[i].to(f),
                                         mask) for i in range(case["BH"])])
    if op == "decode":
        k, v, q = t
        scale = 1.0 / math.sqrt(case["D"])
        return torch.stack([_softmax_out(torch.matmul(q[i].to(f), k[i].to(f)) * scale,
                                         v[i].to(f)) for i in range(case["B"])])
    if op == "scan":
        cb, x, dt, dA, C, D, prev = t
        return _scan64(case, cb, x, dt, dA, C, D, prev)
    x, dt, A, B, C, D = t
    dA, cb, prev = _ssd_stages(case, x, dt, A, B, C, f)
    if op == "prologue":
        return dA, cb, prev
    y = _scan64(case, cb, x, dt.view(dA.shape), dA, C, D, prev)
    return y, dA, cb, prev
