"""Performance cases of kq4: the q4 / Q8_0 matmul family as an inference engine calls it.

A case is one of six kinds of call, each through the public binding (kestrel-llm_amd/kq4.py):

  step     one decode step of `layers` decoder layers (and the lm_head): per layer the fused QKV,
           O + residual, fused gate/up and down + residual, captured once as a HIP graph and
           replayed per token, as a decode loop runs it. `fused` = the layer's RMSNorms and SiLU
           go through the fused entry points, as an engine that keeps everything in HBM does
  mat      one eager matmul call of `n` tokens over one to three matrices that share the activation
           (O, QKV, gate/up, down), with or without residual, SiLU product or RMSNorm
  q8       the same over Q8_0 weights, the prefill format of dual VQF files and the q8 mode
  moe      a whole MoE FFN layer: router logits, top-k, expert FFN, combine
  host     the host-pointer drop-in call: numpy activations in and out, weights cached on the GPU

Model shapes are those of Qwen3-VL-2B, Qwen3-8B and Qwen3-30B-A3B (synth.py) or generic. Weights
have uniform 4-bit (int8) codes with |N(0, sigma)| f16 block scales; activations are N(0, 1) with a
few outlier channels, as hidden states have.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("kestrel-llm_amd"))
import kq4  # noqa: E402

EPS = 1e-6
SIGMA = 0.02
DEV = "cuda"


def listed():
    return [
        # one token of Qwen3-VL-2B: all 28 layers' linear set and the lm_head, the headline loop
        dict(name="decode_2b_m1", kind="step", hidden=2048, heads=16, kv=8, ffn=6144, layers=28,
             vocab=151936, n=1, fused=False),
        # continuous batching, 8 sequences of a Qwen3-8B: norms and SiLU fused (8 layers, so that
        # the weights stream from HBM)
        dict(name="decode_8b_m8", kind="step", hidden=4096, heads=32, kv=8, ffn=12288, layers=8,
             vocab=0, n=8, fused=True),
        # the smallest call, eager: the 2B O projection of one token with its residual
        dict(name="o_proj_2b_m1", kind="mat", cols=2048, rows="2048", n=1, res=True, pre="none"),
        # a wide decode batch or a speculative draft: 13 tokens of the 8B gate/up pair
        dict(name="gate_up_8b_m13", kind="mat", cols=4096, rows="12288,12288", n=13, res=False,
             pre="none"),
        # a short prompt of odd length: 8B norm + QKV (an ASM main segment and a one-token tail)
        dict(name="qkv_8b_m77", kind="mat", cols=4096, rows="4096,1024,1024", n=77, res=False,
             pre="norm"),
        # a prefill chunk of 512 tokens: 8B SiLU + down + residual, the longest K
        dict(name="down_8b_m512", kind="mat", cols=12288, rows="4096", n=512, res=True,
             pre="silu"),
        # a full prefill chunk: 8B gate/up, the largest call of the engine
        dict(name="gate_up_8b_m2048", kind="mat", cols=4096, rows="12288,12288", n=2048, res=False,
             pre="none"),
        # Q8_0 prefill, the 8B gate over a ragged 1000-token chunk
        dict(name="q8_gate_8b_m1000", kind="q8", cols=4096, rows="12288", n=1000, res=False),
        # one decode token of a Qwen3-30B-A3B MoE layer
        dict(name="moe_30b_t1", kind="moe", d=2048, ef=768, experts=128, tk=8, n=1),
        # a decode batch through the same layer: every expert active, few tokens each
        dict(name="moe_30b_t64", kind="moe", d=2048, ef=768, experts=128, tk=8, n=64),
        # a prefill chunk through the same layer: about 64 tokens an expert
        dict(name="moe_30b_t1024", kind="moe", d=2048, ef=768, experts=128, tk=8, n=1024),
        # the drop-in op as the C engine calls it: host pointers, 2B gate/up of one token
        dict(name="host_gate_up_2b_m1", kind="host", cols=2048, rows="6144,6144", n=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same kinds: sizes log-uniform over the listed range, odd ones among
    them (rows any multiple of 4 or 8, K any multiple of 32, any token count)."""
    kind = rng.choice(["step", "mat", "mat", "mat", "mat", "q8", "q8", "moe", "moe", "host"])
    if kind == "step":
        heads = rng.choice([8, 12, 16, 24, 32])
        kv = rng.choice([k for k in (2, 4, 8) if heads % k == 0])
        hidden = 128 * heads if rng.random() < 0.7 else 32 * _log_int(rng, 32, 128)
        return dict(kind="step", hidden=hidden, heads=heads, kv=kv,
                    ffn=32 * _log_int(rng, 64, 384), layers=rng.randint(2, 8),
                    vocab=4 * _log_int(rng, 4000, 38000) if rng.random() < 0.4 else 0,
                    n=rng.randint(1, 16), fused=rng.random() < 0.5)
    if kind == "moe":
        tk = rng.choice([2, 4, 8])
        return dict(kind="moe", d=32 * _log_int(rng, 16, 96), ef=32 * _log_int(rng, 8, 40),
                    experts=rng.choice([16, 32, 60, 64, 128]), tk=tk, n=_log_int(rng, 1, 1024))
    cols = 32 * _log_int(rng, 32, 384)
    if kind == "host":
        rows = [4 * _log_int(rng, 64, 3072) for _ in range(rng.randint(1, 2))]
        return dict(kind="host", cols=cols, rows=",".join(map(str, rows)),
                    n=_log_int(rng, 1, 64))
    n = _log_int(rng, 1, 2048)
    g = 8 if kind == "q8" else 4
    nm = rng.randint(1, 3) if kind == "mat" else rng.randint(1, 2)
    rows = [g * _log_int(rng, 512 // g, 12288 // g) for _ in range(nm)]
    cap = 2 * 12288 * 4096 * 2048
    while cols * n * sum(rows) > cap:
        n = max(1, n * 3 // 4)
    c = dict(kind=kind, cols=cols, rows=",".join(map(str, rows)), n=n, res=rng.random() < 0.5)
    if kind == "mat":
        c["pre"] = rng.choice(["none", "none", "norm", "silu"])
        if c["pre"] == "silu":
            c["rows"] = str(rows[0])
    return c


# ---- inputs --------------------------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + salt * 7919 + 17) & 0x7FFFFFFF)
    return g


def _acts(n, cols, seed, salt):
    """N(0, 1) activations, one channel in 200 six times as large."""
    g = _gen(seed, salt)
    gain = 1.0 + 5.0 * (torch.rand(cols, device=DEV, generator=g) < 0.005).float()
    return torch.randn(n, cols, device=DEV, generator=g) * gain


def _q4(rows, cols, seed, salt):
    """VQF 4x4 tiles, uint8 [rows/4, cols/32, 72]: 4 f16 row scales, then 64 code bytes."""
    g = _gen(seed, salt)
    t = torch.empty(rows // 4, cols // 32, 72, dtype=torch.uint8, device=DEV)
    sc = (torch.randn(rows // 4, cols // 32, 4, device=DEV, generator=g).abs() * SIGMA + 1e-4)
    t[:, :, :8] = sc.half().view(torch.uint8).reshape(rows // 4, cols // 32, 8)
    t[:, :, 8:] = torch.randint(0, 256, (rows // 4, cols // 32, 64), dtype=torch.uint8, device=DEV,
                                generator=g)
    return t


def _q4_f64(t):
    """The weights of 4x4 tiles in 64 bits, [rows, cols] (codes are stored XOR 8)."""
    G, nb, _ = t.shape
    sc = t[:, :, :8].contiguous().view(torch.float16).reshape(G, nb, 4).double()
    qs = t[:, :, 8:].reshape(G, nb, 4, 4, 4)                       # [G][b][k][r][i]
    lo, hi = (qs & 15) ^ 8, (qs >> 4) ^ 8
    half = [h.permute(0, 3, 1, 2, 4).reshape(G, 4, nb, 16) for h in (lo, hi)]
    w = torch.cat(half, 3).double() - 8.0                          # [G][r][b][32]
    return (w * sc.permute(0, 2, 1).unsqueeze(3)).reshape(4 * G, nb * 32)


def _q8(rows, cols, seed, salt):
    """Q8_0 tiles of 8 rows, uint8 [rows/8, cols/32, 272]: 8 f16 row scales, then the codes."""
    g = _gen(seed, salt)
    t = torch.empty(rows // 8, cols // 32, 272, dtype=torch.uint8, device=DEV)
    sc = torch.randn(rows // 8, cols // 32, 8, device=DEV, generator=g).abs() * (SIGMA / 16) + 1e-5
    t[:, :, :16] = sc.half().view(torch.uint8).reshape(rows // 8, cols // 32, 16)
    t[:, :, 16:] = torch.randint(-127, 128, (rows // 8, cols // 32, 256), dtype=torch.int8,
                                 device=DEV, generator=g).view(torch.uint8)
    return t


def _q8_f64(t):
    G, nb, _ = t.shape
    sc = t[:, :, :16].contiguous().view(torch.float16).reshape(G, nb, 8).double()
    qs = t[:, :, 16:].contiguous().view(torch.int8).reshape(G, nb, 8, 8, 4)   # [G][b][k][m][i]
    w = qs.permute(0, 3, 1, 2, 4).reshape(G, 8, nb, 32).double()
    return (w * sc.permute(0, 2, 1).unsqueeze(3)).reshape(8 * G, nb * 32)


def _rows(case):
    return [int(r) for r in case["rows"].split(",")]


def _out(*shape):
    return torch.empty(shape, dtype=torch.float32, device=DEV)


def _step_shapes(c):
    """(weights' name, rows) and K of one layer's four launches."""
    q, kv, h, f = 128 * c["heads"], 128 * c["kv"], c["hidden"], c["ffn"]
    return [("qkv", [q, kv, kv], h), ("o", [h], q), ("gu", [f, f], h), ("down", [h], f)]


def _step_weights(c, seed):
    """The tiles of every layer's matrices, made one at a time: (layer, launch, matrix, tiles)."""
    for layer in range(c["layers"]):
        for k, (_, rows, cols) in enumerate(_step_shapes(c)):
            for m, r in enumerate(rows):
                yield layer, k, m, _q4(r, cols, seed, 100 + 16 * layer + 4 * k + m)
    if c["vocab"]:
        yield c["layers"], 0, 0, _q4(c["vocab"], c["hidden"], seed, 99)


def _step_inputs(c, seed):
    n, h, f = c["n"], c["hidden"], c["ffn"]
    return dict(x=_acts(n, h, seed, 1), attn=_acts(n, 128 * c["heads"], seed, 2),
                gate=_acts(n, f, seed, 3), up=_acts(n, f, seed, 4), res=_acts(n, h, seed, 5),
                norm=1.0 + 0.1 * torch.randn(h, device=DEV, generator=_gen(seed, 6)))


def _prepare_step(c, seed):
    n, L, shapes = c["n"], c["layers"], _step_shapes(c)
    w = {}
    for layer, k, m, t in _step_weights(c, seed):
        rows, cols = 4 * t.shape[0], 32 * t.shape[1]
        w[layer, k, m] = kq4.prepare_dev(t.reshape(-1), rows, cols)
    s = _step_inputs(c, seed)
    # [matrix][layer][token][row], one output tensor per matrix of the layer
    s["out"] = {name: [_out(L, n, r) for r in rows] for name, rows, _ in shapes}
    s["logits"] = _out(n, c["vocab"]) if c["vocab"] else None
    s["w"] = w

    def launches():
        st = torch.cuda.current_stream()
        for layer in range(L):
            for k, (name, rows, cols) in enumerate(shapes):
                ws = [w[layer, k, m] for m in range(len(rows))]
                outs = [o[layer] for o in s["out"][name]]
                if name in ("qkv", "gu") and c["fused"]:
                    kq4.rmsnorm_matmul_multi_dev(outs, s["x"], s["norm"], EPS, ws, rows, cols,
                                                 stream=st)
                elif name in ("qkv", "gu"):
                    kq4.matmul_multi_dev(outs, s["x"], ws, rows, cols, stream=st)
                elif name == "o":
                    kq4.matmul_dev(outs[0], s["attn"], ws[0], rows[0], cols, residual=s["res"],
                                   stream=st)
                elif c["fused"]:
                    kq4.matmul_silu_dev(outs[0], s["gate"], s["up"], ws[0], rows[0], cols,
                                        residual=s["res"], stream=st)
                else:
                    kq4.matmul_dev(outs[0], s["gate"], ws[0], rows[0], cols, residual=s["res"],
                                   stream=st)
        if c["vocab"]:
            kq4.matmul_dev(s["logits"], s["x"], w[L, 0, 0], c["vocab"], c["hidden"], stream=st)

    kq4.workspace_reserve(max(kq4.matmul_workspace_bytes(n, cols) for _, _, cols in shapes))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launches()
    s["graph"] = graph
    return s


def prepare(case, seed):
    kq4.init(0)
    kind, n = case["kind"], case["n"]
    s = dict(case=case)
    if kind == "step":
        s.update(_prepare_step(case, seed))
    elif kind == "moe":
        d, ef, ne = case["d"], case["ef"], case["experts"]
        for i, (name, rows, cols) in enumerate([("G", ne * ef, d), ("U", ne * ef, d),
                                                ("D", d, ne * ef)]):
            s[name] = kq4.prepare_dev(_q4(rows, cols, seed, 10 + i).reshape(-1), rows, cols)
        s["x"] = _acts(n, d, seed, 1)
        s["router"] = torch.randn(ne, d, device=DEV, generator=_gen(seed, 2)) / math.sqrt(d)
        s["y"] = _out(n, d)
        s["sel"] = torch.empty(n, case["tk"], dtype=torch.int32, device=DEV)
        s["pr"] = _out(n, case["tk"])
    elif kind == "host":
        rows, cols = _rows(case), case["cols"]
        s["rows"] = rows
        s["w"] = [_q4(r, cols, seed, 10 + i).reshape(-1).cpu().numpy() for i, r in enumerate(rows)]
        # the engine's key is layer << 32 | projection; a layer of its own per set of inputs
        s["keys"] = [((seed & 0x3FFFFFFF) + 1 << 32) | (4 + i) for i in range(len(rows))]
        for k, w, r in zip(s["keys"], s["w"], rows):
            kq4.check_done(kq4.lib().kq4_weights_upload(k, w.ctypes.data, r, cols), "upload")
        s["x"] = _acts(n, cols, seed, 1).cpu().numpy()
    else:
        rows, cols = _rows(case), case["cols"]
        s["rows"] = rows
        if kind == "q8":
            s["w"] = [kq4.q8_prepare_dev(_q8(r, cols, seed, 10 + i).reshape(-1), r, cols)
                      for i, r in enumerate(rows)]
        else:
            s["w"] = [kq4.prepare_dev(_q4(r, cols, seed, 10 + i).reshape(-1), r, cols)
                      for i, r in enumerate(rows)]
        s["x"] = _acts(n, cols, seed, 1)
        s["out"] = [_out(n, r) for r in rows]
        s["res"] = [_acts(n, r, seed, 30 + i) for i, r in enumerate(rows)] if case["res"] else None
        if case.get("pre") == "silu":
            s["up"] = _acts(n, cols, seed, 2)
        if case.get("pre") == "norm":
            s["norm"] = 1.0 + 0.1 * torch.randn(cols, device=DEV, generator=_gen(seed, 3))
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "step":
        s["graph"].replay()
        out = dict(s["out"])
        if s["logits"] is not None:
            out["logits"] = s["logits"]
        return out
    if kind == "host":
        return kq4.matmul_multi(s["w"], s["rows"], s["x"], c["cols"], wkeys=s["keys"])
    st = torch.cuda.current_stream()
    if kind == "moe":
        kq4.moe_layer_dev(s["y"], s["x"], s["router"], s["G"], s["U"], s["D"], c["experts"],
                          c["tk"], c["d"], c["ef"], sel=s["sel"], pr=s["pr"], stream=st)
        return dict(y=s["y"], sel=s["sel"], pr=s["pr"])
    out, x, w, rows, cols, res = s["out"], s["x"], s["w"], s["rows"], c["cols"], s["res"]
    if kind == "q8":
        if len(rows) == 1:
            kq4.q8_matmul_dev(out[0], x, w[0], rows[0], cols, residual=res and res[0], stream=st)
        else:
            kq4.q8_matmul_multi_dev(out, x, w, rows, cols, residuals=res, stream=st)
    elif c["pre"] == "silu":
        kq4.matmul_silu_dev(out[0], x, s["up"], w[0], rows[0], cols, residual=res and res[0],
                            stream=st)
    elif c["pre"] == "norm":
        kq4.rmsnorm_matmul_multi_dev(out, x, s["norm"], EPS, w, rows, cols, residuals=res,
                                     order=kq4.RMS_SERIAL if c["n"] > 1 else kq4.RMS_CHUNKED,
                                     stream=st)
    elif len(rows) == 1:
        kq4.matmul_dev(out[0], x, w[0], rows[0], cols, residual=res and res[0], stream=st)
    else:
        kq4.matmul_multi_dev(out, x, w, rows, cols, residuals=res, stream=st)
    return out


# ---- what a pass cannot do without ---------------------------------------------------------------

def _mat_work(rows, cols, n, per_weight=18 / 32, res=False, xs=1):
    N = sum(rows)
    return (N * cols * per_weight + 4 * n * cols * xs + 4 * n * N * (2 if res else 1),
            2 * n * N * cols)


def work(case):
    kind, n = case["kind"], case["n"]
    b = f = 0.0
    if kind == "step":
        for name, rows, cols in _step_shapes(case):
            x, y = _mat_work(rows, cols, n, res=name in ("o", "down"),
                             xs=2 if name == "down" and case["fused"] else 1)
            b, f = b + x * case["layers"], f + y * case["layers"]
        if case["vocab"]:
            x, y = _mat_work([case["vocab"]], case["hidden"], n)
            b, f = b + x, f + y
    elif kind == "moe":
        d, ef, ne, tk = case["d"], case["ef"], case["experts"], case["tk"]
        active = ne * (1.0 - (1.0 - tk / ne) ** n)   # experts that some token selects
        b = active * 3 * d * ef * 18 / 32 + 4 * ne * d + 8 * n * d + 8 * n * tk
        f = 2 * n * tk * 3 * d * ef + 2 * n * ne * d
    else:
        xs = 2 if case.get("pre") == "silu" else 1
        b, f = _mat_work(_rows(case), case["cols"], n, 34 / 32 if kind == "q8" else 18 / 32,
                         case.get("res", False), xs)
    return dict(bytes=b, flops=f)


def tolerance(case):
    # fp32 sums of K/32 block terms, in another order; the quantized codes are the same bits. Two
    # orders each up to 3e-7 of the norm from the 64-bit sums (K = 12288) differ by up to 5e-7.
    # MoE: expert ids may differ at router ties.
    return dict(rel=2e-6, max=2e-5, differ=1e-4 if case["kind"] == "moe" else 0.0)


# ---- the same in 64 bits -------------------------------------------------------------------------

def _quant(x, f16_tokens):
    """The activation the op multiplies: int8 codes per 32-block (fp32 division, + 0.5, truncated,
    clamped) times the block scale, f16-rounded for the first f16_tokens tokens; in 64 bits."""
    n, cols = x.shape
    v = x.reshape(n, cols // 32, 32)
    d = v.abs().amax(2, keepdim=True).clamp_min(1e-10) / torch.tensor(127.0, device=x.device)
    q = torch.trunc(v / d + 0.5).clamp(-127, 127).double()
    s = d.double()
    s[:f16_tokens] = d[:f16_tokens].half().double()
    return (q * s).reshape(n, cols)


def _asm(n):
    return (n & ~3) if n > 3 else 0


def _norm(x, w):
    y = x.double()
    rms = 1.0 / torch.sqrt((y * y).mean(1, keepdim=True) + EPS)
    return ((x * rms.float()) * w)   # the normalised input is fp32, as the op hands it on


def _silu(g, u):
    return (g.double() * torch.sigmoid(g.double()) * u.double()).float()


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "step":
        s = _step_inputs(case, seed)
        f16 = _asm(n)
        x = _quant(_norm(s["x"], s["norm"]) if case["fused"] else s["x"], f16)
        ff = _quant(_silu(s["gate"], s["up"]) if case["fused"] else s["gate"], f16)
        inp, res = [x, _quant(s["attn"], f16), x, ff], s["res"].double()
        shapes = _step_shapes(case)
        out = {name: [torch.empty(case["layers"], n, r, dtype=torch.float64, device=DEV)
                      for r in rows] for name, rows, _ in shapes}
        for layer, k, m, t in _step_weights(case, seed):
            if layer == case["layers"]:
                lx = _quant(s["x"], f16)
                out["logits"] = torch.cat([lx @ _q4_f64(p).T for p in t.split(4096)], 1)
                continue
            y = inp[k] @ _q4_f64(t).T
            out[shapes[k][0]][m][layer] = y + res if shapes[k][0] in ("o", "down") else y
        return out
    if kind == "moe":
        return _exact_moe(case, seed)
    rows, cols = _rows(case), case["cols"]
    x = _acts(n, cols, seed, 1)
    if case.get("pre") == "silu":
        x = _silu(x, _acts(n, cols, seed, 2))
    if case.get("pre") == "norm":
        x = _norm(x, 1.0 + 0.1 * torch.randn(cols, device=DEV, generator=_gen(seed, 3)))
    # Q8_0: the f16-rounded scale for every token from two on
    a = _quant(x, (n if n >= 2 else 0) if kind == "q8" else _asm(n))
    out = []
    for i, r in enumerate(rows):
        w = _q8_f64(_q8(r, cols, seed, 10 + i)) if kind == "q8" else _q4_f64(_q4(r, cols, seed,
                                                                                 10 + i))
        y = a @ w.T
        out.append(y + _acts(n, r, seed, 30 + i).double() if case.get("res") else y)
    return [o.cpu().numpy() for o in out] if kind == "host" else out


def _exact_moe(case, seed):
    n, d, ef, ne, tk = case["n"], case["d"], case["ef"], case["experts"], case["tk"]
    x = _acts(n, d, seed, 1)
    router = torch.randn(ne, d, device=DEV, generator=_gen(seed, 2)) / math.sqrt(d)
    logits = x.double() @ router.double().T
    top, sel = torch.sort(logits, dim=1, descending=True, stable=True)
    top, sel = top[:, :tk], sel[:, :tk]
    p = torch.softmax(top, 1)
    a = _quant(x, 0)
    G, U, D = (_q4(r, c, seed, 10 + i) for i, (r, c) in enumerate([(ne * ef, d), (ne * ef, d),
                                                                   (d, ne * ef)]))
    y = torch.zeros(n, d, dtype=torch.float64, device=DEV)
    for e in range(ne):
        tok, rank = torch.nonzero(sel == e, as_tuple=True)
        if not len(tok):
            continue
        g = a[tok] @ _q4_f64(G[e * ef // 4:(e + 1) * ef // 4]).T
        u = a[tok] @ _q4_f64(U[e * ef // 4:(e + 1) * ef // 4]).T
        av = _quant((g * torch.sigmoid(g) * u).float(), 0)
        down = av @ _q4_f64(D[:, e * ef // 32:(e + 1) * ef // 32]).T
        y.index_add_(0, tok, down * p[tok, rank].unsqueeze(1))
    return dict(y=y, sel=sel.to(torch.int32), pr=p)
