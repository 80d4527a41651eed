"""GPU parity of the dense op (quantizer, integer block sums, decode GEMV, prefill GEMM) against
the oracle, through the C ABI.

Bars: activation codes/scales and integer block sums bit-exact; prefill GEMM outputs bit-exact
(it replays the reference chain per output); decode GEMV outputs within
max|got-ref| / max|ref| <= 1e-5 (split-K summation order; the reference's metric,
vllm_safetensors.c:1177-1181), max-abs reported."""
import numpy as np
import pytest

import synth
from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-5


def to_dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def wdev(kq4, torch, w, rows, cols):
    """Device weights as the device API takes them: the stream-layout copy of the VQF tiles."""
    return kq4.prepare_dev(to_dev(torch, w), rows, cols)


def host(t):
    return t.cpu().numpy()


def case(rows, cols, n, seed, sigma=0.02, floor=1e-4):
    w = synth.make_q4_weights(rows, cols, seed, sigma, floor)
    x = synth.make_activations(n, cols, seed + 1)
    return w, x


def test_quantize_bit_exact(kq4, torch_dev, orc):
    torch = torch_dev
    rng = np.random.default_rng(0)
    x = rng.standard_normal((7, 512)).astype(np.float32)
    x[0, :32] = 0
    x[1, :32] *= 1e-30
    x[2, 32:64] = 127.0
    x[2, 40] = -127.0
    x[3, :32] = 1e-41                                   # subnormal inputs
    x[4] *= 1e4
    x[5, 64:96] = np.float32(0.49999997)
    xq_o, xd_o = orc.quantize(x, 512)
    X = to_dev(torch, x)
    xq = torch.empty((7, 512), dtype=torch.int8, device="cuda")
    xd = torch.empty((7, 16), dtype=torch.float32, device="cuda")
    xde = torch.empty_like(xd)
    kq4.quantize_dev(X, xq, xd, xde, chain=kq4.CHAIN_ASM)
    torch.cuda.synchronize()
    assert np.array_equal(host(xq), xq_o)
    assert np.array_equal(host(xd).view(np.uint32), xd_o.view(np.uint32))
    assert np.array_equal(host(xde), xd_o.astype(np.float16).astype(np.float32))


@pytest.mark.parametrize("rows,cols,n", [(8, 64, 1), (20, 160, 3), (64, 2048, 5)])
def test_block_sums_exact(kq4, torch_dev, orc, rows, cols, n):
    torch = torch_dev
    w, x = case(rows, cols, n, 10 + n)
    xq, xd = orc.quantize(x, cols)
    lo_o, hi_o = orc.block_sums(w, xq, rows, cols)
    lo = torch.empty((n, rows, cols // 32), dtype=torch.int32, device="cuda")
    hi = torch.empty_like(lo)
    kq4.block_sums_dev(lo, hi, to_dev(torch, xq), wdev(kq4, torch, w, rows, cols), rows, cols, n)
    torch.cuda.synchronize()
    assert np.array_equal(host(lo), lo_o) and np.array_equal(host(hi), hi_o)


# Workgroup modes: up to 64 row sets (2048 rows) quarter sets, (6144, 2048) half sets, (88000,
# 2048) full sets with two waves for four stages; (256, 12288) and (64, 24576) have more 16-block
# stages than waves (2 and 4 per wave).
GEMV_SHAPES = [(16, 256), (20, 160), (4, 32), (100, 2080), (132, 4096), (256, 12288),
               (64, 24576), (6144, 2048), (2048, 6144), (88000, 2048)]


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("rows,cols", GEMV_SHAPES)
def test_gemv(kq4, torch_dev, orc, rows, cols, n):
    torch = torch_dev
    w, x = case(rows, cols, n, rows + cols + n)
    want = orc.matmul(w, x, rows, cols)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    kq4.matmul_dev(out, to_dev(torch, x), wdev(kq4, torch, w, rows, cols), rows, cols)
    torch.cuda.synchronize()
    r, a = rel_err(host(out), want)
    print(f"gemv rows={rows} cols={cols} n={n}: rel={r:.3e} maxabs={a:.3e}")
    assert r <= TOL


@pytest.mark.parametrize("chain", [1, 2, 3])
def test_gemv_chains_and_residual(kq4, torch_dev, orc, chain):
    torch = torch_dev
    rows, cols, n = 96, 1024, 6
    w, x = case(rows, cols, n, 77, sigma=0.015, floor=0.0)
    res = np.random.default_rng(5).standard_normal((n, rows)).astype(np.float32)
    want = orc.matmul(w, x, rows, cols, residual=res, chain=chain)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    kq4.matmul_dev(out, to_dev(torch, x), wdev(kq4, torch, w, rows, cols), rows, cols,
                   residual=to_dev(torch, res), chain=chain)
    torch.cuda.synchronize()
    r, a = rel_err(host(out), want)
    assert r <= TOL, (r, a)


def test_gemv_multi_qkv(kq4, torch_dev, orc):
    torch = torch_dev
    cols, n = 2048, 4
    rows = [2048, 1024, 1024]
    ws = [synth.make_q4_weights(r, cols, 200 + i) for i, r in enumerate(rows)]
    x = synth.make_activations(n, cols, 300)
    outs = [torch.empty((n, r), dtype=torch.float32, device="cuda") for r in rows]
    kq4.matmul_multi_dev(outs, to_dev(torch, x),
                         [wdev(kq4, torch, w, r, cols) for w, r in zip(ws, rows)], rows, cols)
    torch.cuda.synchronize()
    for o, w, r in zip(outs, ws, rows):
        rr, _ = rel_err(host(o), orc.matmul(w, x, r, cols))
        assert rr <= TOL


@pytest.mark.parametrize("n", [12, 64, 130, 257])
@pytest.mark.parametrize("chain", [0, 1, 2, 3])
def test_gemm_bit_exact(kq4, torch_dev, orc, n, chain):
    torch = torch_dev
    rows, cols = 260, 512
    w, x = case(rows, cols, n, 400 + n)
    res = np.random.default_rng(n).standard_normal((n, rows)).astype(np.float32)
    want = orc.matmul(w, x, rows, cols, residual=res, chain=chain)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    with kq4.options(gemv_chunk_max=8):   # 12 tokens on the GEMM, not two GEMV launches
        kq4.matmul_dev(out, to_dev(torch, x), wdev(kq4, torch, w, rows, cols), rows, cols,
                       residual=to_dev(torch, res), chain=chain)
    torch.cuda.synchronize()
    got = host(out)
    main = (n & ~3) if chain == 0 else n
    exact = np.array_equal(got[:main].view(np.uint32), want[:main].view(np.uint32))
    r, a = rel_err(got, want)
    print(f"gemm n={n} chain={chain}: main bit-exact={exact} rel={r:.3e} maxabs={a:.3e}")
    assert exact
    assert r <= TOL


# The tile planner takes 128x128 tiles from 2 per CU (n = 2048, 4096 rows: 512 tiles), 64x128
# below that (2048 rows; and n = 1152 at K = 8192: 288 tiles of 128x128, one round of 576
# 64x128 tiles); the C-tile chain is capped at 64x128. K = 640 (20 blocks) runs five
# 4-block stages with the next stage's registers prefetched, over two stream-layout stages (the
# second one partial). The oracle is evaluated on sampled outputs: one per 64 x 64 cell (every
# tile, every XCD's range), the last token and row, and random pairs.
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("n,rows,chain,cols", [(2048, 4096, 0, 640), (2048, 4096, 1, 640),
                                               (2048, 4096, 3, 640), (2048, 2048, 2, 640),
                                               (2048, 2048, 3, 640), (300, 2048, 0, 640),
                                               (300, 2000, 0, 672), (1000, 4000, 3, 672),
                                               (1152, 4096, 3, 8192)])
def test_gemm_large_tiles_bit_exact(kq4, torch_dev, orc, n, rows, chain, cols, kind):
    """Both GEMM forms (planner option gemm_kind: 0 token-major activations, 1 activation records) are
    bit-identical to the oracle, also with an odd block count (K = 672: the last 4-block and 2-block
    stages run past K) and a partial last row set."""
    if kind == 1 and chain in (1, 2):
        pytest.skip("this chain has no record form: kind 0 is the same launch")
    torch = torch_dev
    w, x = case(rows, cols, n, 700 + rows + chain)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    with kq4.options(gemm_kind=kind):
        kq4.matmul_dev(out, to_dev(torch, x), wdev(kq4, torch, w, rows, cols), rows, cols,
                       chain=chain)
    torch.cuda.synchronize()
    got = host(out)
    xq, xd = orc.quantize(x, cols)
    rng = np.random.default_rng(rows + chain)
    t0, r0 = np.meshgrid(np.arange(0, n, 64), np.arange(0, rows, 64), indexing="ij")
    tok = np.concatenate([np.minimum(t0.ravel() + rng.integers(0, 64, t0.size), n - 1),
                          [n - 1] * 64, rng.integers(0, n, 2048)]).astype(np.int32)
    row = np.concatenate([np.minimum(r0.ravel() + rng.integers(0, 64, r0.size), rows - 1),
                          rng.integers(0, rows, 64), rng.integers(0, rows, 2048)]).astype(np.int32)
    want = orc.matmul_q_sample(w, xq, xd, rows, cols, n, tok, row, chain=chain)
    assert np.array_equal(got[tok, row].view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("tile", [1, 2, 3, 4])
@pytest.mark.parametrize("chain", [0, 1, 2, 3])
def test_gemm_tile_forms_bit_exact(kq4, torch_dev, orc, tile, chain, kind):
    """Every tile form forced through the planner option gemm_tile (128x128, 64x128, 64x64,
    128x64 tokens x rows; the C-tile chain is capped at 64x128), in both GEMM forms (gemm_kind
    0 token-major activations, 1 activation records, which have the first two tiles), is bit-identical
    to the oracle, with an odd block count (K = 672) and a partial last row set and token tile."""
    if kind == 1 and (chain in (1, 2) or tile > 2):
        pytest.skip("no record form: kind 0 is the same launch")
    torch = torch_dev
    n, rows, cols = 300, 2000, 672
    w, x = case(rows, cols, n, 900 + 10 * tile + chain)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    with kq4.options(gemm_tile=tile, gemm_kind=kind):
        kq4.matmul_dev(out, to_dev(torch, x), wdev(kq4, torch, w, rows, cols), rows, cols,
                       chain=chain)
    torch.cuda.synchronize()
    got = host(out)
    xq, xd = orc.quantize(x, cols)
    rng = np.random.default_rng(tile + chain)
    t0, r0 = np.meshgrid(np.arange(0, n, 32), np.arange(0, rows, 32), indexing="ij")
    tok = np.concatenate([np.minimum(t0.ravel() + rng.integers(0, 32, t0.size), n - 1),
                          [n - 1] * 64, rng.integers(0, n, 1024)]).astype(np.int32)
    row = np.concatenate([np.minimum(r0.ravel() + rng.integers(0, 32, r0.size), rows - 1),
                          rng.integers(0, rows, 64), rng.integers(0, rows, 1024)]).astype(np.int32)
    want = orc.matmul_q_sample(w, xq, xd, rows, cols, n, tok, row, chain=chain)
    assert np.array_equal(got[tok, row].view(np.uint32), want.view(np.uint32))


# (tokens, rows, K, tile of q4 - Q8_0 has the 128 x 128 one only -, K slices); that these run the record
# kernel is checked without a GPU (test_workspace_routes.py)
RECORD_EDGES = [(17, 4, 32, 2, 1), (64, 36, 64, 2, 1), (65, 132, 96, 1, 1), (127, 260, 480, 1, 1),
                (129, 128, 544, 2, 1), (200, 100, 1056, 2, 1), (300, 264, 2080, 1, 2),
                (190, 392, 2592, 2, 4)]


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("n,rows,cols,tile,split", RECORD_EDGES)
def test_gemm_records_match_token_major(kq4, torch_dev, q8, n, rows, cols, tile, split):
    """The record form of the prefill GEMM (gemm_kind = 1) gives the token-major form's bits at the
    edges of its token groups, row sets, stages (odd block counts: a stage past K) and K slices, with
    a tail, a residual and, for q4, activations already quantized."""
    torch = torch_dev
    x = to_dev(torch, synth.make_activations(n, cols, n + cols))
    res = to_dev(torch, synth.make_activations(n, rows, n + 1))
    if q8:
        w = kq4.q8_prepare_dev(synth.make_q8_weights(rows, cols, rows, g=4), rows, cols, g=4)
    else:
        w = wdev(kq4, torch, synth.make_q4_weights(rows, cols, rows), rows, cols)
        xq = torch.empty((n, cols), dtype=torch.int8, device="cuda")
        xd = torch.empty((n, cols // 32), dtype=torch.float32, device="cuda")
        kq4.quantize_dev(x, xq, xd)
    outs = []
    for kind in (0, 1):
        with kq4.options(gemm_kind=kind, gemm_tile=1 if q8 else tile, gemm_split=split):
            o = torch.full((n, rows), float("nan"), dtype=torch.float32, device="cuda")
            (kq4.q8_matmul_dev if q8 else kq4.matmul_dev)(o, x, w, rows, cols, residual=res)
            outs.append(host(o))
            if not q8:
                kq4.matmul_q_dev(o, xq, xd, w, rows, cols, n, residual=res)
                outs.append(host(o))
    torch.cuda.synchronize()
    for o in outs[1:]:
        assert np.array_equal(o.view(np.uint32), outs[0].view(np.uint32))


# Powers of ten for the activations (a token each) and the weight scales (a row each): f16 block scales
# of every kind - normal, subnormal, the smallest, zero; for the activations also past the largest f16
# (1e8: infinite, as the chain's rounding makes them) and an all-zero block's 1e-10 / 127.
TOKEN_GAINS = [1.0, 1e-3, 1e-4, 1e-5, 3e-7, 1e-9, 0.0, 1e4, 1e6, 1e8]
ROW_SCALES = [0.02, 1e-4, 3e-5, 1e-6, 6e-8, 0.0, 1.0, 3e4, -0.02, -3e-6]


def same_bits(a, b):
    """Bit equality, any NaN taken for any other."""
    return np.array_equal(np.where(np.isnan(a), 0, a.view(np.uint32)),
                          np.where(np.isnan(b), 0, b.view(np.uint32))) and \
        np.array_equal(np.isnan(a), np.isnan(b))


@pytest.mark.parametrize("q8,tile", [(False, 1), (False, 2), (True, 1)])
def test_gemm_records_scale_range(kq4, torch_dev, orc, q8, tile):
    """The record form over the f16 range of both scales, each output's terms of one magnitude (a
    token's blocks share a gain, a row's a scale) and, on the tokens past the gains, of mixed ones:
    the oracle's bits and the token-major form's. The matrix unit forms wd * f16r(xd) there, so this
    needs it to take subnormal f16 operands as they are."""
    torch = torch_dev
    n, rows, cols, g = 132, 136, 544, 4
    nb = cols // 32
    rng = np.random.default_rng(17 + tile)
    gain = np.array([TOKEN_GAINS[i % len(TOKEN_GAINS)] for i in range(n)], np.float32)[:, None]
    gain = np.repeat(gain, nb, 1)
    gain[100:] = rng.choice(TOKEN_GAINS[:9], (n - 100, nb))
    x = synth.make_activations(n, cols, 18).reshape(n, nb, 32) * gain[:, :, None]
    x = np.ascontiguousarray(x.reshape(n, cols), np.float32)
    w = synth.make_q8_weights(rows, cols, 19, g=g) if q8 else synth.make_q4_weights(rows, cols, 19)
    sc = np.array([ROW_SCALES[r % len(ROW_SCALES)] for r in range(rows)], np.float32)
    sc = np.repeat(sc.reshape(rows // g, 1, g), nb, 1) * rng.uniform(0.5, 1.0, (rows // g, nb, g))
    w[:, :, :2 * g] = sc.astype(np.float16).view(np.uint8).reshape(rows // g, nb, 2 * g)
    res = synth.make_activations(n, rows, 20)
    if q8:
        want = orc.q8_matmul(w, x, rows, cols, residual=res, chain=kq4.CHAIN_Q8GEMM, g=g)
        W = kq4.q8_prepare_dev(w, rows, cols, g=g)
    else:
        want = orc.matmul(w, x, rows, cols, residual=res, chain=kq4.CHAIN_ASM)
        W = wdev(kq4, torch, w, rows, cols)
    assert np.isfinite(want[gain.max(1) < 1e7]).all() and not np.isfinite(want).all()
    got = []
    for kind in (0, 1):
        o = torch.full((n, rows), float("nan"), dtype=torch.float32, device="cuda")
        with kq4.options(gemm_kind=kind, gemm_tile=tile, gemm_split=1):
            (kq4.q8_matmul_dev if q8 else kq4.matmul_dev)(
                o, to_dev(torch, x), W, rows, cols, residual=to_dev(torch, res),
                chain=kq4.CHAIN_Q8GEMM if q8 else kq4.CHAIN_ASM)
        got.append(host(o))
    bad = [[t for t in range(n) if not same_bits(o[t], want[t])] for o in got]
    assert bad == [[], []], "tokens off the oracle: token-major, records"


@pytest.mark.parametrize("form", ["matmul", "silu", "multi"])
def test_gemm_records_auto_tail(kq4, torch_dev, orc, form):
    """The record form (gemm_kind = 1) with an AUTO-chain tail: 301 tokens are 300 in records (the asm
    chain, bit-exact) and one C-tile token whose codes the same quantizer launch leaves token-major,
    behind the records in the workspace, for the GEMV (within 1e-5), for the plain, SiLU and
    several-matrix calls."""
    torch = torch_dev
    n, cols = 301, 1024
    rows = [512, 256] if form == "multi" else [512]
    ws = [synth.make_q4_weights(r, cols, 950 + i) for i, r in enumerate(rows)]
    x = synth.make_activations(n, cols, 960)
    up = synth.make_activations(n, cols, 961)
    res = [synth.make_activations(n, r, 970 + i) for i, r in enumerate(rows)]
    outs = [torch.empty((n, r), dtype=torch.float32, device="cuda") for r in rows]
    W = [wdev(kq4, torch, w, r, cols) for w, r in zip(ws, rows)]
    with kq4.options(gemm_kind=1):
        if form == "matmul":
            kq4.matmul_dev(outs[0], to_dev(torch, x), W[0], rows[0], cols,
                           residual=to_dev(torch, res[0]))
        elif form == "silu":
            kq4.matmul_silu_dev(outs[0], to_dev(torch, x), to_dev(torch, up), W[0], rows[0],
                                cols, residual=to_dev(torch, res[0]))
        else:
            kq4.matmul_multi_dev(outs, to_dev(torch, x), W, rows, cols,
                                 residuals=[to_dev(torch, r) for r in res])
    torch.cuda.synchronize()
    for o, w, r, rr in zip(outs, ws, rows, res):
        if form == "silu":
            want = orc.matmul_silu(w, x, up, r, cols, residual=rr)
        else:
            want = orc.matmul(w, x, r, cols, residual=rr)
        got = host(o)
        assert np.array_equal(got[:300].view(np.uint32), want[:300].view(np.uint32)), form
        e, a = rel_err(got[300:], want[300:])
        print(f"record tail {form} rows={r}: tail rel={e:.3e} maxabs={a:.3e}")
        assert e <= TOL


@pytest.mark.parametrize("split", [2, 3, 4, 8])
@pytest.mark.parametrize("chain", [0, 1, 2, 3])
def test_gemm_split_k(kq4, torch_dev, orc, chain, split):
    """Split K forced through the planner option gemm_split: K = 4096 (128 blocks) in 2 slices of
    64 blocks, 3 of 48 (the last one 32), 4 of 32 or 8 of 16, each slice its own chain from zero, added in
    slice order with the residual last. Every output within 1e-5 of the oracle's single chain
    (the split is not bit-identical to it), repeat calls bit-identical, for
    every chain, a 301-token batch (AUTO: a 1-token C-tile tail on the GEMV) and two matrices of
    different heights in one call."""
    torch = torch_dev
    n, cols = 301, 4096
    rows = [384, 136]
    ws = [synth.make_q4_weights(r, cols, 1000 + r + chain) for r in rows]
    x = synth.make_activations(n, cols, 1010 + split)
    res = [synth.make_activations(n, r, 1020 + i) for i, r in enumerate(rows)]
    W = [wdev(kq4, torch, w, r, cols) for w, r in zip(ws, rows)]
    X = to_dev(torch, x)
    R = [to_dev(torch, r) for r in res]
    outs = [torch.empty((n, r), dtype=torch.float32, device="cuda") for r in rows]
    again = [torch.empty_like(o) for o in outs]
    with kq4.options(gemm_split=split):
        kq4.matmul_multi_dev(outs, X, W, rows, cols, residuals=R, chain=chain)
        kq4.matmul_multi_dev(again, X, W, rows, cols, residuals=R, chain=chain)
    torch.cuda.synchronize()
    for o, a2, w, r, rr in zip(outs, again, ws, rows, res):
        got = host(o)
        assert np.array_equal(got.view(np.uint32), host(a2).view(np.uint32))
        want = orc.matmul(w, x, r, cols, residual=rr, chain=chain)
        e, a = rel_err(got, want)
        same = (got.view(np.uint32) == want.view(np.uint32)).mean()
        print(f"split={split} chain={chain} rows={r}: rel={e:.3e} maxabs={a:.3e} "
              f"bit-identical {same:.3f}")
        assert e <= TOL


# The planner's K splits over 64-token tiles (small token counts, K >= 128 blocks: 64 x 64 tiles
# for one token tile, 64 x 128 beyond, up to 8 slices of >= 32 blocks), and the same forms
# forced: sampled outputs (every 64 x 64 cell, the last token and row, random pairs) within 1e-5
# of the oracle's single chain, repeat calls bit-identical.
@pytest.mark.parametrize("form", ["planner", (2, 8), (3, 4), (2, 3)])
@pytest.mark.parametrize("n,rows,cols,chain", [(24, 1024, 12288, 0), (64, 2048, 6144, 3),
                                               (100, 4096, 4096, 2), (200, 1000, 8192, 0),
                                               (33, 640, 4096, 3)])
def test_gemm_small_batch_splits(kq4, torch_dev, orc, n, rows, cols, chain, form):
    torch = torch_dev
    w, x = case(rows, cols, n, 1100 + n + rows)
    res = synth.make_activations(n, rows, 1101 + n)
    W, X, R = wdev(kq4, torch, w, rows, cols), to_dev(torch, x), to_dev(torch, res)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    again = torch.empty_like(out)
    opts = {} if form == "planner" else dict(gemm_tile=form[0], gemm_split=form[1])
    with kq4.options(**opts):
        kq4.matmul_dev(out, X, W, rows, cols, residual=R, chain=chain)
        kq4.matmul_dev(again, X, W, rows, cols, residual=R, chain=chain)
    torch.cuda.synchronize()
    got = host(out)
    assert np.array_equal(got.view(np.uint32), host(again).view(np.uint32))
    xq, xd = orc.quantize(x, cols)
    rng = np.random.default_rng(n + rows)
    t0, r0 = np.meshgrid(np.arange(0, n, 64), np.arange(0, rows, 64), indexing="ij")
    tok = np.concatenate([np.minimum(t0.ravel() + rng.integers(0, 64, t0.size), n - 1),
                          [n - 1] * 64, rng.integers(0, n, 2048)]).astype(np.int32)
    row = np.concatenate([np.minimum(r0.ravel() + rng.integers(0, 64, r0.size), rows - 1),
                          rng.integers(0, rows, 64), rng.integers(0, rows, 2048)]).astype(np.int32)
    want = orc.matmul_q_sample(w, xq, xd, rows, cols, n, tok, row, residual=res, chain=chain)
    e = np.abs(got[tok, row].astype(np.float64) - want).max() / np.abs(want).max()
    print(f"small-batch split {form} n={n} rows={rows} cols={cols} chain={chain}: rel={e:.3e}")
    assert e <= TOL


@pytest.mark.parametrize("tile", [1, 2])
@pytest.mark.parametrize("split", [1, 2])
def test_gemm_prio_same_outputs(kq4, torch_dev, orc, split, tile):
    """The pipelined GEMM's issue priority by progress through K (planner option gemm_prio: 0
    off, 1 on, -1 the planner's choice), on the 128 x 128 and 64 x 128 forms, only reorders the
    SIMDs' issue between workgroups: the outputs of the three settings are bit-identical, on a
    small launch (128 x 128: the planner leaves it off; checked against the oracle, bit for bit
    unsplit, within 1e-5 in 2 K slices) and on a whole round of workgroups."""
    torch = torch_dev
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    cases = [(301, 384, 4096, True), (256, 128 * ncu, 2048, False)]
    for n, rows, cols, check in cases:
        w = synth.make_q4_weights(rows, cols, 1040 + rows)
        x = synth.make_activations(n, cols, 1041)
        W, X = wdev(kq4, torch, w, rows, cols), to_dev(torch, x)
        got = {}
        for prio in (0, 1, -1):
            out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
            with kq4.options(gemm_prio=prio, gemm_split=split, gemm_tile=tile):
                kq4.matmul_dev(out, X, W, rows, cols, chain=kq4.CHAIN_ASM)
            torch.cuda.synchronize()
            got[prio] = host(out)
        for prio in (1, -1):
            assert np.array_equal(got[prio].view(np.uint32), got[0].view(np.uint32)), (n, rows, prio)
        if check:
            want = orc.matmul(w, x, rows, cols, chain=kq4.CHAIN_ASM)
            e, a = rel_err(got[1], want)
            print(f"prio tile={tile} split={split} n={n} rows={rows}: rel={e:.3e} maxabs={a:.3e}")
            if split == 1:
                assert np.array_equal(got[1].view(np.uint32), want.view(np.uint32))
            assert e <= TOL


def test_q8_gemm_prio_same_outputs(kq4, torch_dev, orc):
    """The progress priority on the q8 GEMM (Q8_0 weights, the unfused GEMM chain): every
    gemm_prio setting gives the same bits, on a whole round of two workgroups per CU (the planner
    turns it on) and on a small launch checked against the oracle."""
    torch = torch_dev
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    for n, rows, cols, check in [(96, 256, 2048, True), (256, 128 * ncu, 1024, False)]:
        tiles = synth.make_q8_weights(rows, cols, 1050 + rows)
        x = synth.make_activations(n, cols, 1051)
        W = kq4.q8_prepare_dev(tiles, rows, cols)
        X = to_dev(torch, x)
        got = {}
        for prio in (0, 1, -1):
            out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
            with kq4.options(gemm_prio=prio, gemm_tile=1):
                kq4.q8_matmul_dev(out, X, W, rows, cols)
            torch.cuda.synchronize()
            got[prio] = host(out)
        for prio in (1, -1):
            assert np.array_equal(got[prio].view(np.uint32), got[0].view(np.uint32)), (n, rows, prio)
        if check:
            want = orc.q8_matmul(tiles, x, rows, cols)
            assert np.array_equal(got[1].view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("split", [1, 4])
def test_q8_gemm_split_k(kq4, torch_dev, orc, split):
    """Q8_0 weights (8-block stages): K = 4096 in 4 slices of 32 blocks, within 1e-5 of the
    oracle's GEMM chain; unsplit, bit-identical."""
    torch = torch_dev
    n, rows, cols = 96, 256, 4096
    tiles = synth.make_q8_weights(rows, cols, 1030)
    x = synth.make_activations(n, cols, 1031)
    W = kq4.q8_prepare_dev(tiles, rows, cols)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    with kq4.options(gemm_split=split):
        kq4.q8_matmul_dev(out, to_dev(torch, x), W, rows, cols)
    torch.cuda.synchronize()
    got = host(out)
    want = orc.q8_matmul(tiles, x, rows, cols)
    e, a = rel_err(got, want)
    print(f"q8 split={split}: rel={e:.3e} maxabs={a:.3e}")
    if split == 1:
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert e <= TOL


# 9-16 tokens: q4 batches in one launch of the decode GEMV's 16-token kernel (the tokens past n
# padding), for every chain, several matrices with residuals, fp32 and pre-quantized
# activations: within 1e-5 of the oracle (whose AUTO chain puts the first n & ~3 tokens on the
# ASM scale rounding, as the reference's whole-batch dispatch does), the pre-quantized call bit
# for bit the fp32 one, and repeat launches bit-identical.
@pytest.mark.parametrize("n", [9, 12, 13, 16])
@pytest.mark.parametrize("chain", [0, 1, 2, 3])
def test_gemv_wide(kq4, torch_dev, orc, n, chain):
    torch = torch_dev
    rows, cols = [256, 100], 2080
    ws = [synth.make_q4_weights(r, cols, 1400 + r + n) for r in rows]
    x = synth.make_activations(n, cols, 1410 + n + chain)
    res = [synth.make_activations(n, r, 1420 + i) for i, r in enumerate(rows)]
    W = [wdev(kq4, torch, w, r, cols) for w, r in zip(ws, rows)]
    X, R = to_dev(torch, x), [to_dev(torch, r) for r in res]
    assert kq4.gemm_plan(n, rows[0], cols, chain=chain) == (0, 0)   # on the GEMV
    outs = [torch.full((n + 1, r), 7.0, dtype=torch.float32, device="cuda") for r in rows]
    kq4.matmul_multi_dev([o[:n] for o in outs], X, W, rows, cols, residuals=R, chain=chain)
    again = [torch.empty((n, r), dtype=torch.float32, device="cuda") for r in rows]
    kq4.matmul_multi_dev(again, X, W, rows, cols, residuals=R, chain=chain)
    xq, xd = orc.quantize(x, cols)
    outq = torch.empty((n, rows[0]), dtype=torch.float32, device="cuda")
    kq4.matmul_q_dev(outq, to_dev(torch, xq), to_dev(torch, xd), W[0], rows[0], cols, n,
                     residual=R[0], chain=chain)
    torch.cuda.synchronize()
    for o, p, w, r, rr in zip(outs, again, ws, rows, res):
        got = host(o)
        assert np.all(got[n] == 7.0)   # nothing stored past the n tokens
        got = got[:n]
        assert np.array_equal(got.view(np.uint32), host(p).view(np.uint32))
        e, a = rel_err(got, orc.matmul(w, x, r, cols, residual=rr, chain=chain))
        print(f"gemv wide n={n} chain={chain} rows={r}: rel={e:.3e} maxabs={a:.3e}")
        assert e <= TOL
    assert np.array_equal(host(outq).view(np.uint32), host(outs[0][:n]).view(np.uint32))


# The 16-token kernel's launch shapes through the planner options: 2 or 3 whole sets per
# workgroup (the last group short), half sets, fewer waves than stages, with the activations
# quantized in the kernel or apart.
@pytest.mark.parametrize("plan", [dict(gemv_hs=0, gemv_rps=2), dict(gemv_hs=0, gemv_rps=3),
                                  dict(gemv_hs=0, gemv_rps=3, gemv_fq=0, gemv_waves=2),
                                  dict(gemv_hs=1, gemv_waves=3), dict(gemv_hs=0, gemv_rps=1)])
@pytest.mark.parametrize("n", [11, 16])
def test_gemv_wide_plans(kq4, torch_dev, orc, n, plan):
    torch = torch_dev
    rows, cols = [256, 100], 2080
    ws = [synth.make_q4_weights(r, cols, 1500 + r + n) for r in rows]
    x = synth.make_activations(n, cols, 1510 + n)
    res = [synth.make_activations(n, r, 1520 + i) for i, r in enumerate(rows)]
    W = [wdev(kq4, torch, w, r, cols) for w, r in zip(ws, rows)]
    X, R = to_dev(torch, x), [to_dev(torch, r) for r in res]
    outs = [torch.empty((n, r), dtype=torch.float32, device="cuda") for r in rows]
    with kq4.options(**plan):
        kq4.matmul_multi_dev(outs, X, W, rows, cols, residuals=R)
    torch.cuda.synchronize()
    for o, w, r, rr in zip(outs, ws, rows, res):
        e, a = rel_err(host(o), orc.matmul(w, x, r, cols, residual=rr))
        print(f"gemv wide plan {plan} n={n} rows={r}: rel={e:.3e} maxabs={a:.3e}")
        assert e <= TOL


def test_gemm_from_prequantized(kq4, torch_dev, orc):
    torch = torch_dev
    rows, cols, n = 128, 1024, 40
    w, x = case(rows, cols, n, 501)
    xq, xd = orc.quantize(x, cols)
    want = orc.matmul_q(w, xq, xd, rows, cols)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    kq4.matmul_q_dev(out, to_dev(torch, xq), to_dev(torch, xd), wdev(kq4, torch, w, rows, cols),
                     rows, cols, n)
    torch.cuda.synchronize()
    assert np.array_equal(host(out), want)


# Launch shapes of the GEMV set through the planner options (include/kq4.h kq4_set_option):
# whole sets grouped 2 or 3 per workgroup (the last group short), half / quarter sets, wave
# counts that leave a wave with fewer stages than the others, with the activations quantized in
# the kernel or apart, with a residual.
# The last three: waves taking 3 of the 6 stages, all 6, and a mix of 2 and 1 (pre-quantized).
GEMV_PLANS = [dict(gemv_hs=0, gemv_rps=2), dict(gemv_hs=0, gemv_rps=3),
              dict(gemv_hs=0, gemv_rps=3, gemv_waves=2), dict(gemv_hs=1, gemv_waves=3),
              dict(gemv_hs=2, gemv_waves=5), dict(gemv_hs=0, gemv_rps=2, gemv_fq=0),
              dict(gemv_hs=1, gemv_waves=2), dict(gemv_hs=2, gemv_waves=1),
              dict(gemv_hs=0, gemv_waves=4, gemv_fq=0)]


@pytest.mark.parametrize("n", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("plan", range(len(GEMV_PLANS)))
def test_gemv_plans(kq4, torch_dev, orc, plan, n):
    torch = torch_dev
    rows, cols = 32 * 7 + 4, 32 * 16 * 5 + 64            # 8 row sets (last short), 6 stages
    w, x = case(rows, cols, n, 1000 + plan + n)
    res = np.random.default_rng(plan).standard_normal((n, rows)).astype(np.float32)
    want = orc.matmul(w, x, rows, cols, residual=res)
    wd = wdev(kq4, torch, w, rows, cols)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    again = torch.empty_like(out)
    with kq4.options(**GEMV_PLANS[plan]):
        kq4.matmul_dev(out, to_dev(torch, x), wd, rows, cols, residual=to_dev(torch, res))
        kq4.matmul_dev(again, to_dev(torch, x), wd, rows, cols, residual=to_dev(torch, res))
    torch.cuda.synchronize()
    got = host(out)
    r, a = rel_err(got, want)
    print(f"plan {GEMV_PLANS[plan]} n={n}: rel={r:.3e} maxabs={a:.3e}")
    assert r <= TOL
    assert np.array_equal(got.view(np.uint32), host(again).view(np.uint32))   # deterministic


@pytest.mark.parametrize("plan", range(len(GEMV_PLANS)))
def test_gemv_plans_multi_matrix(kq4, torch_dev, orc, plan):
    """Three matrices in one launch (fused QKV): groups of each matrix stay within it."""
    torch = torch_dev
    cols, n = 2048, 4
    rows = [2048 + 96, 1024 + 32, 1024 + 32]
    ws = [synth.make_q4_weights(r, cols, 1200 + i) for i, r in enumerate(rows)]
    x = synth.make_activations(n, cols, 1300 + plan)
    outs = [torch.empty((n, r), dtype=torch.float32, device="cuda") for r in rows]
    with kq4.options(**GEMV_PLANS[plan]):
        kq4.matmul_multi_dev(outs, to_dev(torch, x),
                             [wdev(kq4, torch, w, r, cols) for w, r in zip(ws, rows)], rows, cols)
    torch.cuda.synchronize()
    for o, w, r in zip(outs, ws, rows):
        rr, _ = rel_err(host(o), orc.matmul(w, x, r, cols))
        assert rr <= TOL


# Seeded random shapes across the dense op's whole surface: rows a multiple of 4 (partial row
# sets and tiles), K a multiple of 32 from one block up (partial stream stages), 1-300 tokens
# (the decode GEMV up to 16, in launches of 8 beyond 8, the prefill GEMM beyond, with the AUTO
# chain's C-tile tail), every chain, with and without a residual. Below K = 2048 the planner
# never splits K, so there the GEMM's main segment is checked bit for bit; every output within
# 1e-5.
RANDOM_CASES = 32


@pytest.mark.parametrize("i", range(RANDOM_CASES))
def test_random_shapes(kq4, torch_dev, orc, i):
    torch = torch_dev
    rng = np.random.default_rng(7000 + i)
    rows = 4 * int(rng.integers(1, 257))
    cols = 32 * int(rng.integers(1, 97))
    n = int(rng.integers(1, 9)) if i % 2 == 0 else int(rng.integers(9, 301))
    chain = int(rng.integers(0, 4))
    w, x = case(rows, cols, n, 7100 + i)
    res = rng.standard_normal((n, rows)).astype(np.float32) if i % 3 else None
    want = orc.matmul(w, x, rows, cols, residual=res, chain=chain)
    out = torch.empty((n, rows), dtype=torch.float32, device="cuda")
    kq4.matmul_dev(out, to_dev(torch, x), wdev(kq4, torch, w, rows, cols), rows, cols,
                   residual=None if res is None else to_dev(torch, res), chain=chain)
    torch.cuda.synchronize()
    got = host(out)
    r, a = rel_err(got, want)
    exact = None
    if n > kq4.get_option("gemv_chunk_max") and cols < 2048:   # on the GEMM, K unsplit
        main = (n & ~3) if chain == 0 else n
        exact = np.array_equal(got[:main].view(np.uint32), want[:main].view(np.uint32))
    print(f"random case {i}: rows={rows} cols={cols} n={n} chain={chain} "
          f"residual={res is not None}: rel={r:.3e} maxabs={a:.3e} main bit-exact={exact}")
    assert exact is not False
    assert r <= TOL
