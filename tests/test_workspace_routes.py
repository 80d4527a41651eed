"""The host side of the matmul calls without a GPU: which kernels a call launches and what it asks
of the allocator, when the workspace can grow, cannot (memory full) or must not (a capturing
stream). libkq4.so runs on a stand-in for the HIP runtime (tests/c/hip_standin.c): memory is
addresses nobody reads, a launch is a line in a log. Planned for a 256-CU MI355X. The outputs of
both forms of the prefill GEMM are compared on the GPU (test_gpu_matmul.py, test_gpu_graph.py)."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "kestrel-llm_amd")

PRELUDE = """
import ctypes, json, sys
sys.modules["torch"] = None       # its libraries would bind to the stand-in too
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
hip.standin_limit.argtypes = [ctypes.c_size_t]
hip.standin_used.restype = ctypes.c_size_t
hip.standin_log.restype = ctypes.c_char_p
sys.path.insert(0, sys.argv[2])
import kq4
k = kq4.lib()
assert k.kq4_init(0) == 0, kq4.last_error()
BASE = 1 << 40                    # "device" addresses, far apart; host ones are never read either

def at(i):
    return BASE + (i << 36)

def ptrs(n, first):
    return (ctypes.c_void_p * n)(*[at(first + i) for i in range(n)])

def call(form, n, rows, cols, chain=0):
    \"\"\"One device call of `form` over the matrices of `rows`: (return code, kernels, hipMallocs).\"\"\"
    hip.standin_clear()
    before, m = hip.standin_mallocs(), len(rows)
    r = (ctypes.c_int * m)(*rows)
    outs, ws, x = ptrs(m, 1), ptrs(m, 8), at(0)
    if form == "x":
        rc = k.kq4_matmul_multi_dev(m, outs, None, ws, r, cols, x, n, chain, None)
    elif form == "q":
        rc = k.kq4_matmul_multi_q_dev(m, outs, None, ws, r, cols, x, at(16), n, chain, None)
    elif form == "silu":
        rc = k.kq4_matmul_silu_dev(at(1), x, at(16), None, at(8), rows[0], cols, n, chain, None)
    elif form == "norm":
        rc = k.kq4_rmsnorm_matmul_multi_dev(m, outs, None, ws, r, cols, x, at(16), 1e-6, 1, None, n,
                                            chain, None)
    elif form == "q8":
        rc = k.kq4_q8_matmul_multi_dev(m, outs, None, ws, r, cols, x, n, chain, None)
    elif form == "noalloc":
        rc = k.kq4_matmul_noalloc_dev(at(1), x, None, at(8), rows[0], cols, n, chain, None)
    lines = hip.standin_log().decode().split("\\n")[:-1]
    return rc, [s.split(" ")[0] for s in lines], hip.standin_mallocs() - before

def records(kernels):
    return any("kq4_gemm_rec_kernel" in s for s in kernels)

def token_major(kernels):
    return any("kq4_gemm_kernel" in s for s in kernels)

def up(b):
    return (b + 255) // 256 * 256

def need(form, n, rows, cols):
    \"\"\"Workspace bytes of the token-major form: codes, scales and the partial sums of K splits.\"\"\"
    main = n if form == "q8" else n & ~3
    part = max((kq4.gemm_plan(n, r, cols, q8=form == "q8", ncu=256)[1] - 1) * main * r * 4
               for r in rows)
    return up(n * cols) + up(n * cols // 8) + up(part)

def reserve_exactly(b):           # growth takes a quarter more than asked
    b = (4 * b + 4) // 5
    assert k.kq4_workspace_reserve(b) == 0
"""


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("standin") / "hip_standin.so")
    r = subprocess.run(["gcc", "-std=gnu11", "-O1", "-Wall", "-Wextra", "-Werror", "-fPIC", "-shared",
                        "-I/opt/rocm/include", os.path.join(ROOT, "tests", "c", "hip_standin.c"),
                        "-o", so], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(body, **args):
        """`body` in a process of its own on the stand-in; returns what it leaves in `result`."""
        prog = PRELUDE + "".join(f"{n} = {v!r}\n" for n, v in args.items()) + body + \
            "\nprint('RESULT ' + json.dumps(result))\n"
        env = {n: v for n, v in os.environ.items() if not n.startswith("KQ4_")}
        p = subprocess.run([sys.executable, "-c", prog, so, PKG], capture_output=True, text=True,
                           env=env, timeout=120)
        assert p.returncode == 0, p.stdout + p.stderr
        line = [s for s in p.stdout.splitlines() if s.startswith("RESULT ")]
        return json.loads(line[-1][7:])
    return run


# calls the record form takes when the workspace holds the records, which need more than the token-major
# form: whole 64-token groups (520 tokens, 1000), and after the norm, beside the codes it wrote
REC_CALLS = [("x", 520, [12288], 4096), ("silu", 520, [4096], 12288),
             ("norm", 1024, [4096, 1024, 1024], 4096), ("q8", 1000, [12288], 4096),
             ("x", 200, [2048], 4096)]        # (the one test_gpu_graph.py captures)


@pytest.mark.parametrize("form,n,rows,cols", REC_CALLS)
def test_full_memory_takes_the_token_major_form(standin, form, n, rows, cols):
    """Memory that holds the token-major operands and not the records: the call runs token-major, as
    it does in a workspace that was large enough before. hipMalloc's refusal, which the runtime keeps
    as the thread's last error, is not taken for a failed launch."""
    res = standin("""
reserve_exactly(need(form, n, rows, cols))
hip.standin_limit(hip.standin_used())
full = call(form, n, rows, cols)
hip.standin_limit(1 << 40)
assert k.kq4_workspace_reserve(kq4.matmul_workspace_bytes(n, cols)) == 0
room = call(form, n, rows, cols)
result = [full[0], token_major(full[1]), records(full[1]), room[0], records(room[1])]
""", form=form, n=n, rows=rows, cols=cols)
    assert res[:3] == [0, True, False]        # done, token-major
    assert res[3:] == [0, True]               # the same call with room: records


def test_refused_allocation_does_not_fail_the_next_call(standin):
    """A call that fails for lack of memory says so, and the next call, whose workspace fits, runs."""
    res = standin("""
assert k.kq4_workspace_reserve(1 << 20) == 0
hip.standin_limit(hip.standin_used())
big = call("x", 4096, [4096], 12288)
small = call("x", 6, [4096], 4096, 0)
result = [big[0], big[1], small[0], len(small[1]) > 0]
""")
    assert res == [-3, [], 0, True]           # KQ4_ENOMEM with nothing launched; then done


def test_refused_weight_upload_does_not_fail_the_next_call(standin):
    """The same for the host-pointer calls' buffers: an upload without memory for its device copy, one
    without memory for the staging, then a device call that needs none."""
    res = standin("""
import numpy as np
w = np.zeros(1024 * 128 * 72, np.uint8)       # 4096 x 4096
assert k.kq4_workspace_reserve(1 << 20) == 0
room = hip.standin_used()
hip.standin_limit(room)
a = k.kq4_weights_upload(1 << 32, w.ctypes.data, 4096, 4096)      # no staging
b = call("x", 6, [4096], 4096)
hip.standin_limit(room + w.size + w.size // 4 + 4096)
c = k.kq4_weights_upload(1 << 32, w.ctypes.data, 4096, 4096)      # staging, no copy
d = call("x", 6, [4096], 4096)
hip.standin_limit(1 << 40)
e = k.kq4_weights_upload(1 << 32, w.ctypes.data, 4096, 4096)
result = [a, b[0], c, d[0], e]
""")
    assert res == [0, 0, 0, 0, 1]


@pytest.mark.parametrize("form,n,rows,cols", REC_CALLS)
def test_fallback_is_quiet(standin, form, n, rows, cols):
    """A call done token-major for want of workspace is no failure: it leaves the last failure's text
    alone, with memory full and on a capturing stream. Full memory is asked once: later calls leave
    the allocator alone until the workspace has grown or kq4_workspace_trim gave memory back."""
    res = standin("""
reserve_exactly(need(form, n, rows, cols))
call("x", -5, [64], 64)
text = kq4.last_error()
hip.standin_capture(1)
cap = call(form, n, rows, cols)
hip.standin_capture(0)
hip.standin_limit(hip.standin_used())
full = [call(form, n, rows, cols) for _ in range(3)]
same = kq4.last_error() == text
hip.standin_limit(1 << 40)
assert k.kq4_workspace_trim() == 0
room = call(form, n, rows, cols)
result = [same, "-5" in text, [cap[0], records(cap[1]), cap[2]],
          [[c[0], records(c[1]), c[2]] for c in full], [room[0], records(room[1]), room[2]]]
""", form=form, n=n, rows=rows, cols=cols)
    assert res == [True, True, [0, False, 0], [[0, False, 1], [0, False, 0], [0, False, 0]],
                   [0, True, 1]]


def test_noalloc_without_room_for_records_is_quiet(standin):
    """kq4_matmul_noalloc_dev's fixed scratch (64 MiB) holds 68 tokens x 464384 columns token-major, and
    not the records of their two 64-token groups with the K split's partial sums."""
    res = standin("""
call("x", -5, [64], 64)
text = kq4.last_error()
a = call("noalloc", 68, [128], 464384)
b = call("noalloc", 68, [128], 460000)       # those fit
result = [kq4.last_error() == text, a[0], records(a[1]), a[2], b[0], records(b[1]), b[2]]
""")
    assert res == [True, 0, False, 0, 0, True, 0]


# the largest batch an engine reserves for: every GEMV batch, the 16-token kernel, the prefill GEMM
@pytest.mark.parametrize("most", [1, 2, 3, 4, 5, 7, 8, 12, 16, 17, 68, 77, 300, 1000])
def test_reserved_workspace_holds_every_call_up_to_it(standin, most):
    """kq4_workspace_reserve(kq4_matmul_workspace_bytes(most, cols)), then calls of up to `most` tokens
    on a capturing stream: none needs more, and each takes the kernels it takes with all the workspace
    it may want. (The sizes are the largest K and, for the K splits' partial sums, few and many rows.)"""
    res = standin("""
cols = 4096
def calls():
    out = []
    for n in sorted({1, 2, 3, 4, 5, 6, 8, 9, 16, 17, 33, 67, 130, 1000, most - 1, most}):
        if n < 1 or n > most:
            continue
        for rows in ([12288, 12288], [4096, 1024, 1024], [256]):
            for form in ("x", "q", "silu", "norm", "q8"):
                for c in (cols, 2080):
                    out.append([form, n, rows, c, *call(form, n, rows[:1] if form == "silu" else rows, c)])
    return out
assert k.kq4_workspace_reserve(kq4.matmul_workspace_bytes(most, cols)) == 0
reserve_only = hip.standin_used()
hip.standin_capture(1)
got = calls()
hip.standin_capture(0)
assert k.kq4_workspace_reserve(1 << 32) == 0
want = calls()
result = [[g, w[4:]] for g, w in zip(got, want) if g[4:] != w[4:] or g[4] != 0]
""", most=most)
    assert res == []


# (form, tokens, rows, K) -> records: laying out codes that are already quantized (from the caller or the
# norm) costs time in proportion to tokens x K, which few rows do not earn back
@pytest.mark.parametrize("form,n,rows,cols,want", [
    ("q", 4096, [512], 12288, False), ("q", 2048, [1024], 12288, False),
    ("q", 4096, [1024, 512], 8192, False), ("norm", 4096, [512], 8192, False),
    ("norm", 1024, [4096], 4096, False), ("q", 2048, [2048], 8192, False),
    ("norm", 77, [4096, 1024, 1024], 4096, False),
    ("q", 2048, [12288], 4096, True), ("norm", 2048, [12288, 12288], 4096, True),
    ("norm", 2048, [4096, 1024, 1024], 4096, True), ("q", 4096, [4096], 4096, True),
    ("x", 4096, [512], 12288, True), ("silu", 2048, [1024], 12288, True)])
def test_record_layout_of_quantized_codes(standin, form, n, rows, cols, want):
    res = standin("""
assert k.kq4_workspace_reserve(1 << 32) == 0
a = call(form, n, rows, cols)
assert k.kq4_set_option(b"gemm_kind", 1) == 0
b = call(form, n, rows, cols)
result = [a[0], records(a[1]), token_major(a[1]), b[0], records(b[1])]
""", form=form, n=n, rows=rows, cols=cols)
    assert res == [0, want, not want, 0, True]


# (tokens, experts, columns) -> the tiled router logits: past one round of the few-token kernel's
# workgroups (512), past two where the columns are many
@pytest.mark.parametrize("T,ne,d,want", [
    (64, 128, 1024, False), (65, 128, 1024, True), (512, 16, 32, False), (513, 16, 32, True),
    (65, 128, 2048, False), (96, 128, 2048, False), (112, 128, 2048, False), (113, 128, 2048, True),
    (128, 128, 3072, False), (129, 128, 3072, True), (513, 8, 8192, False), (1024, 128, 2048, True)])
def test_router_logits_kernel(standin, T, ne, d, want):
    res = standin("""
rc = k.kq4_moe_router_logits_dev(at(0), at(1), at(2), T, ne, d, None)
result = [rc, hip.standin_log().decode()]
""", T=T, ne=ne, d=d)
    assert res[0] == 0 and res[1].count("\n") == 1
    assert ("logits_tiled_kernel" in res[1]) == want


def test_forced_forms_of_the_records(standin):
    """gemm_kind = 1 takes the record kernel for every ASM and Q8GEMM launch, at the forced tile where
    there is one (gemm_tile) and the form has it: 128 x 128, q4 also 64 x 128. A tile it does not have
    runs token-major, as do the other chains and gemm_kind = 0. The calls the GPU tests force
    through it run it."""
    from test_gpu_matmul import RECORD_EDGES
    res = standin("""
import re
assert k.kq4_workspace_reserve(1 << 32) == 0

def forced(form, n, rows, cols, chain, kind, tile, split=-1):
    for o, v in ((b"gemm_kind", kind), (b"gemm_tile", tile), (b"gemm_split", split)):
        assert k.kq4_set_option(o, v) == 0
    rc, names, _ = call(form, n, rows, cols, chain)
    assert rc == 0
    m = re.search(r"kq4_gemm_rec_kernelILi(\\d)ELi4ELi(\\d)", " ".join(names))
    return [64 * int(m[1]) // 2, int(m[2])] if m else None       # tokens of the tile, q8

result = dict(
    edges=[[forced("q8" if q8 else f, n, [rows], cols, 0, 1, 1 if q8 else tile, split)
            for f in (["x"] if q8 else ["x", "q"])]
           for n, rows, cols, tile, split in edges for q8 in (False, True)],
    tiles=[[forced(f, 300, [2000], 672, c, kind, tile) for tile in (0, 1, 2, 3, 4)]
           for f, c, kind in [("x", 3, 1), ("x", 0, 1), ("q8", 4, 1), ("x", 2, 1), ("x", 1, 1),
                              ("q8", 2, 1), ("x", 3, 0), ("q8", 4, 0)]],
    small=[forced("x", 24, [64], 256, 3, 1, 0), forced("q8", 24, [64], 256, 4, 1, 0),
           forced("x", 24, [64], 256, 3, -1, 0)],
    # a forced tile under the planner's choice of form, K split
    split4=forced("x", 512, [4096], 12288, 3, -1, 4, 4))
""", edges=RECORD_EDGES)
    want = []
    for n, rows, cols, tile, split in RECORD_EDGES:
        want += [[[64 if tile == 2 else 128, 0]] * 2, [[128, 1]]]
    assert res["edges"] == want
    q4 = [[128, 0], [64, 0], None, None]
    tm = [None] * 5
    assert res["tiles"][0][1:] == q4 and res["tiles"][1][1:] == q4
    assert res["tiles"][0][0] and res["tiles"][1][0]
    assert res["tiles"][2] == [[128, 1], [128, 1], None, None, None]
    assert res["tiles"][3:] == [tm] * 5
    assert res["small"] == [[64, 0], [128, 1], None] and res["split4"] is None


# (form, tokens, rows, K) -> tokens of the record kernel's tile, 0 = token-major: the shapes the rule's
# comment gives figures for (Qwen3-8B gate, QKV and down, Qwen3-VL-2B gate, Q8_0 gate) and its edges
RECORD_TILES = [
    ("x", 512, 12288, 4096, 64), ("x", 768, 12288, 4096, 128), ("x", 2048, 12288, 4096, 128),
    ("x", 2048, 6144, 4096, 128), ("x", 24, 6144, 4096, 0), ("x", 128, 6144, 2048, 0),
    ("silu", 96, 4096, 12288, 64), ("silu", 256, 4096, 12288, 64), ("silu", 512, 4096, 12288, 128),
    ("silu", 768, 4096, 12288, 64), ("q8", 512, 12288, 4096, 0), ("q8", 768, 12288, 4096, 128),
    ("q8", 1000, 12288, 4096, 128), ("q8", 2048, 12288, 4096, 128), ("x", 64, 12288, 4096, 0)]


@pytest.mark.parametrize("form,n,rows,cols,tile", RECORD_TILES)
def test_record_rule(standin, form, n, rows, cols, tile):
    res = standin("""
import re
assert k.kq4_workspace_reserve(1 << 32) == 0
rc, names, _ = call(form, n, [rows], cols)
m = re.search(r"kq4_gemm_rec_kernelILi(\\d)", " ".join(names))
result = [rc, 32 * int(m[1]) if m else 0, token_major(names)]
""", form=form, n=n, rows=rows, cols=cols)
    assert res == [0, tile, tile == 0]
