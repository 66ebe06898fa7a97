"""The prefill GEMM's tile shapes: cases for each, at their edges (one row, one
token, a tile's rows and tokens +- 1, K shares with and without a block) and
over several rounds of their buffers, rows past 32-bit offsets, pointers of
the smallest alignment, and recording into a graph.

Bounds as for the other GEMM tests: f16 weights (three roundings of 2^-11
each) keep the Frobenius error below 1e-3 and each element within
1e-2 sum|w||a| / sqrt(K)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from modgrad_amd import _lib
from tests.gpu_util import dev, empty_f32, host, ptr, random_q4k_bytes

pytestmark = pytest.mark.gpu

def note(msg: str) -> None:
    print(f"[case] {msg}", flush=True)


@pytest.fixture(scope="module")
def L():
    return _lib.load()


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def check(L, orc, n, bpr, m, woff=0, aoff=0, coff=0):
    rng = np.random.default_rng(n + 17 * bpr + 1009 * m + woff)
    w = random_q4k_bytes(rng, n * bpr)
    a = rng.standard_normal((m, bpr * 256)).astype(np.float16)
    wt = dev(np.concatenate([np.zeros(woff, np.uint8), w]))
    at = dev(np.concatenate([np.zeros(aoff, np.uint8), a.view(np.uint8).ravel()]))
    ct = empty_f32(m * n + coff // 4)
    _lib.check("gemm", L.launch_gemm_q4k_f16(ptr(wt) + woff, ptr(at) + aoff, ptr(ct) + coff, n, bpr,
                                             m, None))
    rows = None
    if n > 600:
        rows = np.unique(np.concatenate([rng.choice(n, size=160, replace=False),
                                         np.arange(48), np.arange(n - 48, n)])).astype(np.int32)
    C = host(ct)[coff // 4:].reshape(m, n)
    assert np.all(np.isfinite(C))
    C = C if rows is None else C[:, rows]
    C_ref, A = orc.gemm_f16(w, a.view(np.uint16), n, bpr, rows=rows)
    assert np.all(np.abs(C - C_ref) <= 1e-2 * A / np.sqrt(bpr * 256))
    assert np.linalg.norm(C - C_ref) <= 1e-3 * np.linalg.norm(C_ref)


# rows, tokens and K shares of a tile -> the cases that take it on 256 CUs
# (asserted by tests/test_gemm_tile_pick.py): at its edges, and last one of
# 4 to 17 blocks whose token buffers, register sets and scale tables all come
# round again in every K share, the shares unequal
CASES = {
    (32, 16, 4): [(1, 1, 1), (17, 3, 16), (33, 5, 15), (1000, 6, 17), (33, 29, 15)],
    (32, 32, 4): [(1000, 1, 129), (4001, 9, 33), (806, 13, 149)],
    (32, 48, 4): [(8003, 5, 33), (1032, 13, 225)],
    (64, 48, 2): [(2001, 1, 129), (16001, 1, 1), (4001, 3, 129), (1168, 11, 291)],
    (64, 80, 2): [(8003, 2, 97), (16001, 3, 49), (1852, 11, 388)],
    (128, 48, 2): [(20479, 2, 1), (16001, 3, 81), (30001, 2, 47), (30001, 3, 47), (60001, 2, 1),
                   (3344, 7, 325)],
    (128, 64, 2): [(30001, 1, 49), (16001, 3, 97), (3238, 7, 436)],
    (128, 80, 2): [(16001, 2, 129), (30001, 1, 79), (4695, 7, 389)],
    (160, 48, 1): [(20479, 1, 17), (6660, 7, 269)],
    (160, 48, 2): [(37888, 26, 33), (5458, 17, 321)],
    (160, 80, 2): [(20479, 2, 127), (20479, 3, 97), (5387, 7, 416)],
    (224, 128, 1): [(56001, 4, 100), (7001, 4, 1021), (13156, 4, 489)],
    (336, 80, 1): [(85007, 3, 79), (42001, 1, 5), (42001, 3, 127), (6301, 4, 489)],
    (336, 128, 1): [(30001, 1, 161), (85007, 2, 81), (60001, 3, 127), (14360, 5, 416)],
}


@pytest.mark.parametrize("n,bpr,m", [c for cases in CASES.values() for c in cases])
def test_gemm_tile_shapes(L, orc, n, bpr, m):
    note(f"gemm tiles n={n} bpr={bpr} m={m}")
    check(L, orc, n, bpr, m)


def test_gemm_rows_past_32_bit_offsets(L):
    # 2^27 values a row: offsets inside a tile pass 32 bits (64-bit ones then).
    # The weights of the last 64 blocks of every row are the only nonzero ones,
    # so the reference is that of a 64-block product.
    import torch
    n, bpr, m, tail = 3, 524288, 2, 64
    note(f"gemm n={n} bpr={bpr} m={m}")
    rng = np.random.default_rng(27)
    w = torch.zeros((n, bpr, 144), dtype=torch.uint8, device="cuda")
    wt = random_q4k_bytes(rng, n * tail)
    w[:, -tail:] = dev(wt).view(n, tail, 144)
    a = torch.ones((m, bpr * 256), dtype=torch.float16, device="cuda")
    at = rng.standard_normal((m, tail * 256)).astype(np.float16)
    a[:, -tail * 256:] = torch.from_numpy(at).cuda()
    ct = empty_f32(m * n)
    _lib.check("gemm", L.launch_gemm_q4k_f16(ptr(w), ptr(a), ptr(ct), n, bpr, m, None))
    got = host(ct).reshape(m, n)
    ws, as_, small = dev(wt), dev(at.view(np.uint16)), empty_f32(m * n)
    _lib.check("gemm", L.launch_gemm_q4k_f16(ptr(ws), ptr(as_), ptr(small), n, tail, m, None))
    # the same weights, rounded the same (a row's exponent starts at its first
    # nonzero block): only the order of the f32 sums differs, by K shares
    want = host(small).reshape(m, n)
    assert np.all(np.isfinite(got)) and np.linalg.norm(want) > 0
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)


# weights at an odd byte, activations at an odd f16, C at a 4-byte address:
# the token copies then go through registers
@pytest.mark.parametrize("n,bpr,m", [(100, 3, 33), (2001, 5, 129), (30001, 3, 161)])
@pytest.mark.parametrize("woff,aoff,coff", [(1, 0, 0), (0, 2, 4), (3, 10, 8)])
def test_gemm_unaligned_pointers(L, orc, n, bpr, m, woff, aoff, coff):
    note(f"gemm n={n} bpr={bpr} m={m} offsets {woff} {aoff} {coff}")
    check(L, orc, n, bpr, m, woff, aoff, coff)


# ... over several rounds of the buffers that those registers go to
@pytest.mark.parametrize("tile", CASES)
def test_gemm_unaligned_activations(L, orc, tile):
    n, bpr, m = CASES[tile][-1]
    note(f"gemm tile {tile} n={n} bpr={bpr} m={m}, A at +2")
    check(L, orc, n, bpr, m, 0, 2, 0)


CAPTURE = """
import ctypes, sys, torch
sys.path.insert(0, sys.argv[1])
from modgrad_amd import _lib
L = _lib.load()
gen = torch.Generator(device="cuda"); gen.manual_seed(5)
jobs = []
for n, bpr, m in ((1000, 6, 17), (8003, 2, 97), (30001, 1, 161)):
    w = torch.randint(0, 256, (n * bpr, 144), dtype=torch.uint8, device="cuda", generator=gen)
    w[:, :4] = torch.full((n * bpr, 2), 1e-3, device="cuda").half().view(torch.uint8)
    a = torch.randn(m, bpr * 256, device="cuda", generator=gen).half()
    jobs.append((w, a, torch.zeros(m, n, device="cuda"), n, bpr, m))
torch.cuda.synchronize()
def run(stream):
    for w, a, c, n, bpr, m in jobs:
        assert L.launch_gemm_q4k_f16(w.data_ptr(), a.data_ptr(), c.data_ptr(), n, bpr, m,
                                     ctypes.c_void_p(stream)) == 0
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g):  # the library's first call in this process
    run(torch.cuda.current_stream().cuda_stream)
for i in range(4):
    for j in jobs:
        j[1].copy_(torch.randn(j[1].shape, device="cuda", generator=gen).half())
        j[2].fill_(float("nan"))
    g.replay()
    torch.cuda.synchronize()
    got = [j[2].clone() for j in jobs]
    run(0)
    torch.cuda.synchronize()
    assert all(torch.equal(a, j[2]) for a, j in zip(got, jobs)), i
print("replays equal")
"""


def test_gemm_first_call_in_a_graph():
    note("gemm recorded into a graph as the library's first call, 4 replays")
    r = subprocess.run([sys.executable, "-c", CAPTURE, ROOT], capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0 and "replays equal" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


# A off 16 bytes takes the loader's registers: within twice the time of the
# direct copies (median of 9; 0.95 to 1.35 measured, and 2.6 to 4.5 when the
# loader waited for two pieces at a time)
@pytest.mark.parametrize("n,bpr,m", [(3584, 14, 160), (4608, 14, 512), (18944, 14, 512), (2304, 26, 2048)])
def test_gemm_unaligned_activations_time(L, n, bpr, m):
    import torch
    note(f"gemm time n={n} bpr={bpr} m={m}, A at +0 and +2")
    wt = dev(random_q4k_bytes(np.random.default_rng(1), n * bpr))
    at = dev(np.random.default_rng(2).standard_normal(m * bpr * 256 + 8).astype(np.float16))
    ct = empty_f32(m * n)

    def us(off, reps=20):
        t = []
        for _ in range(9):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(reps):
                _lib.check("gemm", L.launch_gemm_q4k_f16(ptr(wt), ptr(at) + off, ptr(ct), n, bpr, m, None))
            e[1].record()
            e[1].synchronize()
            t.append(e[0].elapsed_time(e[1]) / reps * 1e3)
        return float(np.median(t))

    us(0, 3), us(2, 3)
    aligned, off2 = us(0), us(2)
    print(f"aligned {aligned:.1f} us, at +2 {off2:.1f} us", flush=True)
    assert off2 <= 2.0 * aligned
