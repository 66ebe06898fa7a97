"""Q6_K matvec on Q8_1 activations (launch_matvec_q6k_dp4a): the matrix-core
kernel at the edges of its shapes (one block, blocks per wavefront + 1, table
items per thread, the longest row that its LDS takes and the one past it: 90
blocks up to 4096 rows on 256 CUs, 89 above; ragged row groups), int8
activations at any byte, the extreme int8 values, and a non-finite scale.

Bound: the integer dots are exact, so y differs from the oracle's float
evaluation only by the f32 rounding of its terms and their sum: 2^-20 of the
sum of the terms' magnitudes covers rows of up to 92 blocks."""
import numpy as np
import pytest

from modgrad_amd import _lib
from tests.gpu_util import dev, empty_f32, host, ptr, random_kquant_bytes

pytestmark = pytest.mark.gpu


def note(msg: str) -> None:
    print(f"[case] {msg}", flush=True)


def run(orc, n, bpr, xq, xd, xoff=0, woff=0):
    L = _lib.load()
    w = random_kquant_bytes(np.random.default_rng(n + 31 * bpr), n * bpr, 210)
    wt = dev(np.concatenate([np.zeros(woff, np.uint8), w]))
    qt = dev(np.concatenate([np.zeros(xoff, np.int8), xq]))
    dt, yt = dev(xd), empty_f32(n)
    _lib.check("q6k dp4a", L.launch_matvec_q6k_dp4a(ptr(wt) + woff, ptr(qt) + xoff, ptr(dt), ptr(dt),
                                                    ptr(yt), n, bpr))
    y_ref, absterm = orc.gemv_q6k_dp4a(w, xq, xd, n, bpr)
    return host(yt), y_ref, absterm


@pytest.mark.parametrize("n,bpr", [(8, 1), (24, 3), (136, 13), (40, 14), (48, 15), (16, 16), (520, 17),
                                   (24, 32), (24, 33), (3584, 74), (16, 64), (16, 65), (16, 90),
                                   (4096, 90), (4112, 90), (16, 91), (16, 92),
                                   (9600, 16), (70000, 2), (17, 8), (33, 5)])
def test_q6k_dp4a_shapes(orc, n, bpr):
    note(f"q6k dp4a n={n} bpr={bpr}")
    rng = np.random.default_rng(n + bpr)
    xq = rng.integers(-127, 128, size=bpr * 256).astype(np.int8)
    xd = rng.uniform(1e-3, 2e-2, size=bpr * 8).astype(np.float32)
    y, y_ref, a = run(orc, n, bpr, xq, xd)
    assert np.all(np.abs(y.astype(np.float64) - y_ref) <= 2.0 ** -20 * a)


@pytest.mark.parametrize("xoff,woff", [(1, 0), (7, 0), (0, 2), (3, 1)])
def test_q6k_dp4a_offsets(orc, xoff, woff):
    note(f"q6k dp4a offsets {xoff} {woff}")
    n, bpr = 136, 20
    rng = np.random.default_rng(3)
    xq = rng.integers(-127, 128, size=bpr * 256).astype(np.int8)
    xd = rng.uniform(1e-3, 2e-2, size=bpr * 8).astype(np.float32)
    y, y_ref, a = run(orc, n, bpr, xq, xd, xoff, woff)
    assert np.all(np.abs(y.astype(np.float64) - y_ref) <= 2.0 ** -20 * a)


@pytest.mark.parametrize("value", [127, -127, -128, 0])
def test_q6k_dp4a_extreme_values(orc, value):
    # every product of one sign: the largest integer dots
    note(f"q6k dp4a constant {value}")
    n, bpr = 64, 6
    y, y_ref, a = run(orc, n, bpr, np.full(bpr * 256, value, np.int8), np.full(bpr * 8, 0.01, np.float32))
    assert np.all(np.abs(y.astype(np.float64) - y_ref) <= 2.0 ** -20 * a)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_q6k_dp4a_nonfinite_scale(orc, bad):
    # no clamp in the Q6_K formula: every row comes out non-finite
    note(f"q6k dp4a scale {bad}")
    n, bpr = 40, 3
    xq = np.ones(bpr * 256, np.int8)
    xd = np.full(bpr * 8, 0.01, np.float32)
    xd[5] = bad
    y, _, _ = run(orc, n, bpr, xq, xd)
    assert not np.any(np.isfinite(y))
