"""The prefill GEMM's weights keep f16's full precision whatever the spread of
the block and sub-block scales in a row: activations are scaled against the
weights here (large where the weights are small), so that no part of a row
hides another's rounding.

Bound: the GEMM rounds d*sc, dmin*m and the weight to f16, as normal numbers.
The same three roundings in numpy (one power of two per block, nothing
subnormal) give the error that the format allows; the GEMM's may exceed it by
2 % (subnormal leftovers of sub-blocks far below their block's largest) plus
the rounding of the f32 sums, 2e-6 of the result. Beside it the bounds of the
other GEMM tests: 1e-3 Frobenius, 1e-2 sum|w||a| / sqrt(K) an element."""
import numpy as np
import pytest

from modgrad_amd import _lib
from tests.gpu_util import dev, empty_f32, host, ptr

pytestmark = pytest.mark.gpu

# one shape for each way a row's header is decoded and a rescale runs: 16 rows
# a wavefront (four lanes a header) and K shares of 5 blocks, 32 rows (two
# lanes) and shares of 7, 48 rows with all of K in both orders, 48 rows in one
SHAPES = [(200, 20, 40), (4608, 14, 512), (18944, 14, 256), (18944, 14, 512)]


def block_scales(kind, rng, bpr):
    b = np.arange(bpr)
    if kind == "falling":  # e has to rise again
        return np.where(b < bpr // 4, 64.0, 1.0)
    if kind == "slope":  # never far from the block before
        return 2.0 ** (-7 + 14 * b[::-1] / bpr)
    if kind == "rising":
        return 2.0 ** (-7 + 14 * b / bpr)
    if kind == "mixed":
        return 2.0 ** rng.uniform(-7, 7, bpr)
    if kind == "zeros":  # blocks without a weight between small and large ones
        return np.where(b % 3 == 1, 0.0, np.where(b < bpr // 2, 32.0, 1.0))
    return np.ones(bpr)


def f16(x):
    return x.astype(np.float16).astype(np.float64)


def pack(d, dm, sc, mn, qs):
    """Q4_K blocks from d, dmin [nb], 8 six-bit scales and mins [nb, 8], qs."""
    out = np.empty((d.size, 144), np.uint8)
    out[:, 0:4] = np.stack([d, dm], 1).astype(np.float16).view(np.uint8)
    out[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    out[:, 8:12] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    out[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    out[:, 16:] = qs
    return out.ravel()


@pytest.mark.parametrize("n,bpr,m", SHAPES)
@pytest.mark.parametrize("kind", ["even", "falling", "slope", "rising", "mixed", "zeros", "sub"])
def test_gemm_small_weights_under_large_activations(kind, n, bpr, m):
    print(f"[case] gemm range {kind} n={n} bpr={bpr} m={m}", flush=True)
    rng = np.random.default_rng(n + m + len(kind))
    s = block_scales(kind, rng, bpr)
    d = (rng.uniform(0.6, 1.6, (n, bpr)) * s * 2.0 ** -6).astype(np.float16)
    dm = (d.astype(np.float32) * 7).astype(np.float16)
    sc = rng.integers(32, 64, (n, bpr, 8), dtype=np.uint8)
    if kind == "sub":  # sub-blocks 2^0 .. 2^-5 of the block's largest
        sc = np.broadcast_to(np.array([63, 1, 16, 4, 2, 33, 8, 63], np.uint8), sc.shape)
    qs = rng.integers(0, 256, (n * bpr, 128), dtype=np.uint8)
    w = pack(d.ravel(), dm.ravel(), sc.reshape(-1, 8), sc.reshape(-1, 8), qs)
    a = rng.standard_normal((m, bpr, 8, 32))
    a /= np.where(s > 0, s, 1.0)[None, :, None, None]
    if kind == "sub":
        a /= sc[0, 0].astype(float)[None, None, :, None] / 32
    a = a.astype(np.float16).reshape(m, -1)

    wt, at, ct = dev(w), dev(a.view(np.uint16)), empty_f32(m * n)
    _lib.check("gemm", _lib.load().launch_gemm_q4k_f16(ptr(wt), ptr(at), ptr(ct), n, bpr, m, None))
    rows = np.sort(rng.choice(n, size=96, replace=False))
    C = host(ct).reshape(m, n)[:, rows].astype(np.float64)
    assert np.all(np.isfinite(C))

    def products(dd, q, mm):  # [rows, K] -> [m, rows]
        return a.astype(np.float64) @ (dd * q - mm).reshape(rows.size, -1).T

    qr = qs.reshape(n, bpr, 4, 1, 32)[rows]
    q = np.concatenate([qr & 15, qr >> 4], 3).reshape(rows.size, bpr, 8, 32).astype(np.float64)
    ds = (d[rows].astype(np.float64)[..., None] * sc[rows])[..., None]
    ms = (dm[rows].astype(np.float64)[..., None] * sc[rows])[..., None]
    ref = products(ds, q, ms)
    up = np.exp2(10.0 - np.log2(np.where(s > 0, s, 1.0)).round())[None, :, None, None]
    rounded = f16(f16(ds * up) * q - f16(ms * up)) / up
    allowed = np.linalg.norm(products(rounded, 1.0, 0.0) - ref)
    err, size = np.linalg.norm(C - ref), np.linalg.norm(ref)
    print(f"error {err / size:.3e}, of the format {allowed / size:.3e}", flush=True)
    assert err <= np.hypot(1.02 * allowed, 2e-6 * size)
    assert err <= 1e-3 * size
    absdot = np.abs(a.astype(np.float64)) @ np.abs(ds * q - ms).reshape(rows.size, -1).T
    assert np.all(np.abs(C - ref) <= 1e-2 * absdot / np.sqrt(bpr * 256))
