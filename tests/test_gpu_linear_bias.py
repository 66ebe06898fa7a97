"""launch_matvec_q4k_bias_ex: the same bits as the matvec followed by the bias
add, where it is one kernel (flattened rows of whole sub-blocks, every unit
size) and where it is two (whole blocks, and rows of odd length)."""
import numpy as np
import pytest

from modgrad_amd import _lib
from tests.gpu_util import dev, empty_f32, host, ptr, random_q4k_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,off", [(8, 32, 0), (8, 96, 0), (16, 160, 4), (12, 64, 0), (6, 128, 0),
                                     (4864, 896, 0), (1002, 896, 12), (31, 256, 0), (512, 1024, 0),
                                     (256, 33, 0), (9, 65536 + 256, 0), (264, 14112, 0)])
def test_bias_is_the_two_launch_sequence(n, k, off):
    print(f"[case] bias n={n} k={k} off={off}", flush=True)
    L = _lib.load()
    rng = np.random.default_rng(n + k)
    wt = dev(random_q4k_bytes(rng, n * k // 256))
    xt = dev(rng.standard_normal(k).astype(np.float32))
    bt = dev(np.concatenate([np.zeros(off // 4, np.float32), rng.standard_normal(n).astype(np.float32)]))
    two, one = empty_f32(n), empty_f32(n + off // 4)
    _lib.check("matvec", L.launch_matvec_q4k_ex(ptr(wt), ptr(xt), ptr(two), n, k, _lib.LAYOUT_FLAT, None))
    _lib.check("add", L.launch_residual_add_ex(ptr(two), ptr(bt) + off, n, None))
    _lib.check("bias", L.launch_matvec_q4k_bias_ex(ptr(wt), ptr(xt), ptr(bt) + off, ptr(one) + off, n, k,
                                                   _lib.LAYOUT_FLAT, None))
    a, b = host(two), host(one)[off // 4:]
    assert np.all(np.isfinite(a))
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_bias_refuses_what_the_matvec_refuses():
    L = _lib.load()
    t = empty_f32(64)
    p = ptr(t)
    for args in ((0, p, p, p, 8, 32), (p, 0, p, p, 8, 32), (p, p, 0, p, 8, 32), (p, p, p, 0, 8, 32),
                 (p, p, p + 2, p, 8, 32), (p, p + 2, p, p, 8, 32), (p, p, p, p, 0, 32), (p, p, p, p, 8, 0),
                 (p, p, p, p, 3, 32)):
        assert L.launch_matvec_q4k_bias_ex(*args, _lib.LAYOUT_FLAT, None) == _lib.hipErrorInvalidValue
    assert L.launch_matvec_q4k_bias_ex(p, p, p, p, 8, 32, 7, None) == _lib.hipErrorInvalidValue
