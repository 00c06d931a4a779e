"""The 192-row tile of the prefill's BF16 GEMM (prefill.hip, launch_gemm_e
takes it where the 128-row tile needs another round of the chip and the
256-row one would leave more of it idle): exact on small integers, whose
products and sums f32 holds, with ragged last tiles in both directions, one
K step (fewer than the tile's buffers) and an odd number of them."""
import numpy as np
import pytest

import yue2_rs_amd as y2

pytestmark = pytest.mark.gpu


def _bf16(a):
    return (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)


@pytest.mark.parametrize("M,N,K", [(2048, 5120, 64), (1921, 5001, 192), (2100, 5100, 320)])
def test_gemm_small_integers_exact(gpu, M, N, K):
    rng = np.random.default_rng(M + N + K)
    x = rng.integers(-8, 9, (M, K)).astype(np.float32)
    w = rng.integers(-8, 9, (N, K)).astype(np.float32)
    x16, w16, out = _bf16(x), _bf16(w), np.empty((M, N), np.float32)
    print(M, N, K, flush=True)
    rc = y2.lib().yue2_hip_selftest_gemm(x16.ctypes.data, w16.ctypes.data, out.ctypes.data, M, N, K)
    assert rc == 0, y2.lib().yue2_hip_last_error().decode()
    assert np.array_equal(out, x @ w.T)
