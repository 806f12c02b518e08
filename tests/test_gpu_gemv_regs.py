"""The 16-bit linears of 2 to 15 rows with the activations in registers (rows of
192 elements or more; shorter ones are the fused GEMV's), against the float64 product with the fp32 bound of tests/test_gpu_kernels.py:
one, two and three chunks per lane and their edges, both row tiles and a short
second one, odd outputs, a single pair of them and more than one pass of the
grid."""
import numpy as np
import pytest

import edgecore_amd as ec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,K,N", [(4, 8, 1), (5, 504, 7), (8, 512, 9), (15, 520, 63), (4, 1016, 700), (9, 1024, 33),
                                   (7, 1032, 100), (8, 1536, 2), (13, 1528, 5001), (2, 896, 8193), (3, 768, 9001),
                                   (4, 184, 33), (4, 192, 1), (11, 200, 5000), (2, 184, 8200), (3, 192, 8200)])
def test_rows_in_registers(M, K, N, bf16):
    rng = np.random.default_rng(M + K + N)
    A = rng.normal(0, 1, (M, K)).astype(np.float32)
    if bf16:
        B = (rng.normal(0, 0.02, (N, K)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        Bf = (B.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    else:
        B = rng.normal(0, 0.02, (N, K)).astype(np.float16).view(np.uint16)
        Bf = B.view(np.float16).astype(np.float64)
    got = (ec.gemm_bf16_fp32 if bf16 else ec.gemm_fp16_fp32)(A, B)
    want = A.astype(np.float64) @ Bf.T
    bound = 2.0 * K * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(Bf).T) + 1e-30
    assert np.all(np.abs(got - want) <= bound)


def test_values_not_finite():
    """A weight that is not finite reaches its own output alone, also from the
    end of a row whose length is no multiple of the lanes' chunks."""
    A = np.ones((8, 520), np.float32)
    B = np.full((20, 520), 0.5, np.float16)
    B[3, 519], B[7, 0], B[11, 512] = np.inf, np.nan, -np.inf
    got = ec.gemm_fp16_fp32(A, B.view(np.uint16))
    assert np.isposinf(got[:, 3]).all() and np.isnan(got[:, 7]).all() and np.isneginf(got[:, 11]).all()
    rest = [n for n in range(20) if n not in (3, 7, 11)]
    assert (got[:, rest] == 260.0).all()
