"""GEMMs whose rows are no whole number of 16-byte chunks, or whose operands lie
at any address: the matrix-core kernels' unaligned loads and the mask of the
chunk that a row ends in, against the oracle (int8: bit for bit; 16-bit: the
fp32 bound of tests/test_gpu_kernels.py, also for rows whose values are far
apart or tiny), and, for values that are not finite, the class (finite, which
infinity, NaN) of an fp32 sum."""
import numpy as np
import pytest

import edgecore_amd as ec
import oracle

pytestmark = pytest.mark.gpu

# rows: one, both skinny fragments and their edges, the tiles' edges; widths:
# one byte (element) past and short of a chunk, a 64-byte step, a 128-byte stage;
# int8 tiles of 32 rows, 64 (600 x 9001: 710 blocks) and 128 (1000 x 6900: 432)
SHAPES = [(1, 17, 33), (1, 1001, 777), (15, 31, 16), (16, 65, 100), (17, 1000, 129), (32, 127, 15), (33, 129, 40),
          (64, 1000, 130), (65, 255, 257), (300, 1023, 700), (130, 4097, 65), (600, 1001, 9001), (1000, 33, 6900)]


def _dev(fn, out_shape, *args):
    out = ec.DeviceBuffer(4 * int(np.prod(out_shape)))
    try:
        assert fn(out.ptr, *args) == 0, ec.last_error()
        assert ec.lib().ec_sync() == 0
        return out.to_array(np.float32, out_shape)
    finally:
        out.close()


def _at(a, off):
    """A device copy of `a` that starts `off` bytes into its allocation."""
    raw = np.concatenate([np.zeros(off, np.uint8), np.ascontiguousarray(a).view(np.uint8).reshape(-1)])
    return ec.DeviceBuffer.from_array(raw)


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_int8_bit_exact(M, K, N):
    rng = np.random.default_rng(M + 3 * K + N)
    A = rng.integers(-128, 128, (M, K)).astype(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    a_s, b_s = rng.uniform(1e-4, 1e-1, M).astype(np.float32), rng.uniform(1e-4, 1e-2, N).astype(np.float32)
    bias = rng.normal(0, 0.02, N).astype(np.float32) if M % 2 else None
    got = ec.gemm_int8(A, a_s, B, b_s, bias)
    assert np.array_equal(got.view(np.uint32), oracle.gemm_int8(A, a_s, B, b_s, bias).view(np.uint32))


@pytest.mark.parametrize("M,K,N", [(3, 96, 40), (20, 128, 130), (40, 128, 130), (40, 100, 33)])
@pytest.mark.parametrize("oa,ob", [(1, 0), (0, 3), (8, 4)])
def test_int8_any_address(M, K, N, oa, ob):
    rng = np.random.default_rng(M + K + N + oa)
    A = rng.integers(-128, 128, (M, K)).astype(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    a_s = rng.uniform(1e-4, 1e-1, M).astype(np.float32)
    bufs = [_at(A, oa), ec.DeviceBuffer.from_array(a_s), _at(B, ob)]
    try:
        got = _dev(ec.lib().ec_gemm_int8_dev, (M, N), bufs[0].ptr + oa, bufs[1].ptr, bufs[2].ptr + ob, None, None, M,
                   K, N)
    finally:
        for b in bufs:
            b.close()
    assert np.array_equal(got.view(np.uint32), oracle.gemm_int8(A, a_s, B, None, None).view(np.uint32))


def _bits(x, bf16):
    if not bf16:
        return np.asarray(x, np.float16).view(np.uint16)
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


# 16-bit: up to 16 and 32 rows without stages, above and for wide outputs the
# tiles; one, two, three and more stages of 64
W16_SHAPES = SHAPES[:-2] + [(5, 8, 3), (3, 17, 16400), (32, 129, 16385), (33, 63, 65), (70, 193, 200)]


@pytest.mark.parametrize("M,K,N", W16_SHAPES)
@pytest.mark.parametrize("bf16", [False, True])
def test_w16_within_bound(M, K, N, bf16):
    rng = np.random.default_rng(M + K + N + bf16)
    A = rng.normal(0, 1, (M, K)).astype(np.float32)
    B = _bits(rng.normal(0, 0.02, (N, K)), bf16)
    got = (ec.gemm_bf16_fp32 if bf16 else ec.gemm_fp16_fp32)(A, B)
    Bf = (B.astype(np.uint32) << 16).view(np.float32) if bf16 else B.view(np.float16).astype(np.float32)
    want = A.astype(np.float64) @ Bf.astype(np.float64).T
    bound = 2.0 * K * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(Bf).astype(np.float64).T)
    assert np.all(np.abs(got - want) <= bound)


def _in_order(A, Bf):
    """The fp32 FMA sum over k in order (a product of 24 and at most 11 bits is
    exact in float64)."""
    s = np.zeros((A.shape[0], Bf.shape[0]), np.float32)
    for k in range(A.shape[1]):
        s = (A[:, k, None].astype(np.float64) * Bf[None, :, k].astype(np.float64) + s).astype(np.float32)
    return s


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M", [5, 20, 64])
@pytest.mark.parametrize("K", [9, 17, 33, 101, 1001])
@pytest.mark.parametrize("rows", ["normal", 1e8, 1e10, 1e-36, 1e-40])
def test_w16_activations_keep_their_bits(M, K, rows, bf16):
    """Rows with one value 1e8 or 1e10 times the others (it meets zero weights,
    so the others make the result) and rows down to subnormal values: the fp32
    bound, 2^-149 per product for what underflows, and an error against 64 bits
    that is no larger than that of the fp32 sum in order (5%: the two round
    differently)."""
    N = 200
    rng = np.random.default_rng(K + M)
    A, W = rng.normal(0, 1, (M, K)).astype(np.float32), rng.normal(0, 0.02, (N, K)).astype(np.float32)
    if rows in (1e8, 1e10):
        A[:, 2], W[:, 2] = rows, 0.0
    elif rows != "normal":
        A, W = (A * np.float64(rows)).astype(np.float32), W * 50
    B = _bits(W, bf16)
    Bf = (B.astype(np.uint32) << 16).view(np.float32) if bf16 else B.view(np.float16).astype(np.float32)
    got = (ec.gemm_bf16_fp32 if bf16 else ec.gemm_fp16_fp32)(A, B)
    want = A.astype(np.float64) @ Bf.astype(np.float64).T
    mag = np.abs(A).astype(np.float64) @ np.abs(Bf).astype(np.float64).T
    assert np.all(np.abs(got - want) <= 2.0 * K * 2.0 ** -24 * mag + K * 2.0 ** -149)
    assert np.linalg.norm(got - want) <= 1.05 * np.linalg.norm(_in_order(A, Bf) - want)


@pytest.mark.parametrize("off", [2, 6, 8])
@pytest.mark.parametrize("M,K,N", [(3, 96, 40), (20, 128, 130), (40, 128, 130), (40, 100, 33)])
def test_w16_any_address(M, K, N, off):
    """Weights and activations that start anywhere (multiples of their size)."""
    rng = np.random.default_rng(M + K + N + off)
    A = rng.normal(0, 1, (M, K)).astype(np.float32)
    B = rng.normal(0, 0.02, (N, K)).astype(np.float16)
    oa = 4 * (off // 4)
    bufs = [_at(A, oa), _at(B.view(np.uint16), off)]
    try:
        got = _dev(ec.lib().ec_gemm_fp16_fp32_dev, (M, N), bufs[0].ptr + oa, bufs[1].ptr + off, M, K, N)
    finally:
        for b in bufs:
            b.close()
    want = A.astype(np.float64) @ B.astype(np.float64).T
    assert np.all(np.abs(got - want) <= 2.0 * K * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64).T))


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
@pytest.mark.parametrize("shape", [dict(arch="gpt2", embd=36, heads=2, ffn=147), dict(arch="qwen2", embd=36, heads=2, kv_heads=1, ffn=147)],
                         ids=["gpt2", "qwen2"])
def test_forward_of_ragged_widths(tmp_path, shape, precision):
    """Models whose every linear is ragged: each epilogue (bias, residual, GELU,
    SwiGLU) at 1, 5, 20 and 70 rows against the oracle's logits."""
    path = tmp_path / "m.ecm"
    ec.synth(path, layers=2, ctx=128, vocab=300, precision=precision, seed=3, **shape)
    om = oracle.OracleModel(path, 1, 128)
    with ec.Model(path, 1, 128) as m:
        for n in (1, 5, 20, 70):
            toks, pos, sl = np.arange(n) * 7 % 300, np.arange(n), np.zeros(n, np.int32)
            got, _ = m.forward(toks, pos, sl)
            assert np.abs(got - om.forward(toks, pos, sl)).max() <= 1e-4
    om.close()


@pytest.mark.parametrize("M", [5, 40])
@pytest.mark.parametrize("bf16", [False, True])
def test_w16_not_finite(M, bf16):
    """Infinities and NaN in single activations and weights: every output is
    of the class that the fp32 sum over its row gives (finite ones within the
    bound)."""
    K, N = 101, 50
    rng = np.random.default_rng(M + bf16)
    A = rng.normal(0, 1, (M, K)).astype(np.float32)
    W = rng.normal(0, 0.02, (N, K)).astype(np.float32)
    A[0, 3], A[1, K - 1], A[2, 50] = np.inf, -np.inf, np.nan
    W[0, 100], W[7, 3], W[9, 20] = np.inf, -np.inf, np.nan
    W[11, 3] = 0.0  # meets the infinity of row 0
    B = _bits(W, bf16)
    Bf = (B.astype(np.uint32) << 16).view(np.float32) if bf16 else B.view(np.float16).astype(np.float32)
    got = (ec.gemm_bf16_fp32 if bf16 else ec.gemm_fp16_fp32)(A, B)
    with np.errstate(invalid="ignore"):
        want = (A[:, None, :].astype(np.float64) * Bf[None].astype(np.float64)).sum(2)
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert inf.any() and np.array_equal(got[inf], want[inf].astype(np.float32))
    mag = np.where(np.isfinite(A), np.abs(A), 0).astype(np.float64) @ np.where(np.isfinite(Bf), np.abs(Bf), 0).T
    assert np.all(np.abs(got[fin] - want[fin]) <= 2.0 * K * 2.0 ** -24 * mag[fin])


# rows of whole 16-byte chunks that end inside a 128-byte stage of the tile
# kernel: one chunk past and short of a stage, each row tile, split K (few
# tiles, from 44 stages, 16-bit 16), 2 to 4 stage buffers
STAGE_SHAPES = [(33, 16, 40), (40, 112, 130), (40, 144, 130), (64, 2064, 200), (130, 4848, 129), (64, 5520, 200),
                (130, 6000, 129), (500, 11664, 896), (600, 1008, 9001)]


@pytest.mark.parametrize("M,K,N", STAGE_SHAPES)
def test_int8_partial_stage(M, K, N):
    test_int8_bit_exact(M, K, N)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,K,N", [(M, K // 2, N) for M, K, N in STAGE_SHAPES])
def test_w16_partial_stage(M, K, N, bf16):
    rng = np.random.default_rng(M + K + N)
    A = rng.normal(0, 1, (M, K)).astype(np.float32)
    B = (rng.normal(0, 0.02, (N, K)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) if bf16 else \
        rng.normal(0, 0.02, (N, K)).astype(np.float16).view(np.uint16)
    Bf = (B.astype(np.uint32) << 16).view(np.float32) if bf16 else B.view(np.float16).astype(np.float32)
    got = (ec.gemm_bf16_fp32 if bf16 else ec.gemm_fp16_fp32)(A, B)
    want = A.astype(np.float64) @ Bf.T.astype(np.float64)
    bound = 2.0 * K * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(Bf.T).astype(np.float64)) + 1e-30
    assert np.all(np.abs(got - want) <= bound)
