"""The device attention kernels alone against the oracle's per-row attention
(src/gpt2.c:527-557 GPT-2, 744-777 Qwen2 GQA) on the same seeded q and fp16
caches, through ec_attention_dev.

Bar: the kernels keep the reference's order for every float operation; the
one difference is the double sum of the exponentials, added in a tree order,
whose last bits can move a probability's float rounding in rare ties.  So
almost every element is bit-identical (at least 99.9% asserted) and none is
further than 1e-5 from the oracle (values are O(1))."""
import numpy as np
import pytest

import edgecore_amd as ec
import oracle

pytestmark = pytest.mark.gpu


def _f16(x):
    return np.asarray(x, np.float32).astype(np.float16).view(np.uint16)


def _case(seed, M, H, KVH, hd, C, nslots):
    rng = np.random.default_rng(seed)
    kc = _f16(rng.normal(0, 1, (nslots, C, KVH * hd)))
    vc = _f16(rng.normal(0, 1, (nslots, C, KVH * hd)))
    q = rng.normal(0, 1, (M, H * hd)).astype(np.float32)
    return rng, q, kc, vc


def _check(got, want, rows):
    g, w = got[rows], want[rows]
    assert np.isfinite(g).all()
    err = np.abs(g - w).max()
    exact = (g == w).mean()
    print(f"rows {len(rows)}: max-abs {err:.3e}, bit-identical {exact:.6f}")
    assert err <= 1e-5, err
    assert exact >= 0.999, exact


def _rows(rng, M, k):
    edge = [0, 1, 15, 16, 17, 63, 64, 65, 127, 128, M // 2, M - 17, M - 16, M - 2, M - 1]
    return np.unique(np.concatenate([[r for r in edge if 0 <= r < M], rng.choice(M, min(k, M), replace=False)]))


def test_prefill_qwen2_05b_2048():
    """The 2048-token prompt of the prefill benchmark (Qwen2-0.5B heads: 14
    query heads, 2 KV heads, head_dim 64): 16 tokens per block, the whole-tile
    and partial-tile paths and the diagonal tiles."""
    M, H, KVH, hd = 2048, 14, 2, 64
    rng, q, kc, vc = _case(1, M, H, KVH, hd, M, 1)
    pos, slot = np.arange(M), np.zeros(M)
    got = ec.attention_dev(q, kc, vc, pos, slot, H, KVH, path=0)
    rows = _rows(rng, M, 160)
    want = oracle.attention_rows(q, kc, vc, pos, slot, H, KVH, rows=rows)
    _check(got, want, rows)


@pytest.mark.parametrize("H,KVH,hd,M,p0,window,nslots,slot", [
    (14, 2, 64, 200, 100, 48, 2, 1),   # mid-cache start, sliding window, second slot
    (14, 2, 64, 333, 0, 0, 1, 0),      # ragged last block
    (12, 2, 128, 300, 17, 0, 1, 0),    # head_dim 128: one token per wave
    (4, 4, 32, 150, 0, 0, 1, 0),       # head_dim 32, GPT-2-style heads (KVH = H)
    (4, 4, 64, 700, 0, 100, 1, 0),     # window spanning tiles
])
def test_prefill_shapes(H, KVH, hd, M, p0, window, nslots, slot):
    C = p0 + M + 8
    rng, q, kc, vc = _case(M + hd, M, H, KVH, hd, C, nslots)
    pos = p0 + np.arange(M)
    sl = np.full(M, slot)
    got = ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=window, path=0)
    want = oracle.attention_rows(q, kc, vc, pos, sl, H, KVH, window=window)
    _check(got, want, np.arange(M))


@pytest.mark.parametrize("hd,window", [(64, 0), (128, 0), (64, 300)])
def test_decode_kernel_long_positions(hd, window):
    """The per-token kernel: 8 tokens in 4 slots at positions up to 2047."""
    H, KVH, C, ns = 14, 2, 2048, 4
    rng, q, kc, vc = _case(5 + hd, 8, H, KVH, hd, C, ns)
    pos = np.array([2047, 2000, 1536, 1023, 511, 64, 3, 0])
    sl = np.array([0, 1, 2, 3, 0, 1, 2, 3])
    got = ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=window, path=1)
    want = oracle.attention_rows(q, kc, vc, pos, sl, H, KVH, window=window)
    _check(got, want, np.arange(8))


@pytest.mark.parametrize("H,KVH,hd,window", [(12, 2, 128, 0), (12, 2, 128, 700), (16, 1, 128, 0), (6, 6, 128, 0)])
def test_decode_scores_pass_equals_per_token_kernel(H, KVH, hd, window):
    """The long-context decode form of head_dim 128 (path 2: a scores pass
    per token, KV group and 256 positions, then the per-token kernel's
    softmax and sums on those scores) against the per-token kernel (path 1)
    bit for bit, and against the oracle: GQA groups of 6 and 16 heads and
    GPT-2-style heads, with and without a window; 8 tokens in 4 slots at
    positions up to 2047."""
    C, ns = 2048, 4
    rng, q, kc, vc = _case(77 + hd + H + window, 8, H, KVH, hd, C, ns)
    pos = np.array([2047, 2000, 1536, 1023, 511, 256, 3, 0])
    sl = np.array([0, 1, 2, 3, 0, 1, 2, 3])
    one = ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=window, path=1)
    two = ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=window, path=2)
    assert np.array_equal(one.view(np.uint32), two.view(np.uint32))
    want = oracle.attention_rows(q, kc, vc, pos, sl, H, KVH, window=window)
    _check(two, want, np.arange(8))


def test_attention_dev_rejects_bad_arguments():
    H, KVH, hd, C = 4, 2, 64, 32
    _, q, kc, vc = _case(9, 4, H, KVH, hd, C, 1)
    with pytest.raises(ec.EdgeCoreError):
        ec.attention_dev(q, kc, vc, [0, 1, 2, 40], [0, 0, 0, 0], H, KVH)        # position past the cache
    with pytest.raises(ec.EdgeCoreError):
        ec.attention_dev(q, kc, vc, [0, 1, 3, 4], [0, 0, 0, 0], H, KVH, path=0)  # not consecutive
    with pytest.raises(ec.EdgeCoreError):
        ec.attention_dev(q, kc, vc, [0, 1, 2, 3], [0, 0, 1, 0], H, KVH)          # slot outside the cache


# the two prefill kernels at the edges of the matrix-core one: 16 tokens per
# block (1, 15, 17, 33 of them), 64-position tiles, 1 (span 512), 2 (1024), 4
# (2048) and 8 (4096) of them per wave, and past that the other kernel, which
# also takes what is at most 256 of its 8-token blocks (the rows of few heads);
# head_dim 128 takes the matrix-core one from 192 blocks on
@pytest.mark.parametrize("H,KVH,hd,M,p0,window", [
    (2, 1, 64, 1, 0, 0), (2, 1, 64, 15, 49, 0), (2, 2, 64, 17, 48, 0), (3, 1, 64, 33, 479, 0), (2, 1, 64, 33, 480, 0),
    (2, 1, 64, 20, 2028, 0), (2, 1, 64, 21, 2028, 0), (1, 1, 64, 16, 4080, 0), (1, 1, 64, 16, 4081, 0),
    (2, 1, 64, 40, 700, 1), (2, 1, 64, 70, 0, 497), (2, 1, 64, 70, 430, 498), (2, 1, 32, 33, 500, 0),
    (2, 2, 32, 17, 2100, 0), (96, 8, 128, 31, 0, 0), (96, 8, 128, 32, 490, 0), (96, 8, 128, 17, 1000, 300),
    (96, 8, 128, 17, 2040, 0),
    (257, 1, 64, 1, 0, 0), (130, 2, 64, 15, 49, 0), (86, 2, 64, 17, 48, 0), (128, 2, 64, 16, 500, 0),
    (130, 2, 64, 16, 500, 0), (54, 2, 64, 33, 479, 0), (54, 2, 64, 33, 480, 0), (86, 2, 64, 20, 1004, 0),
    (86, 2, 64, 21, 1004, 0), (86, 2, 64, 20, 2028, 0), (86, 2, 64, 21, 2028, 0), (130, 1, 64, 16, 4080, 0),
    (130, 1, 64, 16, 4081, 0), (54, 2, 64, 40, 700, 1), (30, 2, 64, 70, 0, 497), (30, 2, 64, 70, 430, 498),
    (30, 2, 64, 70, 900, 1009), (30, 2, 64, 70, 900, 1010), (54, 2, 32, 33, 500, 0), (86, 2, 32, 17, 1000, 0),
    (86, 2, 32, 17, 2100, 0), (96, 8, 128, 32, 700, 0), (96, 8, 128, 17, 3000, 0)])
def test_prefill_matrix_core_edges(H, KVH, hd, M, p0, window):
    rng, q, kc, vc = _case(M + p0 + hd + window, M, H, KVH, hd, p0 + M, 2)
    pos, sl = p0 + np.arange(M), np.ones(M)
    got = ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=window, path=0)
    want = oracle.attention_rows(q, kc, vc, pos, sl, H, KVH, window=window)
    _check(got, want, np.arange(M))


@pytest.mark.parametrize("hd,H", [(64, 2), (64, 60), (128, 96)])
def test_prefill_value_not_finite_outside_a_tokens_range(hd, H):
    """An infinity in the last position's value reaches that position's token
    alone, and one before a window no token inside it."""
    M, KVH, window = 40, 2, 20
    _, q, kc, vc = _case(hd, M, H, KVH, hd, M, 1)
    vc[0, M - 1] = 0x7C00
    vc[0, 0] = 0xFC00
    pos, sl = np.arange(M), np.zeros(M)
    got = ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=window, path=0)
    want = oracle.attention_rows(q, kc, vc, pos, sl, H, KVH, window=window)
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    _check(got, want, np.arange(window, M - 1))


@pytest.mark.parametrize("path,H", [(0, 2), (0, 88), (1, 2), (2, 2)])
@pytest.mark.parametrize("window", [2 ** 31 - 1, 2 ** 31 - 8, 2 ** 30])
def test_window_beyond_every_position(window, path, H):
    """A window that reaches past every position, up to the largest int, is no
    window (more than 512 positions: several score tiles per wave)."""
    M, KVH, hd, p0 = 20, 1, 64, 700
    _, q, kc, vc = _case(window % 1000 + path, M, H, KVH, hd, p0 + M, 1)
    pos, sl = p0 + np.arange(M), np.zeros(M)
    got = ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=window, path=path)
    assert np.array_equal(got, ec.attention_dev(q, kc, vc, pos, sl, H, KVH, window=0, path=path))
    _check(got, oracle.attention_rows(q, kc, vc, pos, sl, H, KVH), np.arange(M))
