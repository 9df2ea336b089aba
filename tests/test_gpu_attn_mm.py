"""The matrix-core int8 attention (grouped query heads; prompt rows over one
block) at the sizes where its tiles, masks and ring arithmetic can go wrong,
against the oracle's attend_step.

Tolerance: a score is a dot of at most 64 products summed in fp32 and two
products, |score| < 16 for these N(0, 1) draws, so two summation orders
differ by at most 16 * 66 * 2^-24 = 6.3e-5 in a score in the worst case and
by its square root's share (8e-6) in any draw; an output is a mean of
|v| < 5 under weights off by that much, twice (numerator and sum): 2e-5
bounds the draws with room, against the 1e-4 bar of the entry point.
"""
import numpy as np
import pytest
import torch

import needle_amd as nd
import oracle as O
from conftest import dev, host

pytestmark = pytest.mark.gpu
TOL = 2e-5


def _block(ctx, rng, H, KVH, QK, cap, npos, count=1, k_size=1.0, v_size=1.0):
    """Blocks whose every byte and scale is garbage (NaN) until written."""
    g = nd.kv_geom(H, KVH, QK, 64, cap)
    blk, nb = nd.kv_alloc(g, count)
    blk.fill_(0xff)
    for i in range(count):
        k = (rng.normal(size=(npos, KVH * QK)) * k_size).astype(np.float32)
        v = (rng.normal(size=(npos, KVH * 64)) * v_size).astype(np.float32)
        # the last `cap` positions only: earlier ones would race for a slot
        p0 = max(0, npos - cap)
        pos = torch.arange(p0, npos, dtype=torch.int32, device="cuda")
        nd.kv_write(ctx, g, blk[i * nb:], 0, pos, dev(k[p0:]), dev(v[p0:]))
    return g, blk, nb


def _want(g, block, q, lo, hi):
    if lo < 0 or hi < lo or hi - lo >= g.cap:
        return np.full(g.num_heads * 64, np.nan, np.float32)
    k, ks, v, vs = nd.kv_unpack(g, block)
    return O.attend_step_i8(q, k.reshape(-1), ks.reshape(-1), v.reshape(-1), vs.reshape(-1), g.cap, lo, hi,
                            g.num_heads, g.num_kv_heads, g.qk_head_dim, 64)


def _check(ctx, g, blk, nb, lo, hi, q, quant, shared, tol=TOL):
    lo, hi = np.asarray(lo, np.int32), np.asarray(hi, np.int32)
    got = host(nd.attend_step_i8(ctx, g, blk, 0 if shared else nb, dev(lo), dev(hi), dev(q), quant_query=quant))
    b = host(blk)
    qq = O.quant_rows(q, len(lo), g.num_heads, g.qk_head_dim).reshape(q.shape) if quant else q
    for i in range(len(lo)):
        want = _want(g, b[:nb] if shared else b[i * nb:(i + 1) * nb], qq[i], int(lo[i]), int(hi[i]))
        assert np.array_equal(np.isnan(got[i]), np.isnan(want)), i
        if not np.isnan(want).any():
            assert np.max(np.abs(got[i] - want)) <= np.broadcast_to(tol, len(lo))[i], (i, int(lo[i]), int(hi[i]))


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("H,KVH,QK", [(12, 2, 48), (16, 2, 64), (6, 2, 64), (8, 2, 48), (4, 2, 48)])
@pytest.mark.parametrize("cap,spans", [
    (1, [(0, 0)]), (17, [(0, 16), (20, 36), (3, 3)]), (31, [(40, 70), (69, 70)]), (32, [(33, 64), (64, 64)]),
    (128, [(0, 127), (100, 227), (127, 127)]), (129, [(0, 128), (100, 228), (5, 36)]),
    (2048, [(0, 2047), (1, 33), (100, 131), (2040, 2047)]), (1000, [(500, 1499), (999, 1001), (1480, 1499)])])
def test_decode_grouped(ctx, H, KVH, QK, cap, spans, quant):
    """One row a block: ragged spans, wrapped rings, rings below a chunk."""
    rng = np.random.default_rng(cap + H + quant)
    g, blk, nb = _block(ctx, rng, H, KVH, QK, cap, max(h for _, h in spans) + 1, len(spans))
    q = rng.normal(size=(len(spans), H * QK)).astype(np.float32)
    _check(ctx, g, blk, nb, *zip(*spans), q, quant, False)


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("sessions", [150, 600])
def test_decode_many_sessions(ctx, sessions, quant):
    """Enough sessions for both block widths, each its own ragged span."""
    rng = np.random.default_rng(sessions)
    g, blk, nb = _block(ctx, rng, 12, 2, 48, 96, 96, sessions)
    hi = rng.integers(0, 96, sessions)
    lo = np.array([rng.integers(0, h + 1) for h in hi])
    q = rng.normal(size=(sessions, 12 * 48)).astype(np.float32)
    _check(ctx, g, blk, nb, lo, hi, q, quant, False)


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("H,KVH,QK", [(12, 2, 48), (12, 12, 64), (6, 2, 64), (8, 4, 64)])
@pytest.mark.parametrize("seq,window", [(2, 0), (15, 4), (33, 0), (257, 64), (1500, 100)])
def test_prompt_rows(ctx, H, KVH, QK, seq, window, quant):
    """A prompt's rows over one block, both tile widths (few rows, many)."""
    rng = np.random.default_rng(seq + H)
    g, blk, nb = _block(ctx, rng, H, KVH, QK, seq, seq)
    rows = np.arange(seq) if seq <= 300 else np.arange(seq - 1100, seq)
    lo = np.maximum(rows + 1 - window, 0) if window else 0 * rows
    q = rng.normal(size=(len(rows), H * QK)).astype(np.float32)
    if seq > 300:  # every row runs; the oracle checks some
        got = host(nd.attend_step_i8(ctx, g, blk, 0, dev(lo.astype(np.int32)), dev(rows.astype(np.int32)),
                                     dev(q), quant_query=quant))
        qq = O.quant_rows(q, len(rows), H, QK).reshape(q.shape) if quant else q
        for i in list(range(0, len(rows), 97)) + [len(rows) - 1]:
            assert np.max(np.abs(got[i] - _want(g, host(blk), qq[i], int(lo[i]), int(rows[i])))) <= TOL, i
    else:
        _check(ctx, g, blk, nb, lo, rows, q, quant, True)


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("H,QK", [(12, 64), (32, 48)])
@pytest.mark.parametrize("cap", [30, 512, 513])
@pytest.mark.parametrize("over", [0, 1])
def test_few_rows_of_one_head_each(ctx, H, QK, cap, over, quant):
    """One query head a kv head, as many (row, head) pairs as CUs and a row
    more, rings on both sides of a split: wrapped, windowed and bad spans."""
    rng = np.random.default_rng(cap + H)
    rows = torch.cuda.get_device_properties(0).multi_processor_count // H + over
    g, blk, nb = _block(ctx, rng, H, H, QK, cap, 2 * cap)
    hi = 2 * cap - 1 - np.arange(rows) % cap
    lo = np.maximum(hi + 1 - rng.integers(1, cap + 1, rows), cap)
    lo[0], hi[0], lo[1] = cap, 2 * cap - 1, hi[1] + 1
    q = rng.normal(size=(rows, H * QK)).astype(np.float32)
    _check(ctx, g, blk, nb, lo, hi, q, quant, True)


@pytest.mark.parametrize("H,KVH,QK,cap", [(12, 12, 64, 40000), (8, 1, 64, 34000), (12, 12, 64, 1100),
                                          (12, 12, 64, 2700), (12, 2, 48, 1100), (8, 1, 64, 1500)])
def test_merge_of_split_spans(ctx, H, KVH, QK, cap):
    """One session, its span split over two to more than 64 blocks: whole, a few
    positions (most partials empty), an end, and a bad one."""
    rng = np.random.default_rng(cap + KVH)
    g, blk, nb = _block(ctx, rng, H, KVH, QK, cap, cap)
    for lo, hi in [(0, cap - 1), (5, 7), (cap - 300, cap - 1), (cap // 3, cap // 2), (9, 8)]:
        q = rng.normal(size=(1, H * QK)).astype(np.float32)
        _check(ctx, g, blk, nb, [lo], [hi], q, False, False)


@pytest.mark.parametrize("quant", [False, True])
def test_shared_block_any_spans(ctx, quant):
    """Rows over one ring in any order with spans that share nothing, among
    them bad ones (NaN, that row alone) and positions far apart."""
    H, KVH, QK, cap = 12, 2, 48, 200
    rng = np.random.default_rng(5)
    g, blk, nb = _block(ctx, rng, H, KVH, QK, cap, 450)
    far = 200 * 5_000_000  # a multiple of cap: the same slots
    spans = [(250, 449), (449, 449), (far + 60, far + 99), (300, 310), (-1, 5), (400, 399), (250, 450),
             (255, 260), (2 ** 31 - 48, 2 ** 31 - 1), (251, 252), (far, far + 199), (0, 0)]
    q = rng.normal(size=(len(spans), H * QK)).astype(np.float32)
    _check(ctx, g, blk, nb, *zip(*spans), q, quant, True)


def test_nan_query_stays_with_its_head(ctx):
    """A NaN in one head's query makes that head's output NaN, no other's."""
    rng = np.random.default_rng(6)
    g, blk, nb = _block(ctx, rng, 12, 2, 48, 64, 64)
    for quant in (False, True):
        q = rng.normal(size=(3, 12 * 48)).astype(np.float32)
        q[1, 7 * 48 + 20] = np.nan
        for shared in (True, False):
            blks = blk if shared else torch.cat([blk] * 3)
            out = host(nd.attend_step_i8(ctx, g, blks, 0 if shared else nb, dev(np.zeros(3, np.int32)),
                                         dev(np.full(3, 63, np.int32)), dev(q), quant_query=quant))
            bad = np.isnan(out.reshape(3, 12, 64)).all(-1)
            assert bad[1, 7] and bad.sum() == 1 and np.isnan(out).sum() == 64


@pytest.mark.parametrize("H,KVH,QK", [(12, 2, 48), (8, 4, 64)])
@pytest.mark.parametrize("shared", [False, True])
def test_quantised_query_of_subnormal_scale(ctx, shared, H, KVH, QK):
    """Heads whose absmax / 127 is subnormal, so that its inverse is infinite:
    every nonzero element has a code and the head is finite; a zero element
    (0 * inf) makes its head NaN, no other; a scale that rounds to zero is a
    query of zeros."""
    rng = np.random.default_rng(QK + shared)
    n = 5
    g, blk, nb = _block(ctx, rng, H, KVH, QK, 64, 64, 1 if shared else n)
    q = rng.uniform(0.2, 1.0, (n, H, QK)) * rng.choice([-1.0, 1.0], (n, H, QK))
    q[0] *= 1e-38
    q[1] *= 3.6e-37
    q[2, ::2] *= 1e-38
    q[3] *= 1e-38
    q[3, 2, 7] = 0.0
    q[4] *= 5e-44
    q = q.astype(np.float32)
    assert np.count_nonzero(q) == q.size - 1
    _check(ctx, g, blk, nb, [0, 3, 0, 31, 10], [63, 40, 31, 63, 10], q.reshape(n, -1), True, shared)


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("k_size,q_size", [(6e36, 1.6e-37), (3e-34, 3e33)])
def test_scores_of_unlike_sizes(ctx, shared, quant, k_size, q_size):
    """Keys near the largest floats against a query near the smallest, and the
    other way round: N(0, 1) scores whose factors lie far from 1, so a product
    of two of the three (dot, K scale, query scale) can overflow, or a small
    query's pieces lose bits, where the reference's order does not."""
    rng = np.random.default_rng(int(quant) + 2 * int(shared))
    n = 5
    g, blk, nb = _block(ctx, rng, 12, 2, 48, 64, 64, 1 if shared else n, k_size=k_size)
    q = (rng.normal(size=(n, 12 * 48)) * q_size).astype(np.float32)
    _check(ctx, g, blk, nb, [0, 3, 0, 31, 10], [63, 40, 31, 63, 10], q, quant, shared)


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("H,KVH,QK", [(12, 2, 48), (16, 2, 64)])
@pytest.mark.parametrize("v_size", [1e-25, 1e-31, 1e-35, 1e-36])
def test_small_values_keep_their_bits(ctx, shared, quant, H, KVH, QK, v_size):
    """The error of N(0, 1) values times their size, down to 1e-36, where the
    oracle's own weights (shares of a V scale, v / 127) are subnormal and its
    results 3e-6 off 64 bits.  Past position 700 the values are N(0, 1): spans of both kinds,
    of one and across the change, beside slots no row reads."""
    rng = np.random.default_rng(QK + int(shared))
    cap = 1000
    spans = [(0, 699), (3, 690), (640, 760), (700, 999), (0, 999), (31, 63), (699, 700), (698, 698)]
    size = np.where(np.arange(cap) < 700, v_size, 1.0)[:, None]
    g, blk, nb = _block(ctx, rng, H, KVH, QK, cap, cap, 1 if shared else len(spans), v_size=size)
    q = rng.normal(size=(len(spans), H * QK)).astype(np.float32)
    lo, hi = zip(*spans)
    _check(ctx, g, blk, nb, lo, hi, q, quant, shared, TOL * np.array([v_size if h < 700 else 1.0 for h in hi]))
