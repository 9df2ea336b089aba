"""The f16 matrix-core Cactus-Quants matmul at its tile edges, against the
same product in 64 bits.

Tolerance: both operands are carried to 2^-23 of themselves and the cross term
left out is below 2^-22 of the product: 2^-21 of it in all, 8 units of 2^-24, in
the worst case.  A product sum adds at most 96 fp32 roundings in a step of 32
columns' three products and one a step and a group after it; errors of either
sign add as their square root.  16 units of sum |x w| bound every draw here: by
a factor of two where one product makes most of a sum, of ten or more elsewhere.
"""
import numpy as np
import pytest
import torch

import needle_amd as nd
from conftest import dev, host
from cq_cases import TERNARY, levels_for, random_case

pytestmark = pytest.mark.gpu
CB = np.concatenate([np.sort(np.random.default_rng(b).normal(0, 0.1, 1 << b)) for b in (2, 3, 4)]).astype(np.float32)
TOL = 16 * 2.0 ** -24


def _weights64(c):
    lv = levels_for(c.bits, c.group, c.codebook).astype(np.float64)
    u = lv[c.idx].reshape(c.out, c.num_groups, c.group) * c.norms_f32.astype(np.float64)[:, :, None]
    return u.reshape(c.out, c.in_pad)


def _weight(ctx, c):
    return nd.CqWeight(ctx, c.blob, c.out, c.in_feat, c.group, c.bits, c.codebook)


def _check(ctx, c, gw, xh, r0, rows):
    got = host(gw.matmul_rows_prepared(dev(xh), xh.shape[0], r0, rows)).reshape(xh.shape[0], rows)
    w = _weights64(c)[r0:r0 + rows]
    x = xh.astype(np.float64)
    want, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    assert np.all(np.abs(got - want) <= TOL * mag + 1e-37), np.max(np.abs(got - want) / (mag + 1e-300))


@pytest.mark.parametrize("bits", [2, 3, 4, TERNARY])
@pytest.mark.parametrize("out,inn,group,batch,r0,rows", [
    (1, 1, 128, 1, 0, 1), (64, 128, 128, 16, 0, 64), (65, 200, 128, 17, 0, 65), (300, 768, 128, 15, 7, 193),
    (300, 700, 256, 33, 1, 299), (130, 1024, 1024, 65, 0, 130), (520, 512, 512, 9, 3, 517),
    (4100, 384, 128, 130, 0, 4100), (8192, 256, 128, 520, 0, 8192)])
def test_tiles(ctx, bits, out, inn, group, batch, r0, rows):
    """One row to several tiles of every tile shape, ragged in all three."""
    rng = np.random.default_rng(out + inn + bits)
    c = random_case(rng, out, inn, group, bits, CB)
    xh = rng.normal(size=(batch, c.in_pad)).astype(np.float32)
    _check(ctx, c, _weight(ctx, c), xh, r0, rows)


@pytest.mark.parametrize("bits", [2, 3, 4, TERNARY])
def test_scales(ctx, bits):
    """Rows and 128-column groups whose sizes lie from subnormal to the
    largest floats, a wide range within a group, and a zero group."""
    rng = np.random.default_rng(bits)
    c = random_case(rng, 96, 512, 128, bits, CB)
    xh = rng.normal(size=(40, 512)).astype(np.float32)
    scale = np.float32(2.0) ** rng.integers(-140, 118, size=(40, 4, 1)).astype(np.float32)
    xh = (xh.reshape(40, 4, 128) * scale).astype(np.float32)
    xh[:, 1, ::3] *= np.float32(2.0 ** -12)
    xh[5, 2] = 0
    xh = xh.reshape(40, 512)
    # a row with one large group: the small groups vanish beside it in fp32 too
    got = host(_weight(ctx, c).matmul_rows_prepared(dev(xh), 40, 0, 96)).reshape(40, 96)
    w, x = _weights64(c), xh.astype(np.float64)
    want, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    ok = mag < 1e38
    assert np.all(np.abs(got - want)[ok] <= TOL * mag[ok] + 1e-43)


@pytest.mark.parametrize("bits", [2, 3, 4])
def test_not_finite(ctx, bits):
    """An infinity or NaN reaches its own row's outputs and no other's."""
    rng = np.random.default_rng(10 + bits)
    c = random_case(rng, 200, 300, 128, bits, CB)
    xh = rng.normal(size=(70, c.in_pad)).astype(np.float32)
    xh[3, 17], xh[66, 299], xh[20, 5] = np.inf, -np.inf, np.nan
    got = host(_weight(ctx, c).matmul_rows_prepared(dev(xh), 70, 0, 200)).reshape(70, 200)
    w = _weights64(c)
    with np.errstate(invalid="ignore"):
        want = xh.astype(np.float64) @ w.T
    for r in range(70):
        if r == 20:
            assert np.isnan(got[r]).all()
        elif r in (3, 66):
            assert np.array_equal(got[r], want[r].astype(np.float32), equal_nan=True)
        else:
            assert np.all(np.abs(got[r] - want[r]) <= TOL * (np.abs(xh[r]).astype(np.float64) @ np.abs(w).T))


@pytest.mark.parametrize("bits", [2, 3, 4, TERNARY])
@pytest.mark.parametrize("out,inn,group,batch", [(300, 768, 128, 70), (130, 700, 256, 5), (4100, 512, 512, 130),
                                                 (8192, 256, 128, 200)])
def test_rows_that_are_not_finite(ctx, bits, out, inn, group, batch):
    """Infinities of one sign and both, across groups, in the last column, whole
    groups of them, and NaN: the infinities and NaN of the product in 64 bits;
    the finite rows beside them keep their bits."""
    rng = np.random.default_rng(out + bits)
    c = random_case(rng, out, inn, group, bits, CB)
    gw = _weight(ctx, c)
    xh = rng.normal(size=(batch, c.in_pad)).astype(np.float32)
    run = lambda: host(gw.matmul_rows_prepared(dev(xh), batch, 0, out)).reshape(batch, out)
    finite = run()
    last, far = c.in_pad - 1, min(group + 3, c.in_pad - 2)
    xh[0, 7] = np.inf
    xh[1, last] = -np.inf
    xh[2, [5, far]] = np.inf
    xh[3, [5, far]] = np.inf, -np.inf
    xh[4, far] = np.nan
    odd = [0, 1, 2, 3, 4]
    if batch > 5:
        xh[17, :128] = np.where(rng.random(128) < 0.5, np.inf, -np.inf)
        xh[batch - 1, last - 127:] = np.inf
        odd += [17, batch - 1]
    got = run()
    w = _weights64(c)
    with np.errstate(invalid="ignore"):
        want = xh[odd].astype(np.float64)[:, None, :] * w[None] if out * c.in_pad < 300000 else None
        if want is not None:
            want = want.sum(-1)
        else:  # the elements that are not finite decide
            want = np.stack([(xh[r].astype(np.float64)[k] * w[:, k]).sum(-1)
                             for r in odd for k in [~np.isfinite(xh[r])]])
    assert np.array_equal(got[odd], want.astype(np.float32), equal_nan=True)
    rest = np.setdiff1d(np.arange(batch), odd)
    assert np.array_equal(got[rest].view(np.uint32), finite[rest].view(np.uint32))


@pytest.mark.parametrize("bits", [2, 3, 4, TERNARY])
@pytest.mark.parametrize("size", [2.0 ** 10, 2.0 ** 17, 2.0 ** 24, 2.0 ** 31])
def test_one_large_value_in_a_group(ctx, bits, size):
    """A piece ends at 2^-24 where a group's largest activation is 2^14 to
    2^15: an element is carried to 2^-23 of itself or to 2^-39 of its group's
    largest, whichever is more, and it shows where the largest meets a level of
    zero."""
    rng = np.random.default_rng(bits)
    c = random_case(rng, 300, 512, 128, bits, CB)
    xh = rng.normal(size=(40, 512)).astype(np.float32)
    xh[:, [3, 200, 300, 400]] *= np.float32(size)
    got = host(_weight(ctx, c).matmul_rows_prepared(dev(xh), 40, 0, 300)).reshape(40, 300)
    w, x = _weights64(c), xh.astype(np.float64)
    want, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    top = np.abs(x).reshape(40, 4, 128).max(-1)
    floor = top @ np.abs(w).reshape(300, 4, 128).sum(-1).T
    assert np.all(np.abs(got - want) <= TOL * mag + 2.0 ** -39 * floor)
