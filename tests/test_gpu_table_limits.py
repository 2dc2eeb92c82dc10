"""Error tables at the limits of float: elements whose squares are past the
largest float, elements above the level maximum or exponent that the caller
gives, infinities and NaN. Bit-exact against the oracle, where it defines the
table, else against the terms summed by math.fsum."""
import math

import numpy as np
import pytest
import torch

import oracle_bind as ob
from test_gpu_exact_tables import spread

pytestmark = pytest.mark.gpu


def squared_terms(x, nb, m):
    """the table's terms element by element (entries 0..nb), exactly rounded sums"""
    le = math.frexp(m)[1]
    bins = [[] for _ in range(nb + 1)]
    for v in x[np.isfinite(x) & (x != 0)]:
        diff = le - math.frexp(float(v))[1] + 23 - nb
        low, index = (diff, nb) if diff > 0 else (0, nb + diff)
        if index <= 0:
            continue
        for k in range(index + 1):
            b = low + index - k  # mantissa bits 0..b are cleared, all of x past bit 22
            keep = np.uint32((0xffffffff << (b + 1)) & 0xffffffff) if b < 23 else np.uint32(0)
            d = np.float32(v - (np.float32(v).view(np.uint32) & keep).view(np.float32)) if b < 23 else v
            with np.errstate(over="ignore"):
                bins[k].append(min(float(d * d), 2.0 ** 128))  # as an infinite square counts
    return np.array([math.fsum(t) for t in bins])


# an infinite square counts as 2^128 in the oracle (the bit pattern read as a number)
@pytest.mark.parametrize("scale", [63, 64, 69, 95, 96, 97, 110, 126])
@pytest.mark.parametrize("n,nb,low", [(1, 32, 0), (3, 32, 0), (8193, 32, 20), (20000, 32, 80), (20000, 1, 30), (20000, 9, 100)])
def test_squares_past_float(gpu, n, nb, low, scale):
    from prodm_amd import mdr
    x = spread(n, 11 * n + nb, low, scale)
    m = ob.maxabs(x)
    want = ob.collect_squared(x, nb, m)
    assert np.array_equal(mdr.collect_squared(torch.from_numpy(x).to(gpu), nb, m), want)


def test_largest_float(gpu):
    from prodm_amd import mdr
    x = spread(9000, 4, 140, 127 - 6)
    x[::7] = np.finfo(np.float32).max
    m = ob.maxabs(x)
    assert np.array_equal(mdr.collect_squared(torch.from_numpy(x).to(gpu), 32, m), ob.collect_squared(x, 32, m))


def test_terms_restatement():
    """the restatement used below agrees with the oracle where both hold"""
    for x in (spread(500, 2, 60), spread(500, 2, 60, 100)):
        nb = 32
        assert np.array_equal(squared_terms(x, nb, ob.maxabs(x)), ob.collect_squared(x, nb, ob.maxabs(x)))
    x = spread(500, 2, 60)
    for nb in (1, 8, 23, 24):
        assert np.array_equal(squared_terms(x, nb, ob.maxabs(x)), ob.collect_squared(x, nb, ob.maxabs(x)))


@pytest.mark.parametrize("nb", [1, 8, 23, 32])
@pytest.mark.parametrize("n,low,down", [(700, 0, 2), (3000, 40, 3), (3000, 10, 30)])
def test_squared_above_the_maximum(gpu, n, nb, low, down):
    from prodm_amd import mdr
    x = spread(n, n + nb, low)
    m = math.ldexp(ob.maxabs(x), -down)
    assert np.array_equal(mdr.collect_squared(torch.from_numpy(x).to(gpu), nb, m), squared_terms(x, nb, m))


@pytest.mark.parametrize("enc,nb", [(0, 32), (0, 9), (1, 24), (1, 9)])
@pytest.mark.parametrize("n,low,down", [(700, 0, 2), (8193, 40, 3), (20000, 100, 1)])
def test_encoder_above_the_exponent(gpu, enc, nb, n, low, down):
    from prodm_amd import mdr
    x = spread(n, n + nb + enc, low)
    e = ob.frexp_exp(ob.maxabs(x), np.float32) - down
    got = mdr.level_errors(torch.from_numpy(x).to(gpu), e, nb, enc)
    assert np.array_equal(got, ob.fused_level_errors(x, e, nb, "nb" if enc == 0 else "gb", mode="exact"))


@pytest.mark.parametrize("n,low", [(5, 0), (8193, 30), (20000, 100)])
def test_infinities_and_nan_are_left_out(gpu, n, low):
    from prodm_amd import mdr
    x = spread(n, n + 17, low)
    m, e = ob.maxabs(x), ob.frexp_exp(ob.maxabs(x), np.float32)
    bad = x.copy()
    bad[[0, n - 1]] = np.nan
    bad[n // 3] = np.inf
    bad[n // 4] = -np.inf
    zeroed = np.where(np.isfinite(bad), bad, np.float32(0))
    d = torch.from_numpy(bad).to(gpu)
    for nb in (7, 32):
        assert np.array_equal(mdr.collect_squared(d, nb, m), ob.collect_squared(zeroed, nb, m))
        for enc in (0, 1):
            want = ob.fused_level_errors(zeroed, e, nb, "nb" if enc == 0 else "gb", mode="exact")
            assert np.array_equal(mdr.level_errors(d, e, nb, enc), want)


@pytest.mark.parametrize("enc,nb", [(0, 32), (1, 32), (1, 31), (1, 5)])
@pytest.mark.parametrize("n", [1, 8193, 70001])
@pytest.mark.parametrize("lo,width", [(0.5, 0.5), (270.0, 60.0), (4294967040.0, 0.0), (2.0 ** 31, 2.0 ** 31 - 256)])
def test_encoder_top_binade(gpu, enc, nb, n, lo, width):
    """every element's top digit set"""
    from prodm_amd import mdr
    x = (lo + width * np.random.default_rng(n).random(n)).astype(np.float32)
    x[::3] *= -1
    e = ob.frexp_exp(ob.maxabs(x), np.float32)
    got = mdr.level_errors(torch.from_numpy(x).to(gpu), e, nb, enc)
    assert np.array_equal(got, ob.fused_level_errors(x, e, nb, "nb" if enc == 0 else "gb", mode="exact"))


@pytest.mark.parametrize("scale", [0, -145, 70])
def test_squared_many_above_the_maximum(gpu, scale):
    """a whole wave's elements past the bound, spread over more exponents than the window holds"""
    from prodm_amd import mdr
    x = spread(9000, 21, 0, scale)
    x[:2048] *= np.exp2(np.random.default_rng(4).integers(0, 40 if scale < 60 else 1, 2048)).astype(np.float32)
    m = math.ldexp(1.0, scale - 2)
    assert np.array_equal(mdr.collect_squared(torch.from_numpy(x).to(gpu), 32, m), squared_terms(x, 32, m))
