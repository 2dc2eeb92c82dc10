"""Error tables (exactly rounded sums) where the FP64 accumulators' ranges end:
chunks of 8192 elements, several chunks per workgroup, elements far below the
last plane (summed once for every entry), subnormal data, an exponent below the
data's, infinities and NaN left out as before. Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

import oracle_bind as ob

pytestmark = pytest.mark.gpu


def spread(n, seed, low, scale=0):
    """magnitudes over 2^-low .. 1, times 2^scale, some zero"""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(n) * np.exp2(rng.uniform(-low, 0, n))
    x[rng.random(n) < 0.1] = 0
    x[n // 2] = 1.9
    return np.ldexp(x, scale).astype(np.float32)


CASES = [(1, 32, 0, 0), (8191, 32, 20, 0), (8193, 16, 40, 0), (24593, 32, 100, 0), (24593, 1, 30, 0), (65537, 8, 60, 3),
         (20000, 32, 60, -100), (20000, 24, 30, -140), (20000, 32, 20, 60), (500003, 31, 34, 0)]


@pytest.mark.parametrize("n,nb,low,scale", CASES)
def test_squared(gpu, n, nb, low, scale):
    from prodm_amd import mdr
    x = spread(n, 5 * n + nb, low, scale)
    m = ob.maxabs(x)
    assert np.array_equal(mdr.collect_squared(torch.from_numpy(x).to(gpu), nb, m), ob.collect_squared(x, nb, m))


@pytest.mark.parametrize("enc", [0, 1])
@pytest.mark.parametrize("n,nb,low,scale", CASES)
def test_encoder(gpu, enc, n, nb, low, scale):
    from prodm_amd import mdr
    x = spread(n, 7 * n + nb, low, scale)
    e = ob.frexp_exp(ob.maxabs(x), np.float32)
    got = mdr.level_errors(torch.from_numpy(x).to(gpu), e, nb, enc)
    assert np.array_equal(got, ob.fused_level_errors(x, e, nb, "nb" if enc == 0 else "gb", mode="exact"))


def test_chunks_per_workgroup(gpu):
    """more than 2048 chunks of 8192: several per workgroup"""
    from prodm_amd import mdr
    n, nb = 2050 * 8192 + 3, 4
    x = spread(n, 3, 24)
    m, e = ob.maxabs(x), ob.frexp_exp(ob.maxabs(x), np.float32)
    d = torch.from_numpy(x).to(gpu)
    assert np.array_equal(mdr.collect_squared(d, nb, m), ob.collect_squared(x, nb, m))
    assert np.array_equal(mdr.level_errors(d, e, nb, 0), ob.fused_level_errors(x, e, nb, "nb", mode="exact"))


@pytest.mark.parametrize("off", [0, 1])
def test_misaligned(gpu, off):
    from prodm_amd import mdr
    x = spread(10001, 9, 30)
    full = torch.zeros(x.size + 1, dtype=torch.float32, device=gpu)
    full[off:off + x.size] = torch.from_numpy(x).to(gpu)
    m = ob.maxabs(x)
    assert np.array_equal(mdr.collect_squared(full[off:off + x.size], 32, m), ob.collect_squared(x, 32, m))
