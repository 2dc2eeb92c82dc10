"""maxabs at the ends of its 16-byte loads and workgroups, off a 16-byte line,
with NaN, infinities and zeros, and from several threads at once."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [0, 1, 3, 4, 5, 255, 4096, 4097, 512 * 4096 - 1, 512 * 4096 + 5, 3_000_001])
@pytest.mark.parametrize("shift", [0, 1])
def test_maxabs(gpu, dt, n, shift):
    from prodm_amd import mdr
    rng = np.random.default_rng(n + shift)
    x = rng.standard_normal(n + shift).astype(dt)
    if n:
        x[shift + n - 1] = -9.5
    if n > 4:
        x[shift + n // 2] = np.nan
    d = torch.from_numpy(x).to(gpu)[shift:]
    assert mdr.maxabs(d) == (float(np.nanmax(np.abs(x[shift:]))) if n else 0.0)
    if n > 4:
        d[2] = float("-inf")
        assert mdr.maxabs(d) == float("inf")
    if n:
        assert mdr.maxabs(torch.zeros_like(d)) == 0.0


def test_threads(gpu):
    from prodm_amd import mdr
    xs = [torch.full((100_003,), float(i + 1), device=gpu) for i in range(8)]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                if mdr.maxabs(xs[i]) != i + 1:
                    bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
