"""PerBit sign insertion: runs of 32 elements whose first 1 bits meet in one
plane (none, the edges of the word, all of them), byte for byte against the
oracle."""
import numpy as np
import pytest
import torch

import oracle_bind as ob
from prodm_amd import mdr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("sign", [1, -1, 0])
def test_perbit_flags_of_one_plane(gpu, dt, sign):
    nb = 8 * np.dtype(dt).itemsize
    rng = np.random.default_rng(3)
    masks = [0, 1, 1 << 31, (1 << 31) | 1, 3 << 30, 0xFFFFFFFF, 0x55555555, 0xAAAAAAAA, 0x7FFFFFFF]
    masks += [int(m) for m in rng.integers(0, 1 << 32, 70)]
    flag = np.array([[m >> j & 1 for j in range(32)] for m in masks], bool).reshape(-1)
    s = rng.choice([-1.0, 1.0], flag.size) if sign == 0 else float(sign)
    # flagged elements start in plane 1, the others in planes 2 to 9
    mag = np.where(flag, rng.uniform(0.25, 0.5, flag.size), rng.uniform(0.001, 0.25, flag.size))
    x = (mag * s).astype(dt)
    x[-1] = 0.75  # the level's exponent, 0
    streams, sizes = mdr.perbit_encode(torch.from_numpy(x).cuda(), 0, nb, True)
    torch.cuda.synchronize()
    mine, ref = mdr.perbit_streams(streams, sizes), ob.pb_encode(x, 0, nb)
    assert [len(r) for r in ref] == list(sizes.cpu().numpy())
    for p in range(nb):
        assert mine[p] == ref[p], p
