"""Line solves of long lines against the oracle, at the ends of the classes:
dim 2 of 2048 | 2049 and 18432 | 18433 coarse nodes, dims 1 / 0 of 576 | 577,
1152 | 1153, 2304 | 2305 and 4608 | 4609, with whole and partial groups of lines.
Tolerances as for the other geometries."""
import numpy as np
import pytest
import torch

import oracle_bind as ob
from test_gpu_mgard import TD, TOL, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [[4095], [5, 4097], [16385], [36863], [3, 36865],
                                  [1151, 5], [1153, 35], [1537, 35], [5, 1537, 35], [1537, 5, 33], [2303, 33],
                                  [2305, 35], [4607, 5], [4609, 35], [9215, 5], [9217, 9]])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_long_lines(gpu, dims, dt):
    from prodm_amd import mdr
    rng = np.random.default_rng(len(dims) + dims[0])
    u = (rng.standard_normal(int(np.prod(dims))) + 3.0).astype(dt)
    ref = ob.decompose(u, dims, 1)
    got = mdr.decompose(torch.from_numpy(u).to(gpu), dims, 1).cpu().numpy()
    assert rel(got, ref) <= TOL[dt], rel(got, ref)
    rec = mdr.recompose(torch.from_numpy(ref).to(gpu), dims, 1).cpu().numpy()
    assert rel(rec, ob.recompose(ref, dims, 1)) <= TOL[dt]
    assert rel(rec, u) <= 8 * TOL[dt]
