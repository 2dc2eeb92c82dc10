"""The adjoint against the oracle where its 8 x 8 x 64 tiles end: extents at and
one step past a tile along each dim, inactive dims, 3-node dims (both ends in
one stencil), boxes inside a larger array."""
import numpy as np
import pytest
import torch

import oracle_bind as ob

pytestmark = pytest.mark.gpu

TD = {np.float32: torch.float32, np.float64: torch.float64}


@pytest.mark.parametrize("dims,L", [([3, 3, 3], 1), ([7, 9, 63], 1), ([9, 7, 65], 1), ([17, 17, 129], 2), ([15, 3, 131], 1),
                                    ([65], 3), ([127], 1), ([9, 65], 2), ([1, 17, 67], 1), ([17, 1, 33], 2),
                                    ([33, 17, 1], 2)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_adjoint_tiles(gpu, dims, L, dt):
    from prodm_amd import mdr
    rng = np.random.default_rng(sum(dims) + L)
    g = rng.standard_normal(int(np.prod(dims))).astype(dt)
    ref = ob.recompose_adjoint(g.astype(np.float64), dims, L)
    # float32: the FP64 result rounded once; float64: some 100 roundings of FP64 through the solves
    tol = (2.0 ** -23 if dt == np.float32 else 1e-13) * max(1.0, float(np.max(np.abs(ref))))
    got = mdr.recompose_adjoint(torch.from_numpy(g).to(gpu), dims, L).cpu().numpy()
    assert np.max(np.abs(got.astype(np.float64) - ref)) <= tol
    if len(dims) == 3:
        # the same box inside a larger array
        full = [dims[0] + 1, dims[1] + 2, dims[2] + 3]
        st = [full[1] * full[2], full[2], 1]
        big = torch.zeros(full, dtype=TD[dt], device=gpu)
        big[:dims[0], :dims[1], :dims[2]] = torch.from_numpy(g.reshape(dims)).to(gpu)
        box = mdr.recompose_adjoint(big, dims, L, strides=st)[:dims[0], :dims[1], :dims[2]]
        assert np.array_equal(box.cpu().numpy().ravel(), got)
