"""Levels of a plan that are launched together (up to 2^21 elements each, 16 of
them) against the same plan with every level launched by itself, as it is with
stage timing on: the same kernel bodies, so planes, coefficients and fields
agree bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,L", [
    ([1, 1], 2),            # levels without elements
    ([9, 9, 9], 0),
    ([3], 1),
    ([65, 33, 1], 3),
    ([2 ** 18 + 1], 18),    # small levels past the largest set
    ([129, 65, 65], 3),
    ([161, 129, 129], 4),   # a larger finest level
    ([2897, 2897], 1),      # no small level
    ([3585, 3201], 3),      # two larger levels
])
@pytest.mark.parametrize("enc,dt", [(0, torch.float32), (0, torch.float64), (1, torch.float32), (1, torch.float64),
                                    (2, torch.float32)])
@pytest.mark.parametrize("hier", [0, 1])
def test_sets_match_single_levels(gpu, dims, L, enc, dt, hier):
    from prodm_amd import capi, mdr
    nb = 32 if dt == torch.float32 else 64
    n = int(np.prod(dims))
    gen = torch.Generator(device=gpu).manual_seed(5)
    x = torch.sin(torch.arange(n, device=gpu, dtype=torch.float64) * 0.013)
    x = (x + 1e-3 * torch.randn(n, device=gpu, dtype=torch.float64, generator=gen)).to(dt)
    a, b = (mdr.Plan(dims, L, nb, dt, enc, hier) for _ in range(2))
    b.profile(True)
    if np.prod(dims) == 1:
        # a level without elements has no planes; its retrieve from loaded
        # level bounds (no planes read) is a field of zeros
        for p in (a, b):
            with pytest.raises(capi.ProdmError):
                p.refactor(x)
            p.set_level_max(0, 1.0)
            assert not p.retrieve([0] * (L + 1)).any()
            p.close()
        return
    a.refactor(x)
    b.refactor(x)
    for l in range(L + 1):
        assert a.level_info(l) == b.level_info(l)
        assert torch.equal(a.coefficients(l), b.coefficients(l)), l
        for p in (0, nb // 2, nb - 1):
            assert a.plane_stream(l, p) == b.plane_stream(l, p), (l, p)
    pick = np.random.default_rng(7)
    for ks in ([nb] * (L + 1), [int(k) for k in pick.integers(0, nb + 1, L + 1)], [0] * (L + 1)):
        u, v = a.retrieve(ks).clone(), b.retrieve(ks).clone()
        torch.cuda.synchronize()
        assert torch.equal(u.view(torch.uint8), v.view(torch.uint8)), ks
    if enc < 2:
        # captured: replays against the eager field, eager work between them
        side = torch.cuda.Stream()
        ks = [nb - 2] * (L + 1)
        want = a.retrieve(ks).clone()
        out = torch.empty_like(want)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(3):
                a.refactor_graph(x)
                a.retrieve_graph(ks, out)
                torch.cuda.synchronize()
                assert torch.equal(out.view(torch.uint8), want.view(torch.uint8))
                out.zero_()
                a.refactor(x * 0)
    a.close()
    b.close()
