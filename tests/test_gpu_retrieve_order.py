"""Retrieves of plans with levels between the small ones and a large finest one,
whose decodes wait for the finest's: eager and captured calls, other plane
counts in turn, against the per-level launches on one stream."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,L,dt", [([8193, 8193], 8, torch.float32), ([513, 513, 257], 6, torch.float64)])
def test_finest_first(gpu, dims, L, dt):
    from prodm_amd import mdr
    nb = 32 if dt == torch.float32 else 64
    gen = torch.Generator(device=gpu)
    gen.manual_seed(3)
    n = 1
    for d in dims:
        n *= d
    x = torch.randn(n, dtype=dt, device=gpu, generator=gen)
    plan = mdr.Plan(dims, L, nb, dt)
    ks = [[nb] * (L + 1), [nb // 2 + l % 3 for l in range(L + 1)], [0] * L + [nb // 4]]
    plan.refactor(x)
    plan.profile(True)
    want = [plan.retrieve(k).clone() for k in ks]
    plan.profile(False)
    stream, out = torch.cuda.Stream(), torch.empty_like(x)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(2):
            for k, w in zip(ks, want):
                assert torch.equal(plan.retrieve(k), w)
                for _ in range(2):
                    out.zero_()
                    plan.retrieve_graph(k, out)
                    assert torch.equal(out, w)
    plan.close()
