"""What the encoders return does not depend on what the allocator hands out:
buffers taken from memory full of ones give the same planes, pad words (zero),
recording planes and word counts as buffers from cleared memory."""
import pytest
import torch

from prodm_amd import mdr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,nb", [(torch.float32, 32), (torch.float32, 6), (torch.float64, 64)])
@pytest.mark.parametrize("n", [1, 32, 33, 65, 8192 * 3 + 5, 1 << 20, (1 << 20) + 33])
def test_encoders_write_what_they_return(gpu, dt, nb, n):
    x = torch.sin(torch.arange(n, device=gpu, dtype=torch.float64) * 0.37).to(dt)
    got = []
    for fill in (-1, 0):
        blocks = [torch.full((s,), fill, dtype=torch.int32, device=gpu) for s in (1 << 8, 1 << 16, 1 << 23)]
        del blocks  # the next allocations come from these
        got.append([mdr.negabinary_encode(x, 1, nb), *mdr.grouped_encode(x, 1, nb)])
    torch.cuda.synchronize()
    for a, b in zip(*got):
        assert torch.equal(a, b)
    nw = -(-n // (32 if dt == torch.float32 else 64))
    assert not got[0][0][:, nw:].any()
