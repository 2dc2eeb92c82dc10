"""The adjoint of boxes that it copies before it writes: input and output that
share memory (shifted by some elements, or side by side in one array), rows
that lie 1 GiB apart. The same values as from arrays of their own."""
import ctypes as C

import pytest
import torch

from prodm_amd import capi, mdr

pytestmark = pytest.mark.gpu

CASES = [([65], 3), ([9, 65], 2), ([17, 9, 137], 3), ([33, 65, 65], 4), ([5, 6, 70], 0)]


def adjoint(g, out, dims, L, strides=None):
    lib, u32 = capi.lib(), C.c_uint32 * len(dims)
    ws = torch.empty(lib.prodm_recompose_adjoint_workspace_bytes(u32(*dims), len(dims), L), dtype=torch.uint8, device=g.device)
    fn = lib.prodm_recompose_adjoint_f32 if g.dtype == torch.float32 else lib.prodm_recompose_adjoint_f64
    capi.check(fn(g.data_ptr(), out.data_ptr(), u32(*dims), len(dims), L, u32(*strides) if strides else None,
                  ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "adjoint")
    torch.cuda.synchronize()


def field(dims, dt, gpu):
    n = 1
    for d in dims:
        n *= d
    gen = torch.Generator(device=gpu)
    gen.manual_seed(n)
    return torch.randn(n, dtype=dt, device=gpu, generator=gen)


@pytest.mark.parametrize("dims,L", CASES)
@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
@pytest.mark.parametrize("shift", [1, -1, 64, -30])
def test_shifted(gpu, dims, L, dt, shift):
    g = field(dims, dt, gpu)
    want = mdr.recompose_adjoint(g, dims, L)
    buf = torch.zeros(g.numel() + abs(shift), dtype=dt, device=gpu)
    a, b = max(0, -shift), max(0, shift)
    src, out = buf[a:a + g.numel()], buf[b:b + g.numel()]
    src.copy_(g)
    adjoint(src, out, dims, L)
    assert torch.equal(out, want)


@pytest.mark.parametrize("dims,L", [c for c in CASES if len(c[0]) > 1])
def test_side_by_side(gpu, dims, L):
    g = field(dims, torch.float32, gpu)
    want = mdr.recompose_adjoint(g, dims, L)
    full = list(dims[:-1]) + [2 * dims[-1]]
    st = [1] * len(dims)
    for d in range(len(dims) - 2, -1, -1):
        st[d] = st[d + 1] * full[d + 1]
    both = torch.zeros(full, device=gpu)
    src, out = both[..., :dims[-1]], both[..., dims[-1]:]
    src.copy_(g.view(dims))
    adjoint(src, out, dims, L, st)
    assert torch.equal(out.reshape(-1), want) and torch.equal(src.reshape(-1), g)


def test_rows_far_apart(gpu):
    dims, st = [3, 3, 65], [3 << 28, 1 << 28, 1]
    g = field(dims, torch.float32, gpu)
    want = mdr.recompose_adjoint(g, dims, 1)
    n = 2 * st[0] + 2 * st[1] + dims[2]
    src, out = (torch.empty(n, device=gpu) for _ in range(2))
    src.as_strided(dims, st).copy_(g.view(dims))
    adjoint(src, out, dims, 1, st)
    assert torch.equal(out.as_strided(dims, st).reshape(-1), want)
