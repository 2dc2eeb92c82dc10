"""GroupedBP where the summing of rows by the workgroups themselves ends (768
workgroups of 8192 elements): streams and progressive decodes against the
oracle on both sides of it."""
import numpy as np
import pytest
import torch

import oracle_bind as ob
from test_gpu_bitplane import TD, bits, make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,nb", [(np.float32, 32), (np.float64, 41)])
@pytest.mark.parametrize("n", [768 * 8192, 768 * 8192 + 1, 300 * 8192 - 77])
def test_both_sides(gpu, dt, nb, n):
    from prodm_amd import mdr
    x = make_data(n, dt, n, zeros=0.2)
    x[n // 2:n // 2 + 30000] = 0
    e = ob.frexp_exp(ob.maxabs(x), dt)
    rb, planes, words = mdr.grouped_encode(torch.from_numpy(x).to(gpu), e, nb)
    got = mdr.grouped_streams(rb, planes, words, TD[dt])
    ref = ob.gb_encode(x, e, nb)
    assert all(g == r for g, r in zip(got, ref))
    dev = [torch.frombuffer(bytearray(s) if s else bytearray(8), dtype=torch.uint8).to(gpu) for s in ref]
    dec, odec = mdr.GroupedDecoder(TD[dt]), ob.GBDecoder(dt)
    start = 0
    for k in (2, nb - 9, 7):
        g = dec.decode(0, dev[start:start + k], n, e, start, k).cpu().numpy()
        o = odec.decode(0, ref[start:start + k], n, e, start, k)
        assert np.array_equal(bits(g), bits(o)), (start, k)
        start += k
    dec.close()
