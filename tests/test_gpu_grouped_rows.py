"""GroupedBP at the sizes where its waves, workgroups (8192 elements) and scan
groups (256 workgroups) end, with inputs that start off a 16-byte line, NaN
and infinities, and an exponent below the data's (magnitudes past the top
plane): streams and progressive decodes bit-exact against the oracle."""
import numpy as np
import pytest
import torch

import oracle_bind as ob
from test_gpu_bitplane import TD, bits, make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,nb", [(np.float32, 32), (np.float32, 7), (np.float64, 64), (np.float64, 33)])
@pytest.mark.parametrize("n,shift,low,odd", [(2047, 0, 0, False), (2048, 1, 0, True), (2049, 0, 3, False),
                                             (8191, 3, 0, True), (8193, 0, 2, True), (16385, 1, 0, False),
                                             (256 * 8192 + 65, 0, 0, False), (513 * 8192 + 1, 1, 1, False)])
def test_grouped_edges(gpu, dt, nb, n, shift, low, odd):
    from prodm_amd import mdr
    x = make_data(n, dt, 31 + n, zeros=0.2)
    x[n // 2:n // 2 + 300] = 0  # whole blocks without a word
    e = ob.frexp_exp(ob.maxabs(x), dt) - low
    if odd:
        x[[n // 3, n - 1]] = np.nan
        x[n // 5] = -np.inf
    full = torch.zeros(n + shift, dtype=TD[dt], device=gpu)
    full[shift:] = torch.from_numpy(x).to(gpu)
    rb, planes, words = mdr.grouped_encode(full[shift:], e, nb)
    got = mdr.grouped_streams(rb, planes, words, TD[dt])
    ref = ob.gb_encode(x, e, nb)
    for p in range(nb):
        assert got[p] == ref[p], f"plane {p}"
    dev = [torch.frombuffer(bytearray(s) if s else bytearray(8), dtype=torch.uint8).to(gpu) for s in ref]
    dec, odec = mdr.GroupedDecoder(TD[dt]), ob.GBDecoder(dt)
    start = 0
    for k in (1, nb // 2, nb - 1 - nb // 2):
        g = dec.decode(0, dev[start:start + k], n, e, start, k).cpu().numpy()
        o = odec.decode(0, ref[start:start + k], n, e, start, k)
        assert np.array_equal(bits(g), bits(o)), (start, k)
        start += k
    dec.close()
