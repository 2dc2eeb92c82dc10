"""GroupedBP streams that lie at any byte of a larger buffer, as slices of a
file's bytes do: the same values as from buffers of their own."""
import numpy as np
import pytest
import torch

import oracle_bind as ob
from test_gpu_bitplane import TD, bits, make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,nb", [(np.float32, 32), (np.float64, 64)])
@pytest.mark.parametrize("n", [33, 2049, 8192 * 3 + 5])
@pytest.mark.parametrize("off", [1, 2, 3, 4, 7])
def test_streams_at_any_byte(gpu, dt, nb, n, off):
    from prodm_amd import mdr
    x = make_data(n, dt, 7 + n + off, zeros=0.1)
    e = ob.frexp_exp(ob.maxabs(x), dt)
    ref = ob.gb_encode(x, e, nb)
    at, blob = [], bytearray(off)
    for s in ref:
        at.append(len(blob))
        blob += s + bytes(1 + len(at) % 3)
    file = torch.frombuffer(blob + bytes(64), dtype=torch.uint8).to(gpu)
    dev = [file[a:a + len(s)] for a, s in zip(at, ref)]
    dec, odec = mdr.GroupedDecoder(TD[dt]), ob.GBDecoder(dt)
    start = 0
    for k in (3, nb // 2, nb - 3 - nb // 2):
        g = dec.decode(0, dev[start:start + k], n, e, start, k).cpu().numpy()
        o = odec.decode(0, ref[start:start + k], n, e, start, k)
        assert np.array_equal(bits(g), bits(o)), (start, k)
        start += k
    dec.close()
