"""The host PerBit decoder where its 64-element groups, thread pipeline (from
4096 group planes) and windows (2^14 groups) end, against the oracle bit for
bit: remainders of every kind, dense and sparse signs, progressive calls,
scales past the normal range, and streams one word short."""
import numpy as np
import pytest
import torch

import oracle_bind as ob
from prodm_amd import capi, mdr
from test_host_perbit import TD, field, level_exp


@pytest.mark.parametrize("dt,nb,n,steps,scale", [
    (np.float32, 32, 63, [32], 0), (np.float32, 32, 64, [1, 31], 0), (np.float32, 31, 65, [31], 0),
    (np.float32, 32, 8191, [32], 0), (np.float32, 32, 8193, [5, 27], 0), (np.float64, 64, 9000, [64], 0),
    (np.float32, 32, 100003, [2, 30], 0), (np.float64, 50, 70001, [1, 49], 0), (np.float32, 8, 2 ** 20 + 65, [8], 0),
    (np.float32, 32, 9001, [16, 16], -130), (np.float64, 64, 9001, [64], -1000),
])
def test_groups(dt, nb, n, steps, scale):
    x = np.ldexp(field(n, dt, nb + n), scale).astype(dt)
    x[n // 4:n // 2] = np.abs(x[n // 4:n // 2]) + np.ldexp(dt(0.5), scale)  # a run whose first 1 bits fall together
    e = level_exp(x)
    streams = ob.pb_encode(x, e, nb)
    mine, ref = mdr.PerBitDecoder(TD[dt]), ob.PBDecoder(dt)
    start = 0
    for k in steps:
        a = mine.decode(1, streams[start:start + k], n, e, start, k)
        b = ref.decode(1, streams[start:start + k], n, e, start, k)
        assert a.tobytes() == b.tobytes(), (start, k)
        start += k
    mine.close()


def test_short_stream_in_threads():
    n, nb = 20001, 32
    x = field(n, np.float32, 5)
    e = level_exp(x)
    streams = list(ob.pb_encode(x, e, nb))
    streams[17] = streams[17][:-8]
    dec = mdr.PerBitDecoder(torch.float32)
    with pytest.raises(capi.ProdmError, match="stream 17 is shorter"):
        dec.decode(0, streams, n, e, 0, nb)
    dec.close()
