"""The vector quantizers over rows that start at any address and end off 8 columns: bit-exact
with the oracle, and nothing written past the last row (guard bytes)."""
import numpy as np
import pytest
import torch

from gpu_util import host
from test_oracle import same_bits

pytestmark = pytest.mark.gpu
F16, F32 = torch.float16, torch.float32


def _data(rows, k, seed):
    x = np.random.default_rng(seed).normal(0, 1, (rows, k)).astype(np.float32)
    x[0, 0], x[-1, -1] = np.nan, 9.0
    if rows > 2:
        x[1] = 0
    return x


# one step, a step and a remainder, every thread count of the dispatch on both sides of 256 rows
@pytest.mark.parametrize("xdt", [F32, F16])
@pytest.mark.parametrize("m,k", [(3, 8), (3, 9), (5, 15), (1, 7), (300, 1003), (257, 2049), (256, 6151), (260, 8955),
                                 (256, 12301), (17, 2047), (16, 8955), (4, 16391), (3, 24579), (2, 40003), (2, 65535)])
def test_act_quant_any(dev, nq, orc, m, k, xdt):
    from nanoinfer_amd import _lib
    buf = torch.empty(m * k + 1, dtype=xdt, device=dev)
    x = buf[1:].view(m, k)  # off 16-byte alignment
    x.copy_(torch.from_numpy(_data(m, k, m + k)))
    q, s = orc.act_quant(host(x.float()))
    out = torch.full((m * k + 16,), 85, dtype=torch.int8, device=dev)
    sc = torch.empty(m, device=dev)
    _lib.check(_lib.load().nq_act_quant_i8(x.data_ptr(), 1 if xdt == F16 else 0, m, k, out.data_ptr() + 3, sc.data_ptr(),
                                           torch.cuda.current_stream().cuda_stream))
    assert same_bits(host(out[3:3 + m * k].view(m, k)), q) and same_bits(host(sc), s)
    assert bool((out[:3] == 85).all()) and bool((out[3 + m * k:] == 85).all())


@pytest.mark.parametrize("group", [8, 16, 32, 64, 128, 256, 512])
@pytest.mark.parametrize("n,k", [(1, 1), (3, 7), (5, 8), (4, 33), (9, 259), (7, 1003), (3, 2054)])
def test_quantize_q4g_any(dev, nq, orc, n, k, group):
    from nanoinfer_amd import _lib
    w = _data(n, k, n * k + group)
    q, s = orc.quantize_q4g(w, group)
    buf = torch.empty(n * k + 1, device=dev)
    wd = buf[1:].view(n, k)
    wd.copy_(torch.from_numpy(w))
    rb, nb = (k + 1) // 2, (k + group - 1) // group
    for sdt, code in ((F32, 0), (F16, 1)):
        out = torch.full((n * rb + 8,), 0x55, dtype=torch.uint8, device=dev)
        sc = torch.empty((n, nb), dtype=sdt, device=dev)
        _lib.check(_lib.load().nq_quantize_q4g(wd.data_ptr(), n, k, group, out.data_ptr() + 1, sc.data_ptr(), code,
                                               torch.cuda.current_stream().cuda_stream))
        assert same_bits(host(out[1:1 + n * rb].view(n, rb)), q)
        assert same_bits(host(sc), s.astype(np.float16) if sdt == F16 else s)
        assert int(out[0]) == 0x55 and bool((out[1 + n * rb:] == 0x55).all())
