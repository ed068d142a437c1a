"""The activation quantiser on rows of odd length and rows that start at any
4-byte boundary, at the lengths where its width changes: every i8 value, scale
and row sum equals the oracle's, and nothing is written past a row."""
import numpy as np
import pytest
import torch

import oracle
import xtern

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("mode", [xtern.XT_QUANT_AVX512, xtern.XT_QUANT_SCALAR])
@pytest.mark.parametrize("M,K,shift", [(3, 4, 1), (3, 5, 0), (2, 17, 3), (3, 1023, 0), (2, 1027, 1), (2, 2049, 0),
                                       (3, 2051, 2), (2, 4099, 0), (2, 8191, 1), (2, 8196, 1), (2, 16383, 0),
                                       (2, 16384, 1), (40, 1003, 0)])
def test_quantize_any_row(M, K, shift, mode):
    print(f"[case] quantize M={M} K={K} shift={shift} mode={mode}", flush=True)
    rng = np.random.default_rng(K + shift)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[0] = np.round(x[0] * 4) / 4       # ties at scale 4
    x[0, K - 1] = 127.0 / 4             # the maximum in the last element
    x[1] = 0.0
    buf = torch.zeros(M * K + shift, device=DEV)
    buf[shift:] = torch.from_numpy(x.ravel()).to(DEV)
    q = torch.full((M * K + 8,), 99, dtype=torch.int8, device=DEV)
    inv = torch.empty(M, device=DEV)
    rs = torch.empty(M, dtype=torch.int32, device=DEV)
    lib = xtern.lib()
    rc = lib.xt_quantize_i8_rowsum(buf[shift:].data_ptr(), M, K, q.data_ptr(), inv.data_ptr(), rs.data_ptr(), mode,
                                   torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    got, gi, gr = q.cpu().numpy(), inv.cpu().numpy(), rs.cpu().numpy()
    assert (got[M * K:] == 99).all()
    for m in range(M):
        qo, io = oracle.quantize(x[m], mode)
        assert np.array_equal(got[m * K:(m + 1) * K], qo)
        assert gi[m].view(np.int32) == np.float32(io).view(np.int32)
        assert gr[m] == int(qo.astype(np.int64).sum())
