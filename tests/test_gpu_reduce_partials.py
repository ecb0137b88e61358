"""Sums of K splits (K > 2048) on the GEMV: columns past, at and short of a
workgroup's 1024, columns that are no multiple of 4, outputs not 8-byte
aligned. Against 64-bit products: f16 results of fp32 sums (2^-11 each)."""
import numpy as np
import pytest

import oracle
import synth
from nemo_amd import _lib, runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,shift", [(1, 4, 0), (3, 1024, 0), (17, 1028, 0), (5, 1021, 0), (16, 2052, 1), (160, 128, 0)])
def test_split_sums(torch_cuda, m, n, shift):
    torch = torch_cuda
    k = 4096 + 256
    raw = synth.random_q4k(91 + n, n * k // 256)
    x16 = synth.normal(92 + m, m * k).astype(np.float16).reshape(m, k)
    w = rt.QuantWeight(12, n, k, raw.tobytes())
    dx = torch.from_numpy(x16.view(np.int16).copy()).cuda()
    out = torch.full((m * n + 8,), 0x1234, dtype=torch.int16, device="cuda")
    w.matmul(dx.data_ptr(), m, out.data_ptr() + 2 * shift, _lib.MATMUL_GEMV)
    torch.cuda.synchronize()
    assert (out[:shift] == 0x1234).all() and (out[shift + m * n:] == 0x1234).all()
    y = out[shift:shift + m * n].cpu().numpy().view(np.float16).astype(np.float64).reshape(m, n)
    want = x16.astype(np.float64) @ oracle.dequantize(12, raw).reshape(n, k).astype(np.float64).T
    assert np.linalg.norm(y - want) <= 1e-3 * np.linalg.norm(want)
