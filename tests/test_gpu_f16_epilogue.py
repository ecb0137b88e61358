"""The f16 GEMM's stores: 16 bytes per lane where rows, columns and the output
pointer allow it, value by value elsewhere, bit for bit what the fused kernel
stores."""
import numpy as np
import pytest

import synth
from nemo_amd import _lib, runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,shift", [
    (1, 8, 256, 0),        # one run of 8 columns
    (257, 1000, 256, 0),   # whole runs, columns that end inside a tile
    (257, 1004, 512, 0),   # rows of 1004 values: not 16-byte aligned
    (383, 256, 256, 1),    # an output that starts 2 bytes past alignment
    (640, 2560, 768, 0),   # 128 x 256 tiles (32 x 32 x 16 MFMAs)
    (640, 2560, 768, 1),
])
def test_two_pass_stores(torch_cuda, m, n, k, shift):
    torch = torch_cuda
    raw = synth.random_q4k(77 + m + n, n * k // 256)
    x16 = synth.normal(78 + m, m * k).astype(np.float16)
    w = rt.QuantWeight(12, n, k, raw.tobytes())
    dx = torch.from_numpy(x16.view(np.int16).copy()).cuda()
    fused = torch.zeros(m * n, dtype=torch.int16, device="cuda")
    out = torch.full((m * n + 16,), 0x1234, dtype=torch.int16, device="cuda")
    w.matmul(dx.data_ptr(), m, fused.data_ptr(), _lib.MATMUL_GEMM)
    w.matmul(dx.data_ptr(), m, out.data_ptr() + 2 * shift, _lib.MATMUL_TWO_PASS)
    torch.cuda.synchronize()
    assert torch.equal(out[shift:shift + m * n], fused)
    assert (out[:shift] == 0x1234).all() and (out[shift + m * n:] == 0x1234).all()
