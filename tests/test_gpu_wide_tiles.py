"""The 64 MI x 128 tiles of passes past the GEMV: every tile height, one to
five 256-value blocks of K (the pipeline's ends), rows that fill a tile or one
row of it, outputs that 16-byte stores do not fit. Bit for bit the 64-row
tiles' and the two-pass GEMM's results (same f16 operands, same order), and
the oracle's within the projection bar."""
import numpy as np
import pytest

import oracle
import synth
from nemo_amd import _lib, runtime as rt

pytestmark = pytest.mark.gpu
GEN = {12: synth.random_q4k, 14: synth.random_q6k, 2: synth.random_q40}


@pytest.mark.parametrize("type_", [12, 14, 2])
@pytest.mark.parametrize("m,n,k,shift", [
    (161, 128, 256, 0),      # 64-row tiles, one block
    (193, 384, 512, 0),      # two blocks
    (320, 256, 768, 1),      # three, an output 2 bytes past alignment
    (200, 16384, 256, 0),    # 128-row tiles
    (256, 12800, 1280, 0),   # five blocks
    (384, 16384, 256, 0),    # 192-row tiles
    (321, 16384, 512, 0),
    (380, 16384, 768, 0),
    (500, 16384, 256, 0),    # 256-row tiles
    (512, 16384, 768, 0),
    (1025, 16384, 512, 0),   # several rounds of them, one row in the last
])
def test_wide_tiles_bit_identical(torch_cuda, type_, m, n, k, shift):
    torch = torch_cuda
    seed = 311 + m + n + k + type_
    raw = GEN[type_](seed, n * k // (32 if type_ == 2 else 256))
    x16 = synth.normal(seed + 1, m * k).astype(np.float16).reshape(m, k)
    w = rt.QuantWeight(type_, n, k, raw.tobytes())
    dx = torch.from_numpy(x16.view(np.int16).copy()).cuda()
    outs = []
    for algo in (_lib.MATMUL_AUTO, _lib.MATMUL_GEMM_MID, _lib.MATMUL_TWO_PASS):
        out = torch.full((m * n + 8,), 0x7E00, dtype=torch.int16, device="cuda")
        w.matmul(dx.data_ptr(), m, out.data_ptr() + 2 * shift, algo)
        torch.cuda.synchronize()
        assert (out[:shift] == 0x7E00).all() and (out[shift + m * n:] == 0x7E00).all()
        outs.append(out[shift:shift + m * n])
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    cols = np.sort(synth.randint(seed + 2, min(n, 64), 0, n))
    w64 = oracle.dequantize(type_, raw).reshape(n, k)[cols].astype(np.float64)
    y = outs[0].cpu().numpy().view(np.float16).reshape(m, n)[:, cols].astype(np.float64)
    want = x16.astype(np.float64) @ w64.T
    assert np.linalg.norm(y - want) <= 2e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("type_,k", [(12, 512), (14, 256), (2, 768)])
def test_rows_off_16_bytes(torch_cuda, type_, k):
    """X that starts 2 bytes past alignment takes the 64-row tiles: the same bits."""
    torch = torch_cuda
    m, n = 200, 384
    raw = GEN[type_](407 + type_, n * k // (32 if type_ == 2 else 256))
    w = rt.QuantWeight(type_, n, k, raw.tobytes())
    x16 = torch.from_numpy(synth.normal(408, m * k).astype(np.float16).view(np.int16).copy())
    outs = []
    for shift in (0, 1):
        dx = torch.zeros(m * k + 8, dtype=torch.int16, device="cuda")
        dx[shift:shift + m * k] = x16.cuda()
        out = torch.full((m, n), 0x7E00, dtype=torch.int16, device="cuda")
        w.matmul(dx.data_ptr() + 2 * shift, m, out.data_ptr(), _lib.MATMUL_AUTO)
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
