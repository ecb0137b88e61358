"""The decoders' output mappings at the edges of a workgroup's blocks, one
output at a time: bit-exact with the oracle, nothing written past the end."""
import numpy as np
import pytest

import oracle
import synth
from nemo_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("type_,gen,size", [(12, synth.random_q4k, 144), (14, synth.random_q6k, 210),
                                            (2, synth.random_q40, 18)])
@pytest.mark.parametrize("nb", [1, 31, 33, 255, 256, 257, 515])
@pytest.mark.parametrize("half", [True, False])
def test_dequantize_one_output_bit_exact(torch_cuda, type_, gen, size, nb, half):
    torch = torch_cuda
    raw = gen(2500 + type_ + nb, nb).copy()
    raw.reshape(nb, size)[1::2, {12: 1, 14: 209, 2: 1}[type_]] ^= 0x80  # scales of both signs
    expect = oracle.dequantize(type_, raw)
    d_raw = torch.from_numpy(raw).cuda()
    out = torch.full((expect.size + 64,), 7.0, dtype=torch.float16 if half else torch.float32, device="cuda")
    p = out.data_ptr()
    rt.dequantize_device(type_, d_raw.data_ptr(), expect.size, 0 if half else p, p if half else 0)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(got[expect.size:] == 7.0)
    want = expect.astype(np.float16) if half else expect
    bits = np.uint16 if half else np.uint32
    assert np.array_equal(got[:expect.size].view(bits), want.view(bits))
