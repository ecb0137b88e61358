"""The f16 GEMM's stores: 16 bytes per lane where rows, columns and the output
pointer allow it, value by value elsewhere, bit for bit what the fused kernel
stores; and SwiGLU on gates from 0 to past the f16 range."""
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


# the GEMV, fused tiles of 128 and 192 rows, f16 tiles of 384 x 256, and of 256 x 256 with a rest of 128 x 256
@pytest.mark.parametrize("n", [12, 200, 700, 1200, 2400])
@pytest.mark.parametrize("scale", [0.01, 4.0, 2500.0])  # gates of about 0.1, 32 and 20000
def test_swiglu_over_the_gate_range(torch_cuda, n, scale):
    """One layer whose attention adds nothing (zero output projection), so the
    gate and up rows follow from the embeddings alone. They are f16-rounded
    sums, at most one f16 step (2^-10) from the 64-bit ones: silu's slope is at
    most 1.1, which bounds the product's difference."""
    H, F, V = 256, 8192, 300
    dims = rt.make_dims(hidden=H, q_heads=4, kv_heads=2, head_dim=64, intermediate=F, layers=1, vocab=V,
                        merge_after_layer=1)
    tensors = synth.model_tensors(dims, seed=61, embedding_type=1, sigma=0.5)
    typ, d, _ = tensors["blk.0.attn_output.weight"]
    tensors["blk.0.attn_output.weight"] = (typ, d, np.zeros(H * 144, dtype=np.uint8).tobytes())
    ffn_norm = np.full(H, scale, dtype=np.float32)
    tensors["blk.0.ffn_norm.weight"] = (rt.TYPE_F32, [H], ffn_norm.tobytes())
    model = rt.NemotronHipModel(tensors, dims=dims)
    ids = synth.randint(62, n, 1, V).astype(np.uint32)
    plan = model.createPlan(1, n)
    plan.run_sync(ids, [n])
    got = plan.read_buffer("ffn")[: n * F].reshape(n, F).astype(np.float64)

    om = synth.oracle_model(dims, tensors)
    x = np.frombuffer(tensors["token_embd.weight"][2], np.float16).reshape(V, H)[ids].astype(np.float64)
    h = (x / np.sqrt((x * x).mean(1, keepdims=True) + dims.rms_epsilon) * ffn_norm).astype(np.float16).astype(np.float64)
    gate_up = np.asarray(om.gate_up[0], np.float64).reshape(2 * F, H)
    with np.errstate(all="ignore"):
        g64, u64 = h @ gate_up[:F].T, h @ gate_up[F:].T
        g, u = g64.astype(np.float16).astype(np.float64), u64.astype(np.float16).astype(np.float64)
        want = g / (1 + np.exp(-g)) * u
    # values whose rounding to f16 or to infinity is not in doubt (the rows h
    # are within one f16 step of the kernel's, so the sums within 2^-10 of the
    # terms' magnitudes)
    terms_g, terms_u = np.abs(h) @ np.abs(gate_up[:F]).T, np.abs(h) @ np.abs(gate_up[F:]).T
    with np.errstate(all="ignore"):
        bound = 2.0 ** -9 * (1.1 * terms_g * np.abs(u) + 1.1 * np.abs(g) * terms_u) + 2.0 ** -10 * np.abs(want) + 2.0 ** -23
        sure = (np.abs(g64) + 2.0 ** -9 * terms_g < 65000) & (np.abs(u64) + 2.0 ** -9 * terms_u < 65000)
        inside = sure & (np.abs(want) + bound < 65000)
        assert inside.any() or scale > 1000
        assert (np.abs(got - want)[inside] <= bound[inside]).all()
        over = sure & (np.abs(want) - bound > 66000)
        assert np.isinf(got[over]).all() and (np.sign(got[over]) == np.sign(want[over])).all()
        # gates rounded to -infinity: -inf / inf; to +infinity: inf * u
        far = 70000 + 2.0 ** -9 * terms_g
        assert np.isnan(got[g64 < -far]).all()
        plus = (g64 > far) & (np.abs(u64) > 1 + 2.0 ** -9 * terms_u)
        assert np.isinf(got[plus]).all()
        if scale > 1000:
            assert over.any() and (g64 < -far).any() and plus.any()
