"""SwiGLU of every kernel that ends in one, value by value against 64 bits. The
embeddings have one value each and attention adds nothing (zero O
projection), so gate and up values are f16 roundings of single products, known
exactly. The stored f16 has to be the rounding of a value within 5 * 2^-24 of
g / (1 + e^-g) * u (at most 2 units for fp32's expf (1 ulp) and one each for the
sum, the quotient and the product), and it is the one rounding of fp32's g / (1
+ expf(-g)), as torch computes it on the device, times u."""
import numpy as np
import pytest

import oracle
import synth
from nemo_amd import runtime as rt

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("hidden,F,n", [
    (256, 512, 12),       # GEMV
    (256, 512, 160),      # of ten token groups
    (2304, 512, 40),      # K split in two, summed by a kernel of its own
    (256, 256, 161),      # fused tiles of 64 rows,
    (256, 8192, 200),     # of 128,
    (256, 8192, 384),     # of 192
    (256, 8192, 500),     # and 256
    (256, 1536, 1200),    # 64-row tiles with 128-column waves
    (256, 8192, 1200),    # f16 tiles of 384 x 256,
    (256, 8192, 1600),    # of 256 x 256,
    (256, 8192, 2100),    # of 192 x 128
    (256, 8192, 2400),    # and of 256 x 256 with a rest of 128 x 256
])
def test_swiglu_rounding(torch_cuda, hidden, F, n):
    V = 300
    dims = rt.make_dims(hidden=hidden, q_heads=4, kv_heads=2, head_dim=64, intermediate=F, layers=1, vocab=V,
                        merge_after_layer=1)
    tensors = synth.model_tensors(dims, seed=1300 + hidden + F, sigma=0.5)
    typ, d, data = tensors["blk.0.attn_output.weight"]
    tensors["blk.0.attn_output.weight"] = (typ, d, bytes(len(data)))
    column = np.arange(V) * 7 % hidden
    table = np.zeros((V, hidden), np.float16)
    table[np.arange(V), column] = 1
    tensors["token_embd.weight"] = (rt.TYPE_F16, [hidden, V], table.tobytes())
    # gates from 1e-3 to 100, and one column in ten past the f16 range
    power = np.where(synth.uniform(1301, hidden) < 0.1, 3 + synth.uniform(1302, hidden),
                     -3.5 + 4 * synth.uniform(1303, hidden))
    norm = (10.0 ** power).astype(f32)
    tensors["blk.0.ffn_norm.weight"] = (rt.TYPE_F32, [hidden], norm.tobytes())
    model = rt.NemotronHipModel(tensors, dims=dims)
    plan = model.createPlan(1, n)
    ids = synth.randint(1304, n, 0, V)
    plan.run_sync(ids.astype(np.uint32), [n])
    got = plan.read_buffer("ffn").reshape(-1, F)[:n]

    with np.errstate(all="ignore"):
        inv = f32(1) / np.sqrt(f32(1) / f32(hidden) + f32(dims.rms_epsilon))
        h = (inv * norm[column]).astype(np.float16).astype(f32)
        w = oracle.dequantize(12, np.frombuffer(tensors["blk.0.ffn_gate_up.weight"][2], np.uint8))
        w = w.reshape(2 * F, hidden)[:, column].T.astype(np.float16).astype(f32)
        rows = (h[:, None] * w).astype(np.float16).astype(np.float64)  # per id
        g, u = rows[:, :F], rows[:, F:]
        e = np.where(-g > np.log(float(np.finfo(f32).max)), np.inf, np.exp(-g))  # fp32's range
        want = g / (1 + e) * u
        low, high = (want * (1 - 5 * 2.0 ** -24)).astype(np.float16), (want * (1 + 5 * 2.0 ** -24)).astype(np.float16)
        same = (got == low[ids]) | (got == high[ids]) | (np.isnan(got) & np.isnan(want)[ids])
    assert same.all(), f"{np.count_nonzero(~same)} of {same.size} values off"
    with np.errstate(all="ignore"):
        gt = torch_cuda.from_numpy(g.astype(f32)).cuda()
        silu = (gt / (1 + torch_cuda.exp(-gt))).cpu().numpy().astype(np.float64)
        once = (silu * u).astype(np.float16)[ids]  # 35 bits: exact in 64
        same = (got == once) | (np.isnan(got) & np.isnan(once))
    assert same.all(), f"{np.count_nonzero(~same)} of {same.size} values are not rounded once"
    seen = np.unique(ids)
    assert n < 100 or np.isinf(g[seen]).any() and np.isinf(want[seen]).any() and np.isnan(want[seen]).any()
    plan.destroy()
    model.destroy()
