"""RMSNorm bit for bit: the squares of a row are summed in one stated order
(per thread one fused multiply-add a value, in column order, then the wave's
and the workgroup's butterflies), so the whole kernel can be followed in
numpy. The O projections are zero and the down projection has one weight in a
row, so the residual sum is known exactly: the embedding's value plus the f16
of one product."""
import numpy as np
import pytest

import oracle
import synth
from nemo_amd import runtime as rt

pytestmark = pytest.mark.gpu
f32 = np.float32


def fma_square(v, s):
    """float32 fma(v, v, s): the square is exact in 64 bits, the sum rounded
    to odd there, which the second rounding cannot notice."""
    p, s = v.astype(np.float64) ** 2, s.astype(np.float64)
    t = p + s
    b = t - p
    err = (p - (t - b)) + (s - b)
    even = (t.view(np.uint64) & np.uint64(1)) == 0
    odd = np.nextafter(t, np.where(err > 0, np.inf, -np.inf))
    return np.where((err != 0) & even, odd, t).astype(f32)


def wave_sum(v):
    for o in (32, 16, 8, 4, 2, 1):
        v = v + v[:, np.arange(64) ^ o]
    return v[:, 0]


def rmsnorm(v, w, eps):
    """f16 RMSNorm of float32 rows, of which f16 roundings are stored."""
    rows, hidden = v.shape
    columns = -(-hidden // 2048) * 2048
    xs = np.zeros((rows, columns), f32)
    xs[:, :hidden] = v
    xs = xs.reshape(rows, -1, 256, 8)  # [pass][thread][value]
    part = np.zeros((rows, 256), f32)
    for i in range(xs.shape[1]):
        for e in range(8):
            part = fma_square(xs[:, i, :, e], part)
    waves = np.zeros((rows, 64), f32)
    for i in range(4):
        waves[:, i] = wave_sum(part[:, 64 * i:64 * i + 64])
    total = wave_sum(waves)
    inv = f32(1) / np.sqrt(total / f32(hidden) + f32(eps))
    return (v.astype(np.float16).astype(f32) * inv[:, None] * w).astype(np.float16)


def model_of(hidden, F, emb, merge):
    dims = rt.make_dims(hidden=hidden, q_heads=4, kv_heads=2, head_dim=64, intermediate=F, layers=1, vocab=300,
                        merge_after_layer=merge)
    tensors = synth.model_tensors(dims, seed=900 + hidden + F + emb, embedding_type=emb)
    typ, d, data = tensors["blk.0.attn_output.weight"]
    tensors["blk.0.attn_output.weight"] = (typ, d, bytes(len(data)))
    # row r of the down projection: one weight, at column pick[r]
    pick = synth.randint(902 + F, hidden, 0, F)
    blocks = hidden * F // 256
    at = np.arange(hidden) * (F // 256) + pick // 256
    q = np.full((blocks, 256), 32, np.uint8)
    q[at, pick % 256] = synth.randint(903, hidden, 33, 64)
    scale = np.zeros((blocks, 16), np.int8)
    scale[at, (pick % 256) // 16] = synth.randint(904, hidden, 20, 128)
    down = synth.q6k_blocks(np.full(blocks, np.float16(1e-3)).view(np.uint16), scale, q).reshape(-1)
    tensors["blk.0.ffn_down.weight"] = (14, [F, hidden], down.tobytes())
    weight = oracle.dequantize(14, down).reshape(hidden, F)[np.arange(hidden), pick].astype(np.float16).astype(f32)
    return rt.NemotronHipModel(tensors, dims=dims), dims, tensors, pick, weight


def differing(got, want):
    return np.count_nonzero(got.view(np.uint16) != want.view(np.uint16))


@pytest.mark.parametrize("hidden,F,n", [
    (2048, 512, 900),    # f16 residual
    (2048, 2048, 900),   # tiles, K split in two: f16 partial sums
    (2048, 4096, 900),   # in four
    (2048, 4096, 150),   # GEMV, K split in two: fp32 partial sums
    (256, 4096, 400),    # threads without values
    (2304, 2048, 300),   # rows longer than the threads hold
    (4096, 512, 40),
])
def test_residual_norm_bits(torch_cuda, hidden, F, n):
    model, dims, tensors, pick, weight = model_of(hidden, F, 1, merge=1)
    plan = model.createPlan(1, n)
    ids = synth.randint(901, n, 1, dims.vocab)
    plan.run_sync(ids.astype(np.uint32), [n])
    table = np.frombuffer(tensors["token_embd.weight"][2], np.float16).reshape(-1, hidden)
    ffn = plan.read_buffer("ffn").reshape(-1, F)[:n][:, pick].astype(f32)
    v = table[ids].astype(f32) + (ffn * weight).astype(np.float16).astype(f32)
    assert differing(plan.read_buffer("x_full").reshape(-1, hidden)[:n], v.astype(np.float16)) == 0
    want = rmsnorm(v, np.frombuffer(tensors["output_norm.weight"][2], f32), dims.rms_epsilon)
    assert differing(plan.read_buffer("norm_full").reshape(-1, hidden)[:n], want) == 0
    plan.destroy()
    model.destroy()


@pytest.mark.parametrize("hidden,emb", [(256, 1), (2048, 14), (2304, 1), (2304, 14), (4096, 14)])
def test_embedding_norm_bits(torch_cuda, hidden, emb):
    """The first norm, which the embedding lookup writes; the merge comes
    before the layer, so `norm_full` keeps it."""
    n = 40
    model, dims, tensors, _, _ = model_of(hidden, 256, emb, merge=0)
    plan = model.createPlan(1, n)
    ids = synth.randint(901, n, 1, dims.vocab)
    plan.run_sync(ids.astype(np.uint32), [n])
    typ, _, data = tensors["token_embd.weight"]
    table = np.frombuffer(data, np.float16) if typ == 1 else oracle.dequantize(14, np.frombuffer(data, np.uint8))
    v = table.reshape(-1, hidden)[ids].astype(np.float16)
    assert differing(plan.read_buffer("x_full").reshape(-1, hidden)[:n], v) == 0
    want = rmsnorm(v.astype(f32), np.frombuffer(tensors["blk.0.attn_norm.weight"][2], f32), dims.rms_epsilon)
    assert differing(plan.read_buffer("norm_full").reshape(-1, hidden)[:n], want) == 0
    plan.destroy()
    model.destroy()
