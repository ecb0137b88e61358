"""The 64 MI x 128 tiles of passes past the GEMV: every tile height, one to
eight 256-value blocks of K (the pipeline's ends and its steady state), rows
that fill a tile or one row of it, outputs that 16-byte stores do not fit. Bit
for bit the 64-row tiles' and the two-pass GEMM's results (same f16 operands,
same order), and the oracle's within the projection bar. K splits, their f16
and fp32 partial sums and SwiGLU, which only a plan reaches: bit for bit the
rows of a larger pass, which takes other kernels."""
import numpy as np
import pytest

import oracle
import synth
from nemo_amd import _lib, runtime as rt

pytestmark = pytest.mark.gpu
GEN = {12: synth.random_q4k, 14: synth.random_q6k, 2: synth.random_q40}


def tile_rows(m, n):
    """The tile height that the dispatch takes: the cheapest rounds of 256
    workgroups (its rule, kept here so that each case says what it runs)."""
    return min((cost * -(-(-(-m // rows) * (n // 128)) // 256), rows)
               for rows, cost in ((64, 175), (128, 215), (192, 280), (256, 325)))[1]


@pytest.mark.parametrize("type_", [12, 14, 2])
@pytest.mark.parametrize("m,n,k,shift,rows", [
    (161, 128, 256, 0, 64),       # one block
    (193, 384, 512, 0, 64),       # two
    (320, 256, 768, 1, 64),       # three, an output 2 bytes past alignment
    (1152, 128, 2048, 0, 64),     # eight, the most rows
    (200, 16384, 256, 0, 128),
    (256, 12800, 1280, 0, 128),   # five blocks
    (385, 6400, 1024, 0, 128),    # four, one row in the last tile
    (384, 8192, 2048, 0, 128),    # eight
    (384, 16384, 256, 0, 192),
    (321, 16384, 512, 0, 192),
    (380, 16384, 768, 0, 192),
    (577, 8192, 1024, 0, 192),    # one row in the last tile
    (576, 8192, 2048, 0, 192),
    (1025, 16384, 512, 0, 192),   # several rounds
    (500, 16384, 256, 0, 256),
    (512, 16384, 768, 0, 256),
    (769, 8192, 1024, 0, 256),    # one row in the last tile
    (769, 16384, 512, 0, 256),    # and two rounds
    (1024, 8192, 2048, 0, 256),
])
def test_wide_tiles_bit_identical(torch_cuda, type_, m, n, k, shift, rows):
    assert tile_rows(m, n) == rows
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


def _model(kind):
    """One layer before the merge."""
    dims = rt.make_dims(hidden=2048, q_heads=32, kv_heads=8, head_dim=64, intermediate=8192, layers=1, vocab=300,
                        merge_after_layer=1)
    if kind == "q4_k":  # and a Q6_K down projection
        return rt.NemotronHipModel(None, dims=dims, synthetic_seed=5, embedding_type=rt.TYPE_F16), dims
    if kind == "parts":  # separate q, k and v, whose K splits have fp32 partial sums
        dims.q_heads, dims.kv_heads, dims.intermediate = 4, 2, 256
        return rt.NemotronHipModel(synth.model_tensors(dims, seed=6, fused=False), dims=dims), dims
    dims.q_heads, dims.intermediate = 16, 4096
    sizes = {"attn_qkv": (2048, 2048), "attn_output": (2048, 1024), "ffn_gate_up": (8192, 2048),
             "ffn_down": (2048, 4096)}
    tensors = {"token_embd.weight": (rt.TYPE_F16, [2048, 300], synth.normal(7, 300 * 2048).astype(np.float16).tobytes())}
    for name in ("output_norm", "blk.0.attn_norm", "blk.0.ffn_norm"):
        tensors[name + ".weight"] = (rt.TYPE_F32, [2048], np.full(2048, 0.3, np.float32).tobytes())
    for i, (name, (n, k)) in enumerate(sizes.items()):
        tensors[f"blk.0.{name}.weight"] = (2, [k, n], synth.random_q40(8 + i, n * k // 32).tobytes())
    return rt.NemotronHipModel(tensors, dims=dims), dims


@pytest.mark.parametrize("kind", ["q4_k", "parts", "q4_0"])
def test_wide_tiles_in_a_pass(torch_cuda, kind):
    """A request alone runs on the tiles, and in a pass of 1800 tokens on the
    64-row and f16 tiles, with the same K splits."""
    model, dims = _model(kind)
    F, QKV = dims.intermediate, (dims.q_heads + 2 * dims.kv_heads) * 64
    for n in (161, 200, 384, 500, 769, 1024, 1152):
        ids = synth.randint(31 + n, n, 1, 300).astype(np.uint32)
        alone = model.createPlan(1, n)
        alone.run_sync(ids, [n])
        S = max(n, 1800 - n)
        both = np.zeros((2, S), np.uint32)
        both[0, :n], both[1, :1800 - n] = ids, synth.randint(32, 1800 - n, 1, 300)
        pair = model.createPlan(2, S)
        pair.run_sync(both.reshape(-1), [n, 1800 - n])
        for name, width in (("qkv", QKV), ("attention", dims.q_heads * 64), ("ffn", F), ("x_full", 2048),
                            ("norm_full", 2048)):
            a, b = (p.read_buffer(name)[:n * width].view(np.uint16) for p in (alone, pair))
            assert np.count_nonzero(a & 0x7FFF) > a.size // 2  # values, not an empty buffer
            assert np.array_equal(a, b), f"{n} tokens, {name}: {np.count_nonzero(a != b)} of {a.size} differ"
        alone.destroy()
        pair.destroy()
    model.destroy()
