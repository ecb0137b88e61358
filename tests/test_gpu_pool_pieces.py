"""Pooling of requests whose merged rows end at, before and past the batches of
128 and 512 rows in which they are loaded, alone and beside others. Against the
mean of the normalized rows the pass pooled (bar: fp32 sums of f16 rows, n terms
each within 2^-24 of the sum of magnitudes, and three more roundings for the
mean and the scale), and bit for bit: 32 phases of rows in order, the phases in
order, the squares of the means by thread and butterfly."""
import numpy as np
import pytest

import synth
from nemo_amd import runtime as rt
from test_gpu_norm_order import f32, fma_square, wave_sum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [[1], [400], [402], [799, 400, 3, 801, 1], [1203]])
def test_pooling_in_pieces(torch_cuda, lengths):
    H = 256
    dims = rt.make_dims(hidden=H, q_heads=4, kv_heads=2, head_dim=64, intermediate=256, layers=1, vocab=300,
                        merge_after_layer=0)
    model = rt.NemotronHipModel(synth.model_tensors(dims, seed=31, embedding_type=1), dims=dims)
    S = max(lengths)
    plan = model.createPlan(len(lengths), S)
    ids = synth.randint(17, len(lengths) * S, 1, 300).astype(np.uint32)
    got = plan.run_sync(ids, lengths)
    rows = plan.read_buffer("norm_merged").reshape(-1, H).astype(np.float64)
    at = 0
    for b, n in enumerate(rt.contextual_merged_length(v) for v in lengths):
        part = rows[at:at + n]
        at += n
        mean = part.mean(0)
        want = mean / np.linalg.norm(mean)
        bound = (n + 4) * 2.0 ** -24 * np.abs(part).mean(0).max() / np.linalg.norm(mean) + 2.0 ** -22
        assert np.abs(got[b] - want).max() <= bound, f"request {b}"


@pytest.mark.parametrize("hidden,lengths", [
    (256, [1, 2]),
    (256, [200, 202, 49, 51]),        # 128, 130, 32 and 33 merged rows
    (256, [800, 802, 1000, 1002]),    # 512, 514, 640 and 642
    (2304, [30, 1203]),               # more columns than the threads keep
])
def test_pooling_order(torch_cuda, hidden, lengths):
    dims = rt.make_dims(hidden=hidden, q_heads=4, kv_heads=2, head_dim=64, intermediate=256, layers=1, vocab=300,
                        merge_after_layer=0)
    model = rt.NemotronHipModel(synth.model_tensors(dims, seed=33, embedding_type=1), dims=dims)
    S = max(lengths)
    plan = model.createPlan(len(lengths), S)
    ids = synth.randint(19, len(lengths) * S, 1, 300).astype(np.uint32)
    got = plan.run_sync(ids, lengths)
    rows = plan.read_buffer("norm_merged").reshape(-1, hidden).astype(f32)
    at = 0
    for b, n in enumerate(rt.contextual_merged_length(v) for v in lengths):
        padded = np.zeros((-(-n // 32) * 32, hidden), f32)
        padded[:n] = rows[at:at + n]
        at += n
        phases = np.zeros((32, hidden), f32)
        for r in padded.reshape(-1, 32, hidden):
            phases = phases + r
        total = phases[0]
        for phase in phases[1:]:
            total = total + phase
        mean = total / f32(n)
        columns = np.zeros(-(-hidden // 256) * 256, f32)
        columns[:hidden] = mean
        part = np.zeros((1, 256), f32)
        for c in columns.reshape(-1, 1, 256):
            part = fma_square(c, part)
        waves = np.zeros((1, 64), f32)
        waves[0, :4] = wave_sum(part.reshape(4, 64))
        want = mean * (f32(1) / np.sqrt(wave_sum(waves)[0]))
        assert np.array_equal(got[b].view(np.uint32), want.view(np.uint32)), f"request {b}"
    plan.destroy()
    model.destroy()
