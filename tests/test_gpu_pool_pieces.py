"""Pooling in pieces of 256 rows: requests whose merged rows end at, before and
past a piece, alone and beside others, against the mean of the normalized rows
the pass pooled. Bar: fp32 sums of f16 rows, n terms each within 2^-24 of the
sum of magnitudes, and three more roundings for the mean and the scale."""
import numpy as np
import pytest

import synth
from nemo_amd import runtime as rt

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
