"""The attention of passes that hold a request longer than one staging round:
64-key rounds with 1, 2 and odd counts of 32-key blocks, last keys that fill a
block or one key of it, (query tile, head) pairs that do not fill a workgroup,
sampled keys, and short requests beside long ones. Against the oracle's
attention of the pass's own QKV projection: probabilities and results are
rounded to f16 (2^-11 each), sums are fp32."""
import numpy as np
import pytest

import oracle
import synth
from nemo_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,q_heads,kv_heads,lengths,threshold", [
    (64, 4, 4, [257], 2048),                        # one head per KV head
    (64, 8, 1, [289, 1], 2048),                     # eight
    (64, 20, 4, [320, 31, 33, 96], 2048),           # five
    (64, 4, 2, [1000, 64, 65, 97, 700], 2048),
    (64, 4, 2, [301, 302, 303, 99, 2], 98),         # every third key
    (128, 2, 2, [129, 32], 2048),
    (128, 6, 2, [500, 63, 1, 160, 161], 2048),      # three
    (128, 6, 2, [385, 386, 100, 130], 99),
])
def test_long_attention(torch_cuda, hd, q_heads, kv_heads, lengths, threshold):
    H, V = 256, 300
    dims = rt.make_dims(hidden=H, q_heads=q_heads, kv_heads=kv_heads, head_dim=hd, intermediate=256, layers=1, vocab=V,
                        merge_after_layer=1, kv_stride_threshold=threshold)
    tensors = synth.model_tensors(dims, seed=810 + hd + q_heads, sigma=0.08)
    model = rt.NemotronHipModel(tensors, dims=dims)
    S = max(lengths)
    plan = model.createPlan(len(lengths), S)
    plan.run_sync(synth.randint(811, len(lengths) * S, 1, V).astype(np.uint32), lengths)
    QW, KW = q_heads * hd, kv_heads * hd
    qkv = plan.read_buffer("qkv").reshape(-1, QW + 2 * KW)
    att = plan.read_buffer("attention").reshape(-1, QW).astype(np.float64)
    od = synth.oracle_model(dims, tensors).dims
    at = 0
    for b, n in enumerate(lengths):
        raw = qkv[at:at + n]
        q, k = oracle.rope(raw, np.arange(n), oracle.rope_table(n, hd, od.rope_theta), od)
        want = oracle.attention(q, k, raw[:, QW + KW:].reshape(n, kv_heads, hd), od, threshold, 3)
        want = np.asarray(want, np.float64).reshape(n, QW)
        err = np.linalg.norm(att[at:at + n] - want) / np.linalg.norm(want)
        assert err <= 2e-3, f"request {b} of {n} tokens: {err}"
        at += n
    plan.destroy()
    model.destroy()
