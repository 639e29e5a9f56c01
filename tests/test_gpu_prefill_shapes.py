"""GPU parity of whole prefills at the sizes where their launches change: one
query row, partial blocks of queries, partial work-groups of the fused pooling
and key-norm launch, and selections split into few and many key segments.
Against the float64 oracle, with the tolerance of the 16-bit attention.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from vecattention_amd import VecAttention_prefill
from vecattention_amd.synth import make_inputs

pytestmark = pytest.mark.gpu

DTN = {torch.bfloat16: "bfloat16", torch.float16: "float16"}
# name, B, Hq, Hk, S, D, dtype, causal, qps, bk, G, chunk, threshold
CASES = [
    ("one-row", 1, 2, 1, 1, 128, torch.bfloat16, True, 64, 16, 1, 1024, 0.9),
    ("short-block", 1, 2, 2, 63, 64, torch.float16, True, 64, 16, 1, 1024, 0.9),
    ("block-and-a-row", 1, 4, 2, 65, 128, torch.bfloat16, False, 64, 16, 4, 1024, 0.5),
    ("nine-blocks", 2, 3, 1, 64 * 8 + 1, 128, torch.float16, True, 64, 16, 16, 1024, 0.5),
    ("qps128-tail", 1, 2, 2, 128 * 9 + 127, 64, torch.bfloat16, True, 128, 128, 1, 16384, 0.9),
    ("many-groups-of-8-blocks", 1, 28, 4, 64 * 37 - 35, 128, torch.bfloat16, True, 64, 16, 1, 8192,
     0.9),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_prefill_matches_oracle(case):
    name, B, Hq, Hk, S, D, dtype, causal, qps, bk, G, chunk, th = case
    print("[case] prefill shapes", name, flush=True)
    q, k, v = make_inputs(B, Hq, Hk, S, D, dtype, seed=11)
    k[:, :, S // 2] *= 8.0  # one long key sets the head's norm bound
    dev = "cuda:0"
    kd = k.transpose(1, 2).contiguous().to(dev).transpose(1, 2)  # (B, S, H, D) memory
    out = VecAttention_prefill(q.to(dev), kd, v.to(dev), threshold=th, q_pooling_size=qps,
                               k_local_size=bk, group_k_block=G, causal=causal, chunk_size=chunk)
    torch.cuda.synchronize()
    want, _ = orc.prefill(q, k, v, th, qps, bk, G, causal, chunk, 64, DTN[dtype])
    err = np.abs(out.float().cpu().numpy() - want)
    assert err.max() <= 2e-2 and err.mean() <= 2e-3, (err.max(), err.mean())
