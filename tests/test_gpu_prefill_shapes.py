"""GPU parity of whole prefills at the sizes where their launches change: one
query row, partial blocks of queries, partial work-groups of the fused pooling
and key-norm launch, and selections split into few and many key segments.
Against the float64 oracle, with the tolerance of the 16-bit attention.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from vecattention_amd import VecAttention_prefill, stages, threshold_to_gap
from vecattention_amd import _native as nat
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


# Launches of few work-groups cut their selections into more segments, and
# causal chunks cut only the keys they see: every kernel's unit (64 keys, the
# group span, 768 keys for a 48-key span, 256-key chunks) and the two-pass form.
SPLIT_CASES = [
    # name, B, Hq, Hk, S, D, dtype, causal, qps, bk, G, chunk, threshold
    ("g1-ragged", 1, 4, 2, 2333, 128, torch.bfloat16, True, 64, 16, 1, 1024, 0.9),
    ("g1-under-two-segments", 1, 2, 2, 200, 64, torch.bfloat16, True, 64, 16, 1, 1024, 0.9),
    ("g16-chunks", 1, 4, 4, 3000, 128, torch.float16, True, 64, 16, 16, 512, 0.5),
    ("long-groups-causal-chunks", 1, 2, 2, 5000, 64, torch.bfloat16, True, 64, 64, 32, 1024, 0.5),
    # chunks of 64 rows share launches
    ("merged-chunks", 1, 2, 1, 8400, 128, torch.bfloat16, True, 64, 16, 4, 4096, 0.6),
    ("merged-tail-qps128", 1, 2, 2, 128 * 129 + 5, 64, torch.float16, True, 128, 128, 1, 16384, 0.9),
    ("one-group-causal", 1, 2, 2, 1700, 128, torch.bfloat16, True, 64, 16, 8192, 512, 0.4),
    ("one-group-noncausal", 1, 3, 3, 4050, 128, torch.bfloat16, False, 64, 16, 8192, 2048, 0.4),
    ("one-group-short", 1, 3, 3, 130, 64, torch.float16, False, 64, 32, 8192, 2048, 0.4),
    ("span48", 1, 2, 1, 3100, 128, torch.bfloat16, True, 64, 16, 3, 1024, 0.8),
    ("tiles128", 1, 2, 2, 5003, 128, torch.float16, True, 128, 128, 1, 2048, 0.9),
    ("tiles256", 1, 2, 2, 2900, 64, torch.bfloat16, False, 128, 256, 2, 1024, 0.7),
    ("two-batches-chunks", 2, 4, 2, 3000, 128, torch.bfloat16, True, 64, 16, 4, 1024, 0.6),
    ("three-batches-one-group", 3, 2, 2, 2500, 64, torch.float16, False, 64, 16, 8192, 1024, 0.4),
    ("two-batches-tiles128", 2, 2, 1, 2700, 128, torch.bfloat16, True, 128, 128, 1, 1024, 0.9),
    ("fp32-chunks", 1, 2, 2, 2500, 64, torch.float32, True, 64, 16, 16, 512, 0.5),
    ("fp32-one-group-causal", 1, 2, 2, 1500, 64, torch.float32, True, 64, 16, 8192, 512, 0.4),
]


# Non-causal prefills of 8192 keys or more over kv heads that do not divide the
# 8 XCDs take the attention's items from queues, one per launch (the last case
# has more launches than queues): per-head thresholds far apart.
QUEUE_CASES = [
    ("three-heads", 1, 3, 3, 8200, 128, torch.bfloat16, False, 64, 16, 8192, 4096, 0.2),
    ("sixteen-kv-heads-qps128", 1, 16, 16, 8192, 64, torch.float16, False, 128, 16, 16, 8192, 0.5),
    ("gqa-five-kv-heads", 1, 10, 5, 8321, 128, torch.bfloat16, False, 64, 32, 4, 2048, 0.5),
    # batches: 16 kv heads in all, 15, and 9 (three of each of three batches)
    ("two-batches-of-8", 2, 8, 8, 8300, 64, torch.bfloat16, False, 64, 16, 16, 4096, 0.5),
    ("three-batches-gqa", 3, 10, 5, 8200, 128, torch.float16, False, 64, 16, 8192, 8192, 0.4),
    ("three-batches-of-3", 3, 3, 3, 8193, 64, torch.bfloat16, False, 128, 32, 4, 8192, 0.5),
    ("staged-form", 1, 12, 12, 65600, 128, torch.bfloat16, False, 64, 16, 8192, 128, 0.6),
]


@pytest.mark.parametrize("case", QUEUE_CASES, ids=[c[0] for c in QUEUE_CASES])
def test_queued_attention_equals_static(case):
    name, B, Hq, Hk, S, D, dtype, causal, qps, bk, G, chunk, th = case
    print("[case] queued attention", name, flush=True)
    q, k, v = (x.to("cuda:0") for x in make_inputs(B, Hq, Hk, S, D, dtype, seed=13))
    Sq = min(S, chunk * 66)  # more launches than queues in the last case
    q = q[:, :, :Sq]
    ths = torch.linspace(th, 0.95, Hq, device="cuda:0")
    out = VecAttention_prefill(q, k, v, threshold=ths, q_pooling_size=qps, k_local_size=bk,
                               group_k_block=G, causal=causal, chunk_size=chunk)
    _, gaps = threshold_to_gap(ths, B, Hq, q.device)
    scaled, _ = stages.pool_scaled(q, qps)
    want = torch.empty_like(out)
    segk = stages.segment_keys(S, bk, G)
    for c0 in range(0, Sq, chunk):
        J0, nc = c0 // qps, -(-min(chunk, Sq - c0) // qps)
        counts, idx = stages.select_segments(scaled[:, :, J0:J0 + nc], k, J0, 0.0, gaps, causal,
                                             qps, bk, G, causal, segk)
        stages.sparse_attention(q, k, v, want, J0, nc, counts, idx, causal, qps, segk=segk)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("case", SPLIT_CASES, ids=[c[0] for c in SPLIT_CASES])
def test_split_prefill_equals_unsplit_stages(case):
    # The prefill's output is, bit for bit, that of the unsplit selection on
    # the exact kernel followed by the attention over its lists.
    name, B, Hq, Hk, S, D, dtype, causal, qps, bk, G, chunk, th = case
    print("[case] split prefill", name, flush=True)
    q, k, v = (x.to("cuda:0") for x in make_inputs(B, Hq, Hk, S, D, dtype, seed=12))
    out = VecAttention_prefill(q, k, v, threshold=th, q_pooling_size=qps, k_local_size=bk,
                               group_k_block=G, causal=causal, chunk_size=chunk)
    gap, _ = threshold_to_gap(th, B, Hq, q.device)
    scaled, _ = stages.pool_scaled(q, qps)
    want = torch.empty_like(out)
    for c0 in range(0, S, chunk):
        J0, nc = c0 // qps, -(-min(chunk, S - c0) // qps)
        counts, idx = stages.select_rows(scaled[:, :, J0:J0 + nc], k, J0, gap, None, causal, qps,
                                         bk, G, causal, kernel=nat.VA_SEL_EXACT)
        stages.sparse_attention(q, k, v, want, J0, nc, counts, idx, causal, qps)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
