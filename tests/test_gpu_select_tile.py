"""The selection over tiles of 128 keys that are groups of their own (run on an
MI355X) against the fp64 kernel, lists bit for bit: partial tiles and rows,
segments, and inputs that send most rows to the exact path (gap 0, where every
tile's maximum is ambiguous, and duplicated keys, which tie).
"""
import pytest
import torch

from vecattention_amd import _native as nat
from vecattention_amd import stages

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# name, B, Hq, Hk, Sk, D, dtype, causal, J0, nc, segk, gap, duplicates
CASES = [
    ("one-row", 1, 2, 1, 128, 128, torch.bfloat16, False, 0, 1, 0, 0.5, False),
    ("tail-of-one-key", 1, 2, 2, 1025, 128, torch.float16, False, 0, 33, 0, 0.4, False),
    ("rows129-segments", 2, 2, 1, 1500, 64, torch.bfloat16, False, 0, 129, 256, 0.3, False),
    ("causal-chunk", 1, 4, 2, 128 * 30, 128, torch.bfloat16, True, 7, 23, 512, 0.3, False),
    ("gap0", 1, 2, 2, 900, 128, torch.bfloat16, False, 0, 40, 0, 0.0, False),
    ("ties", 1, 2, 1, 1000, 64, torch.float16, True, 0, 8, 0, 0.0, True),
    ("all-ambiguous", 1, 1, 1, 384, 128, torch.bfloat16, False, 0, 5, 0, 0.0, True),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_tile_lists_equal_exact_lists(case):
    name, B, Hq, Hk, Sk, D, dtype, causal, J0, nc, segk, gap, dup = case
    print("[case] tile selection", name, flush=True)
    qps, bk, G = 128, 128, 1
    g = torch.Generator().manual_seed(9)
    qs = (0.1 * torch.randn(B, Hq, nc, D, generator=g)).to(dtype).to(DEV)
    k = torch.randn(B, Hk, Sk, D, generator=g)
    if dup:
        k = k[:, :, torch.arange(Sk) % (3 if name == "all-ambiguous" else 50)]
    k = k.to(dtype).to(DEV)
    want, wi = stages.select_rows(qs, k, J0, gap, None, causal, qps, bk, G, causal,
                                  kernel=nat.VA_SEL_EXACT)
    if segk:
        got, gi = stages.select_segments(qs, k, J0, gap, None, causal, qps, bk, G, causal, segk)
    else:
        got, gi = stages.select_rows(qs, k, J0, gap, None, causal, qps, bk, G, causal,
                                     kernel=nat.VA_SEL_MFMA)
    want, wi, got, gi = want.cpu(), wi.cpu(), got.cpu(), gi.cpu()
    nseg = got.shape[-1] if segk else 1
    got = got.reshape(B * Hq, nc, nseg)
    assert torch.equal(want.reshape(B * Hq, nc), got.sum(-1)) and int(want.sum()) > 0
    smin = qps if causal else 0
    for bh in range(B * Hq):
        for jr in range(nc):
            o = stages.row_offset(Sk, qps, causal, causal, J0, nc, bh, jr)
            parts = [gi[o + s0:o + s0 + int(got[bh, jr, s])] for s in range(nseg)
                     for s0 in [max(s * segk, smin) - smin if segk else 0]]
            assert torch.equal(wi[o:o + int(want.reshape(B * Hq, nc)[bh, jr])], torch.cat(parts))
