"""The two-pass selection (one group per row) on the MFMA kernels against the
fp64 kernel, lists bit for bit (run on an MI355X): the maxima pass hands on up
to four candidate tiles per row and segment, or an exact maximum where more
keys tie for it (duplicated keys; gap 0 makes every decision depend on it).
"""
import pytest
import torch

from vecattention_amd import _native as nat
from vecattention_amd import stages

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# name, B, Hq, Hk, Sk, D, dtype, qps, bk, causal, J0, nc, segk, gap, distinct keys (0: all)
CASES = [
    ("random-tail", 1, 3, 3, 2001, 128, torch.bfloat16, 64, 16, False, 0, 33, 256, 0.3, 0),
    ("one-row-one-chunk", 1, 2, 1, 130, 64, torch.float16, 64, 32, False, 0, 1, 64, 0.3, 0),
    ("pairs-of-ties", 1, 2, 2, 1600, 128, torch.bfloat16, 64, 16, False, 0, 40, 320, 0.0, 800),
    ("many-ties", 2, 2, 1, 1000, 64, torch.bfloat16, 64, 16, False, 0, 7, 128, 0.0, 7),
    ("all-equal", 1, 1, 1, 300, 128, torch.float16, 64, 64, False, 0, 3, 64, 0.0, 1),
    ("causal-ties", 1, 4, 2, 64 * 30, 128, torch.bfloat16, 64, 32, True, 5, 25, 192, 0.1, 300),
    ("rows129-bk64", 1, 2, 2, 1300, 64, torch.float16, 64, 64, False, 0, 129, 512, 0.2, 0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_two_pass_lists_equal_exact_lists(case):
    name, B, Hq, Hk, Sk, D, dtype, qps, bk, causal, J0, nc, segk, gap, distinct = case
    print("[case] maxima pass", name, flush=True)
    G = 8192
    g = torch.Generator().manual_seed(10)
    qs = (0.1 * torch.randn(B, Hq, nc, D, generator=g)).to(dtype).to(DEV)
    k = torch.randn(B, Hk, distinct or Sk, D, generator=g)
    k = k[:, :, torch.arange(Sk) % k.shape[2]].to(dtype).to(DEV)
    want, wi = stages.select_rows(qs, k, J0, gap, None, causal, qps, bk, G, causal,
                                  kernel=nat.VA_SEL_EXACT)
    got, gi = stages.select_segments(qs, k, J0, gap, None, causal, qps, bk, G, causal, segk)
    want, wi, got, gi = want.cpu().reshape(-1), wi.cpu(), got.cpu(), gi.cpu()
    nseg = got.shape[-1]
    got = got.reshape(-1, nseg)
    assert torch.equal(want, got.sum(-1)) and int(want.sum()) > 0
    smin = qps if causal else 0
    for r in range(B * Hq * nc):
        o = stages.row_offset(Sk, qps, causal, causal, J0, nc, r // nc, r % nc)
        parts = [gi[o + s0:o + s0 + int(got[r, s])] for s in range(nseg)
                 for s0 in [max(s * segk, smin) - smin]]
        assert torch.equal(wi[o:o + int(want[r])], torch.cat(parts)), r


@pytest.mark.parametrize("D,dtype,bk,causal", [(128, torch.bfloat16, 16, False),
                                               (64, torch.bfloat16, 32, True)])
def test_tied_rows_sum_in_order(D, dtype, bk, causal):
    # The first and the last feature cancel at 2^58 and the sum in between is
    # rounded to what fp64 holds beside them, so the scores are ties whose value
    # depends on the order of the sum; the error bound makes every key a
    # candidate, and every row takes the exact scores of whole segments.
    print("[case] maxima pass, order of the sum", D, flush=True)
    qps, G, segk, Sk, nc = 64, 8192, 256, 64 * 34, 34
    g = torch.Generator().manual_seed(18)
    qs = torch.randn(1, 2, nc, D, generator=g) * 8
    k = torch.randn(1, 2, Sk, D, generator=g) * 8
    qs[..., 0] = qs[..., -1] = 2.0 ** 29
    k[..., 0], k[..., -1] = 2.0 ** 29, -(2.0 ** 29)
    qs, k = qs.to(dtype).to(DEV), k.to(dtype).to(DEV)
    want, wi = stages.select_rows(qs, k, 0, 0.0, None, causal, qps, bk, G, causal,
                                  kernel=nat.VA_SEL_EXACT)
    got, gi = stages.select_segments(qs, k, 0, 0.0, None, causal, qps, bk, G, causal, segk)
    want, wi, got, gi = want.cpu().reshape(-1), wi.cpu(), got.cpu(), gi.cpu()
    nseg = got.shape[-1]
    got = got.reshape(-1, nseg)
    assert torch.equal(want, got.sum(-1)) and int(want.max()) > 1
    smin = qps if causal else 0
    for r in range(2 * nc):
        o = stages.row_offset(Sk, qps, causal, causal, 0, nc, r // nc, r % nc)
        parts = [gi[o + s0:o + s0 + int(got[r, s])] for s in range(nseg)
                 for s0 in [max(s * segk, smin) - smin]]
        assert torch.equal(wi[o:o + int(want[r])], torch.cat(parts)), r
