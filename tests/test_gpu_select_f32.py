"""The fp32 selection on the fp64 matrix cores against the vector fp64 kernel
(run on an MI355X): the same lists bit for bit, for every tile size and form.

Keys at an address that is not a multiple of 16 bytes take the vector kernel
(sequential fused multiply-adds), aligned ones the matrix cores; both get the
same values.  The inputs spread their exponents and cancel, so that a sum in
any other order, or one that is not fused, would round differently for a part
of the scores, and gap 0 and ties make a changed score change a list.
"""
import pytest
import torch

from vecattention_amd import _native as nat
from vecattention_amd import stages

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
# name, B, Hq, Hk, Sk, D, qps, bk, G, causal, J0, nc, segk, gap
CASES = [
    ("rows8-tail", 12, 8, 8, 700, 64, 64, 16, 4, False, 0, 8, 0, 0.5),
    ("rows17-causal", 6, 8, 4, 64 * 20, 128, 64, 16, 16, True, 3, 17, 0, 0.5),
    ("gap0-groups-of-16", 4, 8, 4, 1000, 128, 64, 16, 1, False, 0, 33, 0, 0.0),
    ("tiles32-split", 2, 4, 2, 1500, 64, 64, 32, 16, False, 0, 40, 512, 0.25),
    ("tiles128-causal", 12, 8, 8, 128 * 12, 128, 128, 128, 2, True, 0, 12, 0, 0.5),
    ("tiles256-split", 2, 6, 3, 2100, 128, 256, 256, 1, False, 0, 9, 512, 0.1),
    ("one-group-two-pass", 1, 3, 3, 2333, 128, 64, 16, 8192, False, 0, 37, 256, 0.5),
    ("one-group-two-pass-causal", 1, 2, 2, 64 * 40, 64, 64, 16, 8192, True, 0, 40, 320, 0.5),
    ("wide", 4, 16, 16, 2048, 128, 64, 16, 16, False, 0, 33, 256, 0.5),
    ("wide-two-pass", 4, 16, 8, 2040, 64, 64, 16, 8192, False, 0, 34, 256, 0.5),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_matrix_core_lists_equal_vector_lists(case):
    name, B, Hq, Hk, Sk, D, qps, bk, G, causal, J0, nc, segk, gap = case
    print("[case] fp32 selection", name, flush=True)
    g = torch.Generator().manual_seed(3)
    qs = torch.randn(B, Hq, nc, D, generator=g)
    k = torch.randn(B, Hk, Sk, D, generator=g)
    # exponents over 2^16 that pair up to scores of one size, and duplicates
    e = torch.randint(-8, 9, (D,), generator=g).float()
    qs, k = qs * torch.exp2(e), k * torch.exp2(-e)
    k[:, :, 1::2, : D // 2] *= 64.0
    k[:, :, 1::2, D // 2:] = -k[:, :, 1::2, : D // 2] * (1 + 2.0 ** -20)
    k[:, :, 5 % Sk] = k[:, :, 0]
    qs, ka = qs.to(DEV), k.to(DEV)
    flat = torch.empty(k.numel() + 1, device=DEV)
    flat[1:] = ka.reshape(-1)
    ku = flat[1:].view(B, Hk, Sk, D)
    assert ka.data_ptr() % 16 == 0 and ku.data_ptr() % 16 == 4
    got = []
    for kk, matrix in ((ka, 1), (ku, 0)):
        assert nat.lib().va_select_exact_matrix_cores(nat.ptr(kk), *kk.stride()[:3], B, Hq, Sk, D,
                                                      nc, segk) == matrix
        if segk:
            cnt, idx = stages.select_segments(qs, kk, J0, gap, None, causal, qps, bk, G, causal,
                                              segk)
        else:
            cnt, idx = stages.select_rows(qs, kk, J0, gap, None, causal, qps, bk, G, causal)
        got.append((cnt.cpu(), idx.cpu()))
    (ca, ia), (cu, iu) = got
    assert torch.equal(ca, cu) and int(ca.sum()) > 0
    nseg = ca.shape[-1] if segk else 1
    smin = qps if causal else 0
    for bh in range(B * Hq):
        for jr in range(nc):
            off = stages.row_offset(Sk, qps, causal, causal, J0, nc, bh, jr)
            for s in range(nseg):
                n = int(ca.reshape(B * Hq, nc, nseg)[bh, jr, s])
                o = off + (max(s * segk, smin) - smin if segk else 0)
                assert torch.equal(ia[o:o + n], iu[o:o + n]), (bh, jr, s)
