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
    ("skips-first-block", 1, 2, 2, 1500, 128, torch.bfloat16, False, 0, 35, 0, 0.4, False),
    ("skips-first-block-segments", 2, 2, 1, 1000, 64, torch.float16, False, 0, 20, 256, 0.4, False),
    ("skips-every-key", 1, 2, 2, 100, 64, torch.bfloat16, False, 0, 3, 0, 0.4, False),
    ("all-ambiguous", 1, 1, 1, 384, 128, torch.bfloat16, False, 0, 5, 0, 0.0, True),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_tile_lists_equal_exact_lists(case):
    name, B, Hq, Hk, Sk, D, dtype, causal, J0, nc, segk, gap, dup = case
    print("[case] tile selection", name, flush=True)
    qps, bk, G = 128, 128, 1
    wo_init = causal or name.startswith("skips")
    g = torch.Generator().manual_seed(9)
    qs = (0.1 * torch.randn(B, Hq, nc, D, generator=g)).to(dtype).to(DEV)
    k = torch.randn(B, Hk, Sk, D, generator=g)
    if dup:
        k = k[:, :, torch.arange(Sk) % (3 if name == "all-ambiguous" else 50)]
    k = k.to(dtype).to(DEV)
    want, wi = stages.select_rows(qs, k, J0, gap, None, causal, qps, bk, G, wo_init,
                                  kernel=nat.VA_SEL_EXACT)
    if segk:
        got, gi = stages.select_segments(qs, k, J0, gap, None, causal, qps, bk, G, wo_init, segk)
    else:
        got, gi = stages.select_rows(qs, k, J0, gap, None, causal, qps, bk, G, wo_init,
                                     kernel=nat.VA_SEL_MFMA)
    want, wi, got, gi = want.cpu(), wi.cpu(), got.cpu(), gi.cpu()
    nseg = got.shape[-1] if segk else 1
    got = got.reshape(B * Hq, nc, nseg)
    assert torch.equal(want.reshape(B * Hq, nc), got.sum(-1))
    assert (int(want.sum()) > 0) == (name != "skips-every-key")
    smin = min(qps, Sk) if wo_init else 0
    for bh in range(B * Hq):
        for jr in range(nc):
            o = stages.row_offset(Sk, qps, causal, wo_init, J0, nc, bh, jr)
            parts = [gi[o + s0:o + s0 + int(got[bh, jr, s])] for s in range(nseg)
                     for s0 in [max(s * segk, smin) - smin if segk else 0]]
            assert torch.equal(wi[o:o + int(want.reshape(B * Hq, nc)[bh, jr])], torch.cat(parts))


@pytest.mark.parametrize("segk", [0, 256])
@pytest.mark.parametrize("qps,bk,G", [(128, 128, 1), (64, 16, 16)], ids=["tiles128", "wave"])
def test_dense_rows_of_2_to_25_slots(qps, bk, G, segk):
    # 32 rows of that stride are 2^32 bytes: the lists of a full wave and of the
    # row after it.
    B, H, Sk, D, nc, stride = 1, 1, 700, 64, 33, 1 << 25
    print("[case] dense rows", qps, segk, flush=True)
    g = torch.Generator().manual_seed(17)
    qs = (0.1 * torch.randn(B, H, nc, D, generator=g)).bfloat16().to(DEV)
    k = torch.randn(B, H, Sk, D, generator=g).bfloat16().to(DEV)
    want, wi = stages.select_rows(qs, k, 0, 0.5, None, False, qps, bk, G, False,
                                  kernel=nat.VA_SEL_EXACT)
    wi = wi.view(nc, Sk)
    idx = torch.full((nc * stride,), -1, dtype=torch.int32, device=DEV)
    args = (qs, k, 0, 0.5, None, False, qps, bk, G, False)
    if segk:
        got, _ = stages.select_segments(*args, segk, dense_stride=stride, indices=idx)
    else:
        got, _ = stages.select_rows(*args, dense_stride=stride, indices=idx)
    got = got.reshape(nc, -1)
    assert torch.equal(got.sum(-1), want.reshape(nc)) and int(want.min()) > 0
    rows = idx.view(nc, stride)
    for r in range(nc):
        parts = [rows[r, s * segk:s * segk + int(n)] for s, n in enumerate(got[r])]
        assert torch.equal(torch.cat(parts), wi[r, :int(want[0, 0, r])]), r
