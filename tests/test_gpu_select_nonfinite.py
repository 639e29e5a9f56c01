"""Selections with infinities, NaNs and values near overflow (run on an MI355X):
the 16-bit kernels, whose decisions read signs and bit patterns of score
differences, against the fp64 kernel, which compares exact scores: lists bit
for bit.  A score of NaN is never selected and moves no maximum.  Rows that end
inside a wave's 32, causal limits before and after the odd key, segments and
the two-pass form; and the fp32 kernels against each other.
"""
import math

import pytest
import torch

from vecattention_amd import _native as nat
from vecattention_amd import stages

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF, FP = torch.bfloat16, torch.float16
# name, B, Hq, Hk, Sk, D, dtype, qps, bk, G, causal, J0, nc, segk (0: unsplit)
FORMS = [
    ("tiles128-causal", 1, 4, 2, 128 * 21, 128, BF, 128, 128, 1, True, 0, 21, 0),
    ("tiles128-causal-segments", 2, 2, 1, 128 * 38, 64, FP, 128, 128, 1, True, 1, 37, 512),
    ("tiles128", 1, 2, 2, 1100, 128, FP, 128, 128, 1, False, 0, 33, 0),
    ("wave-causal", 1, 4, 2, 64 * 40, 128, BF, 64, 16, 16, True, 3, 37, 0),
    ("wave-bk32-segments", 1, 2, 2, 1500, 64, FP, 64, 32, 4, False, 0, 40, 256),
    ("wave-bk64-causal", 1, 2, 1, 64 * 34, 64, FP, 64, 64, 2, True, 0, 34, 0),
    ("wave-groups-of-16", 1, 2, 1, 64 * 35, 128, BF, 64, 16, 1, True, 0, 35, 512),
    ("two-pass-causal", 1, 2, 2, 64 * 40, 128, BF, 64, 16, 8192, True, 0, 40, 320),
    ("two-pass", 1, 3, 3, 2333, 64, FP, 64, 32, 8192, False, 0, 37, 256),
    ("64-row-span48", 1, 2, 1, 64 * 36, 128, BF, 64, 16, 3, True, 0, 36, 0),
    ("64-row-bk256", 1, 2, 2, 2100, 64, FP, 256, 256, 2, False, 0, 9, 0),
]
ODD = ["inf-key", "minus-inf-key", "nan-key", "huge-keys", "nan-row", "inf-row", "gaps"]


def _odd_values(odd, qs, k, Hq):
    """Plants the odd values: keys late in K (the last head's), rows of head 0."""
    gaps = None
    Sk, top = k.shape[2], torch.finfo(k.dtype).max
    if odd == "inf-key":
        k[:, -1, (3 * Sk) // 4, 5] = math.inf
    elif odd == "minus-inf-key":
        k[:, -1, Sk // 2, 3] = -math.inf
    elif odd == "nan-key":
        k[:, -1, Sk // 2, 7] = math.nan
        k[:, -1, Sk // 2 + 3, 7] = -math.nan
    elif odd == "huge-keys":
        # bf16: squared norms past fp32; fp16: the type's largest values
        k[:, -1, Sk // 3] = top / 1e18 if k.dtype == BF else top
        k[:, -1, (2 * Sk) // 3] = -top / 1e18 if k.dtype == BF else -top
    elif odd == "nan-row":
        qs[:, 0, qs.shape[2] // 2, 1] = math.nan
    elif odd == "inf-row":
        qs[:, 0, qs.shape[2] - 1, 2] = math.inf
    else:
        gaps = torch.full((qs.shape[0], Hq), 0.5, device=DEV)
        gaps[:, 0], gaps[:, -1] = math.inf, math.nan
    return gaps


def _lists(counts, indices, B, Hq, nc, Sk, qps, causal, J0, segk):
    counts, indices = counts.cpu().reshape(B * Hq, nc, -1), indices.cpu()
    smin = qps if causal else 0
    out = []
    for bh in range(B * Hq):
        for jr in range(nc):
            o = stages.row_offset(Sk, qps, causal, causal, J0, nc, bh, jr)
            out.append(torch.cat([
                indices[o + s0:o + s0 + int(counts[bh, jr, s])] for s in range(counts.shape[2])
                for s0 in [max(s * segk, smin) - smin if segk else 0]]))
    return out


@pytest.mark.parametrize("odd", ODD)
@pytest.mark.parametrize("form", FORMS, ids=[f[0] for f in FORMS])
def test_lists_equal_exact_lists(form, odd):
    name, B, Hq, Hk, Sk, D, dtype, qps, bk, G, causal, J0, nc, segk = form
    print("[case] odd values", name, odd, flush=True)
    g = torch.Generator().manual_seed(15)
    qs = (0.1 * torch.randn(B, Hq, nc, D, generator=g)).to(dtype).to(DEV)
    k = torch.randn(B, Hk, Sk, D, generator=g).to(dtype).to(DEV)
    k[:, :, 9] = k[:, :, 8]
    gaps = _odd_values(odd, qs, k, Hq)
    gap = 0.0 if gaps is not None else 0.3
    args = (J0, gap, gaps, causal, qps, bk, G, causal)
    want = _lists(*stages.select_rows(qs, k, *args, kernel=nat.VA_SEL_EXACT), B, Hq, nc, Sk, qps,
                  causal, J0, 0)
    if segk:
        got = stages.select_segments(qs, k, *args, segk)
    else:
        got = stages.select_rows(qs, k, *args)
    got = _lists(*got, B, Hq, nc, Sk, qps, causal, J0, segk)
    assert sum(len(w) for w in want) > 0
    for r, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), (r // nc, r % nc, len(a), len(b))


@pytest.mark.parametrize("segk", [0, 256])
@pytest.mark.parametrize("odd", ["inf-key", "minus-inf-key", "nan-key", "nan-row", "inf-row", "gaps"])
def test_fp32_lists_equal_vector_lists(odd, segk):
    # aligned keys take the matrix cores, keys 4 bytes off the vector kernel
    B, Hq, Hk, Sk, D, qps, bk, G, nc = 4, 8, 4, 1500, 64, 64, 16, 8192 if segk else 4, 50
    print("[case] odd fp32 values", odd, segk, flush=True)
    g = torch.Generator().manual_seed(16)
    qs = (0.1 * torch.randn(B, Hq, nc, D, generator=g)).to(DEV)
    k = torch.randn(B, Hk, Sk, D, generator=g).to(DEV)
    gaps = _odd_values(odd, qs, k, Hq)
    flat = torch.empty(k.numel() + 1, device=DEV)
    flat[1:] = k.reshape(-1)
    lists = []
    for kk, matrix in ((k, 1), (flat[1:].view(k.shape), 0)):
        assert nat.lib().va_select_exact_matrix_cores(nat.ptr(kk), *kk.stride()[:3], B, Hq, Sk, D,
                                                      nc, segk) == matrix
        args = (0, 0.0 if gaps is not None else 0.3, gaps, False, qps, bk, G, False)
        res = (stages.select_segments(qs, kk, *args, segk) if segk
               else stages.select_rows(qs, kk, *args))
        lists.append(_lists(*res, B, Hq, nc, Sk, qps, False, 0, segk))
    assert all(torch.equal(a, b) for a, b in zip(*lists))
