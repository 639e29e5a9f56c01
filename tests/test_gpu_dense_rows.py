"""GPU parity of the 128-row dense attention and its row statistics against
float64, at the edges of its blocks (128 rows, 32 per wave) and tiles (64
keys).  Batches and heads make up the work-groups that the dispatch asks for.
Output tolerance as the other 16-bit attention tests; the row's log-sum-exp
within 2e-5 relative (fp32 accumulation of exact products).
"""
import math

import pytest
import torch

from vecattention_amd import _native as nat
from vecattention_amd import stages

pytestmark = pytest.mark.gpu

# name, B, Hq, Hk, Sq, Sk, D, dtype, causal
CASES = [
    ("one-row", 40, 16, 4, 1, 1, 128, torch.bfloat16, True),
    ("causal-257", 10, 28, 4, 257, 257, 128, torch.bfloat16, True),
    ("causal-127-of-333", 40, 16, 16, 127, 333, 64, torch.float16, True),
    ("causal-129-of-1000", 10, 32, 8, 129, 1000, 128, torch.float16, True),
    ("dense-65-of-63", 24, 16, 8, 65, 63, 128, torch.bfloat16, False),
    ("dense-300-of-321", 8, 16, 16, 300, 321, 64, torch.bfloat16, False),
    ("dense-1-of-700", 24, 16, 2, 1, 700, 128, torch.bfloat16, False),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_dense_attention_and_statistics(case):
    name, B, Hq, Hk, Sq, Sk, D, dtype, causal = case
    print("[case] dense rows", name, flush=True)
    assert nat.lib().va_dense_rows(B, Hq, Sq, causal) == 128
    g = torch.Generator().manual_seed(5)
    q = torch.randn(B, Sq, Hq, D, generator=g).to(dtype).transpose(1, 2)
    k = torch.randn(B, Hk, Sk, D, generator=g)
    k[:, :, Sk // 3] *= 6.0  # the running maximum moves late and by more than its slack
    k, v = k.to(dtype), torch.randn(B, Hk, Sk, D, generator=g).to(dtype)
    qd, kd, vd = q.to("cuda:0"), k.to("cuda:0"), v.to("cuda:0")
    out = stages.dense_attention(qd, kd, vd, causal=causal)
    stats = stages.dense_row_stats(qd, kd, causal)
    torch.cuda.synchronize()
    s = q.double() @ k.double().repeat_interleave(Hq // Hk, 1).transpose(2, 3) / math.sqrt(D)
    if causal:
        see = torch.arange(Sk)[None] <= torch.arange(Sq)[:, None] + Sk - Sq
        s = s.masked_fill(~see, -math.inf)
    want = torch.softmax(s, -1) @ v.double().repeat_interleave(Hq // Hk, 1)
    err = (out.double().cpu() - want).abs()
    assert err.max() <= 2e-2 and err.mean() <= 2e-3, (err.max(), err.mean())
    st = stats.double().cpu()
    lse = (st[..., 0] + torch.log2(st[..., 1])) * math.log(2.0)
    ref = torch.logsumexp(s, -1)
    assert ((lse - ref).abs() <= 2e-5 * ref.abs().clamp(min=1.0)).all()


def test_keys_past_the_end_add_nothing():
    # Key rows behind the tensors' ends hold infinities; the last tile's empty
    # slots must not read them.
    B, Hq, Sq, Sk, D = 24, 16, 70, 70, 128
    assert nat.lib().va_dense_rows(B, Hq, Sq, False) == 128
    g = torch.Generator().manual_seed(6)
    q = torch.randn(B, Hq, Sq, D, generator=g).bfloat16().to("cuda:0")
    kv = [torch.full((B, Hq, Sk + 58, D), math.inf) for _ in range(2)]
    for x in kv:
        x[:, :, :Sk] = torch.randn(B, Hq, Sk, D, generator=g)
    k, v = (x.bfloat16().to("cuda:0")[:, :, :Sk] for x in kv)
    out = stages.dense_attention(q, k, v, causal=False)
    want = torch.softmax(q.double() @ k.double().transpose(2, 3) / math.sqrt(D), -1) @ v.double()
    assert (out.double() - want).abs().max() <= 2e-2


# name, Hq, Hk, S, D, dtype, causal: all heads at once take the 128-row form,
# one head at a time the 64-row form (too few work-groups).
ERROR_CASES = [
    ("causal-bf16", 28, 4, 3000, 128, torch.bfloat16, True),
    ("causal-fp16-d64", 32, 8, 2600, 64, torch.float16, True),
    ("dense-bf16", 28, 4, 2048, 128, torch.bfloat16, False),
]


@pytest.mark.parametrize("case", ERROR_CASES, ids=[c[0] for c in ERROR_CASES])
def test_error_is_no_larger_than_the_64_row_forms(case):
    # Both forms round their probabilities to 16 bits against a running
    # maximum; the 64-row form has two of them per row.  The bound is the
    # 64-row form's own error against float64 on the same inputs.
    name, Hq, Hk, S, D, dtype, causal = case
    print("[case] dense error", name, flush=True)
    assert nat.lib().va_dense_rows(1, Hq, S, causal) == 128
    assert nat.lib().va_dense_rows(1, 1, S, causal) == 64
    g = torch.Generator().manual_seed(14)
    q, k, v = (torch.randn(1, h, S, D, generator=g).to(dtype).to("cuda:0") for h in (Hq, Hk, Hk))
    both = stages.dense_attention(q, k, v, causal=causal)
    err = torch.zeros(2, dtype=torch.float64)
    for h in range(Hq):
        kh, vh = (x[:, h // (Hq // Hk):][:, :1] for x in (k, v))
        one = stages.dense_attention(q[:, h:h + 1], kh, vh, causal=causal)
        s = q[0, h].double() @ kh[0, 0].double().T / math.sqrt(D)
        if causal:
            s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
        want = torch.softmax(s, -1) @ vh[0, 0].double()
        for i, got in enumerate((both[0, h], one[0, 0])):
            err[i] += (got.double() - want).square().sum().cpu()
    assert err[0] <= err[1], err.sqrt()
