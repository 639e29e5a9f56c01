"""The tuner's bf16 copies of fp32 tensors (run on an MI355X): the values torch
rounds to, and None as soon as one value is not a bf16 value."""
import pytest
import torch

from vecattention_amd.tuner import _bf16_copies

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 2047, 2056, 100003])
def test_bf16_copies(n):
    print("[case] bf16 copies", n, flush=True)
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, generator=g).bfloat16()
    special = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), 1e-40, 3.0])[:n]
    x[:special.numel()] = special.bfloat16()
    x = x.float().to("cuda:0")
    (c, d) = _bf16_copies(x, x.flip(0))
    assert torch.equal(c.view(torch.int16), x.to(torch.bfloat16).view(torch.int16))
    assert torch.equal(d.float(), x.flip(0))
    for bad in (1.0 + 2.0 ** -9, float("nan"), 1e-45):
        for at in {0, n - 1, n // 2}:
            y = x.clone()
            y[at] = bad
            assert _bf16_copies(x, y) is None and _bf16_copies(y, x) is None, (bad, at)
    assert torch.equal(_bf16_copies(x[1:], x[1:])[0].float(), x[1:]) if n > 1 else True  # unaligned
