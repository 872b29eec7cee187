"""The all-heads aggregate with four waves a target (small launches) and with one
(large ones), on both sides of the line between them."""

import pytest
import torch

from gm_attention_amd import _native

pytestmark = pytest.mark.gpu

LINE = 7 << 19  # targets x 16-byte output pieces (40 or more) up to which a target takes four waves


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d_out,n", [(1, 4, 1), (8, 20, 9), (6, 20, 700), (16, 20, 333), (48, 16, 65),
                                       (16, 64, LINE // 256), (16, 64, LINE // 256 + 1),
                                       (1, 32, LINE // 40), (1, 32, LINE // 40 + 1)])
def test_aggregate_on_both_sides_of_the_line(H, d_out, n, dtype, cuda):
    """Degrees of no edge, fewer than a wave's step, quarters that end early and
    rows of thousands, against float64 sums: n products added in any order are
    within (n + 4) 2^-24 of the sum of their magnitudes (one rounding a
    product, n sums from zero, three joins of quarters)."""
    g = torch.Generator().manual_seed(n + H)
    degree = torch.tensor([0, 1, 3, 4, 5, 8, 13, 16, 17], dtype=torch.long).repeat(-(-n // 9))[:n]
    if n < 1000:
        degree[n // 2] = 3001
        degree[n - 1] = 2048
    row_ptr = torch.zeros(n + 1, dtype=torch.long)
    row_ptr[1:] = degree.cumsum(0)
    E = int(row_ptr[-1])
    rows = torch.randn(H, E, d_out, generator=g).to(dtype)
    alpha, inv = torch.rand(E, H, generator=g), torch.randperm(E, generator=g)
    rows, alpha, inv, row_ptr, degree = (t.to(cuda) for t in (rows, alpha, inv, row_ptr, degree))
    got = _native.aggregate_heads(rows, inv, alpha, row_ptr, 1)
    target = torch.repeat_interleave(torch.arange(n, device=cuda), degree)
    for h in range(H):
        terms = alpha[:, h, None].double() * rows[h, inv].double()
        want = torch.zeros(n, d_out, dtype=torch.float64, device=cuda).index_add_(0, target, terms)
        size = torch.zeros(n, d_out, dtype=torch.float64, device=cuda).index_add_(0, target, terms.abs())
        bound = (degree + 4)[:, None].double() * 2.0 ** -24 * size
        assert bool(((got[:, h].double() - want).abs() <= bound).all()), (h, float((got[:, h] - want).abs().max()))
