"""The radial depthwise forward at the edges of its groups of sixteen copies and
tiles of sixteen edges, against the sums of its definition in float64."""

import pytest
import torch

from gm_attention_amd import _native

pytestmark = pytest.mark.gpu

DEGREES = [0, 1, 15, 16, 17, 33, 0, 100, 2]


@pytest.mark.parametrize("basis", [4, 6, 8])
@pytest.mark.parametrize("a0,orders", [(4, []), (0, [2]), (12, [1, 2, 2]), (16, [2, 1, 2, 1]), (20, [1] * 5 + [2] * 3),
                                       (32, [2] * 15), (32, [1, 2] * 8), (8, [2, 1, 1, 2, 2]), (28, [1] * 9)])
def test_partial_and_mixed_groups_over_ragged_rows(a0, orders, basis, cuda):
    """Frequencies mixed within a group, tiles' columns in any order, dead copies in
    the last group, scalars short of a tile, rows of no edge to several tiles.
    A message's terms are within a few ulp of their magnitudes: the features'
    exponentials (2 ulp), 17 products of the readout and about ten operations a
    copy, so 64 x 2^-24 of the magnitudes' sum bounds the row's error, with one more a sum
    over at most 100 edges."""
    g = torch.Generator().manual_seed(a0 + len(orders) + basis)
    nc, ns, n = len(orders), -(-a0 // 16), len(DEGREES)
    D = a0 + 8 * nc
    rnd = lambda *s: torch.randn(*s, generator=g)
    R = torch.zeros(18, 16, 17)
    R[:ns] = rnd(ns, 16, 17)
    if a0 % 16:
        R[ns - 1, a0 % 16:] = 0
    R[2:2 + nc] = rnd(nc, 16, 17)
    lane = torch.arange(64)
    rf = torch.stack([R[:, lane % 16, 4 * (lane // 16) + s] for s in range(4)], 1).contiguous()
    order = torch.randperm(nc, generator=g)
    tiles = torch.tensor([orders, (a0 + 8 * order).tolist()], dtype=torch.int32).reshape(2, nc)
    row_ptr = torch.zeros(n + 1, dtype=torch.long)
    row_ptr[1:] = torch.tensor(DEGREES).cumsum(0)
    E = int(row_ptr[-1])
    source = torch.randint(n, (E,), generator=g)
    gamma, phi, rho = 3 * rnd(E, 1), 3 * rnd(E, 1), torch.rand(E, generator=g)
    k = torch.arange(5.0)
    phases = lambda x: torch.stack((torch.cos(x * k), torch.sin(x * k)), -1).contiguous()
    transport, angular = phases(gamma), phases(phi)
    w, v, w1, b1 = torch.rand(E, generator=g), rnd(n, D), rnd(16, basis), rnd(16)
    centers, width = [i / (basis - 1) for i in range(basis)], 1.0 / basis
    got = _native.conv_radial_forward(v.to(cuda), rf.to(cuda), R[..., 16].reshape(-1).contiguous().to(cuda), w1.to(cuda),
                                      b1.to(cuda), centers, width, transport.to(cuda), angular.to(cuda), rho.to(cuda),
                                      w.to(cuda), row_ptr.to(cuda), source.to(cuda), a0, ns, tiles).cpu().double()
    f = lambda x: x.double()
    s = f(rho)[:, None] ** 2
    basis_ = torch.exp(-0.5 * ((s - torch.tensor(centers).double()) / width) ** 2)
    pre = basis_ @ f(w1).t() + f(b1)
    h = torch.cat((pre * torch.sigmoid(pre), torch.ones(E, 1).double()), 1)
    C = torch.einsum("mrk,ek->emr", f(R), h)
    size = torch.einsum("mrk,ek->emr", f(R).abs(), h.abs() + (basis_ @ f(w1).abs().t() + f(b1).abs()).max())
    x = f(v)[source]
    message, magnitude = torch.zeros(E, D).double(), torch.zeros(E, D).double()
    for m in range(ns):
        c = slice(16 * m, min(16 * m + 16, a0))
        message[:, c] = C[:, m, :c.stop - c.start] * x[:, c]
        magnitude[:, c] = size[:, m, :c.stop - c.start] * x[:, c].abs()
    for m in range(nc):
        q, col = orders[m], int(tiles[1, m])
        A, B = torch.view_as_complex(C[:, 2 + m].reshape(E, 4, 2, 2).contiguous()).unbind(-1)
        z = torch.view_as_complex(x[:, col:col + 8].reshape(E, 4, 2).contiguous())
        z = z * torch.view_as_complex(f(transport))[:, q, None]
        p = (s ** q) * torch.view_as_complex(f(angular))[:, 2 * q, None]
        message[:, col:col + 8] = torch.view_as_real(A * z + p * B * z.conj()).reshape(E, 8)
        magnitude[:, col:col + 8] = (size[:, 2 + m].reshape(E, 4, 4).sum(-1) * z.abs()).repeat_interleave(2, 1)
    target = torch.repeat_interleave(torch.arange(n), torch.tensor(DEGREES))
    add = lambda t: torch.zeros(n, D).double().index_add_(0, target, f(w)[:, None] * t)
    want, bound = add(message), 164 * 2.0 ** -24 * add(magnitude)
    assert bool((got[torch.tensor(DEGREES) == 0] == 0).all())
    assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() - bound).max())
