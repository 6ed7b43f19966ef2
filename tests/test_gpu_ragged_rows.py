"""GPU: rows that the vector width does not divide, at any alignment.

Widths around one vector (the last lane's vector overlaps its neighbour), around a slice, and
odd ones; rows off every alignment (views one element into their buffer); guard elements
around every output; outputs that are one of the inputs, which take a dividing vector instead.
An element's value does not depend on the vector width: it is compared with the oracle at the
parity bar and, bit for bit, with the same values in aligned rows.
"""
from __future__ import annotations

import pytest
import torch

from helpers import announce, assert_parity
from oracle import sihc_oracle as O
from sihc_hip import launch

pytestmark = pytest.mark.gpu

GUARD = 64


def _off(t):
    """t's values in a packed view that starts one element into its buffer."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    return buf[1:].copy_(t.reshape(-1)).view(t.shape)


class Out:
    """A packed output one element off alignment, with sentinels on both sides."""

    def __init__(self, shape, dtype):
        n = 1
        for s in shape:
            n *= s
        self.buf = torch.full((n + 2 * GUARD + 1,), 7.0, dtype=dtype, device="cuda")
        self.t = self.buf[GUARD + 1:GUARD + 1 + n].view(shape)

    def check(self):
        assert (self.buf[:GUARD + 1] == 7).all() and (self.buf[-GUARD:] == 7).all()
        return self.t


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("slots", [4, 16])
@pytest.mark.parametrize("channels", [3, 8, 9, 15, 67, 129, 130, 259, 1001])
def test_ragged_rows(dtype, slots, channels):
    announce(f"ragged rows C={channels} slots={slots} {dtype}")
    gen = torch.Generator().manual_seed(channels * slots)
    k, b, g, c, events = O.cell_edge(slots), 2, 5, channels, 5

    def draw(*shape, scale=1.0):
        return (scale * torch.randn(*shape, generator=gen)).to(dtype)

    x, z = draw(b, k * g, k * g, c), [draw(b, g * g, c) for _ in range(events)]
    w = (1 / slots + 0.1 * draw(events, c, slots).float()).to(dtype)
    xo, zo, wd = _off(x.cuda()), [_off(t.cuda()) for t in z], w.cuda()

    outs = [Out((b, g * g, c), dtype) for _ in range(events)]
    launch.read(xo, wd, out=[o.t for o in outs])
    aligned = launch.read(x.cuda(), wd)
    for o, a, want in zip(outs, aligned, O.read(x, w)):
        assert_parity(o.check(), want, dtype, what="read")
        assert torch.equal(o.t, a)

    out = Out(x.shape, dtype)
    launch.write(xo, zo, wd, out=out.t)
    want = O.write(x, z, w)
    assert_parity(out.check(), want, dtype, what="write")
    inplace = x.cuda().clone()
    launch.write(inplace, zo, wd, out=inplace)  # every element read and written by one lane
    assert torch.equal(inplace, out.t)

    x1, z1 = launch.event_forward(xo, zo[0], wd[0], wd[1])
    rx, rz = O.event_forward(x, z[0], w[0], w[1])
    assert_parity(x1, rx, dtype, what="event x")
    assert_parity(z1, rz, dtype, what="event z")
    got = launch.event_backward(_off(x1), zo[1], xo, zo[0], wd[0], wd[1])
    want = O.event_backward(x1.cpu(), z[1], x, z[0], w[0], w[1])
    for name, a, e, kind in zip(("dX", "ddz", "dbeta", "dalpha"), got, want, ("elementwise",) * 2 + ("reduced",) * 2):
        assert_parity(a, e.to(dtype), dtype, what=name, kind=kind)
    gx = _off(x1)
    same = launch.event_backward(gx, zo[1], xo, zo[0], wd[0], wd[1], grad_x=gx)  # dX over its gradient
    assert torch.equal(same[0], got[0]) and torch.equal(same[1], got[1])

    for active in (1, 2, 3, 5):
        gamma = draw(active, c).float()
        t = launch.triangular(zo[4], zo[:active], gamma.cuda())
        assert_parity(t, O.triangular_torch(z[4], z[:active], gamma), dtype, what="triangular")
        assert torch.equal(t, launch.triangular(z[4].cuda(), [u.cuda() for u in z[:active]], gamma.cuda()))
        dg = O.triangular_gamma_grad(z[4], z[:active])
        assert_parity(launch.triangular_gamma_grad(zo[4], zo[:active], None, out_dtype=torch.float32), dg,
                      torch.float32, what="dgamma")
        ddz, fused = launch.triangular_backward(zo[4], zo[:active], gamma.cuda(), out_dtype=torch.float32)
        assert_parity(fused, dg, torch.float32, what="fused dgamma")
        for j in range(active):
            assert torch.equal(ddz[j].cpu(), (z[4].float() * gamma[j]).to(dtype))

    index = torch.stack([torch.randperm(g * g, generator=gen) for _ in range(b)]).to(torch.int32)
    cells = launch.gather_cells(xo, index.cuda(), slots)
    assert torch.equal(cells.cpu(), O.gather_cells(x, index, slots))
    back = Out(x.shape, dtype)
    launch.scatter_cells(_off(cells), index.cuda(), out=back.t)
    assert torch.equal(back.check(), x.cuda())
    back = Out(x.shape, dtype)
    launch.scatter_add_cells(_off(cells), index.cuda(), out=back.t)
    assert torch.equal(back.check(), x.cuda())
