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
from sihc_hip._lib import check, lib, ptr_array

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


# Tokens for which the launches hold more blocks than a device has CUs, so that rows a vector does
# not divide take it all the same (smaller grids keep a dividing one).
MANY = (64, 16)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("channels", [24, 67, 130, 259])
def test_ragged_rows_of_large_grids(dtype, channels):
    """Reads, writes, triangular and the per-event backward at 16,384 tokens: the oracle's values,
    and the bits of whole rows one element off alignment."""
    announce(f"ragged rows, large grid C={channels} {dtype}")
    gen = torch.Generator().manual_seed(channels)
    (b, g), c, events = MANY, channels, 3

    def draw(*shape, scale=1.0):
        return (scale * torch.randn(*shape, generator=gen)).to(dtype)

    x, z = draw(b, 2 * g, 2 * g, c), [draw(b, g * g, c) for _ in range(events)]
    w, gamma = (0.25 + 0.1 * draw(events, c, 4).float()).to(dtype), draw(events, c).float()
    xd, zd, wd, gd = x.cuda(), [t.cuda() for t in z], w.cuda(), gamma.cuda()
    outs = [Out((b, g * g, c), dtype) for _ in range(events)]
    launch.read(_off(xd), wd, out=[o.t for o in outs])
    for o, want, a in zip(outs, O.read(x, w), launch.read(xd, wd)):
        assert_parity(o.check(), want, dtype, what="read")
        assert torch.equal(o.t, a)
    out = Out(x.shape, dtype)
    launch.write(_off(xd), [_off(t) for t in zd], wd, out=out.t)
    assert_parity(out.check(), O.write(x, z, w), dtype, what="write")
    assert torch.equal(out.t, launch.write(xd, zd, wd))
    for active in (1, 3):
        got = launch.triangular(_off(zd[2]), [_off(t) for t in zd[:active]], gd[:active].contiguous())
        assert_parity(got, O.triangular_torch(z[2], z[:active], gamma[:active]), dtype, what="triangular")
    got = launch.event_backward(_off(xd), _off(zd[1]), xd, zd[0], wd[0], wd[1])
    want = O.event_backward(x, z[1], x, z[0], w[0], w[1])
    for name, a, e, kind in zip(("dX", "ddz", "dbeta", "dalpha"), got, want, ("elementwise",) * 2 + ("reduced",) * 2):
        assert_parity(a, e.to(dtype), dtype, what=name, kind=kind)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("batch", [16, 64])  # 32-lane reads from three blocks per CU
@pytest.mark.parametrize("channels,events", [(67, 12), (131, 12), (131, 20), (195, 20)])
def test_ragged_rows_of_many_events(dtype, batch, channels, events):
    """Both sides of the lines at which many-event reads and writes keep a dividing vector."""
    announce(f"ragged rows, batch {batch} C={channels} E={events} {dtype}")
    gen = torch.Generator().manual_seed(channels + events)
    x = torch.randn(batch, 32, 32, channels, generator=gen).to(dtype)
    z = [torch.randn(batch, 256, channels, generator=gen).to(dtype) for _ in range(events)]
    w = (0.25 + 0.1 * torch.randn(events, channels, 4, generator=gen)).to(dtype)
    outs = [Out(z[0].shape, dtype) for _ in range(events)]
    launch.read(_off(x.cuda()), w.cuda(), out=[o.t for o in outs])
    for o, want in zip(outs, O.read(x, w)):
        assert_parity(o.check(), want, dtype, what="read")
    out = Out(x.shape, dtype)
    launch.write(_off(x.cuda()), [_off(t.cuda()) for t in z], w.cuda(), out=out.t)
    assert_parity(out.check(), O.write(x, z, w), dtype, what="write")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,updates", [(1, 9), (1, 32), (4, 4), (4, 5), (4, 11), (64, 5)])
def test_ragged_triangular_backward_of_few_rows(dtype, rows, updates):
    """Both sides of the lines up to which many updates keep a dividing vector."""
    gen = torch.Generator().manual_seed(updates)
    grad, *z = (torch.randn(rows, 256, 67, generator=gen).to(dtype) for _ in range(updates + 1))
    gamma = torch.randn(updates, 67, generator=gen)
    got, dgamma = launch.triangular_backward(grad.cuda(), [t.cuda() for t in z], gamma.cuda())
    want, dwant = O.triangular_backward(grad, z, gamma)
    for a, e in zip(got, want):
        assert_parity(a, e, dtype, what="dz")
    assert_parity(dgamma, dwant, torch.float32, what="dgamma", kind="reduced")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("channels", [67, 130, 259])
def test_outputs_that_are_inputs(dtype, channels):
    """Every entry point that lets an output be one of its inputs, at widths whose last lane
    overlaps its neighbour where it is not: the bits of the call with its own output."""
    announce(f"in place C={channels} {dtype}")
    gen = torch.Generator(device="cuda").manual_seed(channels)
    (b, g), c, L = MANY, channels, lib()
    code, m, st = launch.dtype_code(dtype), b * g * g, launch._stream(torch.device("cuda"))

    def draw(*shape):
        return torch.empty(*shape, device="cuda").normal_(generator=gen).to(dtype)

    x, y, z = draw(b, 2 * g, 2 * g, c), draw(b, 2 * g, 2 * g, c), [draw(b, g * g, c) for _ in range(5)]
    w = draw(2, c, 4)
    p = torch.Tensor.data_ptr

    gammas = {a: torch.empty(a, c, device="cuda").normal_(generator=gen) for a in (1, 2, 3, 5)}
    for active, gamma in gammas.items():
        want = launch.triangular(z[0], z[:active], gamma)
        for over in (0, active - 1, None):  # over an update (the base is z[0] too), or over a base of its own
            base, ups = z[0].clone(), [t.clone() for t in z[:active]]
            out = base if over is None else ups[over]
            check(L.sihc_triangular(p(base), ptr_array(map(p, ups)), p(gamma), p(out), active, m, c, code, 0, st))
            assert torch.equal(out, want)
        wdz, wdg = launch.triangular_backward(z[4], z[:active], gamma, out_dtype=torch.float32)
        ws = launch._workspace(L.sihc_triangular_gamma_grad_workspace_size(active, m, c), x.device)
        for over in ("updates", "gradient") if active == 1 else ("updates",):
            grad, ups, dg = z[4].clone(), [t.clone() for t in z[:active]], torch.empty_like(wdg)
            outs = ups if over == "updates" else [grad]
            check(L.sihc_triangular_backward(p(grad), ptr_array(map(p, ups)), p(gamma), ptr_array(map(p, outs)), p(dg),
                                             active, m, c, code, 0, 0, p(ws), ws.numel() * 4, st))
            assert all(torch.equal(a, e) for a, e in zip(outs, wdz))
            # narrower lanes sum other rows together: 64 roundings of a random chain
            bound = 64 * 2 ** -24 * torch.stack([(z[4].float() * t.float()).abs().sum((0, 1)) for t in z[:active]])
            assert ((dg - wdg).abs() <= bound).all()

    want_x, want_z = launch.event_forward(x, z[0], w[0], w[1])
    for over_x, over_z in ((True, False), (False, True), (True, True)):
        xi, zi = x.clone(), z[0].clone()
        xo, zo = xi if over_x else torch.empty_like(x), zi if over_z else torch.empty_like(zi)
        check(L.sihc_event_forward(p(xi), p(zi), p(w[0]), p(w[1]), p(xo), p(zo), b, g, 2, c, None, code, st))
        assert torch.equal(xo, want_x) and torch.equal(zo, want_z)

    want = launch.event_backward(y, z[1], x, z[0], w[0], w[1])
    ws = launch._workspace(L.sihc_event_backward_workspace_size(b, g, 2, c), x.device)
    for over in ("gx", "x", "dz", "gz"):
        gx, gz, xi, dz = y.clone(), z[1].clone(), x.clone(), z[0].clone()
        ox = {"gx": gx, "x": xi}.get(over, torch.empty_like(x))
        oz = {"dz": dz, "gz": gz}.get(over, torch.empty_like(dz))
        ob, oa = torch.empty_like(w[0]), torch.empty_like(w[1])
        check(L.sihc_event_backward(p(gx), p(gz), p(xi), p(dz), p(w[0]), p(w[1]), p(ox), p(oz), p(ob), p(oa), b, g, 2, c,
                                    None, code, code, p(ws), ws.numel() * 4, st))
        assert torch.equal(ox, want[0]) and torch.equal(oz, want[1])
        assert_parity(ob, want[2].cpu(), dtype, what="dbeta", kind="reduced")
        assert_parity(oa, want[3].cpu(), dtype, what="dalpha", kind="reduced")
