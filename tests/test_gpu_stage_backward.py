"""GPU: the matrix-core weight gradient and the one-pass backward of the read and the write.

Event counts at the edges of the 4-event groups and of the dispatch (one pass up to 24 events
for the read and 8 for the write, two kernels past them; 9 and more bf16 events at 16 slots on
the pipelined kernel), widths below, at and around one vector and one 64- or 128-channel slice
(the last channel group moved back over its neighbour), rows at odd alignments, token counts
that leave groups of 1 to 3 tokens, state permutations, both element types.
Weight gradients are fp32 sums of exact (bf16) or once-rounded products: the fp32 bar against
the oracle's float64 sums. The other gradients are one element's fp32 sum rounded once: the
elementwise bar.
"""
from __future__ import annotations

import pytest
import torch

from helpers import announce, assert_parity
from oracle import sihc_oracle as O
from sihc_hip import launch

pytestmark = pytest.mark.gpu


def _inputs(slots, events, b, g, c, dtype, with_index, seed):
    k = O.cell_edge(slots)
    gen = torch.Generator().manual_seed(seed)

    def draw(*shape):
        return torch.randn(*shape, generator=gen).to(dtype)

    x = draw(b, k * g, k * g, c)
    z = [draw(b, g * g, c) for _ in range(events)]
    w = (1.0 / slots + 0.1 * torch.randn(events, c, slots, generator=gen)).to(dtype)
    index = None
    if with_index:
        index = torch.stack([torch.randperm(g * g, generator=gen) for _ in range(b)]).to(torch.int32)
    return x, z, w, index


def _place(cells, index, slots):
    """Carrier whose cell index[b, n] is cells[b, n]."""
    return O.cells_to_high(cells) if index is None else O.scatter_cells(cells, index)


def _token_order(x, index, slots):
    return x if index is None else O.cells_to_high(O.gather_cells(x, index, slots))


GEOMS = [  # batch, grid, channels, index
    (2, 5, 8, False), (1, 3, 3, False), (3, 5, 67, True), (1, 7, 129, False), (2, 16, 136, True), (1, 4, 1153, False),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("slots,events", [(4, e) for e in (1, 2, 4, 5, 8, 9, 13, 16, 17, 20, 21, 24, 25, 29, 32)] +
                         [(16, e) for e in (1, 4, 5, 8, 9, 12, 13, 17, 24, 25, 32)])
@pytest.mark.parametrize("geom", GEOMS, ids=[f"b{b}-g{g}-c{c}{'-index' if i else ''}" for b, g, c, i in GEOMS])
def test_weight_grad_and_stage_backward(dtype, slots, events, geom):
    b, g, c, with_index = geom
    announce(f"stage backward slots={slots} E={events} b={b} g={g} c={c} index={with_index} {dtype}")
    x, z, w, index = _inputs(slots, events, b, g, c, dtype, with_index, 31 * events + c + slots)
    xd, zd, wd = x.cuda(), [t.cuda() for t in z], w.cuda()
    idx = None if index is None else index.cuda()
    dw = O.weight_grad(_token_order(x, index, slots), z, slots)
    assert_parity(launch.weight_grad(xd, zd, wd, index=idx, out_dtype=torch.float32), dw, torch.float32, what="dw")

    gx, ga = launch.read_backward(xd, zd, wd, index=idx, out_dtype=torch.float32)
    assert_parity(ga, dw, torch.float32, what="dalpha")
    zero = torch.zeros(b, g * O.cell_edge(slots), g * O.cell_edge(slots), c, dtype=dtype)
    want = O.write(zero, z, w, add_x=False)
    assert_parity(gx, _place(O.high_to_cells(want, slots), index, slots), dtype, what="dx")

    gz, gb = launch.write_backward(xd, zd, wd, index=idx, out_dtype=torch.float32)
    assert_parity(gb, dw, torch.float32, what="dbeta")
    for e, t in enumerate(O.read(_token_order(x, index, slots), w)):
        assert_parity(gz[e], t, dtype, what=f"ddz[{e}]")
    # fixed order: the same bits again
    gx2, ga2 = launch.read_backward(xd, zd, wd, index=idx, out_dtype=torch.float32)
    assert torch.equal(gx, gx2) and torch.equal(ga, ga2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("events", [1, 3, 6, 8, 21])
def test_infinities_stay_in_their_token_event_and_channel(dtype, events):
    # Repeated tail tokens and lanes past the last event load real rows: an Inf there must
    # reach only the gradients it belongs to.
    announce(f"stage backward Inf E={events} {dtype}")
    b, g, c, ch = 1, 5, 67, 66  # 25 tokens: the last group holds one
    x, z, w, _ = _inputs(4, events, b, g, c, dtype, False, events)
    z[-1][0, -1, ch] = float("inf")
    gx, ga = launch.read_backward(x.cuda(), [t.cuda() for t in z], w.cuda(), out_dtype=torch.float32)
    bad = ~torch.isfinite(ga.cpu())
    assert bad[-1, ch].all() and bad.sum() == 4
    cells = O.high_to_cells(gx.cpu(), 4)
    bad = ~torch.isfinite(cells)
    assert bad[0, -1, :, ch].all() and bad.sum() == 4
    x[0, -1, -1, ch] = float("inf")  # slot 3 of the last token
    z[-1][0, -1, ch] = 1.0
    gz, gb = launch.write_backward(x.cuda(), [t.cuda() for t in z], w.cuda(), out_dtype=torch.float32)
    bad = ~torch.isfinite(gb.cpu())
    assert bad[:, ch, 3].all() and bad.sum() == events
    for t in gz:
        bad = ~torch.isfinite(t.cpu())
        assert bad[0, -1, ch] and bad.sum() == 1


def test_long_chunks_walk_every_group():
    # 65,925 tokens: chunks of many interleaved 8-token groups, 5 tokens in the last one.
    announce("stage backward long")
    x, z, w, _ = _inputs(4, 5, 293, 15, 24, torch.bfloat16, False, 1)
    gx, ga = launch.read_backward(x.cuda(), [t.cuda() for t in z], w.cuda(), out_dtype=torch.float32)
    assert_parity(ga, O.weight_grad(x, z, 4), torch.float32, what="dalpha")
    assert_parity(gx, O.write(torch.zeros_like(x), z, w, add_x=False), torch.bfloat16, what="dx")
