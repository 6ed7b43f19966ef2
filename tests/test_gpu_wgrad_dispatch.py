"""GPU: weight gradients on both sides of the lines at which their kernels change.

Sizes (batches of 16 x 16 workspaces) just below and at each line of tokens x channels, and the
event counts at the ends of each range, with and without a state index. Expected values are
float64 sums of the same inputs. A chain of n random products keeps its partial sums near sqrt(n),
so its n roundings come to about 6 * 2^-24 of the sum of magnitudes for n up to 1,024; the bound
is 64 * 2^-24, and a token lost or counted twice is at least 2^-16 of it."""
from __future__ import annotations

import pytest
import torch

from helpers import announce
from sihc_hip import launch

pytestmark = pytest.mark.gpu

BF, F32 = torch.bfloat16, torch.float32
# (dtype, slots, channels, batches around a line, events)
LINES = [
    (BF, 4, 512, (31, 32), (17, 24)),          # 4 Mi: pipelined, two parts
    (BF, 4, 768, (127, 128), (18, 19)),        # 24 Mi: two parts, one, to 18 events
    (BF, 4, 1024, (191, 192), (19, 25, 32)),   # 48 Mi: two parts, one
    (BF, 4, 627, (26, 27), (17, 24, 25, 32)),  # ragged rows: no pipelined kernel
    (F32, 4, 320, (15, 16), (20, 21, 29, 32)),  # 1.25 Mi: k_wgrad, one part, two from 29
    (BF, 16, 768, (31, 32, 127, 128), (1, 4, 5, 8)),  # 6 and 24 Mi: pipelined, matrix cores
    (BF, 16, 512, (127, 128), (5, 8)),         # 16 Mi for up to 512 channels
    (F32, 16, 288, (15, 16, 32), (13, 16, 17, 32)),  # 1.125 and 2.25 Mi: k_wgrad16, matrix cores
    (F32, 16, 256, (7, 8), (13, 16)),          # 0.5 Mi
    (BF, 16, 291, (15, 16), (20, 21, 32)),     # ragged rows at 1.125 Mi
]


@pytest.mark.parametrize("dtype,slots,channels,batches,events", LINES,
                         ids=[f"{str(d)[6:]}-s{s}-c{c}-e{e[0]}" for d, s, c, _, e in LINES])
def test_weight_gradient_on_both_sides_of_a_line(dtype, slots, channels, batches, events):
    k = 2 if slots == 4 else 4
    gen = torch.Generator(device="cuda").manual_seed(channels + slots)
    for batch in batches:
        announce(f"wgrad line dtype={dtype} slots={slots} C={channels} b={batch}")
        x = torch.empty(batch, 16 * k, 16 * k, channels, device="cuda").normal_(generator=gen).to(dtype)
        z = [torch.empty(batch, 256, channels, device="cuda").normal_(generator=gen).to(dtype)
             for _ in range(max(events))]
        index = torch.stack([torch.randperm(256, device="cuda", generator=gen) for _ in range(batch)]).to(torch.int32)
        cells = x.view(batch, 16, k, 16, k, channels).permute(0, 1, 3, 2, 4, 5).reshape(batch, 256, slots, channels)
        for count in events:
            for idx in (None, index):
                got = launch.weight_grad(x, z[:count], None, index=idx, out_dtype=torch.float32, slots=slots)
                rows = cells if idx is None else cells[torch.arange(batch, device="cuda")[:, None], idx.long()]
                for e in {0, 1, count // 2, count - 1}:
                    if e >= count:
                        continue
                    ze = z[e].double()
                    for s in {0, slots // 2, slots - 1}:
                        prod = rows[:, :, s].double() * ze
                        err = (got[e, :, s].double() - prod.sum((0, 1))).abs()
                        assert (err <= 64 * 2 ** -24 * prod.abs().sum((0, 1))).all(), (batch, count, e, s)
                if idx is None:
                    again = launch.weight_grad(x, z[:count], None, out_dtype=torch.float32, slots=slots)
                    assert torch.equal(got, again)
        del x, z, cells
