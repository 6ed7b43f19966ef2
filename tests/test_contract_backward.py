"""CPU: the registered backward ops refuse operands that do not fit before any launch.

A backward receives its saved tensors through the caller's saved-tensor hooks, which may
return another type, shape or device than was saved. Each op is called with GPU tensors that
hold no memory (fake tensors) and a launcher that only records the call.
"""
from __future__ import annotations

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from sihc_hip import event_ops as EV
from sihc_hip import indexed as IX
from sihc_hip import kernels as LK
from sihc_hip import launch
from sihc_hip import sublayer_kernels as SK

B, G, C, E, S = 2, 4, 8, 3, 4
BF, F32 = torch.bfloat16, torch.float32


def _t(*shape, dtype=F32, device="cuda:0"):
    return torch.empty(*shape, dtype=dtype, device=device)


def _operands():
    """name -> (op, launcher, operands that fit, {position: replacements that do not})"""
    x, z = _t(B, 2 * G, 2 * G, C), [_t(B, G * G, C) for _ in range(E)]
    w, gamma, idx = _t(E, C, S), _t(E, C), _t(B, G * G, dtype=torch.int32)
    one, cells = _t(C, S), _t(B, G * G, S, C)
    bad_x = [x.to(BF), _t(B, 2 * G, 2 * G, C + 1), _t(B - 1, 2 * G, 2 * G, C), x.transpose(1, 2), x.cpu()]
    bad_z = [[t.to(BF) for t in z], z[:2], [z[0], z[1], _t(B, G * G, C - 1)], [z[0], z[1], _t(B, G * G, 2 * C)[..., :C]],
             [t.cpu() for t in z]]
    bad_w = [w.to(BF), _t(E, C - 1, S), _t(E - 1, C, S), w.cpu()]
    bad_idx = [idx.long(), idx.cpu(), _t(B, G * G - 1, dtype=torch.int32), idx.t()]
    bad_gamma = [_t(E, C + 1), _t(E - 1, C), gamma.double(), gamma.cpu()]
    bad_one = [one.to(BF), _t(C - 1, S), one.cpu()]
    lx = _t(B, 32, 32, C)
    lz, lw = [_t(B, 256, C) for _ in range(12)], [_t(C, S) for _ in range(12)]
    return {
        "read": (SK._read_grads, "read_backward", (x, z, w), {0: bad_x, 1: bad_z, 2: bad_w}),
        "write": (SK._write_grads, "write_backward", (x, z, w), {0: bad_x, 1: bad_z, 2: bad_w}),
        "weights": (SK._weights_backward, "weight_grad", (x, z, w), {0: bad_x, 1: bad_z, 2: bad_w}),
        "triangular": (SK._tri_backward, "triangular_backward", (z[0], z, gamma), {1: bad_z, 2: bad_gamma}),
        "gamma": (SK._tri_gamma_backward, "triangular_gamma_grad", (z[0], z, gamma), {1: bad_z, 2: bad_gamma}),
        "event": (EV._event_backward, "event_backward", (x, z[0], x, z[1], one, one),
                  {0: bad_x, 1: [t[-1] for t in bad_z[2:]], 2: bad_x, 3: [t[-1] for t in bad_z[2:]], 4: bad_one,
                   5: bad_one}),
        "indexed_read": (IX._indexed_read_grads, "read_backward", (x, z, w, idx), {0: bad_x, 1: bad_z, 3: bad_idx}),
        "indexed_write": (IX._indexed_write_grads, "write_backward", (x, z, w, idx), {1: bad_z, 2: bad_w, 3: bad_idx}),
        "indexed_weights": (IX._indexed_weight_grad, "weight_grad", (x, z, w, idx), {1: bad_z, 3: bad_idx}),
        "gather": (IX._gather_cells, "gather_cells", (x, idx, S), {1: bad_idx}),
        "scatter": (IX._scatter_cells, "scatter_cells", (cells, idx), {0: [_t(B, 7, S, C)], 1: bad_idx}),
        "scatter_add": (IX._scatter_add_cells, "scatter_add_cells", (cells, idx), {0: [_t(B, 7, S, C)], 1: bad_idx}),
        "grad_dz": (LK.final_accumulate_p8_12_grad_dz_ptr_traceable, "read", (lx, *lw),
                    {0: [_t(B, 64, 64, C), lx.transpose(1, 2)], 3: [_t(C - 1, S), lw[0].cpu()]}),
        "grad_beta": (LK.final_accumulate_p8_12_grad_beta_ptr_traceable, "weight_grad", (lx, *lz),
                      {0: [_t(B, 64, 64, C), lx.transpose(1, 2)],
                       3: [_t(B, 255, C), lz[0].cpu(), _t(B, 256, 2 * C)[..., :C]]}),
    }


NAMES = ["read", "write", "weights", "triangular", "gamma", "event", "indexed_read", "indexed_write",
         "indexed_weights", "gather", "scatter", "scatter_add", "grad_dz", "grad_beta"]


@pytest.mark.parametrize("name", NAMES)
def test_operands_that_do_not_fit_are_refused_before_the_launch(name, monkeypatch):
    with FakeTensorMode():
        op, launcher, args, bad = _operands()[name]
        launched = []
        monkeypatch.setattr(launch, launcher, lambda *a, **k: launched.append(a) or (None,) * 4)
        op._init_fn(*args)
        assert len(launched) == 1
        for place, values in bad.items():
            for value in values:
                with pytest.raises(ValueError):
                    op._init_fn(*args[:place], value, *args[place + 1:])
        assert len(launched) == 1
