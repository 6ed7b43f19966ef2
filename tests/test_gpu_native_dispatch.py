"""GPU: the native eager entries of the custom ops against the registered Python ops.

A plain call takes the C++ node (its grad_fn says so) and gives the Python op's bits, forward
and backward. What a registered op lets other machinery see is still seen: dispatch and
function modes, vmap, forward-mode tangents, create_graph, saved-tensor hooks, tensor
subclasses, no_grad and inference mode, version checks; what it refuses is still refused.
"""
from __future__ import annotations

import sys
import threading
import time

import pytest
import torch
import torch._dynamo.compiled_autograd
import torch.utils.checkpoint
from torch.utils._python_dispatch import TorchDispatchMode

from sihc_hip import indexed as ix
from sihc_hip import kernels as legacy
from sihc_hip import sublayer_kernels as sk
from sihc_hip._native import native
from sihc_hip.event_ops import event_write_read

pytestmark = pytest.mark.gpu

B, G, C, E = 2, 16, 24, 3


def _t(*shape, dtype=torch.float32, grad=True):
    return torch.randn(*shape, device="cuda").to(dtype).requires_grad_(grad)


def _calls(dtype):
    """name -> (op, arguments with lists in place, the registered op of the same arguments)"""
    torch.manual_seed(1)
    x, dz = _t(B, 2 * G, 2 * G, C, dtype=dtype), [_t(B, G * G, C, dtype=dtype) for _ in range(12)]
    w, idx = _t(E, C, 4, dtype=dtype), ix.group_index(B, G, 5, 2).cuda()
    ops = torch.ops.sihc
    return {
        "read": (sk.sublayer_read, (x, w), ops.sublayer_read),
        "write": (sk.sublayer_write, (x, dz[:E], w), ops.sublayer_write),
        "triangular": (sk.sublayer_triangular, (dz[0], dz[1:4], _t(3, C)), ops.sublayer_triangular),
        "event": (event_write_read, (x, dz[0], _t(C, 4, dtype=dtype), _t(C, 4, dtype=dtype)), ops.event_write_read),
        "indexed_read": (ix._indexed_read, (x, w, idx), ops.indexed_read),
        "indexed_write": (ix._indexed_write, (x, dz[:E], w, idx), ops.indexed_write),
        "gather": (ix._gather_cells, (x, idx, 4), ops.gather_cells),
        "scatter": (ix._scatter_cells, (_t(B, G * G, 4, C, dtype=dtype), idx), ops.scatter_cells),
        "all_base": (legacy.all_base_p8_12_split_traceable, (x, _t(12, C, 4, dtype=dtype)),
                     ops.all_base_p8_12_split_traceable),
        "final_accumulate": (legacy.final_accumulate_p8_12_traceable,
                             (x, *dz, *(_t(C, 4, dtype=dtype) for _ in range(12))),
                             ops.final_accumulate_p8_12_traceable),
    }


NAMES = ["read", "write", "triangular", "event", "indexed_read", "indexed_write", "gather", "scatter", "all_base",
         "final_accumulate"]


def _flat(v):
    return [t for a in v for t in (_flat(a) if isinstance(a, (list, tuple)) else [a])]


def _leaves(args):
    return [t for t in _flat(args) if isinstance(t, torch.Tensor) and t.requires_grad]


def _outs(r):
    return _flat([r])


def _grads(out, args, seed=3):
    torch.manual_seed(seed)
    up = [torch.randn_like(o) for o in out]
    return torch.autograd.grad(out, _leaves(args), up)


def _is_native(t):
    return "Fn" in type(t.grad_fn).__name__ + t.grad_fn.name() and "GeneratedBackward" not in type(t.grad_fn).__name__


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", NAMES)
def test_same_bits_as_the_registered_op(name, dtype):
    op, args, registered = _calls(dtype)[name]
    out, want = op(*args), registered(*args)
    assert type(out) is type(want)
    out, want = _outs(out), _outs(want)
    assert _is_native(out[0]) and not _is_native(want[0])
    assert all(torch.equal(a, b) for a, b in zip(out, want))
    for a, b in zip(_grads(out, args), _grads(want, args)):
        assert a.dtype == b.dtype and torch.equal(a, b)
    # an unused output's gradient is zeros for both
    a, b = (torch.autograd.grad(_outs(f(*args))[0].float().square().sum(), _leaves(args), allow_unused=True)
            for f in (op, registered))
    assert all((p is None and q is None) or torch.equal(p, q) for p, q in zip(a, b))
    with torch.no_grad():
        r = _outs(op(*args))
        assert r[0].grad_fn is None and all(torch.equal(p, q) for p, q in zip(r, want))
    with torch.inference_mode():
        r = _outs(op(*args))
        assert r[0].is_inference() and all(torch.equal(p, q) for p, q in zip(r, want))


@pytest.mark.parametrize("name", NAMES)
def test_modes_and_transforms_still_see_the_op(name):
    op, args, _ = _calls(torch.float32)[name]

    class Count(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, a=(), kw=None):
            self.seen += str(func).startswith("sihc.")
            return func(*a, **(kw or {}))

    with Count() as m:
        out = _outs(op(*args))
    assert m.seen >= 1 and not _is_native(out[0])

    class Functions(torch.overrides.TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, a=(), kw=None):
            self.seen += "sihc" in str(func)
            return func(*a, **(kw or {}))

    with Functions() as f:
        op(*args)
    assert f.seen >= 1


def test_backward_under_a_mode_calls_the_registered_ops():
    op, args, _ = _calls(torch.float32)["event"]
    out = op(*args)
    assert _is_native(out[0])
    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), kw=None):
            seen.append(str(func))
            return func(*a, **(kw or {}))

    want = _grads(out, args)
    out = op(*args)
    with Log():
        got = _grads(out, args)
    assert any("event_write_read_backward" in s for s in seen)  # engine threads carry the caller's modes
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_create_graph_keeps_the_differentiable_rule_of_the_write():
    op, (x, dz, beta), registered = _calls(torch.float32)["write"]
    second = []
    for f in (op, registered):
        v = torch.ones_like(x, requires_grad=True)
        (g,) = torch.autograd.grad(f(x, dz, beta), dz[:1], v, create_graph=True)
        second.append(torch.autograd.grad(g.square().sum(), (v, beta)))
    assert all(torch.equal(a, b) for a, b in zip(*second))


def test_saved_tensor_hooks_and_version_checks():
    for name in ("read", "write", "event", "triangular"):
        op, args, _ = _calls(torch.float32)[name]
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.clone(), lambda t: t):
            out = _outs(op(*args))
        assert _is_native(out[0]) and len(packed) >= 2
        _grads(out, args)
    op, (x, w), _ = _calls(torch.float32)["read"]
    out = op(x, w)
    with torch.no_grad():
        w.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        _grads(out, (x, w))


def _with_one_changed(op, args, place, change):
    """op(*args) whose backward gets change(t) in place of the saved tensor number `place`."""
    packed = []

    def pack(t):
        packed.append(t)
        return len(packed) - 1, t

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda v: change(v[1]) if v[0] == place else v[1]):
        return _outs(op(*args)), packed


CHANGES = {"cast": lambda t: t.long() if t.dtype == torch.int32 else
           t.to(torch.bfloat16 if t.dtype == torch.float32 else torch.float32),
           "narrowed": lambda t: t[..., :-1].contiguous(),
           "strided": lambda t: t.repeat_interleave(2, -1)[..., ::2],
           "on the host": lambda t: t.cpu()}


@pytest.mark.parametrize("change", list(CHANGES))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", NAMES)
def test_unpacked_tensors_that_do_not_fit_are_refused(name, dtype, change):
    """An unpack hook may return anything: the backward checks what it got, tensor by tensor,
    before it launches. (Widening bf16 weights or updates is the legacy write's own contract, and
    a gamma may be of either type.)"""
    op, args, _ = _calls(dtype)[name]
    _, saved = _with_one_changed(op, args, None, None)
    for place in range(len(saved)):
        if change == "cast" and (name == "final_accumulate" and dtype == torch.float32
                                 or name == "triangular" and dtype == torch.bfloat16 and place == 0):
            continue
        if change == "strided" and name == "final_accumulate" and place >= 12:
            continue  # its weights are stacked, and so packed, first
        out, _ = _with_one_changed(op, args, place, CHANGES[change])
        assert _is_native(out[0])
        with pytest.raises((ValueError, RuntimeError)):
            _grads(out, args)


@pytest.mark.parametrize("dims", [(2, 3), (2,), (3,)], ids=["both", "weights", "updates"])
def test_bf16_copies_of_the_legacy_write_are_widened(dims):
    """fp32 training whose hooks keep the updates or weights as bf16 copies: the registered op's
    gradients bit for bit (it widens the copies)."""
    op, args, registered = _calls(torch.float32)["final_accumulate"]
    both = []
    for f in (op, registered):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.bfloat16() if t.ndim in dims else t, lambda t: t):
            out = _outs(f(*args))
        both.append(_grads(out, args))
    assert all(a.dtype == b.dtype and torch.equal(a, b) for a, b in zip(*both))


@pytest.mark.parametrize("name", NAMES)
def test_an_error_of_a_saved_tensor_hook_reaches_the_caller_once(name):
    """Checkpointing ends its recomputation by raising from the pack hook of the last tensor."""
    op, args, _ = _calls(torch.float32)[name]
    calls = []

    def pack(t):
        calls.append(t)
        raise KeyError("stop")

    with pytest.raises(KeyError, match="stop"), torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        op(*args)
    assert len(calls) == 1

    def region():
        return _outs(op(*args))

    again = torch.utils.checkpoint.checkpoint(region, use_reentrant=False)
    assert _is_native(again[0])
    assert all(torch.equal(a, b) for a, b in zip(_grads(again, args), _grads(region(), args)))


@pytest.mark.parametrize("name", NAMES)
def test_profiles_show_the_ops_with_their_shapes(name):
    op, args, registered = _calls(torch.float32)[name]
    seen = []
    for f in (op, registered):
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as prof:
            _grads(_outs(f(*args)), args)
        ours = {e.name: e.input_shapes for e in prof.events() if e.name.startswith("sihc::")}
        forward = registered._qualified_op_name
        seen.append((ours[forward], sorted(n for n in ours if "backward" in n or "_add_" in n)))
    assert seen[0] == seen[1] and seen[0][0]


def _read_op(name):
    """An op like sublayer_read with a native entry, for one test's registrations."""
    @torch.library.custom_op(f"sihc_test::{name}", mutates_args=())
    def read(x: torch.Tensor, alpha: torch.Tensor) -> list[torch.Tensor]:
        return sk.sublayer_read(x, alpha)

    torch.library.register_autograd(read, sk._read_backward, setup_context=sk._read_setup)
    return native(read, "sublayer_read")


def test_what_a_program_registers_for_an_op_is_honoured():
    _, (x, w), _ = _calls(torch.float32)["read"]
    want = sk.sublayer_read(x, w)

    def again(op, register, expected):
        assert _is_native(op(x, w)[0])
        register(op)
        got = op(x, w)
        assert not _is_native(got[0])
        assert torch.equal(got[0], expected)

    def kernel(x, alpha):
        return [2 * t for t in sk.sublayer_read(x, alpha)]

    again(_read_op("kernel"), lambda op: op.register_kernel(None, kernel), 2 * want[0])
    again(_read_op("cuda_kernel"), lambda op: op.register_kernel("cuda", kernel), 2 * want[0])
    lib = torch.library.Library("sihc_test", "FRAGMENT")
    again(_read_op("dispatcher_kernel"), lambda op: lib.impl("dispatcher_kernel", kernel, "CUDA"), 2 * want[0])
    again(_read_op("by_name"), lambda op: torch.library.register_kernel("sihc_test::by_name", "cuda", kernel),
          2 * want[0])

    def backward(ctx, grads):
        return torch.full_like(x, 3.0), None

    op = _read_op("rule")
    again(op, lambda op: torch.library.register_autograd("sihc_test::rule", backward), want[0])
    assert (torch.autograd.grad(op(x, w)[0].sum(), x)[0] == 3.0).all()

    op = _read_op("autocast")
    again(op, lambda op: torch.library.register_autocast("sihc_test::autocast", "cuda", torch.bfloat16), want[0])
    with torch.autocast("cuda", torch.bfloat16):
        assert op(x, w)[0].dtype == torch.bfloat16

    op = _read_op("host_kernel")
    op.register_kernel("cpu", kernel)
    assert _is_native(op(x, w)[0])


@pytest.mark.parametrize("name", NAMES)
def test_other_threads_run_during_a_native_call(name):
    """The GIL is free while a call allocates and launches. With a switch interval that no thread
    outlives, another thread runs only where this one gives the GIL up: inside a call."""
    op, args, _ = _calls(torch.float32)[name]
    op(*args)
    entry, inside, stop, seen = op._sihc_entry, [False], [False], []

    def watch():
        while not stop[0]:
            if inside[0]:
                seen.append(1)
            time.sleep(0)

    other, interval = threading.Thread(target=watch), sys.getswitchinterval()
    try:
        sys.setswitchinterval(20.0)
        other.start()
        for _ in range(5000):
            inside[0] = True
            out = entry(*args)
            inside[0] = False
            del out
            if seen:
                break
    finally:
        stop[0] = True
        sys.setswitchinterval(interval)
        other.join()
    assert seen


@pytest.mark.parametrize("name", NAMES)
def test_compiled_autograd_traces_the_native_backward(name):
    """Compiled autograd traces each node's backward with fake tensors, for which the node calls the
    registered ops."""
    op, args, _ = _calls(torch.float32)[name]
    out, leaves = _outs(op(*args)), _leaves(args)
    torch.manual_seed(3)
    up = [torch.randn_like(o) for o in out]
    want = torch.autograd.grad(out, leaves, up, retain_graph=True)
    torch._dynamo.reset()
    with torch._dynamo.compiled_autograd._enable(torch.compile(backend="eager")):
        torch.autograd.backward(out, up)
    # (the write's two gradients may come from two kernels there: other orders of 2,048 products)
    assert all(torch.allclose(t.grad, w, rtol=1e-5, atol=2048 * 2 ** -24) for t, w in zip(leaves, want))


def test_vmap_forward_mode_and_subclasses_take_the_registered_op():
    op, args, registered = _calls(torch.float32)["event"]
    x, *rest = (t.detach() for t in args)
    got = torch.func.vmap(lambda a: op(a, *rest))(torch.stack([x, 2 * x]))
    assert all(torch.equal(a[1], b) for a, b in zip(got, registered(2 * x, *rest)))
    op, (x, w), registered = _calls(torch.float32)["read"]
    import torch.autograd.forward_ad as fw
    with fw.dual_level():
        out = op(fw.make_dual(x.detach(), torch.ones_like(x)), w.detach())
        assert torch.equal(out[0], registered(x.detach(), w.detach())[0])

    class Sub(torch.Tensor):
        pass

    out = op(x.detach().as_subclass(Sub), w.detach())
    assert isinstance(out[0], Sub)
    out = op(x, torch.nn.Parameter(w.detach()))
    assert _is_native(out[0])


def test_refusals_are_unchanged():
    op, (x, w), _ = _calls(torch.float32)["read"]
    with pytest.raises(ValueError, match="contiguous"):
        op(x.transpose(1, 2), w)
    with pytest.raises(ValueError, match="share CUDA device and dtype"):
        op(x, w.bfloat16())
    with pytest.raises(ValueError, match="1..32 events"):
        op(x, w[:, :5].contiguous())
    _, (base, dz, gamma), _ = _calls(torch.float32)["triangular"]
    with pytest.raises(ValueError, match="active updates"):
        sk.sublayer_triangular(base, [dz[0], dz[1][:, :4].contiguous(), dz[2]], gamma)


def test_keywords_other_streams_and_capture():
    op, args, _ = _calls(torch.bfloat16)["event"]
    x, dz, beta, alpha = (t.detach() for t in args)
    want = op(x, dz, beta, alpha)
    got = op(x=x, dz=dz, beta=beta, alpha_next=alpha)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        out = op(*args)
        grads = _grads(out, args)
    s.synchronize()
    ref = _grads(op(*args), args)
    assert all(torch.equal(a, b) for a, b in zip(grads, ref))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = op(x, dz, beta, alpha)
    for k in range(3):
        x.mul_(0.5)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, op(x, dz, beta, alpha)))
