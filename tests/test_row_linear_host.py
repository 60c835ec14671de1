"""Which linears and activations the timestep MLPs may take off the module path
(dit._row_linear): those whose call is exactly their class's forward, in plain
eager mode."""
import contextlib

import pytest
import torch
import torch.nn as nn
from torch.nn.modules import module as nn_module
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from taomate_amd import dit


class _Sub(nn.Linear):
    pass


def _hook(m):
    m.register_forward_hook(lambda *_: None)


def _pre_hook(m):
    m.register_forward_pre_hook(lambda *_: None)


def _own_forward(m):
    base = m.forward
    m.forward = lambda x: base(x) + 1


def _weight_norm(m):
    nn.utils.parametrizations.weight_norm(m)


def test_plain_modules():
    assert dit._is_plain(nn.Linear(4, 4), nn.Linear) and dit._is_plain(nn.SiLU(), nn.SiLU)
    assert not dit._is_plain(_Sub(4, 4), nn.Linear) and not dit._is_plain(nn.GELU(), nn.SiLU)


@pytest.mark.parametrize("change", [_hook, _pre_hook, _own_forward, _weight_norm, nn.Module.compile])
def test_changed_modules_run_as_modules(change):
    lin = nn.Linear(4, 4)
    change(lin)
    assert not dit._is_plain(lin, nn.Linear)


@pytest.mark.parametrize("register", [nn_module.register_module_forward_hook, nn_module.register_module_forward_pre_hook])
def test_global_hooks_run_as_modules(register):
    h = register(lambda *_: None)
    try:
        assert not dit._is_plain(nn.Linear(4, 4), nn.Linear)
    finally:
        h.remove()
    assert dit._is_plain(nn.Linear(4, 4), nn.Linear)


class _Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Function(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@contextlib.contextmanager
def _autocast():
    torch.set_autocast_enabled("cuda", True)
    try:
        yield
    finally:
        torch.set_autocast_enabled("cuda", False)


@pytest.mark.parametrize("ctx", [torch.enable_grad, _autocast, torch.autograd.forward_ad.dual_level, _Dispatch, _Function])
def test_intercepted_ops_run_as_modules(ctx):
    with torch.no_grad():
        assert dit._is_eager()
        with ctx():
            assert not dit._is_eager()
        assert dit._is_eager()


def test_transforms_and_traces_run_as_modules():
    seen = []

    def fn(x):
        seen.append(dit._is_eager())
        return x + 1
    with torch.no_grad():
        torch.vmap(fn)(torch.zeros(3))
        torch.jit.trace(fn, torch.zeros(3), check_trace=False)
    assert seen == [False, False]


class _Tensor(torch.Tensor):
    pass


def test_operands_that_the_row_kernel_does_not_take():
    """CPU, wrong types, subclasses and tensors without storage are declined, not errors."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from taomate_amd import _native
    ok = _native.host().row_operands
    x, w = torch.zeros(2, 64, dtype=torch.bfloat16), torch.zeros(8, 64, dtype=torch.bfloat16)
    with FakeTensorMode():
        fake = torch.empty(2, 64, dtype=torch.bfloat16, device="cuda")
    meta = torch.empty(2, 64, dtype=torch.bfloat16, device="meta")
    for a in (x, x.float(), x.as_subclass(_Tensor), fake, meta, x.to_sparse(), None, 3):
        assert ok(a, w, None) is False
    held = []
    torch.vmap(lambda t: (held.append(t), t)[1])(x)   # a transform's tensor, past its end
    assert ok(held[0], w, None) is False
    with pytest.raises(TypeError):
        ok(x, w)
