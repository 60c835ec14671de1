"""The native call module's argument checks, without a GPU: what the wrappers
refuse and with which error, and how long they hold what they are given."""
import ctypes
import weakref

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from taomate_amd import _native, kernels
from taomate_amd.kernels import KVSegment

x = torch.zeros(1, 4, 64, dtype=torch.bfloat16)
q = torch.zeros(1, 4, 1, 64, dtype=torch.bfloat16)


@pytest.mark.parametrize("call", [
    lambda: kernels.qk_rmsnorm_rope(x, x, None, 1e-6, None, 1, 64),
    lambda: kernels.kv_append(q, q),
    lambda: kernels.kv_append_fp8_pair(q, q, q, q, q, q, 4),
    lambda: kernels.flash_attn(q, [KVSegment(q, q)], q),
    lambda: kernels.adaln(x, n_out=x),
    lambda: kernels.skinny_linear(x[0], x[0]),
])
def test_cpu_tensors_are_refused(call):
    with pytest.raises(ValueError, match="device tensors"):
        call()


def test_wrong_objects_raise_python_errors():
    host = _native.host()
    with pytest.raises(TypeError, match="expected a tensor"):
        kernels.flash_attn(q, [KVSegment(q, q)], "out")
    with pytest.raises(TypeError, match="expected 10 arguments"):
        host.flash_attn(q)
    with pytest.raises(ValueError, match="missing entry point"):
        host.bind({}, RuntimeError)
    with pytest.raises(ValueError, match="device tensors"):   # the refused bind left the calls bound
        kernels.adaln(x, n_out=x)


class _OwnTables:
    """A (cos, sin) argument that nothing but its iteration holds."""

    def __init__(self):
        self.refs = []

    def __iter__(self):
        for _ in range(2):
            t = torch.ones(1, 1, 4, 32)
            self.refs.append(weakref.ref(t))
            yield t


class _Eps:
    """An eps that is read after the tables, and records whether they are still there."""

    def __init__(self, tables):
        self.tables, self.alive = tables, []

    def __float__(self):
        self.alive += [r() is not None for r in self.tables.refs]
        return 1e-6


@pytest.mark.parametrize("side", ["q", "k"])
def test_rope_tables_are_held_for_the_call(side):
    """The call reads the tables long after it took them apart: a pair that the
    caller does not hold (an iterator's, a stacked tensor's rows) stays alive.
    A device tensor without storage stands for the rows; the call ends at its
    missing data pointer."""
    with FakeTensorMode():
        rows = torch.empty(1, 4, 64, dtype=torch.bfloat16, device="cuda")
    tab = _OwnTables()
    eps = _Eps(tab)
    q_tab, k_tab = (tab, None) if side == "q" else (None, tab)
    with pytest.raises(Exception) as e:
        kernels.qk_rmsnorm_rope(rows, rows, None, eps, q_tab, 1, 64, rows, rows, None, 1e-6, k_tab)
    assert "unsupported dtype" not in str(e.value)
    assert eps.alive == [True, True]
    assert [r() for r in tab.refs] == [None, None]   # and no longer than the call


def test_a_segment_without_a_token_dim_is_an_index_error():
    with FakeTensorMode():
        rows = torch.empty(1, 4, 1, 64, dtype=torch.bfloat16, device="cuda")
    flat = torch.zeros(64, dtype=torch.bfloat16)
    with pytest.raises(IndexError):
        kernels.flash_attn(rows, [KVSegment(flat, flat)], rows)


class _Entry:
    def __init__(self, value):
        self.value = value

    def __call__(self):
        return self.value


@pytest.mark.parametrize("have,message", [
    ({"ltx_abi_version": 2, "ltx_last_error": b""}, "ltx_rope_table"),         # an older library of this ABI
    ({"ltx_abi_version": 1}, "ABI version 1, expected 2"),
    ({}, "ltx_abi_version"),                                                   # another library altogether
])
def test_a_library_without_the_entry_points_is_refused(monkeypatch, have, message):
    lib = type("Lib", (), {})()
    for name, value in have.items():
        setattr(lib, name, _Entry(value))
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(ctypes, "CDLL", lambda path: lib)
    with pytest.raises(_native.NativeLibraryError, match=message):
        _native.load()
    assert _native._lib is None
