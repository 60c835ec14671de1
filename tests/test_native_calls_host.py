"""The native call module's argument checks, without a GPU: what the wrappers
refuse and with which error."""
import pytest
import torch

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
