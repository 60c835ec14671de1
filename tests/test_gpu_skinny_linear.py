"""ltx_skinny_linear against float64: row counts of every instance, K at and
around the 512-element chunks, N around the row pairs and past one round of
waves, with and without SiLU and bias."""
import pytest
import torch

from taomate_amd import kernels

from .helpers import gen, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("silu", [False, True], ids=["plain", "silu"])
@pytest.mark.parametrize("M", [1, 2, 3, 8])
@pytest.mark.parametrize("K,N", [(8, 1), (256, 63), (504, 512), (520, 4099), (2048, 17), (4096, 8200)])
def test_skinny_linear(dev, M, K, N, silu):
    g = gen(K + N + M)
    x = randn((M, K), g, torch.bfloat16)
    w = randn((N, K), g, torch.bfloat16, 0.05)
    b = randn((N,), g, torch.bfloat16) if N != 63 else None
    y = kernels.skinny_linear(x.to(dev), w.to(dev), None if b is None else b.to(dev), silu=silu)
    xa = torch.nn.functional.silu(x.float()).to(torch.bfloat16) if silu else x
    ref = xa.double() @ w.double().t() + (0 if b is None else b.double())
    # the output's rounding (2^-9) and, for SiLU, an input whose rounding may
    # fall the other way (2^-8 of one product), over float32 sums
    mag = xa.double().abs() @ w.double().abs().t()
    bound = 2.0 ** -8 * ref.abs() + (2.0 ** -8 * (xa.double().abs()[:, :, None] * w.double().abs().t()[None]).amax(1)
                                     if silu else 0) + 2.0 ** -20 * mag + 1e-6
    assert ((y.double().cpu() - ref).abs() <= bound).all()


def test_skinny_linear_rejections(dev):
    x = torch.zeros(9, 64, device=dev, dtype=torch.bfloat16)
    w = torch.zeros(16, 64, device=dev, dtype=torch.bfloat16)
    from taomate_amd import _native as N
    with pytest.raises(N.NativeCallError, match="M must be"):
        kernels.skinny_linear(x, w)
    with pytest.raises(ValueError, match="skinny_linear"):
        kernels.skinny_linear(x[:2], w[:, :32])
