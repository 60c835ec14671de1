"""The pipelined bf16 attention at the edges of its tiles: query counts around
the 16-query blocks, the 32-query waves and the 128-query tiles, key counts
around the 8-token chunks and the 64-key tiles, output rows that are only
8-byte aligned, and the log-sum-exp output, with V key-major, token-major (the
transposing fragment reads) and in separate tensors, against a float64
reference."""
import math

import pytest
import torch

from taomate_amd import kernels
from taomate_amd.kernels import KVSegment

from .helpers import gen, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vlayout", ["key", "token", "tensors"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq", [1, 15, 16, 17, 33, 127, 129, 256, 385])
@pytest.mark.parametrize("lens", [(1,), (9, 63), (64, 65, 8), (200, 127, 1)], ids=str)
def test_pipelined_edges(dev, D, Lq, lens, vlayout):
    B, H = 2, 3
    g = gen(1000 * D + Lq)
    q = randn((B, Lq, H, D), g, torch.bfloat16)
    n = sum(lens)
    k, v = randn((B, n, H, D), g, torch.bfloat16), randn((B, n, H, D), g, torch.bfloat16)
    cap = sum(-(-m // 8) * 8 + 8 for m in lens)
    ka = torch.zeros(B, cap, H, D, dtype=torch.bfloat16, device=dev)
    va = torch.zeros(B, H, D, cap, dtype=torch.bfloat16, device=dev).permute(0, 3, 1, 2) if vlayout == "key" \
        else torch.zeros_like(ka)
    segs, pos, at = [], 0, 0
    for m in lens:
        if vlayout == "tensors":   # segments that are tensors of their own, each with its batch stride
            segs.append(KVSegment(k[:, at:at + m].to(dev).contiguous(), v[:, at:at + m].to(dev).contiguous()))
            at += m
            continue
        ka[:, pos:pos + m] = k[:, at:at + m].to(dev)
        va[:, pos:pos + m] = v[:, at:at + m].to(dev)
        segs.append(KVSegment(ka[:, pos:pos + m], va[:, pos:pos + m]))
        at += m
        pos += -(-m // 8) * 8 + 8
    s = torch.einsum("bqhd,bkhd->bhqk", q.double(), k.double()) / math.sqrt(D)
    ref = torch.einsum("bhqk,bkhd->bqhd", s.softmax(-1), v.double())
    lse = torch.empty(B, H, Lq, dtype=torch.float32, device=dev)
    # 16-byte aligned rows, then rows offset by 8 bytes (the unstaged stores)
    for off in (0, 4):
        store = torch.full((B, Lq, H * D + 8), float("nan"), dtype=torch.bfloat16, device=dev)
        out = store[..., off:off + H * D].view(B, Lq, H, D)
        kernels.flash_attn(q.to(dev), segs, out, lse=lse, segment_batch_strides=vlayout == "tensors")
        torch.cuda.synchronize()
        # P, the output and the ratio of the rounded P's to the row sum are each
        # off by at most half a bf16 ulp (2^-9) of the largest value
        bound = 3 * 2.0 ** -9 * v.abs().max().item()
        assert (out.double().cpu() - ref).abs().max().item() <= bound
        assert torch.isnan(store[..., :off]).all() and torch.isnan(store[..., off + H * D:]).all()
        assert (lse.double().cpu() - s.logsumexp(-1)).abs().max().item() <= 2.0 ** -9
