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


def _segments(dev, k, v, lens, layout):
    """K and V [B, n, H, D] cut into spans of one store, each at an 8-token offset."""
    B, _, H, D = k.shape
    cap = sum(-(-m // 8) * 8 for m in lens)
    ka = torch.zeros(B, cap, H, D, dtype=torch.bfloat16, device=dev)
    va = torch.zeros(B, H, D, cap, dtype=torch.bfloat16, device=dev).permute(0, 3, 1, 2) if layout == "key" \
        else torch.zeros_like(ka)
    segs, pos, at = [], 0, 0
    for m in lens:
        ka[:, pos:pos + m], va[:, pos:pos + m] = k[:, at:at + m], v[:, at:at + m]
        segs.append(KVSegment(ka[:, pos:pos + m], va[:, pos:pos + m]))
        at += m
        pos += -(-m // 8) * 8
    return segs


@pytest.mark.parametrize("layout,form", [("key", "plain"), ("key", "lens"), ("token", "plain")])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq", [257, 273, 289])
def test_single_tile_workgroups(dev, D, Lq, layout, form):
    """Three q-tiles per head of 128 heads over 19 key tiles: the 4-wave
    workgroups of the 16x16x32 body, whole, with ragged queries and segments,
    output rows of 16- and 8-byte alignment, the log-sum-exp and per-row key
    counts, against float64 on a few heads."""
    B, H, lens = 2, 64, (9, 63, 1000, 1)
    g = torch.Generator(device=dev)
    g.manual_seed(Lq + D)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    n = sum(lens)
    q, k, v = r(B, Lq, H, D), r(B, n, H, D), r(B, n, H, D)
    segs = _segments(dev, k, v, lens, layout)
    counts = [n, 700] if form == "lens" else [n, n]
    lse = torch.empty(B, H, Lq, dtype=torch.float32, device=dev)
    for off in (0, 4):
        store = torch.full((B, Lq, H * D + 8), float("nan"), dtype=torch.bfloat16, device=dev)
        out = store[..., off:off + H * D].view(B, Lq, H, D)
        kernels.flash_attn(q, segs, out, lse=lse, key_lens=counts if form == "lens" else None)
        torch.cuda.synchronize()
        assert torch.isnan(store[..., :off]).all() and torch.isnan(store[..., off + H * D:]).all()
        assert not torch.isnan(out).any()
        for b, h in ((0, 0), (0, 37), (1, 1), (1, H - 1)):
            m = counts[b]
            s = q[b, :, h].double() @ k[b, :m, h].double().t().contiguous() / math.sqrt(D)
            ref = s.softmax(-1) @ v[b, :m, h].double()
            # P, the output and the ratio of the rounded P's to the row sum (half a bf16 ulp each)
            assert (out[b, :, h].double() - ref).abs().max().item() <= 3 * 2.0 ** -9 * v.abs().max().item()
            assert (lse[b, h].double() - s.logsumexp(-1)).abs().max().item() <= 2.0 ** -9


@pytest.mark.parametrize("layout", ["key", "token"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq", [100, 256, 300])
def test_nothing_of_an_earlier_tile_is_read(dev, D, Lq, layout):
    """Partial tiles after a call that leaves NaN in every tile buffer of the
    LDS: the keys past a segment's end have weight 0, so their V must be
    finite (rows past it load zeros, or repeat a chunk of the segment)."""
    B, H, lens = 2, 32, (9, 63, 65, 130, 1)
    nan = torch.full((B, 256, H, D), float("nan"), dtype=torch.bfloat16, device=dev)
    g = torch.Generator(device=dev)
    g.manual_seed(D)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    n = sum(lens)
    q, k, v = r(B, Lq, H, D), r(B, n, H, D), r(B, n, H, D)
    segs, bad = _segments(dev, k, v, lens, layout), _segments(dev, nan, nan, (256,), layout)
    fill_q, out = r(B, 1152, H, D), torch.empty_like(q)
    fill_out = torch.empty_like(fill_q)
    kernels.flash_attn(fill_q, bad, fill_out)
    kernels.flash_attn(q, segs, out)
    torch.cuda.synchronize()
    assert torch.isnan(fill_out).all()
    for b, h in ((0, 0), (1, H - 1)):
        s = q[b, :, h].double() @ k[b, :, h].double().t().contiguous() / math.sqrt(D)
        ref = s.softmax(-1) @ v[b, :, h].double()
        assert (out[b, :, h].double() - ref).abs().max().item() <= 3 * 2.0 ** -9 * v.abs().max().item()
    assert not torch.isnan(out).any()
