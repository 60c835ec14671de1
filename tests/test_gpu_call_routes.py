"""Calls whose route depends on their form, each against the general path or a
reference: plain caches in strides and alignments that are attended in place
or concatenated, key-range splits of partly filled grids, norm rows without
RoPE tables, and the timestep MLPs with and without the row kernel."""
import contextlib
import ctypes
import math

import pytest
import torch

import taomate_amd as T
from taomate_amd import _native, dit, kernels
from taomate_amd.kernels import KVSegment

from .helpers import gen, randn

pytestmark = pytest.mark.gpu


def _attend64(q, k, v):
    s = torch.einsum("bqhd,bkhd->bhqk", q.double(), k.double()) / math.sqrt(q.shape[-1])
    return torch.einsum("bhqk,bkhd->bqhd", s.softmax(-1), v.double())


def _bound(v):
    # P, the output and the ratio of the rounded P's to the row sum: half a bf16 ulp each
    return 3 * 2.0 ** -9 * v.abs().max().item()


def _odd_offset(t):
    """The same values in storage that starts 2 bytes past a 16-byte boundary."""
    s = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    return s[1:1 + t.numel()].view(t.shape).copy_(t)


FORMS = {
    "contiguous": lambda t: t.contiguous(),
    "batch_slice": lambda t: torch.cat([t, t], 1)[:, :t.shape[1]],
    "token_offset": lambda t: torch.cat([t.new_zeros(t.shape[0], 3, *t.shape[2:]), t], 1)[:, 3:],
    "head_major": lambda t: t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3),
    "row_gap": lambda t: torch.cat([t, t], -1)[..., :t.shape[-1]],
    "odd_offset": _odd_offset,
}


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("Lc,L", [(1, 5), (64, 130), (203, 300)])
@pytest.mark.parametrize("kform,vform", [(f, f) for f in FORMS] + [("contiguous", "head_major"),
                                                                 ("contiguous", "odd_offset"),
                                                                 ("batch_slice", "contiguous")])
def test_plain_cache_forms(dev, kform, vform, Lc, L, B):
    """attention_with_cache over plain tensors: every cache form gives the
    result of contiguous cache tensors within the kernels' bf16 rounding."""
    H, D = 4, 64
    g = gen(Lc + L)
    attn = T.CausalLTXAttention(H * D, heads=H, dim_head=D)
    with torch.no_grad():
        for p in attn.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * 0.05)
        attn = attn.to(dev, torch.bfloat16)
        x = randn((B, L, H * D), g, torch.bfloat16).to(dev)
        ck, cv = (randn((B, Lc, H, D), g, torch.bfloat16).to(dev) for _ in range(2))
        want, wk, wv = T.attention_with_cache(attn, x, None, None, None, ck, cv)
        out, nk, nv = T.attention_with_cache(attn, x, None, None, None, FORMS[kform](ck), FORMS[vform](cv))
    torch.cuda.synchronize()
    assert torch.equal(nk, wk) and torch.equal(nv, wv)
    # two roundings of the attention output (2^-8 relative), through to_out
    err = (out.float() - want.float()).norm() / want.float().norm()
    assert err <= 2.0 ** -7, err.item()


@pytest.mark.parametrize("layout", ["key", "token"])
@pytest.mark.parametrize("B,H,D,qtiles,keys", [(2, 32, 64, 3, 4608), (2, 16, 128, 5, 2500), (1, 32, 64, 7, 3000),
                                              (2, 32, 64, 11, 6001), (2, 8, 128, 1, 300)])
def test_split_plans(dev, layout, B, H, D, qtiles, keys):
    """Grids whose last round is partly filled: the planned key-range split
    against float64 on some heads, and the same plan in the no-allocation
    entry point bit for bit."""
    Lq = qtiles * 128 - 37
    g = torch.Generator(device=dev)
    g.manual_seed(keys)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    q, k = r(B, Lq, H, D), r(B, keys, H, D)
    v = r(B, H, D, -(-keys // 8) * 8).permute(0, 3, 1, 2)[:, :keys] if layout == "key" else r(B, keys, H, D)
    out, again = torch.empty_like(q), torch.empty_like(q)
    lse = torch.empty(B, H, Lq, dtype=torch.float32, device=dev)
    kernels.flash_attn(q, [KVSegment(k, v)], out, lse=lse)
    kernels.flash_attn(q, [KVSegment(k, v)], again, noalloc=True)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    for h in (0, H - 1):
        sl = slice(h, h + 1)
        ref = _attend64(q[:, :, sl].cpu(), k[:, :, sl].cpu(), v[:, :, sl].cpu())
        assert (out[:, :, sl].double().cpu() - ref).abs().max().item() <= _bound(v) + 2.0 ** -8 * ref.abs().max().item()


def _fp8_cache(k, v, frame, dev):
    """fp8 codes and scales of K and V, and the values they hold."""
    B, n, H, D = k.shape
    kc, vc = (torch.empty(B, n, H, D, dtype=torch.uint8, device=dev) for _ in range(2))
    ks, vs = (torch.empty(B, H, n // frame, device=dev) for _ in range(2))
    kernels.kv_append_fp8_pair(k, kc, ks, v, vc, vs, frame)
    value = lambda c, s: (c.view(torch.float8_e4m3fn).double()
                          * s.double().transpose(1, 2).repeat_interleave(frame, 1)[..., None])
    return KVSegment(kc, vc, ks, vs), value(kc, ks), value(vc, vs)


def _whole(q, seg, out, frame):
    """The same call without a workspace: every q-tile runs whole, in float32 sums."""
    k, v = seg.k, seg.v
    fp8 = seg.k_scales is not None
    keep = [_native.ptr_array([t.data_ptr()]) for t in (k, v)] + [_native.i64_array([k.shape[1]])] + \
        [_native.ptr_array([t.data_ptr()]) if fp8 else None for t in (seg.k_scales, seg.v_scales)]
    kp, vp, lens, ksp, vsp = (None if a is None else ctypes.cast(a, ctypes.c_void_p) for a in keep)
    _native.call("ltx_flash_attn_fwd", q.data_ptr(), *q.shape, *q.stride()[:3], 1, kp, vp, lens, *k.stride()[:3],
                 *v.stride(), 2 if fp8 else 1, ksp, vsp, *(seg.k_scales.stride()[:2] if fp8 else (0, 0)), frame, None, 0,
                 None, out.data_ptr(), *out.stride()[:3], None, 0.0, None, 0,
                 torch.cuda.current_stream().cuda_stream)


def _split_case(dev, layout, B, Lq, H, D, keys, frame=330):
    """A call with its launch plan and with whole q-tiles: both outputs, their
    root mean square errors against float64 on a few heads."""
    g = torch.Generator(device=dev)
    g.manual_seed(keys + Lq)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    q, k, v = r(B, Lq, H, D), r(B, keys, H, D), r(B, keys, H, D)
    frame = frame if layout == "fp8" else 0
    if layout == "fp8":
        seg, k, v = _fp8_cache(k, v, frame, dev)
    elif layout == "key":
        store = torch.zeros(B, H, D, -(-keys // 8) * 8, dtype=torch.bfloat16, device=dev)
        store[..., :keys] = v.permute(0, 2, 3, 1)
        seg = KVSegment(k, store[..., :keys].permute(0, 3, 1, 2))
    else:
        seg = KVSegment(k, v)
    out, whole = torch.empty_like(q), torch.empty_like(q)
    kernels.flash_attn(q, [seg], out, frame_tokens=frame)
    _whole(q, seg, whole, frame)
    torch.cuda.synchronize()
    err = [0.0, 0.0]
    for b, h in ((0, 0), (B - 1, H - 1), (0, H // 2), (B - 1, 5)):
        p = ((q[b, :, h].double() @ k[b, :, h].double().t().contiguous()) / math.sqrt(D)).softmax(-1)
        ref = p @ v[b, :, h].double()
        for i, o in enumerate((out, whole)):
            err[i] += (o[b, :, h].double() - ref).square().sum().item()
    return out, whole, math.sqrt(err[0]), math.sqrt(err[1])


@pytest.mark.parametrize("keys", [640, 2560, 5120])
@pytest.mark.parametrize("B,H,qtiles", [(2, 32, 1), (1, 32, 3), (2, 32, 3), (1, 32, 7), (2, 32, 9), (2, 32, 11),   # 4-wave
                                        (1, 32, 2), (2, 32, 4), (2, 32, 10), (2, 32, 12), (2, 24, 14)])          # pair units
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("layout,frame", [("key", 0), ("token", 0), ("fp8", 320), ("fp8", 160)])
def test_launch_plan_against_whole_tiles(dev, layout, frame, D, B, H, qtiles, keys):
    """Every kernel (fp8 in frames of whole 64-key tiles and not) with tails of a partial round and behind whole rounds, over
    few and many keys: bf16 partials add one rounding of the output's size to
    the two of P and the output (sqrt(3 / 2) = 1.22 times the error), float32
    partials none."""
    _, _, err, whole = _split_case(dev, layout, B, qtiles * 128 - 20, H, D, keys, frame)
    assert err <= 1.3 * whole


@pytest.mark.parametrize("layout,B,Lq,H,D,keys", [
    ("key", 1, 620, 32, 128, 4000), ("key", 2, 300, 32, 64, 5000), ("key", 2, 620, 32, 64, 5000),
    ("key", 1, 1370, 32, 128, 7000), ("token", 2, 620, 32, 128, 4000), ("token", 1, 300, 32, 64, 2600),
    ("token", 2, 512, 32, 64, 2000), ("token", 2, 1152, 32, 64, 1152), ("token", 1, 2423, 32, 128, 1152),
    ("fp8", 1, 620, 32, 64, 1650), ("fp8", 2, 300, 32, 128, 2640), ("fp8", 2, 620, 32, 128, 3300),
    ("fp8", 1, 1370, 32, 64, 4950)])
def test_split_keeps_float32_sums(dev, layout, B, Lq, H, D, keys):
    """Tails that are split with float32 partials, one case per branch of the
    launch plan: the error against float64 is the whole q-tiles' (bf16
    partials of all rows make it 1.22 times that).  Both share P's rounding
    and the output's; over the 1e5 and more values compared, what is left
    differs by well under 1 %."""
    out, whole, err, err_whole = _split_case(dev, layout, B, Lq, H, D, keys)
    assert not torch.equal(out, whole)   # the plan does split
    assert err <= 1.02 * err_whole


@pytest.mark.parametrize("counts", [(5000, 37), (0, 5000), (1300, 2501)])
def test_key_counts_over_float32_ranges(dev, counts):
    """Per-row key counts where the plan cuts the keys into ranges with float32
    partials: ranges past a row's count hold nothing."""
    B, Lq, H, D, n = 2, 300, 32, 64, 5000
    g = torch.Generator(device=dev)
    g.manual_seed(sum(counts))
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    q, k, v = r(B, Lq, H, D), r(B, n, H, D), r(B, n, H, D)
    store = v.permute(0, 2, 3, 1).contiguous()
    out = torch.empty_like(q)
    lse = torch.empty(B, H, Lq, dtype=torch.float32, device=dev)
    kernels.flash_attn(q, [KVSegment(k, store.permute(0, 3, 1, 2))], out, lse=lse, key_lens=list(counts))
    torch.cuda.synchronize()
    for b, m in enumerate(counts):
        for h in (0, H - 1):
            if m == 0:
                assert (out[b, :, h] == 0).all() and (lse[b, h] == float("-inf")).all()
                continue
            s = q[b, :, h].double() @ k[b, :m, h].double().t().contiguous() / math.sqrt(D)
            ref = s.softmax(-1) @ v[b, :m, h].double()
            assert (out[b, :, h].double() - ref).abs().max().item() <= _bound(v)
            assert (lse[b, h].double() - s.logsumexp(-1)).abs().max().item() <= 2.0 ** -9


@pytest.mark.parametrize("B,L,H,D", [(2, 1, 8, 64), (1, 33, 32, 128), (2, 75, 32, 64)])
def test_norm_without_tables(dev, B, L, H, D):
    """Rows with a norm and a gain but no RoPE tables (the branch-free form)
    equal the rotated form under identity tables bit for bit, also from packed
    q/k/v columns and on one side alone."""
    g = gen(L)
    n = H * D
    y = randn((B, L, 3 * n), g, torch.bfloat16).to(dev)
    gq, gk = (randn((n,), g, torch.bfloat16).to(dev) for _ in range(2))
    eye = (torch.ones(1, H, L, D // 2, dtype=y.dtype, device=dev), torch.zeros(1, H, L, D // 2, dtype=y.dtype, device=dev))
    got, want = ([torch.empty(B, L, n, dtype=y.dtype, device=dev) for _ in range(3)] for _ in range(2))
    for out, tab in ((got, None), (want, eye)):
        kernels.qk_rmsnorm_rope(y[..., :n], out[0], gq, 1e-6, tab, H, D, y[..., n:2 * n], out[1], gk, 1e-6, tab)
        kernels.qk_rmsnorm_rope(y[..., :n], out[2], gq, 1e-6, tab, H, D)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert torch.equal(got[0], got[2])


@pytest.mark.parametrize("form", ["list", "stacked", "iterator"])
def test_table_forms(dev, form):
    """A RoPE table given as a list, one stacked tensor or an iterator (whose
    items only the call holds) rotates as the (cos, sin) tuple does."""
    B, L, H, D = 2, 19, 4, 64
    g = gen(3)
    y = randn((B, L, H * D), g, torch.bfloat16).to(dev)
    gain = randn((H * D,), g, torch.bfloat16).to(dev)
    pair = torch.stack([randn((1, H, L, D // 2), g, torch.bfloat16) for _ in range(2)]).to(dev)
    forms = {"tuple": lambda: (pair[0], pair[1]), "list": lambda: [pair[0], pair[1]], "stacked": lambda: pair,
             "iterator": lambda: (t.clone() for t in pair)}
    got, want = ([torch.empty_like(y) for _ in range(2)] for _ in range(2))
    for out, f in ((got, form), (want, "tuple")):
        kernels.qk_rmsnorm_rope(y, out[0], gain, 1e-6, forms[f](), H, D, y, out[1], gain, 1e-6, forms[f]())
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("rows", [1, 2, 6, 8, 9])
def test_timestep_mlp_routes(dev, rows):
    """AdaLayerNormSingle without grad (the row kernel up to 8 rows) against
    the module path that grad mode, a hook or a replaced activation takes."""
    m = dit.AdaLayerNormSingle(512, 6).to(dev, torch.bfloat16)
    g = gen(rows)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_((torch.randn(p.shape, generator=g) * 0.05).to(dev))
    t = (torch.rand(rows, generator=g) * 1000).to(dev)
    with torch.no_grad():
        out, e = m(t, torch.bfloat16)
    want, we = (z.detach() for z in m(t, torch.bfloat16))
    for a, b in ((out, want), (e, we)):   # a few bf16 roundings through three layers
        assert a.shape == b.shape and ((a - b).float().norm() / b.float().norm()).item() <= 2.0 ** -6
    seen = []
    h = m.linear.register_forward_hook(lambda *_: seen.append(1))
    with torch.no_grad():
        m(t, torch.bfloat16)
    h.remove()
    assert seen == [1]


def _forward_override(m):
    base = m.linear.forward
    m.linear.forward = lambda x: base(x) + 1


def _strided_bias(m):
    m.linear.bias = torch.nn.Parameter(torch.stack([m.linear.bias.detach()] * 2, 1)[:, 0])


@pytest.mark.parametrize("how", ["forward", "strided_bias", "global_hook", "autocast", "tangent"])
def test_timestep_mlp_keeps_what_modules_do(dev, how):
    """What a linear's own call would see or do holds without grad too: a
    replaced forward, a strided bias, a global hook, autocast to fp16 and a
    forward-mode tangent give the module path's result bit for bit."""
    fw = torch.autograd.forward_ad
    m = dit.AdaLayerNormSingle(512, 6).to(dev, torch.bfloat16)
    g = gen(7)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_((torch.randn(p.shape, generator=g) * 0.05).to(dev))
        {"forward": _forward_override, "strided_bias": _strided_bias}.get(how, lambda m: None)(m)
    x = randn((2, 512), g, torch.bfloat16).to(dev)
    seen = []
    hook = torch.nn.modules.module.register_module_forward_hook(lambda *_: seen.append(1)) if how == "global_hook" else None
    try:
        with torch.autocast("cuda", torch.float16, enabled=how == "autocast"), \
                fw.dual_level() if how == "tangent" else contextlib.nullcontext():
            xin = fw.make_dual(x, torch.ones_like(x)) if how == "tangent" else x
            with torch.no_grad():
                out = dit._row_linear(m.linear, xin, m.silu)
                calls = len(seen)
                want = m.linear(m.silu(xin))
            if how == "tangent":
                (out, t), (want, wt) = fw.unpack_dual(out), fw.unpack_dual(want)
                assert torch.equal(t, wt)
    finally:
        if hook is not None:
            hook.remove()
    torch.cuda.synchronize()
    assert out.dtype == want.dtype and torch.equal(out, want)
    assert calls == (2 if how == "global_hook" else 0)


def test_timestep_mlp_takes_the_row_kernel(dev, monkeypatch):
    """Plain modules without grad (and in inference mode): three row linears a
    call up to 8 rows, none beyond or with gradients."""
    m = dit.AdaLayerNormSingle(512, 6).to(dev, torch.bfloat16)
    calls, run = [], kernels.skinny_linear
    monkeypatch.setattr(kernels, "skinny_linear", lambda *a, **k: (calls.append(1), run(*a, **k))[1])
    seen = []
    for ctx, rows in ((torch.no_grad, 2), (torch.inference_mode, 8), (torch.no_grad, 9), (torch.enable_grad, 2)):
        with ctx():
            m(torch.rand(rows, device=dev) * 1000, torch.bfloat16)
        seen.append(len(calls))
    assert seen == [3, 6, 6, 6]
