"""Typed wrappers over the C ABI: torch device tensors in, kernels enqueued on the
current HIP stream.  Shapes and strides are checked before any launch (for the
calls of every layer in csrc/host_calls.cpp, for the others here) so a
malformed call raises instead of reaching the GPU."""
from __future__ import annotations

import ctypes
import math
from typing import List, Optional, Sequence, Tuple

import torch

from . import _native as N

_DT = {torch.float32: N.F32, torch.bfloat16: N.BF16, torch.uint8: N.F8E4M3,
       torch.float8_e4m3fn: N.F8E4M3}


def _code(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}") from None


def _stream(t: torch.Tensor) -> int:
    return torch.cuda.current_stream(t.device).cuda_stream


def _need_gpu(*ts: Optional[torch.Tensor]) -> None:
    for t in ts:
        if t is not None and not t.is_cuda:
            raise ValueError("taomate_amd kernels take device tensors (got a CPU tensor)")


def rope_table(freq_idx: torch.Tensor, grid: Tuple[int, ...], start_frame: int, is_audio: bool,
               max_pos: Sequence[float], dim: int, num_heads: int, batch: int,
               dtype: torch.dtype) -> Tuple[torch.Tensor, torch.Tensor]:
    """ltx_rope_table -> (cos, sin) [batch, H, T, dim/(2H)] on freq_idx's device."""
    _need_gpu(freq_idx)
    assert freq_idx.dtype == torch.float32 and freq_idx.is_contiguous()
    nd = len(grid)
    T = math.prod(grid)
    per = dim // 2 // num_heads
    cos = torch.empty(batch, num_heads, T, per, device=freq_idx.device, dtype=dtype)
    sin = torch.empty_like(cos)
    gf = grid[0]
    gh = grid[1] if nd == 3 else 1
    gw = grid[2] if nd == 3 else 1
    mp = list(max_pos) + [1.0] * (3 - len(max_pos))
    N.call("ltx_rope_table", cos.data_ptr(), sin.data_ptr(), _code(cos), freq_idx.data_ptr(),
           freq_idx.numel(), nd, gf, gh, gw, int(start_frame), int(bool(is_audio)),
           float(mp[0]), float(mp[1]), float(mp[2]), dim, num_heads, batch, _stream(freq_idx))
    return cos, sin


def rope_table_retime(src: Tuple[torch.Tensor, torch.Tensor], freq_idx: torch.Tensor, grid: Tuple[int, int, int],
                      start_frame: int, max_pos_t: float, dim: int, num_heads: int) -> Tuple[torch.Tensor, torch.Tensor]:
    """ltx_rope_table_retime: the video table of ``grid`` at ``start_frame``
    from ``src`` = (cos, sin) [1, H, T, dim/(2H)] of the same grid built for
    another start frame."""
    cs, ss = src
    _need_gpu(freq_idx, cs, ss)
    T = math.prod(grid)
    per = dim // 2 // num_heads
    for t in (cs, ss):
        if t.shape != (1, num_heads, T, per) or not t.is_contiguous() or t.dtype != cs.dtype:
            raise ValueError(f"rope_table_retime: source tables must be contiguous [1, {num_heads}, {T}, {per}]")
    cos = torch.empty_like(cs)
    sin = torch.empty_like(ss)
    N.call("ltx_rope_table_retime", cos.data_ptr(), sin.data_ptr(), cs.data_ptr(), ss.data_ptr(), _code(cos),
           freq_idx.data_ptr(), freq_idx.numel(), grid[0], grid[1], grid[2], int(start_frame), float(max_pos_t),
           dim, num_heads, _stream(freq_idx))
    return cos, sin


def qk_rmsnorm_rope(q_in: torch.Tensor, q_out: torch.Tensor, gamma_q: Optional[torch.Tensor],
                    eps_q: Optional[float], q_tab, H: int, D: int,
                    k_in: Optional[torch.Tensor] = None, k_out: Optional[torch.Tensor] = None,
                    gamma_k: Optional[torch.Tensor] = None, eps_k: Optional[float] = None,
                    k_tab=None, v_in: Optional[torch.Tensor] = None, v_out: Optional[torch.Tensor] = None) -> None:
    """ltx_qk_rmsnorm_rope.  eps None skips the norm; a None table skips RoPE.
    With ``v_in`` [B, L, H, D] and a key-major bf16 ``v_out`` view of the same
    shape (the arena's V slots), the V append rides in the same launch
    (ltx_qk_rmsnorm_rope_v)."""
    (N._host or N.host()).qk_rmsnorm_rope(q_in, q_out, gamma_q, eps_q, q_tab, H, D, k_in, k_out, gamma_k, eps_k,
                                          k_tab, v_in, v_out)


def kv_append(src: torch.Tensor, dst: torch.Tensor, scales: Optional[torch.Tensor] = None,
              frame_tokens: int = 1) -> None:
    """ltx_kv_append: src [B, L, H, D] -> dst [B, L, H, D] view.

    A token-major dst (head dim contiguous) is a bf16 copy or an fp8 quantise
    (``scales`` float32 [B, H, L/frame_tokens], frame index contiguous); a
    key-major dst (token stride 1, the arena's V layout) is a bf16 transpose."""
    (N._host or N.host()).kv_append(src, dst, scales, frame_tokens)


def kv_append_fp8_pair(k: torch.Tensor, k_dst: torch.Tensor, k_scales: torch.Tensor, v: torch.Tensor,
                       v_dst: torch.Tensor, v_scales: torch.Tensor, frame_tokens: int) -> None:
    """ltx_kv_append_fp8_pair: a chunk's bf16 K and V [B, L, H, D] quantised into
    fp8 arena slots in one launch (codes and scales as ``kv_append``)."""
    (N._host or N.host()).kv_append_fp8_pair(k, k_dst, k_scales, v, v_dst, v_scales, frame_tokens)


def kv_gather(src: torch.Tensor, dst: torch.Tensor, spans: Sequence[Tuple[int, int]]) -> None:
    """ltx_kv_gather: dst[:, 0:sum(len)] = cat(src[:, s:s+len] for s, len in spans)."""
    _need_gpu(src, dst)
    if src.dtype != dst.dtype or src.dim() != 4 or dst.dim() != 4 or src.shape[0] != dst.shape[0] \
            or src.shape[2:] != dst.shape[2:]:
        raise ValueError("kv_gather: src/dst layout mismatch")
    if src.stride(3) != 1 or dst.stride(3) != 1:
        raise ValueError("kv_gather: head dim must be contiguous")
    total = sum(int(n) for _, n in spans)
    if total > dst.shape[1]:
        raise ValueError(f"kv_gather: {total} tokens do not fit dst ({dst.shape[1]})")
    for s, n in spans:
        if s < 0 or n < 0 or s + n > src.shape[1]:
            raise ValueError(f"kv_gather: span ({s}, {n}) outside src ({src.shape[1]})")
    B, _, H, D = src.shape
    starts = N.i64_array([s for s, _ in spans])
    lens = N.i64_array([n for _, n in spans])
    N.call("ltx_kv_gather", src.element_size(), B, H, D, src.data_ptr(), src.stride(0),
           src.stride(1), src.stride(2), dst.data_ptr(), dst.stride(0), dst.stride(1),
           dst.stride(2), len(spans), ctypes.cast(starts, ctypes.c_void_p),
           ctypes.cast(lens, ctypes.c_void_p), _stream(src))


class KVSegment:
    """One key/value span for flash_attn: k, v [B, L, H, D] views sharing strides;
    for fp8, k_scales / v_scales are float32 [B, H, L/frame] views."""
    __slots__ = ("k", "v", "k_scales", "v_scales")

    def __init__(self, k, v, k_scales=None, v_scales=None):
        self.k, self.v, self.k_scales, self.v_scales = k, v, k_scales, v_scales


def flash_attn(q: torch.Tensor, segments: List[KVSegment], out: torch.Tensor,
               key_mask: Optional[torch.Tensor] = None, lse: Optional[torch.Tensor] = None,
               scale: Optional[float] = None, frame_tokens: int = 0, noalloc: bool = False,
               key_lens: Optional[Sequence[int]] = None, segment_batch_strides: bool = False) -> None:
    """ltx_flash_attn_fwd.  q/out [B, Lq, H, D] bf16; key_mask float32 [B, Lk] additive.
    ``key_lens`` (B host ints): batch row b attends keys [0, key_lens[b]) only
    (a prefix-per-row padding mask, bf16 key-major V, on the pipelined kernel).
    ``noalloc`` calls ltx_flash_attn_fwd_noalloc instead: no workspace tensor,
    the split partials go to the library's fixed per-device scratch array
    (calls overlapping on one device race on it).
    ``segment_batch_strides``: token-major bf16 segments may be separate
    tensors whose batch strides differ (ltx_flash_attn_fwd_plain), with no
    mask, key counts or ``noalloc``."""
    (N._host or N.host()).flash_attn(q, segments, out, key_mask, lse, scale, frame_tokens, noalloc, key_lens,
                                     segment_batch_strides)


def skinny_linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
                  silu: bool = False) -> torch.Tensor:
    """ltx_skinny_linear: act(x) @ weight.T + bias for x [M <= 8, K <= 4096]
    bf16 (SiLU of x first with ``silu``); K must be a multiple of 8."""
    y = torch.empty(x.shape[0], weight.shape[0], dtype=x.dtype, device=x.device)
    (N._host or N.host()).skinny_linear(x, weight, bias, y, silu)
    return y


def adaln(x: torch.Tensor, y: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None,
          x_out: Optional[torch.Tensor] = None, n_out: Optional[torch.Tensor] = None,
          scale: Optional[torch.Tensor] = None, shift: Optional[torch.Tensor] = None, eps: float = 1e-6) -> None:
    """ltx_adaln on bf16 [B, L, C] rows: x_out = x + y * gate (x + y without a
    gate), n_out = rms_norm(x_out or x) * (1 + scale) + shift (plain rms_norm
    without scale/shift).  gate/scale/shift are [B, 1 or L, C]."""
    (N._host or N.host()).adaln(x, y, gate, x_out, n_out, scale, shift, eps)
