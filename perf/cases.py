"""The work that is timed: what a program built on this package has it do.

Each case is one call (or the few calls that belong together) through the
public entry points, with the sizes of the package's own configurations: the
512x768 chunk (3 latent frames of 16x24 tokens, 32 heads x 128, batch 2 for
classifier-free guidance), the 60-chunk stream's steady state, the audio and
cross-modal attentions, the text cross-attention, the small 8x12 grid, and
other latent grids of the same model.  ``draw`` gives further cases of the same
ranges: other grids (odd ones among them), frame counts, windows, head layouts,
batch sizes and cache types.

Operations:

* ``chunk``    -- q/k norm + RoPE, the K/V append and the attention of a chunk
                  over arena segments (projected rows in hand): the path's core.
* ``layer``    -- ``attention_with_cache``: a whole attention layer.
* ``text``     -- ``CausalLTXAttention`` over the prompt with a padding mask.
* ``residual`` -- gated residual + modulated RMSNorm between two layers.
* ``step``     -- one denoising step of a chunk through the dual-stream model.
"""
import math

import torch
import torch.nn.functional as F

import taomate_amd as T
from taomate_amd import dit, kernels

BF = torch.bfloat16
DEV = "cuda"
EPS = 1e-6


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    video = {"B": 2, "H": 32, "D": 128}
    audio = {"B": 2, "H": 32, "D": 64}
    return [
        # the 512x768 chunk: 1152 queries over anchor | memory | window | current = 4608 keys
        {"name": "chunk 16x24 bf16", "op": "chunk", **video, "gh": 16, "gw": 24, "frames": 3, "segs": "1,2,6",
         "kv": "bf16"},
        # the long stream's steady state: a 12-frame window in four chunks, fp8 cache, 6912 keys
        {"name": "chunk 16x24 fp8 stream", "op": "chunk", **video, "gh": 16, "gw": 24, "frames": 3,
         "segs": "1,2,3,3,3,3", "kv": "fp8"},
        # 480x704 output: frames of 330 tokens, so every segment ends in a partial key tile
        {"name": "chunk 15x22 bf16", "op": "chunk", **video, "gh": 15, "gw": 22, "frames": 3, "segs": "1,2,3,3",
         "kv": "bf16"},
        # 576x1024 output, the largest grid: 1728 queries over 10368 keys
        {"name": "chunk 18x32 fp8", "op": "chunk", **video, "gh": 18, "gw": 32, "frames": 3, "segs": "1,2,3,3,3,3",
         "kv": "fp8"},
        # the first block of a stream: 4 frames, nothing cached yet, the whole layer
        {"name": "layer first block", "op": "layer", "kind": "video", **video, "gh": 16, "gw": 24, "frames": 4,
         "segs": "", "kv": "bf16", "dim": 4096},
        # the same layer with plain-tensor caches, as a caller without arenas holds them
        {"name": "layer plain cache", "op": "layer", "kind": "video", **video, "gh": 16, "gw": 24, "frames": 3,
         "segs": "9", "kv": "dense", "dim": 4096},
        # the smallest model: 192 queries over 768 keys, 8 heads x 64, one sample
        {"name": "layer small 8x12", "op": "layer", "kind": "video", "B": 1, "H": 8, "D": 64, "gh": 8, "gw": 12,
         "frames": 2, "segs": "1,1,4", "kv": "bf16", "dim": 512},
        # audio self-attention: 75 queries over 600 cached
        {"name": "layer audio", "op": "layer", "kind": "audio", **audio, "frames": 75, "segs": "600", "kv": "bf16",
         "dim": 2048},
        # audio queries over the chunk's video tokens (the video-to-audio direction)
        {"name": "layer video to audio", "op": "layer", "kind": "v2a", **audio, "gh": 16, "gw": 24, "frames": 3,
         "audio": 75, "dim": 2048, "ctx_dim": 4096},
        # the prompt: 1024 text keys, two prompts of different length
        {"name": "text cross", "op": "text", **video, "Lq": 1152, "Lt": 1024, "keep": "820,611", "dim": 4096},
        # between two layers of a block
        {"name": "residual + norm", "op": "residual", "B": 2, "L": 1152, "C": 4096},
        # one denoising step of the chunk through two full-width dual-stream blocks
        {"name": "step of two blocks", "op": "step", "layers": 2, "B": 2, "vH": 32, "vD": 128, "aH": 32, "aD": 64,
         "gh": 16, "gw": 24, "frames": 3, "cached": 9, "audio": 75, "audio_cached": 600, "Lt": 1024,
         "keep": "820,820"},
    ]


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= 5.5e11 and w["bytes"] <= 1.2e9:
            return c


def _grid(rng, lo=96, hi=576):
    while True:
        gh, gw = rng.randint(6, 24), rng.randint(8, 32)
        if lo <= gh * gw <= hi:
            return gh, gw


def _draw(rng):
    op = rng.choice(["chunk", "chunk", "chunk", "layer", "layer", "audio", "v2a", "a2v", "text", "residual", "step"])
    B = rng.choice([1, 2, 2])
    H, D = rng.choice([(32, 128), (32, 128), (32, 64), (16, 128), (8, 64)])
    gh, gw = _grid(rng)
    frames = rng.choice([1, 2, 3, 3, 4])
    if op in ("chunk", "layer"):
        window = rng.randint(0, 4)
        segs = ",".join(["1"] + (["2"] if rng.random() < 0.7 else []) + ["3"] * window)
        c = {"op": op, "B": B, "H": H, "D": D, "gh": gh, "gw": gw, "frames": frames}
        if op == "chunk":
            return {**c, "segs": segs, "kv": rng.choice(["bf16", "fp8"])}
        kv = rng.choice(["bf16", "fp8", "dense"])
        cached = sum(_segs(segs))
        return {**c, "kind": "video", "segs": str(cached) if kv == "dense" else segs, "kv": kv, "dim": H * D}
    La = 25 * frames + rng.choice([0, 0, 1])
    if op == "audio":
        return {"op": "layer", "kind": "audio", "B": B, "H": 32, "D": 64, "frames": La,
                "segs": str(25 * rng.randint(1, 60)), "kv": "bf16", "dim": 2048}
    if op in ("v2a", "a2v"):
        return {"op": "layer", "kind": op, "B": B, "H": 32, "D": 64, "gh": gh, "gw": gw, "frames": frames, "audio": La,
                "dim": 2048 if op == "v2a" else 4096, "ctx_dim": 4096 if op == "v2a" else 2048}
    if op == "text":
        Lt = rng.randint(64, 1024)
        keep = ",".join(str(rng.randint(Lt // 2, Lt)) for _ in range(B))
        return {"op": "text", "B": B, "H": H, "D": D, "Lq": frames * gh * gw, "Lt": Lt, "keep": keep, "dim": H * D}
    if op == "residual":
        return {"op": "residual", "B": B, "L": int(round(math.exp(rng.uniform(math.log(25), math.log(2304))))),
                "C": rng.choice([512, 2048, 4096])}
    Lt = rng.randint(128, 1024)
    return {"op": "step", "layers": 1, "B": B, "vH": 8, "vD": 128, "aH": 8, "aD": 64, "gh": gh, "gw": gw,
            "frames": frames, "cached": rng.randint(1, 9), "audio": La, "audio_cached": 25 * rng.randint(1, 24),
            "Lt": Lt, "keep": ",".join(str(rng.randint(Lt // 2, Lt)) for _ in range(B))}


def _segs(text):
    return [int(n) for n in text.split(",")] if text else []


# --------------------------------------------------------------------------
# inputs, from the seed alone
# --------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def __call__(self, *shape, std=1.0, mean=0.0):
        x = torch.randn(*shape, generator=self.g, device=DEV)
        return (x.mul_(std).add_(mean) if std != 1.0 or mean else x).to(BF)


def _rope(grid, dim, heads, start, audio=False, repeat=1):
    """(cos, sin) [1, heads, tokens, dim / (2 heads)] in bf16 at the model's
    positions: seconds / 20 and, for a grid, pixels / 2048, against
    10000^[0, 1] frequencies, axes interleaved, identity pairs in front."""
    nd = len(grid)
    f = torch.arange(grid[0], device=DEV, dtype=torch.float64) + start
    scale, rate = (4, 100.0) if audio else (8, 24.0)
    sec = ((f * scale + 1 - scale).clamp(min=0) + ((f + 1) * scale + 1 - scale).clamp(min=0)) / 2 / rate
    axes = [sec / 20.0]
    if nd == 3:
        axes += [(torch.arange(n, device=DEV, dtype=torch.float64) * 32 + 16) / 2048.0 for n in grid[1:]]
    pos = torch.stack(torch.meshgrid(*axes, indexing="ij"), -1).reshape(-1, nd)
    n = dim // (2 * nd)
    freq = 10000.0 ** torch.linspace(0, 1, n, device=DEV, dtype=torch.float64) * (math.pi / 2)
    ang = (freq[None, :, None] * (pos[:, None, :] * 2 - 1)).reshape(pos.shape[0], -1)
    pad = dim // 2 - ang.shape[1]
    ang = F.pad(ang, (pad, 0)).repeat_interleave(repeat, 0)
    ang = ang.reshape(ang.shape[0], heads, -1).transpose(0, 1)[None]
    return ang.cos().to(BF).contiguous(), ang.sin().to(BF).contiguous()


def _e4m3(x, hw):
    """Codes and scales of frames of ``hw`` tokens: x [B, L, H, D]."""
    B, L, H, D = x.shape
    f = x.float().reshape(B, L // hw, hw, H, D)
    s = f.abs().amax(dim=(2, 4)) / 448.0
    s = torch.where(s > 0, s, torch.ones_like(s))
    codes = (f / s[:, :, None, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return codes.view(torch.uint8).reshape(B, L, H, D), s.permute(0, 2, 1).contiguous()


def _dequant(codes, s, hw):
    B, L, H, D = codes.shape
    v = codes.view(torch.float8_e4m3fn).double().reshape(B, L // hw, hw, H, D)
    return (v * s.permute(0, 2, 1).double()[:, :, None, :, None]).reshape(B, L, H, D)


def _weights(r, names):
    """{name: tensor}: linears ~N(0, 0.02^2) with small biases, norm gains around 1."""
    out = {}
    for n, shape in names:
        if n.endswith("norm.weight"):
            out[n] = r(*shape, std=0.1, mean=1.0)
        else:
            out[n] = r(*shape, std=0.02)
    return out


def _attn_names(c):
    inner, dim, ctx = c["H"] * c["D"], c["dim"], c.get("ctx_dim", c["dim"])
    return [("to_q.weight", (inner, dim)), ("to_q.bias", (inner,)), ("to_k.weight", (inner, ctx)),
            ("to_k.bias", (inner,)), ("to_v.weight", (inner, ctx)), ("to_v.bias", (inner,)),
            ("q_norm.weight", (inner,)), ("k_norm.weight", (inner,)), ("to_out.0.weight", (dim, inner)),
            ("to_out.0.bias", (dim,))]


def _attn_module(c, weights, cross):
    with torch.device("meta"):
        m = T.CausalLTXAttention(c["dim"], context_dim=c.get("ctx_dim", c["dim"]) if cross else None, heads=c["H"],
                                 dim_head=c["D"], norm_eps=EPS)
    m.load_state_dict(weights, assign=True)
    return m.eval()


def _inputs(case, seed):
    c, r = case, _Rand(seed)
    B = c["B"]
    if c["op"] == "residual":
        L, C = c["L"], c["C"]
        return {"x": r(B, L, C), "y": r(B, L, C), "gate": r(B, 1, C), "scale": r(B, 1, C, std=0.3),
                "shift": r(B, 1, C, std=0.3)}
    if c["op"] == "step":
        return _step_inputs(c, r)
    H, D = c["H"], c["D"]
    HD = H * D
    if c["op"] == "text":
        mask = torch.zeros(B, 1, 1, c["Lt"], dtype=BF, device=DEV)
        for b, n in enumerate(_segs(c["keep"])):
            mask[b, ..., n:] = torch.finfo(BF).min
        return {"w": _weights(r, _attn_names(c)), "x": r(B, c["Lq"], c["dim"]), "ctx": r(B, c["Lt"], c["dim"]),
                "mask": mask}
    hw = 1 if c.get("kind") == "audio" else c["gh"] * c["gw"]
    L = c["frames"] * hw
    i = {"hw": hw, "segs": [n * hw for n in _segs(c.get("segs", ""))]}
    # cached keys carry unit rows (they were normalised), values the projection's spread
    cached = sum(i["segs"])
    if cached:
        i["k"], i["v"] = r(B, cached, H, D), r(B, cached, H, D, std=0.02 * math.sqrt(HD))
        if c.get("kv") == "fp8":
            i["kc"], i["ks"] = _e4m3(i["k"], hw)
            i["vc"], i["vs"] = _e4m3(i["v"], hw)
    start = cached // hw
    if c["op"] == "chunk":
        std = 0.02 * math.sqrt(HD)
        i.update(q_lin=r(B, L, HD, std=std), k_lin=r(B, L, HD, std=std), v_lin=r(B, L, HD, std=std),
                 gq=r(HD, std=0.1, mean=1.0), gk=r(HD, std=0.1, mean=1.0),
                 pe=_rope((c["frames"], c["gh"], c["gw"]), HD, H, start))
        return i
    i["w"] = _weights(r, _attn_names(c))
    if c["kind"] == "video":
        i.update(x=r(B, L, c["dim"]), pe=_rope((c["frames"], c["gh"], c["gw"]), HD, H, start))
    elif c["kind"] == "audio":
        i.update(x=r(B, L, c["dim"]), pe=_rope((L,), HD, H, start, True))
    else:
        v_pe, a_pe = _rope((c["frames"],), HD, H, 3, repeat=hw), _rope((c["audio"],), HD, H, 75, True)
        to_audio = c["kind"] == "v2a"
        i.update(x=r(B, c["audio"] if to_audio else L, c["dim"]), ctx=r(B, L if to_audio else c["audio"], c["ctx_dim"]),
                 pe=a_pe if to_audio else v_pe, k_pe=v_pe if to_audio else a_pe)
    return i


def _batched(pe, B):
    return tuple(t.expand(B, -1, -1, -1) for t in pe)


def _arena(c, i, extra):
    """An arena holding the cached segments, each at its own aligned slots, and their spans."""
    hw, fp8 = i["hw"], c["kv"] == "fp8"
    al = hw if fp8 else 8
    up = lambda n: -(-n // al) * al
    cap = sum(up(n) for n in i["segs"]) + up(extra)
    arena = T.KVArena(c["B"], cap, c["H"], c["D"], DEV, c["kv"], frame_tokens=hw)
    spans, pos, at = [], 0, 0
    for n in i["segs"]:
        src = slice(at, at + n)
        if fp8:
            arena.slots("k", pos, n).copy_(i["kc"][:, src])
            arena.slots("v", pos, n).copy_(i["vc"][:, src])
            arena.scale_slots("k", pos, n).copy_(i["ks"][:, :, at // hw:(at + n) // hw])
            arena.scale_slots("v", pos, n).copy_(i["vs"][:, :, at // hw:(at + n) // hw])
        else:
            arena.slots("k", pos, n).copy_(i["k"][:, src])
            arena.slots("v", pos, n).copy_(i["v"][:, src])
        spans.append((pos, n))
        at += n
        pos += up(n)
    return arena, spans, pos


def prepare(case, seed):
    c, i = case, _inputs(case, seed)
    B = c["B"]
    s = {"c": c}
    if c["op"] == "residual":
        s.update(i, x_out=torch.empty_like(i["x"]), n_out=torch.empty_like(i["x"]))
        return s
    if c["op"] == "step":
        return _step_prepare(c, i)
    if c["op"] == "text":
        s.update(m=_attn_module(c, i["w"], True), x=i["x"], ctx=i["ctx"], mask=i["mask"])
        return s
    if c["op"] == "chunk":
        L, H, D = i["q_lin"].shape[1], c["H"], c["D"]
        arena, spans, pos = _arena(c, i, L)
        segs = [kernels.KVSegment(arena.slots("k", a, n), arena.slots("v", a, n), arena.scale_slots("k", a, n),
                                    arena.scale_slots("v", a, n)) for a, n in spans + [(pos, L)]]
        s.update(arena=arena, segs=segs, new=segs[-1], hw=i["hw"], pe=_batched(i["pe"], B), gq=i["gq"], gk=i["gk"],
                 q_lin=i["q_lin"], k_lin=i["k_lin"], v_lin=i["v_lin"].view(B, L, H, D),
                 q=torch.empty_like(i["q_lin"]), k=torch.empty_like(i["k_lin"]),
                 out=torch.empty(B, L, H, D, dtype=BF, device=DEV))
        return s
    cross = "ctx" in i
    s.update(m=_attn_module(c, i["w"], cross), x=i["x"], ctx=i.get("ctx"), pe=_batched(i["pe"], B),
             k_pe=_batched(i["k_pe"], B) if cross else None, ck=None, cv=None)
    if not cross and c["kv"] == "dense":
        s.update(ck=i["k"], cv=i["v"])
    elif not cross:
        arena, spans, _ = _arena(c, i, i["x"].shape[1])
        s.update(arena=arena, ck=T.KVSpanView(arena, "k", spans), cv=T.KVSpanView(arena, "v", spans))
        s["m"].fuse_qkv_()
    return s


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _new_kv(view):
    """The chunk's new cache entries: slots (and scales), or the plain tensor."""
    return [view] if isinstance(view, torch.Tensor) else [list(p) for p in view.pieces()]


@torch.no_grad()
def run(s):
    c = s["c"]
    if c["op"] == "residual":
        kernels.adaln(s["x"], y=s["y"], gate=s["gate"], x_out=s["x_out"], n_out=s["n_out"], scale=s["scale"],
                      shift=s["shift"], eps=EPS)
        return {"x": s["x_out"], "n": s["n_out"]}
    if c["op"] == "chunk":
        H, D, new, q, pe = c["H"], c["D"], s["new"], s["q"], s["pe"]
        B, L = q.shape[:2]
        if c["kv"] == "bf16":
            kernels.qk_rmsnorm_rope(s["q_lin"], q, s["gq"], EPS, pe, H, D, s["k_lin"], new.k, s["gk"], EPS, pe,
                                    v_in=s["v_lin"], v_out=new.v)
            kernels.flash_attn(q.view(B, L, H, D), s["segs"], s["out"])
            return {"q": q, "k": new.k, "v": new.v, "out": s["out"]}
        k = s["k"]
        kernels.qk_rmsnorm_rope(s["q_lin"], q, s["gq"], EPS, pe, H, D, s["k_lin"], k, s["gk"], EPS, pe)
        kernels.kv_append_fp8_pair(k.view(B, L, H, D), new.k, new.k_scales, s["v_lin"], new.v, new.v_scales, s["hw"])
        kernels.flash_attn(q.view(B, L, H, D), s["segs"], s["out"], frame_tokens=s["hw"])
        return {"q": q, "k": new.k, "ks": new.k_scales, "v": new.v, "vs": new.v_scales, "out": s["out"]}
    if c["op"] == "text":
        return {"out": s["m"](s["x"], context=s["ctx"], mask=s["mask"])}
    if c["op"] == "step":
        vo, ao, _ = s["model"].forward_chunk(*s["args"], s["caches"])
        return {"video": vo, "audio": ao}
    out, nk, nv = T.attention_with_cache(s["m"], s["x"], s["ctx"], s["pe"], s["k_pe"], s["ck"], s["cv"])
    return {"out": out, "k": _new_kv(nk), "v": _new_kv(nv)}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    c = case
    B = c["B"]
    if c["op"] == "residual":
        n = B * c["L"] * c["C"]
        return {"bytes": 2 * (4 * n + 3 * B * c["C"]), "flops": 12 * n}
    if c["op"] == "step":
        return _step_work(c)
    H, D = c["H"], c["D"]
    HD = H * D
    if c["op"] == "text":
        Lq, Lt, dim, kept = c["Lq"], c["Lt"], c["dim"], sum(_segs(c["keep"]))
        rows = 2 * B * Lq * dim * HD * 2 + 2 * B * Lt * dim * HD * 2
        return {"bytes": 2 * (4 * dim * HD + 2 * B * Lq * dim + B * Lt * dim), "flops": rows + 4 * HD * Lq * kept}
    if c.get("kind") in ("v2a", "a2v"):
        hw = c["gh"] * c["gw"] * c["frames"]
        Lq, Lk = (c["audio"], hw) if c["kind"] == "v2a" else (hw, c["audio"])
        dim, ctx = c["dim"], c["ctx_dim"]
        return {"bytes": 2 * (2 * HD * (dim + ctx) + 2 * B * Lq * dim + B * Lk * ctx + 2 * B * Lk * HD),
                "flops": 4 * B * (Lq * dim + Lk * ctx) * HD + 4 * B * HD * Lq * Lk}
    hw = 1 if c.get("kind") == "audio" else c["gh"] * c["gw"]
    L, cached = c["frames"] * hw, sum(_segs(c["segs"])) * hw
    esz = 1 if c["kv"] == "fp8" else 2
    attn = 4 * B * HD * L * (cached + L)
    table = 2 * L * HD
    cache = 2 * B * HD * esz * (cached + L)
    if c["op"] == "chunk":
        # rows in, q (an output here) and the attention out, the cache read and the new slots written, the table
        return {"bytes": 2 * B * L * HD * 5 + cache + table, "flops": attn}
    dim = c["dim"]
    return {"bytes": 2 * (4 * dim * HD + 2 * B * L * dim) + cache + table, "flops": 8 * B * L * dim * HD + attn}


def tolerance(case):
    if case["op"] == "residual":
        return {"rel": 4e-3, "max": 4e-2}
    if case["op"] == "step":
        return {"rel": 2e-2, "max": 2e-1}
    return {"rel": 1e-2, "max": 1e-1, "differ": 2e-3}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------
def _norm64(x, w=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _rot64(x, pe, H):
    """Rotate [B, L, H*D] rows: pairs (j, j + D/2) of every head."""
    B, L, HD = x.shape
    cos, sin = (t.double().permute(0, 2, 1, 3)[:, :L] for t in pe)
    x1, x2 = x.view(B, L, H, 2, -1).unbind(3)
    return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1)


def _attend64(q, k, v, keep=None):
    """softmax(q k^T / sqrt(D)) v for [B, L, H, D], a few heads at a time."""
    B, Lq, H, D = q.shape
    out = torch.empty_like(q)
    step = max(1, int(1.5e9 // (8 * Lq * k.shape[1])))
    for b in range(B):
        n = k.shape[1] if keep is None else keep[b]
        for h in range(0, H, step):
            hs = slice(h, h + step)
            qq = q[b, :, hs].transpose(0, 1).contiguous()
            kt = k[b, :n, hs].permute(1, 2, 0).contiguous()
            p = torch.softmax(torch.matmul(qq, kt) / math.sqrt(D), -1)
            out[b, :, hs] = torch.matmul(p, v[b, :n, hs].transpose(0, 1).contiguous()).transpose(0, 1)
    return out


def _lin64(x, w, name):
    return F.linear(x, w[name + ".weight"].double(), w[name + ".bias"].double())


def _layer64(w, H, x, ctx, pe, k_pe, ck, cv, keep=None, quant=None):
    """(out, new k, new v) of an attention layer; ``quant`` stores the new keys and values."""
    B = x.shape[0]
    q, k = _norm64(_lin64(x, w, "to_q"), w["q_norm.weight"]), _norm64(_lin64(ctx, w, "to_k"), w["k_norm.weight"])
    split = lambda t: t.view(B, t.shape[1], H, -1)
    q, k = (_rot64(t, p, H) if p is not None else split(t) for t, p in ((q, pe), (k, k_pe)))
    v = split(_lin64(ctx, w, "to_v"))
    kk, vv = (k, v) if quant is None else (quant(k), quant(v))
    if ck is not None:
        kk, vv = torch.cat([ck, kk], 1), torch.cat([cv, vv], 1)
    o = _attend64(q, kk, vv, keep).flatten(2)
    return _lin64(o, w, "to_out.0"), k, v


@torch.no_grad()
def exact(case, seed):
    c, i = case, _inputs(case, seed)
    if c["op"] == "residual":
        x = i["x"].double() + i["y"].double() * i["gate"].double()
        return {"x": x, "n": _norm64(x) * (1 + i["scale"].double()) + i["shift"].double()}
    if c["op"] == "step":
        return _step_exact(c, i)
    if c["op"] == "text":
        return {"out": _layer64(i["w"], c["H"], i["x"].double(), i["ctx"].double(), None, None, None, None,
                                _segs(c["keep"]))[0]}
    ck = cv = quant = None
    fp8 = c.get("kv") == "fp8"
    if "k" in i:
        ck, cv = i["k"].double(), i["v"].double()
        if fp8:
            ck, cv = _dequant(i["kc"], i["ks"], i["hw"]), _dequant(i["vc"], i["vs"], i["hw"])
    if fp8:
        quant = lambda t: _dequant(*_e4m3(t, i["hw"]), i["hw"])
    if c["op"] == "layer":
        x = i["x"].double()
        ctx = i["ctx"].double() if "ctx" in i else x
        out, k, v = _layer64(i["w"], c["H"], x, ctx, i["pe"], i.get("k_pe", i["pe"]), ck, cv, None, quant)
        stored = lambda t: [[None, _e4m3(t, i["hw"])[1]]] if fp8 else [t] if c.get("kv", "dense") == "dense" else \
            [[t, None]]
        return {"out": out, "k": stored(k), "v": stored(v)}
    H = c["H"]
    B, L, HD = i["q_lin"].shape
    q = _rot64(_norm64(i["q_lin"].double(), i["gq"]), i["pe"], H)
    k = _rot64(_norm64(i["k_lin"].double(), i["gk"]), i["pe"], H)
    v = i["v_lin"].double().view(B, L, H, -1)
    kk, vv = (quant(k), quant(v)) if fp8 else (k, v)
    if ck is not None:
        kk, vv = torch.cat([ck, kk], 1), torch.cat([cv, vv], 1)
    out = {"q": q.flatten(2), "k": k, "v": v, "out": _attend64(q, kk, vv)}
    if fp8:
        out.update(k=None, v=None, ks=_e4m3(k, i["hw"])[1], vs=_e4m3(v, i["hw"])[1])
    return out


# --------------------------------------------------------------------------
# the dual-stream step
# --------------------------------------------------------------------------
def _step_config(c):
    return dit.AVConfig(num_layers=c["layers"], video_dim=c["vH"] * c["vD"], audio_dim=c["aH"] * c["aD"],
                        video_heads=c["vH"], video_d_head=c["vD"], audio_heads=c["aH"], audio_d_head=c["aD"])


def _step_inputs(c, r):
    B, cfg = c["B"], _step_config(c)
    vd, ad, aH = cfg.video_dim, cfg.audio_dim, c["aH"]
    with torch.device("meta"):
        shapes = [(n, tuple(p.shape)) for n, p in dit.AVModel(cfg).named_parameters()]
    w = _weights(r, [(n, s) for n, s in shapes if "scale_shift_table" not in n])
    w.update({n: r(*s, std=1 / math.sqrt(s[-1])) for n, s in shapes if "scale_shift_table" in n})
    hw = c["gh"] * c["gw"]
    L, Lc, La, Lac = c["frames"] * hw, c["cached"] * hw, c["audio"], c["audio_cached"]
    mask = torch.zeros(B, 1, 1, c["Lt"], dtype=BF, device=DEV)
    for b, n in enumerate(_segs(c["keep"])):
        mask[b, ..., n:] = torch.finfo(BF).min
    return {"w": w, "vlat": r(B, L, cfg.in_channels), "alat": r(B, La, cfg.in_channels),
            "sigma": torch.rand(B, generator=r.g, device=DEV) * 0.8 + 0.1, "vctx": r(B, c["Lt"], vd),
            "actx": r(B, c["Lt"], ad), "mask": mask,
            "vk": r(B, Lc, c["vH"], c["vD"]), "vv": r(B, Lc, c["vH"], c["vD"], std=0.02 * math.sqrt(vd)),
            "ak": r(B, Lac, aH, c["aD"]), "av": r(B, Lac, aH, c["aD"], std=0.02 * math.sqrt(ad)),
            "vpe": _rope((c["frames"], c["gh"], c["gw"]), vd, c["vH"], c["cached"]), "ape": _rope((La,), ad, aH, Lac, True),
            "vcross": _rope((c["frames"],), ad, aH, c["cached"], repeat=hw), "across": _rope((La,), ad, aH, Lac, True)}


def _step_prepare(c, i):
    B, cfg = c["B"], _step_config(c)
    with torch.device("meta"):
        model = dit.AVModel(cfg)
    model.load_state_dict(i["w"], assign=True)
    model.eval().fuse_qkv_()
    Lv, La, Lc, Lac = i["vlat"].shape[1], c["audio"], i["vk"].shape[1], c["audio_cached"]
    up = lambda n: -(-n // 8) * 8
    specs = {"video_self": T.ArenaSpec(up(Lc) + up(Lv), c["vH"], c["vD"]),
             "audio_self": T.ArenaSpec(up(Lac) + up(La), c["aH"], c["aD"])}
    caches = []
    for lay in T.init_kv_cache(cfg.num_layers, B, specs, DEV).layers:
        va, aa = lay.video_self_k.arena, lay.audio_self_k.arena
        for arena, n, k, v in ((va, Lc, i["vk"], i["vv"]), (aa, Lac, i["ak"], i["av"])):
            arena.slots("k", 0, n).copy_(k)
            arena.slots("v", 0, n).copy_(v)
        view = lambda arena, which, n: T.KVSpanView(arena, which, [(0, n)])
        caches.append(T.LayerKVCache(video_self_k=view(va, "k", Lc), video_self_v=view(va, "v", Lc),
                                     audio_self_k=view(aa, "k", Lac), audio_self_v=view(aa, "v", Lac)))
    args = (i["vlat"], i["alat"], i["sigma"], i["vctx"], i["actx"], i["mask"], i["mask"], _batched(i["vpe"], B),
            _batched(i["ape"], B), _batched(i["vcross"], B), _batched(i["across"], B))
    return {"c": c, "model": model, "caches": caches, "args": args}


def _step_work(c):
    B, n = c["B"], c["layers"]
    hw = c["gh"] * c["gw"]
    L, Lc, La, Lac, Lt = c["frames"] * hw, c["cached"] * hw, c["audio"], c["audio_cached"], c["Lt"]
    vd, ad, kept = c["vH"] * c["vD"], c["aH"] * c["aD"], sum(_segs(c["keep"]))
    # projections: self (4), text (q, out on the stream's rows, k, v on the prompt's), both cross directions, 4x FFN
    params = 4 * vd * vd + 4 * ad * ad + 4 * vd * vd + 4 * ad * ad + 8 * vd * ad + 8 * vd * vd + 8 * ad * ad
    v_rows = (4 + 2 + 8) * vd * vd + 2 * vd * ad + 2 * vd * ad
    a_rows = (4 + 2 + 8) * ad * ad + 4 * ad * ad
    gemm = 2 * B * (L * v_rows + La * a_rows + Lt * 2 * (vd * vd + ad * ad))
    attn = 4 * (B * vd * L * (Lc + L) + B * ad * La * (Lac + La) + (vd * L + ad * La) * kept + 2 * B * ad * L * La)
    # weights, the cache, and the latents, prompts and outputs once
    io = 2 * (n * params + 2 * n * B * (vd * (Lc + L) + ad * (Lac + La)) + B * Lt * (vd + ad) + 2 * B * 128 * (L + La))
    ada = 2 * (14 * vd * vd + 14 * ad * ad)
    return {"bytes": io + ada, "flops": n * (gemm + attn)}


def _step_exact(c, i):
    B, w = c["B"], {n: t.double() for n, t in i["w"].items()}
    sub = lambda p: {n[len(p):]: t for n, t in w.items() if n.startswith(p)}
    lin = lambda x, n: F.linear(x, w[n + ".weight"], w[n + ".bias"])

    def embed(p, t):
        ang = t[:, None] * torch.exp(-math.log(10000) * torch.arange(128, device=DEV, dtype=torch.float64) / 128)
        e = torch.cat([ang.cos(), ang.sin()], -1)
        e = lin(F.silu(lin(e, p + "emb.timestep_embedder.linear_1")), p + "emb.timestep_embedder.linear_2")
        return lin(F.silu(e), p + "linear"), e

    t = (i["sigma"] * 1000.0).double()
    (v_ts, v_e), (a_ts, a_e) = embed("adaln_single.", t), embed("audio_adaln_single.", t)
    v_ss, a_ss = (embed(f"av_ca_{m}_scale_shift_adaln_single.", t)[0] for m in ("video", "audio"))
    v_g, a_g = (embed(f"av_ca_{m}_gate_adaln_single.", t / 1000.0)[0] for m in ("a2v", "v2a"))
    mod = lambda table, ts: (table[None] + ts.view(B, table.shape[0], -1)).unsqueeze(2).unbind(1)
    keep = _segs(c["keep"])
    vctx, actx = i["vctx"].double(), i["actx"].double()
    vx, ax = lin(i["vlat"].double(), "patchify_proj"), lin(i["alat"].double(), "audio_patchify_proj")
    ffn = lambda x, p: lin(F.gelu(lin(x, p + "net.0.proj"), approximate="tanh"), p + "net.2")
    for n in range(c["layers"]):
        p = f"transformer_blocks.{n}."
        new = []
        for x, ts, pre, H, pe, k, v, ctx in ((vx, v_ts, "", c["vH"], i["vpe"], i["vk"], i["vv"], vctx),
                                             (ax, a_ts, "audio_", c["aH"], i["ape"], i["ak"], i["av"], actx)):
            m = mod(w[p + pre + "scale_shift_table"], ts)
            xn = _norm64(x) * (1 + m[1]) + m[0]
            x = x + _layer64(sub(p + pre + "attn1."), H, xn, xn, pe, pe, k.double(), v.double())[0] * m[2]
            x = x + _layer64(sub(p + pre + "attn2."), H, _norm64(x), ctx, None, None, None, None, keep)[0]
            new.append((x, m))
        (vx, vm), (ax, am) = new
        vn, an = _norm64(vx), _norm64(ax)
        ta, tv = w[p + "scale_shift_table_a2v_ca_audio"], w[p + "scale_shift_table_a2v_ca_video"]
        sa, sv = mod(ta[:4], a_ss), mod(tv[:4], v_ss)
        ga, gv = mod(ta[4:], a_g)[0], mod(tv[4:], v_g)[0]
        aH = c["aH"]
        a2v = _layer64(sub(p + "audio_to_video_attn."), aH, vn * (1 + sv[0]) + sv[1], an * (1 + sa[0]) + sa[1],
                       i["vcross"], i["across"], None, None)[0]
        v2a = _layer64(sub(p + "video_to_audio_attn."), aH, an * (1 + sa[2]) + sa[3], vn * (1 + sv[2]) + sv[3],
                       i["across"], i["vcross"], None, None)[0]
        vx, ax = vx + a2v * gv, ax + v2a * ga
        vx = vx + ffn(_norm64(vx) * (1 + vm[4]) + vm[3], p + "ff.") * vm[5]
        ax = ax + ffn(_norm64(ax) * (1 + am[4]) + am[3], p + "audio_ff.") * am[5]

    def head(x, e, pre):
        m = w[pre + "scale_shift_table"][None] + e[:, None]
        return lin(F.layer_norm(x, (x.shape[-1],), eps=1e-6) * (1 + m[:, 1:]) + m[:, :1], pre + "proj_out")

    return {"video": head(vx, v_e, ""), "audio": head(ax, a_e, "audio_")}
