"""Timing cases of the framework's public calls, from the smallest to the largest.

Each case is one call a program makes per layer and denoising step:

* ``dfs``: ``dfs_attention`` of a Wan-style (video only) or HunyuanVideo-style
  (video, then text with padding) layer, on a step that selects its mask or on
  one that reuses it;
* ``dense``: ``full_attention`` of a warm-up or skipped layer;
* ``heads``: the projections' way into the attention inputs (QK RMSNorm, RoPE,
  head split), in either model's form;
* ``glue``: the adaLN modulation and gated residual around a layer;
* ``layer``: a whole self-attention layer through the Wan processor
  (projections, norm, RoPE, sparse attention, output projection).
"""
import itertools
import math
from types import SimpleNamespace

import torch

from dfsattn_amd import attention_hyvideo, attention_wan, ops
from dfsattn_amd.dit import DiTAttention, wan_rope_freqs
from dfsattn_amd.fullattention import full_attention
from dfsattn_amd.layout import ScoringLayout, hunyuan_policy, wan_policy
from dfsattn_amd.replace_hyvideo import fused_qkv_heads_per_head
from dfsattn_amd.replace_wan import Wan_DFSAttn_Processor2_0, fused_qkv_heads
from dfsattn_amd.utils.order import hilbert3d_perm
from dfsattn_amd.workloads import DfsConfig, drift, smoothed_field, synth_qkv

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
BLOCK = 128
SKIP, INTERVAL = 12, 12  # the drivers' warm-up steps and mask refresh interval

# One layer number per state: a program's layers each keep their own order and mask.
_layers = itertools.count()


def _dfs(name, grid, heads, dim=128, dtype="bf16", operand="f16", text=0, valid=0, tile=16, sparsity=0.3,
         refresh=True):
    f, h, w = grid
    return {"name": name, "kind": "dfs", "f": f, "h": h, "w": w, "heads": heads, "dim": dim, "dtype": dtype,
            "operand": operand, "text": text, "valid": valid, "tile": tile, "sparsity": sparsity,
            "refresh": refresh}


def listed():
    return [
        # the plumbing size, 1,024 tokens and 2 heads: latency and launches
        _dfs("dfs_small", (4, 16, 16), 2, dim=64, dtype="f16"),
        # one latent frame (an image) at the API's default tile of 32
        _dfs("dfs_frame", (1, 45, 80), 12, tile=32),
        # a short clip at 480p on the steps between refreshes, which are most of a run
        _dfs("dfs_clip_cached", (13, 30, 52), 40, sparsity=0.2, refresh=False),
        # the Wan benchmark layer: 75,600 tokens, 40 heads, a fresh mask
        _dfs("dfs_video", (21, 45, 80), 40),
        # bf16 operands (the setting for the reference kernel's precision class), 480p
        _dfs("dfs_bf16_operands", (21, 30, 52), 12, operand="bf16"),
        # the HunyuanVideo benchmark layer: text padded to 256 tokens, 118 of them valid
        _dfs("dfs_hunyuan", (33, 45, 80), 24, text=256, valid=118),
        # odd sizes everywhere: ragged video and text, f16 inputs
        _dfs("dfs_hunyuan_odd", (9, 33, 47), 24, dtype="f16", text=125, valid=93, sparsity=0.4),
        # a dense warm-up step of a short ragged sequence
        {"name": "dense_ragged", "kind": "dense", "length": 8191, "heads": 12, "dim": 128, "dtype": "bf16"},
        # projections to heads, Wan form (norm over all heads, complex RoPE) at the benchmark layer
        {"name": "heads_wan", "kind": "heads", "form": "wan", "f": 21, "h": 45, "w": 80, "text": 0, "heads": 40,
         "dim": 128, "dtype": "bf16"},
        # HunyuanVideo form (norm per head, real RoPE, text not rotated), a short odd clip
        {"name": "heads_hunyuan", "kind": "heads", "form": "hunyuan", "f": 9, "h": 33, "w": 47, "text": 125,
         "heads": 24, "dim": 128, "dtype": "bf16"},
        # modulation before and gated residual after a layer at the benchmark width
        {"name": "glue_wan", "kind": "glue", "rows": 32760, "channels": 5120, "dtype": "bf16"},
        # a whole attention layer of the benchmark width on a short clip
        {"name": "layer_wan", "kind": "layer", "f": 13, "h": 30, "w": 52, "heads": 40, "dim": 128,
         "dtype": "bf16", "sparsity": 0.3},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A latent grid of about log-uniform size between lo and hi tokens."""
    tokens = _log_int(rng, lo, hi)
    h, w = rng.randint(12, 45), rng.randint(16, 80)
    while h * w > tokens:
        h, w = max(8, h * 3 // 4), max(8, w * 3 // 4)
    return max(1, tokens // (h * w)), h, w


def draw(rng):
    kind = rng.choices(["dfs", "dense", "heads", "glue", "layer"], [11, 3, 3, 2, 1])[0]
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    if kind == "dfs":
        while True:
            grid = _grid(rng, 1024, 75600)
            text = rng.randint(20, 300) if rng.random() < 0.4 else 0
            dim = rng.choice([128, 128, 128, 64])
            case = _dfs("", grid, _log_int(rng, 1, 40), dim=dim, dtype=dtype,
                        operand="bf16" if dtype == "bf16" and rng.random() < 0.2 else "f16", text=text,
                        valid=rng.randint(1, text) if text else 0, tile=rng.choice([16, 16, 32]),
                        sparsity=round(rng.uniform(0.1, 0.5), 3), refresh=rng.random() < 0.5)
            del case["name"]
            try:  # the text has to fit the padded scoring layout and the budget
                _policy(case)
            except (RuntimeError, AssertionError):
                continue
            return case
    if kind == "dense":
        length = _log_int(rng, 256, 24000)
        return {"kind": kind, "length": length, "heads": _log_int(rng, 1, 40),
                "dim": rng.choice([128, 128, 64]), "dtype": dtype}
    if kind == "heads":
        f, h, w = _grid(rng, 1024, 75600)
        form = rng.choice(["wan", "hunyuan"])
        return {"kind": kind, "form": form, "f": f, "h": h, "w": w,
                "text": rng.randint(20, 300) if form == "hunyuan" else 0, "heads": _log_int(rng, 2, 40),
                "dim": rng.choice([128, 128, 64]), "dtype": dtype}
    if kind == "glue":
        return {"kind": kind, "rows": _log_int(rng, 1000, 75600), "channels": 64 * rng.randint(8, 80),
                "dtype": dtype}
    f, h, w = _grid(rng, 1024, 20280)
    return {"kind": kind, "f": f, "h": h, "w": w, "heads": rng.choice([8, 12, 24, 40]), "dim": 128,
            "dtype": "bf16", "sparsity": round(rng.uniform(0.15, 0.5), 3)}


# --------------------------------------------------------------------------
# sizes
# --------------------------------------------------------------------------

def _video(case):
    return case["f"] * case["h"] * case["w"]


def _policy(case):
    text = case.get("text", 0)
    layout = ScoringLayout(_video(case) + text, _video(case), case.get("tile", 16))
    return (hunyuan_policy if text else wan_policy)(layout, case["sparsity"])


def _attention_flops(case):
    """Products of the kept block pairs, valid tokens only."""
    pol = _policy(case)
    length = _video(case) + case.get("text", 0)
    counts = torch.as_tensor(pol.row_counts()).tolist()
    sizes = [min(BLOCK, length - BLOCK * i) for i in range(pol.q_blocks)]
    mean_keys = length / pol.k_blocks
    return 4.0 * case["dim"] * case["heads"] * sum(n * s * mean_keys for n, s in zip(counts, sizes))


def work(case):
    kind = case["kind"]
    if kind == "dfs":
        length = _video(case) + case["text"]
        flops = _attention_flops(case)
        if case["refresh"]:  # pooled products of the mask selection
            flops += 2.0 * (length / case["tile"]) ** 2 * case["dim"] * case["heads"]
        return {"bytes": 4 * 2 * case["heads"] * length * case["dim"], "flops": flops}
    if kind == "dense":
        n, d, h = case["length"], case["dim"], case["heads"]
        return {"bytes": 4 * 2 * h * n * d, "flops": 4.0 * h * n * n * d}
    if kind == "heads":
        length, c = _video(case) + case["text"], case["heads"] * case["dim"]
        table = _video(case) * (16 * case["dim"] // 2 if case["form"] == "wan" else 8 * case["dim"])
        return {"bytes": 3 * 2 * 2 * length * c + table, "flops": 20.0 * length * c}
    if kind == "glue":
        n = case["rows"] * case["channels"]
        return {"bytes": 2 * 5 * n, "flops": 12.0 * n}
    length, c = _video(case), case["heads"] * case["dim"]
    return {"bytes": 2 * (2 * length * c + 4 * c * c), "flops": 8.0 * length * c * c + _attention_flops(case)}


def tolerance(case):
    # Two roundings of the same fp32 value to the output type, plus the operands' roundings (f16 or
    # bf16 probabilities, keys and values): about four times the distance from 64-bit results.
    kind, out = case["kind"], case["dtype"]
    if kind == "layer":
        return {"rel": 1.3e-2}
    if kind in ("dfs", "dense"):
        if case.get("operand") == "bf16":
            return {"rel": 9e-3}
        return {"rel": 7e-3 if out == "bf16" else 1.2e-3}
    return {"rel": 7e-3 if out == "bf16" else 1e-3}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32).to(dtype)


def _dfs_inputs(case, seed):
    """(q, k, v) of this step and (q, k) of the step that selected the mask."""
    cfg = DfsConfig("case", (case["f"], case["h"], case["w"]), case["heads"], case["dim"], DTYPES[case["dtype"]],
                    text_len=case["text"], tile=case["tile"], sparsity=case["sparsity"])
    q, k, v = synth_qkv(cfg, device=DEVICE, seed=seed)
    if case["refresh"]:
        return q, k, v, q, k
    gen = _gen(seed + 1)
    return drift(q, 0.02, gen), drift(k, 0.02, gen), v, q, k


def _heads_inputs(case, seed):
    gen = _gen(seed)
    dtype, d = DTYPES[case["dtype"]], case["dim"]
    length, c = _video(case) + case["text"], case["heads"] * d
    x = [_randn(gen, 1, length, c, dtype=dtype) for _ in range(3)]
    width = c if case["form"] == "wan" else d
    norms = [torch.nn.RMSNorm(width, eps=1e-6, device=DEVICE, dtype=dtype).requires_grad_(False) for _ in range(2)]
    for n in norms:
        n.weight.copy_(1.0 + 0.1 * _randn(gen, width))
    grid = (case["f"], case["h"], case["w"])
    freqs = wan_rope_freqs(grid, d).to(DEVICE)
    if case["form"] == "wan":
        rope = freqs
    else:  # real tables, each frequency repeated for its channel pair
        rope = tuple(t.reshape(-1, d // 2).repeat_interleave(2, dim=1).float().contiguous()
                     for t in (freqs.real, freqs.imag))
    return x, norms, rope


def _glue_inputs(case, seed):
    gen = _gen(seed)
    dtype, n, c = DTYPES[case["dtype"]], case["rows"], case["channels"]
    x, y = _randn(gen, 1, n, c, dtype=dtype), _randn(gen, 1, n, c, dtype=dtype)
    scale, shift, gate = (0.3 * _randn(gen, 1, 1, c) for _ in range(3))
    return x, y, scale, shift, gate


def _layer_inputs(case, seed):
    """Hidden states with the locality of video features, and a layer whose query and key
    projections agree in part, as trained ones do."""
    gen = _gen(seed)
    grid, heads, d = (case["f"], case["h"], case["w"]), case["heads"], case["dim"]
    c, length = heads * d, _video(case)
    field = smoothed_field(grid, heads, d, 2.0, gen, DEVICE)
    x = field.transpose(0, 1).reshape(1, length, c)
    x = (x + 0.5 * _randn(gen, 1, length, c)).to(torch.bfloat16)
    attn = DiTAttention(c, heads, 1e-6, device=DEVICE, dtype=torch.bfloat16).requires_grad_(False)
    std = 1.0 / math.sqrt(c)
    shared = _randn(gen, c, c)
    attn.to_q.weight.copy_(std * shared)
    attn.to_k.weight.copy_(std * (0.8 * shared + 0.6 * _randn(gen, c, c)))
    attn.to_v.weight.copy_(std * _randn(gen, c, c))
    attn.to_out[0].weight.copy_(std * _randn(gen, c, c))
    for lin in (attn.to_q, attn.to_k, attn.to_v, attn.to_out[0]):
        lin.bias.copy_(0.02 * _randn(gen, c))
    for n in (attn.norm_q, attn.norm_k):
        n.weight.copy_(1.0 + 0.1 * _randn(gen, c))
    return x, attn.eval(), wan_rope_freqs(grid, d).to(DEVICE)


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "dfs":
        q, k, v, q0, k0 = _dfs_inputs(case, seed)
        variant = attention_hyvideo if case["text"] else attention_wan
        kw = dict(skip_steps=SKIP, cache_interval=INTERVAL, layer_idx=next(_layers), sparsity=case["sparsity"],
                  sparsity_dcrt=0.0, tile_size=case["tile"], block_size=BLOCK,
                  video_perm=hilbert3d_perm(case["f"], case["h"], case["w"]))
        if case["text"]:
            kw["video_len"] = _video(case)
            # what the processor passes: the valid text, then its padding
            length = _video(case) + case["text"]
            cu = torch.tensor([0, _video(case) + case["valid"], length], dtype=torch.int32, device=DEVICE)
            kw.update(cu_seqlens_q=cu, cu_seqlens_kv=cu.clone(), max_seqlen_q=length, max_seqlen_kv=length)
        step = SKIP if case["text"] else 2 * SKIP  # Wan's counter runs over both guidance passes
        state = {"kind": kind, "variant": variant, "q": q, "k": k, "v": v, "kw": kw,
                 "step": step if case["refresh"] else step + 1,
                 "operand": torch.bfloat16 if case["operand"] == "bf16" else None}
        if not case["refresh"]:  # the mask of the last refresh
            variant.DFS_Attention.operand_dtype = state["operand"]
            variant.dfs_attention(q0, k0, v, step_idx=step, **kw)
        return state
    if kind == "dense":
        gen = _gen(seed)
        shape = (1, case["heads"], case["length"], case["dim"])
        q, k, v = (_randn(gen, *shape, dtype=DTYPES[case["dtype"]]) for _ in range(3))
        return {"kind": kind, "q": q, "k": k, "v": v}
    if kind == "heads":
        x, norms, rope = _heads_inputs(case, seed)
        return {"kind": kind, "form": case["form"], "x": x, "rope": rope, "rope_rows": _video(case),
                "attn": SimpleNamespace(heads=case["heads"], norm_q=norms[0], norm_k=norms[1])}
    if kind == "glue":
        x, y, scale, shift, gate = _glue_inputs(case, seed)
        return {"kind": kind, "x": x, "y": y, "scale": scale, "shift": shift, "gate": gate}
    x, attn, rope = _layer_inputs(case, seed)
    attn.set_processor(Wan_DFSAttn_Processor2_0(
        "dfs", case["sparsity"], 16, BLOCK, hilbert3d_perm(case["f"], case["h"], case["w"]), next(_layers), [],
        SKIP, INTERVAL, 0.0, True, False))
    return {"kind": kind, "x": x, "attn": attn, "rope": rope}


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "dfs":
        variant = state["variant"]
        variant.DFS_Attention.operand_dtype = state["operand"]
        return variant.dfs_attention(state["q"], state["k"], state["v"], step_idx=state["step"], **state["kw"])
    if kind == "dense":
        return full_attention(state["q"], state["k"], state["v"], mode="flash")
    if kind == "heads":
        if state["form"] == "wan":
            return fused_qkv_heads(state["attn"], *state["x"], state["rope"])
        return fused_qkv_heads_per_head(state["attn"], *state["x"], state["rope"], state["rope_rows"])
    if kind == "glue":
        return (ops.adaln_modulate(state["x"], 1e-6, scale=state["scale"], shift=state["shift"]),
                ops.gated_residual(state["x"], state["y"], state["gate"]))
    state["attn"].get_processor().step_idx = 2 * SKIP  # a step that selects its mask
    attention_wan.DFS_Attention.operand_dtype = None
    return state["attn"](state["x"], None, None, state["rope"])


# --------------------------------------------------------------------------
# 64-bit results
# --------------------------------------------------------------------------

def _block_mask(q, k, case):
    """Kept blocks [Qb, Kb] of one head from fp64 q, k in execution order: tile means of the
    padded layout [video | 0 | text | 0], softmax over all key tiles, block sums, top-k."""
    tile, video = case.get("tile", 16), _video(case)
    text, length = case.get("text", 0), q.shape[0]
    d = q.shape[1]
    vblocks, blocks = -(-video // BLOCK), -(-length // BLOCK)

    def padded(x, rows):
        out = x.new_zeros(rows, d)
        out[:video] = x[:video]
        if rows > vblocks * BLOCK and text:
            out[vblocks * BLOCK:vblocks * BLOCK + text] = x[video:]
        return out.reshape(-1, tile, d).mean(1)

    qt, kt = padded(q, vblocks * BLOCK), padded(k, blocks * BLOCK)
    p = torch.softmax(qt @ kt.t().contiguous() / math.sqrt(d), dim=-1)
    per = BLOCK // tile
    score = p.reshape(vblocks, per, blocks, per).sum((1, 3))
    keep = max(1, int(case["sparsity"] * blocks))
    mask = torch.zeros(blocks, blocks, dtype=torch.bool, device=q.device)
    if text:
        cols = video // BLOCK  # video columns; text columns are always kept, text rows are dense
        idx = score[:, :cols].topk(keep - (blocks - cols), dim=-1).indices
        mask[:vblocks].scatter_(1, idx, True)
        mask[:, cols:] = True
        mask[cols:] = True
    else:
        mask.scatter_(1, score.topk(keep, dim=-1).indices, True)
    return mask


def _masked_attention(q, k, v, mask=None, rows=2048):
    """softmax(q k^T / sqrt(d)) v of one head under a block mask counted from the first row and key."""
    out = torch.empty_like(q)
    kt = k.t().contiguous()
    for r in range(0, q.shape[0], rows):
        s = q[r:r + rows] @ kt / math.sqrt(q.shape[1])
        if mask is not None:
            m = mask[r // BLOCK:-(-min(r + rows, q.shape[0]) // BLOCK)]
            m = m.repeat_interleave(BLOCK, 1)[:, :k.shape[0]].repeat_interleave(BLOCK, 0)[:s.shape[0]]
            s.masked_fill_(~m, -math.inf)
        out[r:r + rows] = torch.softmax(s, dim=-1).nan_to_num_(0.0) @ v  # a row without keys is zero
    return out


def _exact_dfs(q, k, v, q0, k0, case, perm):
    """One head, token order in and out."""
    order = torch.cat([perm, torch.arange(_video(case), q.shape[0], device=q.device)])
    mask = _block_mask(q0[order], k0[order], case)
    qe, ke, ve = q[order], k[order], v[order]
    cut = _video(case) + case["valid"] if case.get("text") else q.shape[0]
    o = torch.empty_like(qe)
    o[:cut] = _masked_attention(qe[:cut], ke[:cut], ve[:cut], mask)
    if cut < q.shape[0]:  # the padding attends itself under the mask counted from its own start
        o[cut:] = _masked_attention(qe[cut:], ke[cut:], ve[cut:], mask)
    out = torch.empty_like(o)
    out[order] = o
    return out


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w


def _rotate(x, cos, sin):
    """Pairs (2i, 2i + 1) of the last axis turned by (cos, sin) [.., D/2]."""
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], dim=-1).flatten(-2)


def _wan_heads(x, weight, heads, freqs):
    """[1, L, C] fp64 -> [1, H, L, D]: norm over all channels, then RoPE per head."""
    y = x if weight is None else _rms(x, weight.double())
    y = y.unflatten(2, (heads, -1)).transpose(1, 2)
    if freqs is None:
        return y.contiguous()
    return _rotate(y, freqs.real.reshape(-1, y.shape[-1] // 2), freqs.imag.reshape(-1, y.shape[-1] // 2))


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "dfs":
        q, k, v, q0, k0 = _dfs_inputs(case, seed)
        perm = hilbert3d_perm(case["f"], case["h"], case["w"]).to(DEVICE)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
        for h in range(case["heads"]):
            out[0, h] = _exact_dfs(*(t[0, h].double() for t in (q, k, v, q0, k0)), case, perm)
        return out
    if kind == "dense":
        s = prepare(case, seed)
        return torch.stack([_masked_attention(*(s[n][0, h].double() for n in "qkv"))
                            for h in range(case["heads"])])[None]
    if kind == "heads":
        x, norms, rope = _heads_inputs(case, seed)
        if case["form"] == "wan":
            return tuple(_wan_heads(t.double(), w, case["heads"], f) for t, w, f in
                         zip(x, (norms[0].weight, norms[1].weight, None), (rope, rope, None)))
        out, n = [], _video(case)
        cos, sin = (t.double()[:, 0::2] for t in rope)
        for t, norm in zip(x, (norms[0], norms[1], None)):
            y = t.double().unflatten(2, (case["heads"], -1)).transpose(1, 2)
            if norm is not None:
                y = _rms(y, norm.weight.double())
                y = torch.cat([_rotate(y[:, :, :n], cos, sin), y[:, :, n:]], dim=2)
            out.append(y.contiguous())
        return tuple(out)
    if kind == "glue":
        x, y, scale, shift, gate = (t.double() for t in _glue_inputs(case, seed))
        mean, var = x.mean(-1, keepdim=True), x.var(-1, unbiased=False, keepdim=True)
        return (x - mean) * torch.rsqrt(var + 1e-6) * (1 + scale) + shift, x + y * gate
    x, attn, freqs = _layer_inputs(case, seed)
    heads = case["heads"]

    def project(lin, t):
        return t @ lin.weight.double().t().contiguous() + lin.bias.double()

    q, k, v = (_wan_heads(project(lin, x.double()), w, heads, f) for lin, w, f in
               ((attn.to_q, attn.norm_q.weight, freqs), (attn.to_k, attn.norm_k.weight, freqs),
                (attn.to_v, None, None)))
    perm = hilbert3d_perm(case["f"], case["h"], case["w"]).to(DEVICE)
    o = torch.stack([_exact_dfs(q[0, h], k[0, h], v[0, h], q[0, h], k[0, h], case, perm) for h in range(heads)])
    return project(attn.to_out[0], o.transpose(0, 1).reshape(1, _video(case), -1))
