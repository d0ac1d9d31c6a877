"""Performance cases of the H3 block's hot path, through the calls of the Python binding.

The shapes are those of the two workloads that this repository measures: the 768p block (dim 5120, 40 heads, FFN
13,824, a 32 x 48 x 84 token grid, 512 text rows) and the H3 block at 960 x 544 (dim 5376, 56 heads, FFN 14,336, a
37 x 17 x 30 grid, 435 text rows), and the same blocks on a single image or a short clip, where few rows leave the chip
to launches and latency. Every case is one layer or block of that path; `draw` gives more of the same ranges.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "mako-video_amd"))

import mako_h3 as mh  # noqa: E402

DEV = "cuda"
MODELS = {  # dim, heads, ffn
    "768p": (5120, 40, 13824),
    "h3": (5376, 56, 14336),
}
BF16, F64 = torch.bfloat16, torch.float64


def listed():
    return [
        # The modulated norm of a single 480 x 272 image (1 x 9 x 15 tokens and 77 text rows) on the float residual
        # stream: the smallest call of a step, all latency.
        {"name": "norm_image", "op": "norm", "model": "h3", "rows": 212, "stream": "f32"},
        # The fused modulated norm and gated residual over the 768p batch: the largest streaming call.
        {"name": "norm_residual_768p", "op": "norm_residual", "model": "768p", "rows": 129536},
        # After the QKV projection at 960 x 544: head norms, rotary, gather into cubes and the cube means in one pass.
        {"name": "heads_960x544", "op": "heads", "model": "h3", "t": 37, "h": 17, "w": 30, "text": 435},
        # The sparse selection of a block at 960 x 544, ratio 0.1: pool, select, order.
        {"name": "select_960x544", "op": "select", "model": "h3", "t": 37, "h": 17, "w": 30, "text": 435,
         "ratio": 0.1, "local": 1},
        # Sparse attention at 960 x 544 over rows in the model's order, similar content in q and k.
        {"name": "attn_960x544", "op": "attn", "heads": 56, "t": 37, "h": 17, "w": 30, "text": 435, "ratio": 0.1,
         "layout": "rows", "shared": True},
        # Dense attention at 960 x 544: every cube selected.
        {"name": "attn_dense_960x544", "op": "attn", "heads": 56, "t": 37, "h": 17, "w": 30, "text": 435,
         "ratio": 1.0, "layout": "heads", "shared": True},
        # Sparse attention at 768p, the longest call of the 768p block.
        {"name": "attn_768p", "op": "attn", "heads": 40, "t": 32, "h": 48, "w": 84, "text": 512, "ratio": 0.1,
         "layout": "heads", "shared": False},
        # fc1 with SwiGLU under weight-only int8 over the 768p batch, the largest product.
        {"name": "fc1_w8a16_768p", "op": "fc1", "model": "768p", "rows": 129536, "form": "w8a16"},
        # fc1 with SwiGLU in bf16 at 960 x 544 (odd rows), the default of the 960 x 544 workload.
        {"name": "fc1_bf16_960x544", "op": "fc1", "model": "h3", "rows": 19305, "form": "bf16"},
        # The MLP half of a block on a single 960 x 544 image (1 x 17 x 30 tokens and 435 text rows), int8 weights.
        {"name": "mlp_image_w8a16", "op": "mlp", "model": "h3", "rows": 945, "form": "w8a16"},
        # The QKV projection of a short clip (5 x 17 x 30 tokens and 435 text rows) under int8 weights and activations.
        {"name": "qkv_clip_w8a8", "op": "qkv", "model": "h3", "rows": 2985, "form": "w8a8"},
        # A whole block of a short low-resolution clip (5 x 12 x 20 tokens and 77 text rows), bf16 weights: its
        # modulation vectors from the conditioning, and every layer in turn.
        {"name": "block_clip", "op": "block", "model": "768p", "t": 5, "h": 12, "w": 20, "text": 77, "ratio": 0.25,
         "form": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["norm", "norm_residual", "heads", "select", "attn", "attn", "fc1", "mlp", "qkv", "block"])
    model = rng.choice(list(MODELS))
    form = rng.choice(["w8a16", "bf16", "w8a8"])
    if op == "norm":
        return {"op": op, "model": model, "rows": _log(rng, 77, 40000), "stream": rng.choice(["f32", "bf16"])}
    if op == "norm_residual":
        return {"op": op, "model": model, "rows": _log(rng, 212, 120000)}
    if op in ("fc1", "mlp", "qkv"):
        return {"op": op, "model": model, "rows": _log(rng, 64, 24000), "form": form}
    t, h, w = rng.randint(1, 37), rng.randint(9, 48), rng.randint(15, 84)
    while t * h * w > (4000 if op == "block" else 32000):
        t, h, w = max(1, t * 3 // 4), max(9, h * 7 // 8), max(15, w * 7 // 8)
    c = {"op": op, "t": t, "h": h, "w": w, "text": rng.randint(16, 512)}
    if op != "attn":
        c["model"] = model
    if op == "select":
        c.update(ratio=round(rng.uniform(0.05, 0.5), 3), local=rng.choice([1, 3]))
    elif op == "attn":
        c.update(heads=rng.choice([5, 7, 40, 56]), ratio=rng.choice([0.1, 0.1, 0.2, 0.5, 1.0]),
                 layout=rng.choice(["heads", "rows", "gathered"]), shared=rng.random() < 0.5)
    elif op == "block":
        c.update(ratio=rng.choice([0.1, 0.25, 1.0]), form=form)
    return c


# ---- geometry --------------------------------------------------------------------------------------------------------

def _grid(case):
    return case["t"], case["h"], case["w"]


def _cubes(case):
    t, h, w = _grid(case)
    return -(-t // 4) * -(-h // 4) * -(-w // 4)


def _slots(grid):
    """int64 [cubes][64]: each 4 x 4 x 4 cube's tokens as rows of the frame-major grid, -1 past its edge."""
    t, h, w = grid
    ct, cy, cx = -(-t // 4), -(-h // 4), -(-w // 4)
    rows = torch.full((ct * 4, cy * 4, cx * 4), -1, dtype=torch.int64, device=DEV)
    rows[:t, :h, :w] = torch.arange(t * h * w, device=DEV).view(t, h, w)
    return rows.view(ct, 4, cy, 4, cx, 4).permute(0, 2, 4, 1, 3, 5).reshape(-1, 64).contiguous()


def _means(rows, slots):
    """Float64 means of the cubes' rows, [heads][cubes][128]."""
    have = (slots >= 0)
    picked = rows[:, slots.clamp(min=0)].double() * have[..., None]
    return picked.sum(2) / have.sum(1)[:, None].double()


def _lists(q, k, slots, count):
    """The pass lists of [heads][tokens][128] q and k as a selector gives them (the top `count` cubes of each query
    cube by the score of the cube means, and the cube itself), ascending, padded with -1; and the cubes of each head in
    the order of their lists' middle entries."""
    heads, cubes = q.shape[0], slots.shape[0]
    idx = torch.empty((heads, cubes, count + 1), dtype=torch.int32, device=DEV)
    cnt = torch.empty((heads, cubes), dtype=torch.int32, device=DEV)
    for h in range(heads):
        s = _means(q[h:h + 1], slots)[0] @ _means(k[h:h + 1], slots)[0].T.contiguous()
        sel = torch.zeros((cubes, cubes), dtype=torch.bool, device=DEV)
        sel.scatter_(1, s.topk(count, dim=1).indices, True)
        sel.fill_diagonal_(True)
        js = torch.where(sel, torch.arange(cubes, device=DEV), cubes).sort(dim=1).values
        js = torch.nn.functional.pad(js, (0, 1), value=cubes)[:, :count + 1]
        idx[h] = torch.where(js < cubes, js, -1).int()
        cnt[h] = sel.sum(1).int()
    middle = idx.gather(2, (cnt // 2).long()[..., None])[..., 0]
    return idx, cnt, middle.sort(dim=1, stable=True).indices.int().contiguous()


def _count(case):
    return max(1, math.ceil(case["ratio"] * _cubes(case)))


# ---- inputs ----------------------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, scale=1.0, dtype=BF16):
    """Seeded normals, a slab of rows at a time (the large cases' float rows need not all exist at once)."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 26):
        part = flat[i:i + (1 << 26)]
        part.copy_(torch.randn(part.numel(), generator=g, device=DEV) * scale)
    return out


def _qk(g, heads, grid, text, shared):
    """q and k [heads][tokens + text][128]: normals plus, on the video tokens, four smooth waves over the grid along
    random directions; `shared`: the same waves in q and k, as similar content gives."""
    t, h, w = grid
    video = t * h * w
    pos = torch.stack(torch.meshgrid(torch.arange(t, device=DEV) / t, torch.arange(h, device=DEV) / h,
                                     torch.arange(w, device=DEV) / w, indexing="ij"), -1).view(-1, 3)
    out, waves = [], None
    for _ in range(2):
        x = _randn(g, heads, video + text, 128)
        if waves is None or not shared:
            waves = (torch.randint(0, 3, (heads, 3, 4), generator=g, device=DEV).float(),
                     torch.nn.functional.normalize(torch.randn((heads, 4, 128), generator=g, device=DEV), dim=-1),
                     torch.rand((heads, 1, 4), generator=g, device=DEV) * 2 * math.pi)
        f, u, phase = waves
        for i in range(heads):
            x[i, :video] += (0.5 * torch.cos(2 * math.pi * (pos @ f[i]) + phase[i]) @ u[i]).to(BF16)
        out.append(x)
    return out


def _quant(w):
    """Rows to int8 with a float scale each, the row's largest value at 127."""
    s = w.float().abs().amax(1) / 127.0
    return torch.round(w.float() / s[:, None]).clamp(-127, 127).to(torch.int8), s


def _weight(g, n, k, form):
    w = _randn(g, n, k, scale=0.02)
    return (w, None) if form == "bf16" else _quant(w)


def _vectors(g, dim):
    w = 1 + 0.02 * torch.randn(dim, generator=g, device=DEV)
    return [w] + [0.1 * torch.randn(dim, generator=g, device=DEV) for _ in range(3)]


def _rotary(g, rows):
    a = (torch.rand((rows, 48), generator=g, device=DEV) * 2 - 1) * math.pi
    return torch.cos(a), torch.sin(a)


def _place(x, layout, slots, text):
    """[heads][rows][128] rows as a layout holds them: per head, per row, or gathered cube by cube (zero padding)."""
    if layout == "heads":
        return x
    if layout == "rows":
        return x.permute(1, 0, 2).contiguous().view(x.shape[1], -1)
    pad = torch.zeros((x.shape[0], 1, 128), dtype=x.dtype, device=x.device)
    video = x.shape[1] - text
    dense = torch.arange(video, video + text, device=x.device)
    order = torch.cat([torch.where(slots < 0, x.shape[1], slots).view(-1), dense])
    return torch.cat([x, pad], 1)[:, order].contiguous()


def prepare(case, seed):
    g, op, s = _gen(seed), case["op"], {"case": case}
    if "model" in case:
        dim, heads, ffn = MODELS[case["model"]]
    if op == "norm":
        s["x"] = _randn(g, case["rows"], dim, dtype=torch.float32 if case["stream"] == "f32" else BF16)
        s["vec"] = _vectors(g, dim)
    elif op == "norm_residual":
        s["x"], s["r"] = _randn(g, case["rows"], dim), _randn(g, case["rows"], dim)
        s["vec"] = _vectors(g, dim)
    elif op == "heads":
        grid, text = _grid(case), case["text"]
        rows = grid[0] * grid[1] * grid[2] + text
        s["qkv"] = _randn(g, rows, 3 * heads * 128)
        s["qw"], s["kw"] = (1 + 0.05 * torch.randn(128, generator=g, device=DEV) for _ in range(2))
        s["cos"], s["sin"] = _rotary(g, rows)
        s["map"], _ = mh.cube_map(grid, n_dense=text, video_row0=0, dense_row0=rows - text)
    elif op == "select":
        s["q"], s["k"] = _qk(g, heads, _grid(case), case["text"], True)
        s["args"] = mh.cube_args(heads, _grid(case), head_stride=s["q"].shape[1] * 128, k=_count(case),
                                 local=case["local"])
        s["ws"] = torch.empty(mh.cube_select_workspace_bytes(s["args"]), dtype=torch.uint8, device=DEV)
    elif op == "attn":
        grid, text, n, layout = _grid(case), case["text"], case["heads"], case["layout"]
        q, k = _qk(g, n, grid, text, case["shared"])
        v = _randn(g, n, q.shape[1], 128)
        slots, rows = _slots(grid), q.shape[1]
        count = _count(case)
        s["idx"], s["cnt"], s["order"] = _lists(q, k, slots, count)
        s["q"], s["k"], s["v"] = (_place(x, layout, slots, text) for x in (q, k, v))
        s["out"] = torch.zeros_like(s["q"])
        if layout == "gathered":
            where = {"layout": mh.CUBES_GATHERED, "head_stride": (slots.numel() + text) * 128}
        elif layout == "rows":
            where = {"head_stride": 128, "row_stride": n * 128}
        else:
            where = {"head_stride": rows * 128}
        s["args"] = mh.cube_args(n, grid, k=count, local=1, **where)
        s["dense0"] = slots.numel() if layout == "gathered" else rows - text
    elif op == "fc1":
        s["x"] = _randn(g, case["rows"], dim)
        s["w"], s["ws"] = _weight(g, 2 * ffn, dim, case["form"])
    elif op == "mlp":
        s["h"], s["x"] = _randn(g, case["rows"], dim), _randn(g, case["rows"], dim)
        s["w1"], s["s1"] = _weight(g, 2 * ffn, dim, case["form"])
        s["w2"], s["s2"] = _weight(g, dim, ffn, case["form"])
        s["gate"] = 0.1 * torch.randn(dim, generator=g, device=DEV)
    elif op == "qkv":
        s["x"] = _randn(g, case["rows"], dim)
        s["w"], s["ws"] = _weight(g, 3 * heads * 128, dim, case["form"])
    else:
        grid, text, form = _grid(case), case["text"], case["form"]
        rows = grid[0] * grid[1] * grid[2] + text
        s["x"] = _randn(g, rows, dim)
        s["cond"] = torch.nn.functional.silu(_randn(g, 1, dim // 2))
        s["wada"] = _randn(g, 18 * dim, dim // 2, scale=0.1 / math.sqrt(dim // 2))
        s["n1"], s["n2"] = (1 + 0.02 * torch.randn(dim, generator=g, device=DEV) for _ in range(2))
        s["wqkv"], s["sqkv"] = _weight(g, 3 * heads * 128, dim, form)
        s["wo"], s["so"] = _weight(g, dim, heads * 128, form)
        s["w1"], s["s1"] = _weight(g, 2 * ffn, dim, form)
        s["w2"], s["s2"] = _weight(g, dim, ffn, form)
        s["cos"], s["sin"] = _rotary(g, rows)
        s["args"] = mh.cube_args(heads, grid, head_stride=128, row_stride=heads * 128, k=_count(case), local=1)
        s["ws"] = torch.empty(mh.cube_select_workspace_bytes(s["args"]), dtype=torch.uint8, device=DEV)
        s["att"] = torch.zeros((rows, heads * 128), dtype=BF16, device=DEV)
        # The video's rows take set 0 of the table, the text's set 1.
        s["set"] = torch.zeros(rows, dtype=torch.uint8, device=DEV)
        s["set"][rows - text:] = 1
    return s


# ---- the calls -------------------------------------------------------------------------------------------------------

def _fc1(x, w, ws, form):
    if form == "bf16":
        return mh.gemm_bf16_swiglu(x, w)
    if form == "w8a16":
        return mh.gemm_w8a16_swiglu(x, w, ws)
    return mh.gemm_i8_swiglu(*mh.quant_rows_i8(x), w, ws)


def _operand(x, form):
    return mh.quant_rows_i8(x) if form == "w8a8" else (x, None)


def _residual(x, w, ws, residual, gate, form, **sets):
    a, xs = _operand(x, form)
    return mh.gemm_gate_add(a, w, residual, gate, x_scale=xs, w_scale=ws, **sets)


def run(s):
    case, op = s["case"], s["case"]["op"]
    if op == "norm":
        w, shift, scale, _ = s["vec"]
        return mh.rms_mod_rows(s["x"], w, shift, scale, out_dtype=BF16)
    if op == "norm_residual":
        w, shift, scale, gate = s["vec"]
        return mh.rms_mod_gate_add_rows(s["x"], s["r"], w, shift, scale, gate)
    if op == "heads":
        return mh.heads_partial_pool(s["qkv"], MODELS[case["model"]][1], _grid(case), s["qw"], s["kw"], s["cos"],
                                     s["sin"], map=s["map"])
    if op == "select":
        qc, kc = mh.cube_pool(s["args"], s["q"], s["k"])
        idx, cnt = mh.cube_select(s["args"], qc, kc, workspace=s["ws"])
        return qc, kc, idx, cnt, mh.cube_order(s["args"], idx, cnt)
    if op == "attn":
        return mh.flash_attn_sparse_128(s["args"], s["q"], s["k"], s["v"], s["idx"], s["cnt"], dense_row0=s["dense0"],
                                        n_dense=case["text"], out=s["out"], order=s["order"])
    form = case["form"]
    if op == "fc1":
        return _fc1(s["x"], s["w"], s["ws"], form)
    if op == "mlp":
        # The residual's first value stays with the caller (a step that is cached or guided reads it again).
        return _residual(_fc1(s["h"], s["w1"], s["s1"], form), s["w2"], s["s2"], s["x"].clone(), s["gate"], form)
    if op == "qkv":
        a, xs = _operand(s["x"], form)
        return mh.gemm(a, s["w"], x_scale=xs, w_scale=s["ws"])
    _, heads, _ = MODELS[case["model"]]
    grid, text, x = _grid(case), case["text"], s["x"].clone()
    sets = {"set_of_row": s["set"], "n_sets": 3}
    mod = mh.adaln_mod(s["cond"], s["wada"]).view(3, 6, -1)
    a, xs = _operand(mh.rms_mod_rows(x, s["n1"], mod[:, 0], mod[:, 1], **sets), form)
    qkv = mh.gemm(a, s["wqkv"], x_scale=xs, w_scale=s["sqkv"])
    q, k, v, qc, kc = mh.heads_partial_pool(qkv, heads, grid, None, None, s["cos"], s["sin"], layout="rows",
                                            cube_layout=mh.CUBES_GRID)
    idx, cnt = mh.cube_select(s["args"], qc, kc, workspace=s["ws"])
    order = mh.cube_order(s["args"], idx, cnt)
    att = mh.flash_attn_sparse_128(s["args"], q, k, v, idx, cnt, dense_row0=x.shape[0] - text, n_dense=text,
                                   out=s["att"], order=order)
    _residual(att, s["wo"], s["so"], x, mod[:, 2], form, **sets)
    h = mh.rms_mod_rows(x, s["n2"], mod[:, 3], mod[:, 4], **sets)
    return _residual(_fc1(h, s["w1"], s["s1"], form), s["w2"], s["s2"], x, mod[:, 5], form, **sets)


# ---- what a pass needs -----------------------------------------------------------------------------------------------

def _gemm_work(m, n, k, form, out_bytes):
    a, b = {"bf16": (2, 2), "w8a16": (2, 1), "w8a8": (2, 1)}[form]
    return a * m * k + b * n * k + out_bytes, 2.0 * m * n * k


def _attn_work(heads, tokens, text, cubes, count):
    """q, k, v and the output once; 512 flops for each query and key that it attends, a selected cube at its mean of
    tokens."""
    pairs = tokens * (min(tokens, (count + 1) * tokens / cubes) + text) + text * (tokens + text)
    return 4.0 * heads * (tokens + text) * 256, 512.0 * heads * pairs


def work(case):
    op = case["op"]
    if "model" in case:
        dim, heads, ffn = MODELS[case["model"]]
    if op == "norm":
        n = case["rows"] * dim
        return {"bytes": n * (6 if case["stream"] == "f32" else 4), "flops": 6.0 * n}
    if op == "norm_residual":
        return {"bytes": 6 * case["rows"] * dim, "flops": 8.0 * case["rows"] * dim}
    if op in ("heads", "select", "attn", "block"):
        t, h, w = _grid(case)
        tokens, text, cubes = t * h * w, case["text"], _cubes(case)
    if op == "heads":
        rows = cubes * 64 + text
        return {"bytes": 2 * 3 * heads * 128 * (tokens + text + rows) + 2 * heads * cubes * 512 + (tokens + text) * 384,
                "flops": 10.0 * 3 * heads * 128 * (tokens + text)}
    if op == "select":
        return {"bytes": 2 * heads * tokens * 256 + 2 * heads * cubes * 512 + heads * cubes * (_count(case) + 3) * 4,
                "flops": 2.0 * heads * tokens * 128 + 256.0 * heads * cubes * cubes}
    if op == "attn":
        b, f = _attn_work(case["heads"], tokens, text, cubes, _count(case))
        return {"bytes": b, "flops": f}
    form = case["form"]
    if op == "block":
        m = tokens + text
        parts = [_gemm_work(m, 3 * heads * 128, dim, form, 0), _gemm_work(m, dim, heads * 128, form, 0),
                 _gemm_work(m, 2 * ffn, dim, form, 0), _gemm_work(m, dim, ffn, form, 0),
                 _attn_work(heads, tokens, text, cubes, _count(case)), (18 * dim * dim, 18.0 * dim * dim)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    m = case["rows"]
    if op == "fc1":
        parts = [_gemm_work(m, 2 * ffn, dim, form, 2 * m * ffn)]
    elif op == "mlp":
        parts = [_gemm_work(m, 2 * ffn, dim, form, 2 * m * ffn), _gemm_work(m, dim, ffn, form, 4 * m * dim)]
    else:
        parts = [_gemm_work(m, 3 * heads * 128, dim, form, 2 * m * 3 * heads * 128)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """About four times what the path was measured to differ from `exact` by (its roundings to bf16)."""
    op = case["op"]
    if op == "select":
        return {"rel": 1e-6, "differ": 5e-3}    # float means; cubes whose scores tie within their rounding
    if op == "attn":
        return {"rel": 9.5e-3, "max": 6e-2}     # probabilities and outputs each rounded to bf16
    if op == "block":
        return {"rel": 1e-2, "max": 0.1}        # ten layers that round to bf16, and cubes that tie in the selection
    return {"rel": 7e-3, "max": 3.5e-2}         # each result rounded to bf16 (the MLP's hidden rows before that)


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------

def _f64_norm(x, w, shift, scale):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w.double() * (1 + scale.double()) + shift.double()


def _f64_product(x, w, ws, form, fold=None, step=16384):
    """x w^T in 64 bits, rows in steps (through `fold` when given); under w8a8 of x as its rows quantize."""
    wd = w.double() if ws is None else w.double() * ws.double()[:, None]
    wt = wd.T.contiguous()
    del wd
    out = []
    for i in range(0, x.shape[0], step):
        r = x[i:i + step]
        if form == "w8a8":
            q, s = _quant(r.to(BF16))
            r = q.double() * s.double()[:, None]
        y = r.double() @ wt
        out.append(y if fold is None else fold(y))
    return torch.cat(out)


def _swiglu64(y):
    gate, up = y.chunk(2, dim=1)
    return torch.nn.functional.silu(gate) * up


def _f64_attention(q, k, v, idx, cnt, slots, text):
    """[heads][rows][128] in 64 bits: a cube's queries over its list's tokens and the text, a text row over all rows."""
    heads, rows, _ = q.shape
    video, cubes = rows - text, slots.shape[0]
    dense = torch.arange(video, rows, device=DEV)
    out = torch.zeros((heads, rows, 128), dtype=F64, device=DEV)
    for h in range(heads):
        kd, vd = (torch.cat([x[h].double(), torch.zeros((1, 128), dtype=F64, device=DEV)]) for x in (k, v))
        qd = q[h].double() / math.sqrt(128)
        out[h, video:] = torch.softmax(qd[video:] @ kd[:rows].T.contiguous(), -1) @ vd[:rows]
        step = max(1, (1 << 22) // (idx.shape[2] * 64 + text))
        for c in range(0, cubes, step):
            j = idx[h, c:c + step].long()
            keys = torch.where((j >= 0)[..., None], slots[j.clamp(min=0)], -1).flatten(1)
            keys = torch.cat([keys, dense.expand(keys.shape[0], -1)], 1)
            qs = slots[c:c + step]
            sc = torch.bmm(qd[qs.clamp(min=0)], kd[keys].transpose(1, 2).contiguous())
            sc.masked_fill_((keys < 0)[:, None], -math.inf)
            o = torch.bmm(torch.softmax(sc, -1), vd[keys])
            out[h, qs[qs >= 0]] = o[qs >= 0]
    return out


def _f64_heads(qkv, heads, qw, kw, cos, sin):
    """[3][heads][rows][128]: q and k with their head norms and rotary positions on the first 96 values, v as it is."""
    rows = qkv.shape[0]
    x = qkv.double().view(rows, 3, heads, 128).permute(1, 2, 0, 3).contiguous()
    for i, w in ((0, qw), (1, kw)):
        t = x[i]
        t = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6)
        if w is not None:
            t = t * w.double()
        a, b, c, s = t[..., :48].clone(), t[..., 48:96].clone(), cos.double(), sin.double()
        t[..., :48], t[..., 48:96] = a * c - b * s, b * c + a * s
        x[i] = t
    return x


def exact(case, seed):
    op = case["op"]
    if op in ("attn", "heads", "block"):
        slots = _slots(_grid(case))
    s = prepare(case, seed)
    if op == "norm":
        return _f64_norm(s["x"], *s["vec"][:3])
    if op == "norm_residual":
        w, shift, scale, gate = s["vec"]
        parts = [r.double() + gate.double() * _f64_norm(x, w, shift, scale)
                 for x, r in zip(s["x"].split(16384), s["r"].split(16384))]
        return torch.cat(parts)
    if op == "heads":
        x = _f64_heads(s["qkv"], MODELS[case["model"]][1], s["qw"], s["kw"], s["cos"], s["sin"])
        placed = [_place(t, "gathered", slots, case["text"]) for t in x]
        # The means are of the rows as they are stored, in bf16.
        return (*placed, *(_means(t.to(BF16), slots) for t in x[:2]))
    if op == "select":
        slots = _slots(_grid(case))
        return _means(s["q"], slots), _means(s["k"], slots), None, None, None
    if op == "attn":
        if work(case)["flops"] > 2e13:
            return None
        n, text, layout = case["heads"], case["text"], case["layout"]
        q, k = _qk(g := _gen(seed), n, _grid(case), text, case["shared"])
        v = _randn(g, n, q.shape[1], 128)
        return _place(_f64_attention(q, k, v, s["idx"], s["cnt"], slots, text), layout, slots, text)
    form = case["form"]
    if op == "fc1":
        if case["rows"] > 40000:
            return None
        return _f64_product(s["x"], s["w"], s["ws"], form, _swiglu64)
    if op == "mlp":
        f = _f64_product(s["h"], s["w1"], s["s1"], form, _swiglu64)
        return s["x"].double() + s["gate"].double() * _f64_product(f, s["w2"], s["s2"], form)
    if op == "qkv":
        return _f64_product(s["x"], s["w"], s["ws"], form)
    _, heads, _ = MODELS[case["model"]]
    text, x = case["text"], s["x"].double()
    mod = (s["cond"].double() @ s["wada"].double().T.contiguous()).view(3, 6, -1)
    vec = [mod[s["set"].long(), i] for i in range(6)]
    h = _f64_norm(x, s["n1"], vec[0], vec[1])
    q, k, v = _f64_heads(_f64_product(h, s["wqkv"], s["sqkv"], form), heads, None, None, s["cos"], s["sin"])
    idx, cnt, _ = _lists(q, k, slots, _count(case))
    att = _place(_f64_attention(q, k, v, idx, cnt, slots, text), "rows", slots, text)
    x = x + vec[2] * _f64_product(att, s["wo"], s["so"], form)
    f = _f64_product(_f64_norm(x, s["n2"], vec[3], vec[4]), s["w1"], s["s1"], form, _swiglu64)
    return x + vec[5] * _f64_product(f, s["w2"], s["s2"], form)
