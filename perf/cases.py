"""The work that a user of this framework has it do, as timed cases.

A case is one call, or one chain of calls, through the public entry points of
awa_hip: a single attention layer (plain, with the q/k RMSNorm fused, or as
the four layers of a block's .param graph), a DiT block, or the whole block
loop of a step. The sizes are those of the tests and of the benchmark: latent
grids t x h x w (4x temporal and 8x spatial compression, 2x2 patches), window
counts, 58 or 64 text tokens, 20 heads of 128 features, hidden width 2560 and
SwiGLU width 6912.
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("seedvr2-ncnn_amd"))

import awa_hip as A  # noqa: E402

HEAD_DIM = 128
EPS = 1e-5
DEVICE = "cuda"


def _layer(name, path, grid, windows, text, shifted, dtype, heads=20):
    return {"name": name, "kind": "layer", "path": path, "t": grid[0], "h": grid[1], "w": grid[2], "nt": windows[0],
            "nh": windows[1], "nw": windows[2], "text": text, "shifted": shifted, "dtype": dtype, "heads": heads}


def _block(name, grid, windows, text, shifted, dtype, heads=20, mlp=6912, last=False):
    return {"name": name, "kind": "block", "t": grid[0], "h": grid[1], "w": grid[2], "nt": windows[0],
            "nh": windows[1], "nw": windows[2], "text": text, "shifted": shifted, "dtype": dtype, "heads": heads,
            "mlp": mlp, "last": last}


def _step(name, grid, windows, text, blocks, prefix, heads=20, mlp=6912):
    return {"name": name, "kind": "step", "t": grid[0], "h": grid[1], "w": grid[2], "nt": windows[0],
            "nh": windows[1], "nw": windows[2], "text": text, "blocks": blocks, "prefix": prefix, "heads": heads,
            "mlp": mlp}


def listed():
    return [
        # One 256x256 image in fp32: the smallest layer of the benchmark, where
        # launches and latency count (4 windows of 128 rows).
        _layer("layer_image_f32", "fused", (1, 16, 16), (1, 8, 8), 64, False, "f32"),
        # A 5-frame clip, bf16, shifted windows with partial edges.
        _layer("layer_clip_bf16", "fused", (2, 16, 16), (1, 8, 8), 64, True, "bf16"),
        # The 33-frame 256x256 workload of the benchmark: an fp32 block's layer ...
        _layer("layer_33f_f32", "fused", (9, 16, 16), (3, 8, 8), 64, False, "f32"),
        # ... and a bf16 block's shifted layer.
        _layer("layer_33f_bf16", "fused", (9, 16, 16), (3, 8, 8), 64, True, "bf16"),
        # 49 frames at 720p with the production window counts: 1678-row windows, fp32.
        _layer("layer_720p_f32", "fused", (13, 45, 80), (4, 3, 3), 58, False, "f32"),
        # 121 frames at 720p, bf16, shifted: windows of up to 3298 rows, the largest layer.
        _layer("layer_720p_bf16", "fused", (31, 45, 80), (4, 3, 3), 58, True, "bf16"),
        # 121 frames at 256x256 straight from the QKV projection (q/k RMSNorm
        # in the gather), ragged in time, bf16.
        _layer("qknorm_121f_bf16", "qknorm", (31, 16, 16), (8, 8, 8), 64, True, "bf16"),
        # The four layers as a block's .param graph runs them, one call each, fp32.
        _layer("staged_33f_f32", "staged", (9, 16, 16), (3, 8, 8), 64, True, "f32"),
        # One DiT block of the fp32 prefix at the 33-frame workload.
        _block("block_33f_f32", (9, 16, 16), (3, 8, 8), 64, False, "f32"),
        # One bf16 DiT block at the 33-frame workload, shifted.
        _block("block_33f_bf16", (9, 16, 16), (3, 8, 8), 64, True, "bf16"),
        # One bf16 DiT block of a 256x256 image with the production window
        # counts: 256 tokens, bound by reading the weights.
        _block("block_image_bf16", (1, 16, 16), (4, 3, 3), 64, False, "bf16"),
        # A whole DiT step at the 33-frame workload: 9 fp32 and 23 bf16 blocks.
        _step("step_33f", (9, 16, 16), (3, 8, 8), 64, 32, 9),
    ]


def _intervals(size, window, shifted):
    shift = 0.5 if shifted and window < size else 0.0
    out = []
    for i in range(math.ceil((size - shift) / window) + (1 if shift else 0)):
        a, b = max(int((i - shift) * window), 0), min(int((i - shift + 1.0) * window), size)
        if b > a:
            out.append((a, b))
    return out


def _windows(case, shifted):
    """Window boxes of a layer: w outermost, then h, then t."""
    t, h, w = case["t"], case["h"], case["w"]
    scale = math.sqrt(3600.0 / (h * w))
    wt = -(-min(t, 30) // case["nt"])
    wh = -(-round(h * scale) // case["nh"])
    ww = -(-round(w * scale) // case["nw"])
    return [(a, b, c) for c in _intervals(w, ww, shifted) for b in _intervals(h, wh, shifted)
            for a in _intervals(t, wt, shifted)]


def _attention_flops(case, shifted):
    rows = [(a[1] - a[0]) * (b[1] - b[0]) * (c[1] - c[0]) + case["text"] for a, b, c in _windows(case, shifted)]
    return 4.0 * HEAD_DIM * case["heads"] * sum(n * n for n in rows)


def _gemm_flops(case, last):
    hidden, hd, mlp = _hidden(case), case["heads"] * HEAD_DIM, case["mlp"]
    attn = 2.0 * hidden * 4 * hd
    full = attn + 2.0 * hidden * 3 * mlp
    return _tokens(case) * full + case["text"] * (attn if last else full)


def _tokens(case):
    return case["t"] * case["h"] * case["w"]


def _hidden(case):
    return case["heads"] * HEAD_DIM


def _weights_count(case, last_text):
    hidden, hd = _hidden(case), case["heads"] * HEAD_DIM
    return hidden * 4 * hd + (0 if last_text else 3 * hidden * case["mlp"])


def draw(rng):
    """Another size of the same kinds of work: odd grids, few and many tokens,
    whole and partial windows, both data types."""
    counts = [(1, 8, 8), (3, 8, 8), (8, 8, 8), (4, 3, 3), (2, 4, 4), (3, 5, 6), (2, 3, 8)]
    while True:
        kind = rng.choice(["layer", "layer", "layer", "layer", "block", "block", "block", "step"])
        dtype = rng.choice(["f32", "bf16"])
        most = {"layer": 40000 if dtype == "bf16" else 15000, "block": 9300 if dtype == "bf16" else 4700,
                "step": 1500}[kind]
        grid = (round(math.exp(rng.uniform(0, math.log(31)))), rng.randint(9, 48), rng.randint(9, 48))
        n = grid[0] * grid[1] * grid[2]
        if n > most or n < rng.uniform(0, 1) * 2000:
            continue
        windows, text = rng.choice(counts), rng.choice([64, 58, 64, 77, rng.randint(16, 80)])
        heads = rng.choice([20, 20, 16, 12, 8])
        shifted = rng.random() < 0.5
        if kind == "layer":
            case = _layer("", rng.choice(["fused", "fused", "qknorm", "staged"]), grid, windows, text, shifted, dtype,
                          heads)
        elif kind == "block":
            case = _block("", grid, windows, text, shifted, dtype, heads, heads * 344 + 8 * rng.randint(0, 8),
                          rng.random() < 0.2)
        else:
            blocks = rng.randint(3, 8)
            case = _step("", grid, windows, text, blocks, rng.randint(1, blocks - 1), heads, heads * 344 + 32)
        del case["name"]
        if _attention_flops(case, False) > 4e11:
            continue
        return case


def _torch_type(dtype):
    return torch.float32 if dtype == "f32" else torch.bfloat16


def _normal(gen, shape, dtype, std=1.0):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32).mul_(std).to(_torch_type(dtype))


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _layer_inputs(case, seed):
    gen = _generator(seed)
    d, heads = HEAD_DIM, case["heads"]
    out = {"video": _normal(gen, (_tokens(case), 3, heads, d), case["dtype"]),
           "text": _normal(gen, (case["text"], 3, heads, d), case["dtype"])}
    if case["path"] == "qknorm":
        out["gammas"] = [torch.rand(d, generator=gen, device=DEVICE) + 0.5 for _ in range(4)]
    return out


def _branch(gen, case, dtype, last_text):
    """One branch's weights: GEMM weights N(0, 0.02), Ada vectors around their
    use (scale and gate of order one), as the benchmark's random init."""
    hidden, hd, mlp = _hidden(case), case["heads"] * HEAD_DIM, case["mlp"]
    w = {"qkv": _normal(gen, (3 * hd, hidden), dtype, 0.02), "proj_out": _normal(gen, (hidden, hd), dtype, 0.02),
         "bias": _normal(gen, (hidden,), "f32", 0.02),
         "norm_q": torch.rand(HEAD_DIM, generator=gen, device=DEVICE) + 0.5,
         "norm_k": torch.rand(HEAD_DIM, generator=gen, device=DEVICE) + 0.5}
    if not last_text:
        w["mlp_gate_in"] = _normal(gen, (2 * mlp, hidden), dtype, 0.02)
        w["mlp_out"] = _normal(gen, (hidden, mlp), dtype, 0.02)
        w["ada"] = _normal(gen, (6, hidden), "f32", 0.1)
    return w


def _branch_struct(w):
    has = "ada" in w
    gate = w["mlp_gate_in"] if has else None
    half = gate.numel() // 2 * gate.element_size() if has else 0
    return A.AwaDitBranchWeights(
        w["qkv"].data_ptr(), w["proj_out"].data_ptr(), w["bias"].data_ptr(), gate.data_ptr() if has else None,
        gate.data_ptr() + half if has else None, w["mlp_out"].data_ptr() if has else None, w["norm_q"].data_ptr(),
        w["norm_k"].data_ptr(), w["ada"].data_ptr() if has else None)


def _dit_inputs(case, seed):
    """Activations N(0, 1), the block embedding, and each block's weights."""
    gen = _generator(seed)
    hidden = _hidden(case)
    if case["kind"] == "block":
        dtypes, lasts = [case["dtype"]], [case["last"]]
    else:
        dtypes = ["f32" if b < case["prefix"] else "bf16" for b in range(case["blocks"])]
        lasts = [b == case["blocks"] - 1 for b in range(case["blocks"])]
    return {"video": _normal(gen, (_tokens(case), hidden), dtypes[0]),
            "text": _normal(gen, (case["text"], hidden), dtypes[0]), "emb": _normal(gen, (hidden * 6,), dtypes[0]),
            "dtypes": dtypes, "lasts": lasts,
            "weights": [(_branch(gen, case, dt, False), _branch(gen, case, dt, last))
                        for dt, last in zip(dtypes, lasts)]}


def prepare(case, seed):
    A.init(0)
    if case["kind"] != "layer":
        state = _dit_inputs(case, seed)
        state["case"] = case
        args = (case["t"], case["h"], case["w"], case["nt"], case["nh"], case["nw"], case["text"])
        out = _torch_type(state["dtypes"][-1])
        state["video_out"] = torch.empty(state["video"].shape, device=DEVICE, dtype=out)
        state["text_out"] = torch.empty(state["text"].shape, device=DEVICE, dtype=out)
        state["structs"] = ([_branch_struct(v) for v, _ in state["weights"]],
                            [_branch_struct(t) for _, t in state["weights"]])
        if case["kind"] == "block":
            state["object"] = A.DitBlock(*args, case["shifted"], case["heads"], HEAD_DIM, _hidden(case), case["mlp"],
                                         case["last"],
                                         A.COMPUTE_F32 if case["dtype"] == "f32" else A.COMPUTE_BF16, EPS)
        else:
            state["object"] = A.DitStack(*args, case["blocks"], case["prefix"], case["heads"], HEAD_DIM,
                                         _hidden(case), case["mlp"], EPS)
        return state

    d, heads, tokens, text = HEAD_DIM, case["heads"], _tokens(case), case["text"]
    state = _layer_inputs(case, seed)
    state["case"] = case
    plan = A.Plan(A.LayerParams(case["t"], case["h"], case["w"], case["nt"], case["nh"], case["nw"], text,
                                case["shifted"]), heads=heads)
    plan.upload()
    state["plan"] = plan
    dtype = _torch_type(case["dtype"])
    es = 4 if case["dtype"] == "f32" else 2

    def blob(name, shape, dt, size):
        if name not in state:
            state[name] = torch.empty(shape, device=DEVICE, dtype=dt)
        c, h, w = shape
        return A.mat(state[name].data_ptr(), w, h, c, size, dims=3)

    blobs = {"video": A.mat(state["video"].data_ptr(), d, 3 * heads, tokens, es, dims=3),
             "text": A.mat(state["text"].data_ptr(), d, 3 * heads, text, es, dims=3),
             "video_out": blob("video_out", (tokens, heads, d), dtype, es),
             "text_out": blob("text_out", (text, heads, d), dtype, es)}
    if case["path"] == "staged":
        rows = plan.info.sequence_tokens
        blobs["packed"] = blob("packed", (rows, 3 * heads, d), torch.float32, 4)
        blobs["roped"] = blob("roped", (rows, 3 * heads, d), torch.float32, 4)
        blobs["attended"] = blob("attended", (rows, heads, d), torch.float32, 4)
        n = plan.info.window_count + 1
        state["cu"] = torch.empty(n, device=DEVICE, dtype=torch.float32)
        blobs["cu"] = A.mat(state["cu"].data_ptr(), n, elemsize=4, dims=1)
    if case["path"] == "qknorm":
        state["norm"] = A.AwaQkNorm(*[g.data_ptr() for g in state["gammas"]], EPS)
    state["blobs"] = blobs
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "block":
        state["object"].forward(state["structs"][0][0], state["structs"][1][0], state["video"].data_ptr(),
                                state["text"].data_ptr(), state["emb"].data_ptr(), state["video_out"].data_ptr(),
                                state["text_out"].data_ptr())
        return {"video": state["video_out"], "text": state["text_out"]}
    if case["kind"] == "step":
        state["object"].run(state["structs"][0], state["structs"][1], state["video"].data_ptr(),
                            state["text"].data_ptr(), state["emb"].data_ptr(), state["video_out"].data_ptr(),
                            state["text_out"].data_ptr())
        return {"video": state["video_out"], "text": state["text_out"]}
    plan, b = state["plan"], state["blobs"]
    compute = A.COMPUTE_F32 if case["dtype"] == "f32" else A.COMPUTE_BF16
    out = {"video": state["video_out"], "text": state["text_out"]}
    if case["path"] == "fused":
        plan.forward(b["video"], b["text"], b["video_out"], b["text_out"], compute)
    elif case["path"] == "qknorm":
        plan.forward_qknorm(b["video"], b["text"], state["norm"], b["video_out"], b["text_out"], compute)
    else:
        plan.pack(b["video"], b["text"], b["packed"], b["cu"])
        plan.mmrope(b["packed"], b["roped"])
        plan.window_attention(b["roped"], b["attended"], compute)
        plan.unpack(b["attended"], b["video_out"], b["text_out"])
        out.update(packed=state["packed"], cu=state["cu"], roped=state["roped"], attended=state["attended"])
    return out


def work(case):
    tokens, text = _tokens(case), case["text"]
    if case["kind"] == "layer":
        es = 4 if case["dtype"] == "f32" else 2
        row = case["heads"] * HEAD_DIM
        io = (tokens + text) * 4 * row * es
        if case["path"] == "staged":
            # Each of the four calls reads its input and writes its own output
            # blob: packed and rotated QKV and the attended rows, all fp32.
            rows = tokens + text * len(_windows(case, case["shifted"]))
            io += rows * row * 4 * (2 * 3 + 2 * 3 + 2)
        return {"bytes": io, "flops": _attention_flops(case, case["shifted"])}
    hidden = _hidden(case)
    if case["kind"] == "block":
        es = 4 if case["dtype"] == "f32" else 2
        return {"bytes": es * (_weights_count(case, False) + _weights_count(case, case["last"]) +
                               2 * (tokens + text) * hidden + 6 * hidden),
                "flops": _gemm_flops(case, case["last"]) + _attention_flops(case, case["shifted"])}
    blocks, prefix = case["blocks"], case["prefix"]
    moved = flops = 0.0
    for b in range(blocks):
        last = b == blocks - 1
        moved += (4 if b < prefix else 2) * (_weights_count(case, False) + _weights_count(case, last))
        flops += _gemm_flops(case, last) + _attention_flops(case, b % 2 == 1)
    return {"bytes": moved + (tokens + text) * hidden * (4 + 2) + 24 * hidden, "flops": flops}


def tolerance(case):
    """fp32 paths: sums in another order (layers are 3e-7 to 7e-7 off their
    64-bit results, blocks 2e-6). bf16 paths: roundings of bf16 stores that
    fall the other way (layers are 3e-3 off, blocks 5e-3), and for a step their
    way through every block (1.2e-2 off)."""
    if case["kind"] == "step":
        return {"rel": 3e-2}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2 if case["kind"] == "layer" else 1.5e-2}
    return {"rel": 1e-5}


# ---- the same in 64 bits, from the definitions ----

def _rotate(x, coords):
    """3-D RoPE of features 0..125: 21 interleaved pairs per axis; angles are
    the layer's fp32 products of coordinate and frequency."""
    out = x.clone()
    freq = torch.tensor([10000.0 ** (-2.0 * p / 42) for p in range(21)], device=x.device, dtype=torch.float32)
    for axis in range(3):
        angle = (coords[:, axis].float()[:, None] * freq[None, :]).double()
        cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
        a, b = x[..., 42 * axis:42 * axis + 42:2], x[..., 42 * axis + 1:42 * axis + 42:2]
        out[..., 42 * axis:42 * axis + 42:2] = a * cos - b * sin
        out[..., 42 * axis + 1:42 * axis + 42:2] = b * cos + a * sin
    return out


def _exact_layer(case, shifted, video, text, gammas=None, parts=None):
    """video [N][3][H][d] and text [T][3][H][d] in float64 -> their outputs."""
    dev, n_text = video.device, text.shape[0]
    if gammas is not None:
        def norm(x, gq, gk):
            x = x.clone()
            for i, g in enumerate((gq, gk)):
                x[:, i] *= torch.rsqrt((x[:, i] ** 2).mean(-1, keepdim=True) + EPS) * g.double()
            return x
        video, text = norm(video, gammas[0], gammas[1]), norm(text, gammas[2], gammas[3])
    out_video = torch.zeros(video.shape[0], video.shape[2], video.shape[3], device=dev, dtype=torch.float64)
    out_text = torch.zeros(n_text, video.shape[2], video.shape[3], device=dev, dtype=torch.float64)
    k = torch.arange(n_text, device=dev)
    boxes = _windows(case, shifted)
    for a, b, c in boxes:
        tt, hh, ww = torch.meshgrid(*[torch.arange(*i, device=dev) for i in (a, b, c)], indexing="ij")
        idx = ((tt * case["h"] + hh) * case["w"] + ww).reshape(-1)
        coords = torch.cat([torch.stack([(tt - a[0]).reshape(-1) + n_text, (hh - b[0]).reshape(-1),
                                         (ww - c[0]).reshape(-1)], 1), k[:, None].expand(n_text, 3)])
        x = torch.cat([video[idx], text])
        q, key, v = _rotate(x[:, 0], coords), _rotate(x[:, 1], coords), x[:, 2]
        s = torch.matmul(q.permute(1, 0, 2).contiguous(), key.permute(1, 2, 0).contiguous())
        o = torch.matmul(torch.softmax(s * HEAD_DIM ** -0.5, -1), v.permute(1, 0, 2).contiguous()).permute(1, 0, 2)
        out_video[idx] = o[:len(idx)]
        out_text += o[len(idx):]
        if parts is not None:
            parts["packed"].append(x)
            parts["roped"].append(torch.stack([q, key, v], 1))
            parts["attended"].append(o)
    return out_video, out_text / len(boxes)


def _exact_block(case, shifted, last, wv, wt, xs, emb):
    d, heads = HEAD_DIM, case["heads"]
    e = emb.reshape(-1, 2, 3)
    ws = (wv, wt)

    def rms(x):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)

    def lin(x, w):
        return x @ w.double().t()

    def ada(w, layer):
        return [e[:, layer, i] + w["ada"][3 * layer + i].double() for i in range(3)]

    qkv = []
    for br in range(2):
        x = rms(xs[br])
        if br == 0 or not last:
            shift, scale, _ = ada(ws[br], 0)
            x = x * scale + shift
        qkv.append(lin(x, ws[br]["qkv"]).reshape(-1, 3, heads, d))
    att = _exact_layer(case, shifted, qkv[0], qkv[1], [wv["norm_q"], wv["norm_k"], wt["norm_q"], wt["norm_k"]])
    out = []
    for br in range(2):
        w = ws[br]
        y = lin(att[br].reshape(-1, heads * d), w["proj_out"]) + w["bias"].double()
        if br == 1 and last:
            out.append(2 * (y + xs[br]))
            continue
        y = y * ada(w, 0)[2] + xs[br]
        shift, scale, gate = ada(w, 1)
        a, b = lin(rms(y) * scale + shift, w["mlp_gate_in"]).chunk(2, -1)
        out.append(lin(torch.nn.functional.silu(a) * b, w["mlp_out"]) * gate + y)
    return out


def exact(case, seed):
    if case["kind"] != "layer":
        s = _dit_inputs(case, seed)
        xs = [s["video"].double(), s["text"].double()]
        emb = s["emb"].double()
        for b, (wv, wt) in enumerate(s["weights"]):
            shifted = case["shifted"] if case["kind"] == "block" else b % 2 == 1
            xs = _exact_block(case, shifted, s["lasts"][b], wv, wt, xs, emb)
        return {"video": xs[0], "text": xs[1]}
    s = _layer_inputs(case, seed)
    parts = {"packed": [], "roped": [], "attended": []} if case["path"] == "staged" else None
    video, text = _exact_layer(case, case["shifted"], s["video"].double(), s["text"].double(), s.get("gammas"), parts)
    out = {"video": video, "text": text}
    if parts is not None:
        out.update({name: torch.cat(p) for name, p in parts.items()})
        lengths = torch.tensor([0] + [len(p) for p in parts["packed"]], device=video.device)
        out["cu"] = lengths.cumsum(0).double()
        out["packed"] = out["packed"].reshape(len(out["packed"]), -1, HEAD_DIM)
        out["roped"] = out["roped"].reshape(len(out["roped"]), -1, HEAD_DIM)
    return out
