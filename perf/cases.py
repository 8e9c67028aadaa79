"""Timed cases of the sparse global-attention framework on one MI355X.

``listed()`` holds the fixed cases, ``draw`` more of the same ranges,
``prepare`` builds what a program has in hand before the call, ``run`` is one
pass through the public entry points, ``work`` the bytes and operations the
pass cannot do without, ``tolerance`` what two correct implementations may
differ by, ``exact`` the float64 value of the outputs that have one.

The kinds of case:

* ``layer``: two consecutive global layers of a VGGT- or Pi3-shaped model
  (qkv, fused layout, pooling, selection with the cross-layer ledger, sparse
  attention, projection), as the installed model runs them;
* ``model``: a whole VGGT-shaped aggregator forward, every second layer sparse;
* ``dense``: the dense attention layer (the frame layers of every model, and
  the global layers of the dense mode);
* ``op``: the drop-in operator pair ``predict_attention`` and
  ``block_sparse_attn_cuda`` on given q, k, v;
* ``attend``: V packing and block-sparse attention over given block lists;
* ``predict``: the pooled predictor alone;
* ``mask``: the block map of a cdf threshold;
* ``select``: two layers of the block selection with the ledger.
"""
import math
import os

import torch

from vasc_amd import ops, pipeline
from vasc_amd.aggregator import Aggregator, Attention, RotaryPositionEmbedding2D, grid_positions
from vasc_amd.attention import adaptive_sparse_attention_forward, frame_grid, predict_attention
from vasc_amd.install import sparse_aggregator_from_vggt_layerwise
from vasc_amd.launcher import layer_sparsity, method_environment
from vasc_amd.sparse_wrapper import STATE_KEY, block_sparse_attn_cuda, get_block_mask

HEAD_DIM = 64
SPECIAL = 5  # camera + registers (VGGT), registers (Pi3): both models hold five
GRID = (28, 37)  # patches of a 392x518 frame


def listed():
    h, w = GRID
    return [
        # an image pair, the smallest thing a multi-view model is called with
        dict(name="layer_vasc_2f", kind="layer", backbone="vggt", mode="vasc", frames=2, gh=h, gw=w, sparsity=0.75),
        # a short clip: the layer is a few hundred microseconds, launches and small grids count
        dict(name="layer_vasc_8f", kind="layer", backbone="vggt", mode="vasc", frames=8, gh=h, gw=w, sparsity=0.75),
        # the benchmark's configuration
        dict(name="layer_vasc_32f", kind="layer", backbone="vggt", mode="vasc", frames=32, gh=h, gw=w, sparsity=0.75),
        # a Pi3 sequence whose patch count is no multiple of the key block: protected mixed tail
        dict(name="layer_vasc_pi3_50f", kind="layer", backbone="pi3", mode="vasc", frames=50, gh=h, gw=w,
             sparsity=0.75),
        # a long sequence, the sparsest setting in use
        dict(name="layer_vasc_128f", kind="layer", backbone="vggt", mode="vasc", frames=128, gh=h, gw=w,
             sparsity=0.875),
        # whole aggregator over a short clip
        dict(name="model_8f", kind="model", frames=8, gh=h, gw=w, depth=24, sparsity=0.75),
        # the frame layers of the benchmark's forward: 32 sequences of one frame each
        dict(name="dense_frames_32f", kind="dense", batch=32, tokens=1041, gw=w),
        # the operator called on float16 tensors, as the reference's evaluators hand them over (Top-K mode)
        dict(name="op_topk_fp16_12f", kind="op", mode="topk", dtype="float16", heads=16, frames=12, per_frame=1041,
             sparsity=0.75),
        # the operator on block lists of uneven length at 64k tokens
        dict(name="attend_64k", kind="attend", heads=16, tokens=65536, density=0.25),
        # the predictor at the longest sequence in use
        dict(name="predict_256k", kind="predict", heads=16, tokens=262144),
        # cumulative-probability selection at 64 frames
        dict(name="mask_cdf_64f", kind="mask", heads=16, qblocks=518, kblocks=1036, threshold=0.9, sink=5),
        # selection with the ledger at the longest sequence in use
        dict(name="select_vasc_256k", kind="select", mode="vasc", heads=16, qblocks=2048, kblocks=4096, keep=0.25,
             force_last=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _candidate(rng):
    kind = rng.choice(["layer", "layer", "layer", "dense", "op", "attend", "predict", "mask", "select", "model"])
    grid = GRID if rng.random() < 0.4 else (rng.randint(14, 37), rng.randint(14, 37))
    per = SPECIAL + grid[0] * grid[1]
    if kind == "layer":
        return dict(kind=kind, backbone=rng.choice(["vggt", "pi3"]), mode=rng.choice(["vasc", "vasc", "topk"]),
                    frames=_log_int(rng, 2, 120), gh=grid[0], gw=grid[1],
                    sparsity=rng.choice([0.55, 0.65, 0.75, 0.85, 0.875]))
    if kind == "model":
        return dict(kind=kind, frames=_log_int(rng, 2, 8), gh=grid[0], gw=grid[1], depth=rng.randint(4, 12),
                    sparsity=rng.choice([0.65, 0.75, 0.85]))
    if kind == "dense":
        if rng.random() < 0.6:  # frame layers
            return dict(kind=kind, batch=_log_int(rng, 2, 64), tokens=per, gw=grid[1])
        return dict(kind=kind, batch=1, tokens=per * _log_int(rng, 2, 24), gw=grid[1])
    if kind == "op":
        return dict(kind=kind, mode=rng.choice(["topk", "vasc"]), dtype=rng.choice(["float16", "bfloat16"]),
                    heads=rng.choice([2, 8, 12, 16]), frames=_log_int(rng, 1, 48), per_frame=per,
                    sparsity=rng.choice([0.55, 0.65, 0.75, 0.85]))
    if kind == "attend":
        return dict(kind=kind, heads=rng.choice([2, 8, 12, 16]), tokens=_log_int(rng, 1000, 70000),
                    density=rng.choice([0.1, 0.25, 0.5]))
    tokens = _log_int(rng, 2000, 262144)
    heads = rng.choice([2, 8, 12, 16])
    if kind == "predict":
        return dict(kind=kind, heads=heads, tokens=tokens)
    kb, qb = -(-tokens // 64), -(-tokens // 128)
    if kind == "mask":
        return dict(kind=kind, heads=heads, qblocks=qb, kblocks=kb, threshold=rng.choice([0.5, 0.8, 0.9]),
                    sink=rng.randint(0, 5))
    return dict(kind=kind, mode=rng.choice(["vasc", "vasc", "topk"]), heads=heads, qblocks=qb, kblocks=kb,
                keep=rng.choice([0.125, 0.25, 0.45]), force_last=rng.random() < 0.4)


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        case = _candidate(rng)
        if work(case)["flops"] <= most:
            return case


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _frames_like(g, groups, per_group, width, scale=0.5):
    """[groups * per_group, width] float32: N(0,1) plus a rank-8 component shared by each group (frame)."""
    x = torch.randn(groups, per_group, width, device="cuda", generator=g)
    u = torch.randn(groups, per_group, 8, device="cuda", generator=g)
    v = torch.randn(groups, 8, width, device="cuda", generator=g)
    return (x + scale * (u @ v) / math.sqrt(8)).view(groups * per_group, width)


def _qkv(g, heads, groups, per_group, dtype):
    """q, k, v [1, heads, groups * per_group, 64] in frame-major order."""
    return [torch.stack([_frames_like(g, groups, per_group, HEAD_DIM) for _ in range(heads)]).unsqueeze(0).to(dtype)
            for _ in range(3)]


def _scores(g, heads, qb, kb):
    """Pooled probabilities [1, heads, qb, kb] with the spread (logits of unit scale, nearby blocks alike) and the
    bf16-rounded logits the predictor gives."""
    step = 16  # key blocks of a frame
    q = torch.randn(heads, qb, HEAD_DIM, device="cuda", generator=g)
    q = 0.8 * q + 0.6 * torch.randn(heads, -(-qb // 8), HEAD_DIM, device="cuda",
                                    generator=g).repeat_interleave(8, 1)[:, :qb]
    k = torch.randn(heads, kb, HEAD_DIM, device="cuda", generator=g)
    k = 0.8 * k + 0.6 * torch.randn(heads, -(-kb // step), HEAD_DIM, device="cuda",
                                    generator=g).repeat_interleave(step, 1)[:, :kb]
    logits = (q.bfloat16() @ k.bfloat16().transpose(1, 2).contiguous()) * 0.125
    return torch.softmax(logits.float(), -1).unsqueeze(0)


def _export(backbone, mode):
    """The mode's switches in the environment, where the evaluators put them once for their process."""
    for k in [k for k in os.environ if k.startswith("SPARSE_VGGT_")]:
        del os.environ[k]
    os.environ.update(method_environment(backbone, mode))


def _ratios(backbone, sparsity):
    return layer_sparsity(backbone, sparsity, "paper") or [sparsity] * (24 if backbone == "vggt" else 18)


def _attention(seed, rope, n=1):
    torch.manual_seed(seed)
    with torch.device("cuda"):
        return [Attention(1024, 16, rope=rope).to(torch.bfloat16).eval() for _ in range(n)]


def _lists(g, heads, tokens, density):
    """Block lists of Poisson length per query block, drawn without replacement, ascending."""
    qb, kb = -(-tokens // 128), -(-tokens // 64)
    n = torch.poisson(torch.full((heads, qb), density * kb, device="cuda"), generator=g).long().clamp(1, kb)
    order = torch.argsort(torch.rand(heads, qb, kb, device="cuda", generator=g), -1)
    keep = torch.arange(kb, device="cuda") < n.unsqueeze(-1)
    index = torch.sort(torch.where(keep, order, kb), -1).values
    width = int(n.max())
    return index[..., :width].to(torch.int32).unsqueeze(0).contiguous(), n.to(torch.int32).unsqueeze(0)


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind == "layer":
        N, gh, gw = case["frames"], case["gh"], case["gw"]
        P = SPECIAL + gh * gw
        _export(case["backbone"], case["mode"])
        rope = RotaryPositionEmbedding2D(100.0)
        rope.tables(HEAD_DIM, torch.device("cuda:0"))
        s["attn"] = _attention(seed, rope, 2)
        s["x"] = [_frames_like(g, N, P, 1024).to(torch.bfloat16).unsqueeze(0) for _ in range(2)]
        s["pos"] = grid_positions(N, gh, gw, SPECIAL, "cuda").to(torch.int32).contiguous().view(1, N * P, 2)
        s["ratio"] = _ratios(case["backbone"], case["sparsity"])[0]
        s["routing"] = {}
    elif kind == "model":
        _export("vggt", "vasc")
        torch.manual_seed(seed)
        with torch.device("cuda"):
            model = Aggregator(dim=1024, depth=case["depth"], num_heads=16,
                               intermediate_layer_idx=(case["depth"] // 2, case["depth"] - 1))
        model = model.to(torch.bfloat16).eval()
        model.rope.tables(HEAD_DIM, torch.device("cuda:0"))
        ratios = _ratios("vggt", case["sparsity"])[:case["depth"]]
        sparse_aggregator_from_vggt_layerwise(model, layer_sparsity_ratios=ratios, verbose=False)
        s["model"] = model
        s["images"] = torch.rand(1, case["frames"], 3, 14 * case["gh"], 14 * case["gw"], device="cuda", generator=g)
    elif kind == "dense":
        B, T, gw = case["batch"], case["tokens"], case["gw"]
        rope = RotaryPositionEmbedding2D(100.0)
        s["attn"] = _attention(seed, rope)[0]
        s["x"] = _frames_like(g, B, T, 1024).to(torch.bfloat16).view(B, T, 1024)
        t = torch.arange(T, device="cuda")
        pos = torch.stack([(t - SPECIAL) // gw + 1, (t - SPECIAL) % gw + 1], -1)
        pos = torch.where((t < SPECIAL).unsqueeze(-1), torch.zeros_like(pos), pos)
        s["pos"] = pos.to(torch.int32).expand(B, T, 2).contiguous()
        rope.tables(HEAD_DIM, torch.device("cuda:0"))
    elif kind == "op":
        _export("vggt", case["mode"])
        N, P, H = case["frames"], case["per_frame"], case["heads"]
        q, k, v = _qkv(g, H, N, P, getattr(torch, case["dtype"]))
        order = torch.arange(N * P, device="cuda").view(N, P)
        order = torch.cat([order[:, SPECIAL:].reshape(-1), order[:, :SPECIAL].reshape(-1)])  # [patch; special]
        s["n_patch"] = N * (P - SPECIAL)
        s["q"] = q[:, :, order[:s["n_patch"]]].contiguous()
        s["k"], s["v"] = k[:, :, order].contiguous(), v[:, :, order].contiguous()
        s["routing"] = {}
    elif kind == "attend":
        H, T = case["heads"], case["tokens"]
        s["q"], s["k"], s["v"] = (torch.randn(1, H, T, HEAD_DIM, device="cuda", generator=g).to(torch.bfloat16)
                                  for _ in range(3))
        s["index"], s["count"] = _lists(g, H, T, case["density"])
    elif kind == "predict":
        H, T = case["heads"], case["tokens"]
        s["q"], s["k"], _ = _qkv(g, H, max(1, T // 1041), -(-T // max(1, T // 1041)), torch.bfloat16)
        s["q"], s["k"] = s["q"][:, :, :T].contiguous(), s["k"][:, :, :T].contiguous()
    elif kind == "mask":
        s["score"] = _scores(g, case["heads"], case["qblocks"], case["kblocks"])
    else:
        H, Q, K = case["heads"], case["qblocks"], case["kblocks"]
        s["score"] = [_scores(g, H, Q, K) for _ in range(2)]
        # innovation of a pair of pooled values: 1 - cos like, in [0, 1], larger between frames
        s["iota"] = [torch.rand(1, H, (K + 1) // 2, device="cuda", generator=g).square() for _ in range(2)]
        n_patch = 64 * K - (7 if case["force_last"] else 0)
        s["plan"] = pipeline.LayerPlan.make(n_patch, n_patch + 3 * 64)
        assert s["plan"].k_blocks == K
        s["ledger"] = pipeline.Ledger()
    return s


# --------------------------------------------------------------------- run
def _run_layer(s):
    case, routing = s["case"], s["routing"]
    routing.clear()
    out = []
    with torch.no_grad(), frame_grid(case["gh"], case["gw"]):
        for i in range(2):
            out.append(adaptive_sparse_attention_forward(s["attn"][i], s["x"][i], s["pos"], sparse_ratio=s["ratio"],
                                                         num_special_tokens=SPECIAL, num_heads=16, layer_idx=i,
                                                         routing_state=routing))
    if case["mode"] == "vasc":
        out.append(routing[STATE_KEY])
    return out


def _run_op(s):
    case, n_patch = s["case"], s["n_patch"]
    s["routing"].clear()
    score = predict_attention(s["q"], s["k"][:, :, :n_patch])
    o = block_sparse_attn_cuda(s["q"], s["k"], s["v"], score, sparse_ratio=case["sparsity"], layer_idx=0,
                               routing_state=s["routing"], num_patch_tokens=n_patch)
    return {"score": score, "o": o}


def _run_select(s):
    case, ledger, plan = s["case"], s["ledger"], s["plan"]
    ledger.clear()
    out = {}
    for i in range(2):
        sel = pipeline.select_layer(s["score"][i], s["iota"][i], plan, mode=case["mode"],
                                    sparse_ratio=1.0 - case["keep"], official_mask=not case["force_last"],
                                    ledger=ledger, layer_idx=i)
        out["index%d" % i], out["count%d" % i] = sel["index"], sel["count"]
        if case["mode"] == "vasc":
            out["arrival%d" % i], out["service%d" % i], out["debt%d" % i] = sel["arrival"], sel["service"], sel["debt"]
    return out


def run(s):
    kind = s["case"]["kind"]
    if kind == "layer":
        return _run_layer(s)
    if kind == "model":
        with torch.no_grad():
            outputs, _ = s["model"](s["images"])
        return [t for t in outputs if t is not None]
    if kind == "dense":
        with torch.no_grad():
            return s["attn"](s["x"], pos=s["pos"])
    if kind == "op":
        return _run_op(s)
    if kind == "attend":
        return ops.block_sparse_attn(s["q"], s["k"], ops.pack_v(s["v"]), s["index"], s["count"])
    if kind == "predict":
        return predict_attention(s["q"], s["k"])
    if kind == "mask":
        return get_block_mask(s["score"], s["case"]["sink"], cdf_threshold=s["case"]["threshold"])
    return _run_select(s)


# -------------------------------------------------------------------- work
def _sparse_pairs(n_patch, n_special, sparsity):
    """(query, key) pairs of one head of a sparse layer: patch queries over their budget and the special keys, special
    queries over every key."""
    budget = max(1, int(-(-n_patch // 64) * (1 - sparsity)))
    return n_patch * (min(64 * budget, n_patch) + n_special) + n_special * (n_patch + n_special)


def work(case):
    kind = case["kind"]
    if kind == "layer":
        N, P = case["frames"], SPECIAL + case["gh"] * case["gw"]
        T = N * P
        s = _ratios(case["backbone"], case["sparsity"])[0]
        pairs = 16 * _sparse_pairs(N * (P - SPECIAL), N * SPECIAL, s)
        # x and the output once, the weights of qkv and proj once
        return {"bytes": 2 * (2 * T * 1024 * 2 + 4 * 1024 * 1024 * 2),
                "flops": 2 * (2.0 * T * 1024 * 4096 + 4.0 * HEAD_DIM * pairs)}
    if kind == "model":
        N, P, L = case["frames"], SPECIAL + case["gh"] * case["gw"], case["depth"]
        T = N * P
        pairs = 16 * sum(_sparse_pairs(N * (P - SPECIAL), N * SPECIAL, s)
                         for s in _ratios("vggt", case["sparsity"])[:L])
        pairs += L * 16 * N * P * P
        return {"bytes": N * 3 * 196 * case["gh"] * case["gw"] * 4 + 2 * L * 12 * 1024 * 1024 * 2 + 2 * T * 2048 * 2,
                "flops": 2 * L * 2.0 * T * 1024 * 12288 + 4.0 * HEAD_DIM * pairs}
    if kind == "dense":
        B, T = case["batch"], case["tokens"]
        return {"bytes": 2 * B * T * 1024 * 2 + 4 * 1024 * 1024 * 2,
                "flops": 2.0 * B * T * 1024 * 4096 + 4.0 * HEAD_DIM * 16 * B * T * T}
    if kind == "op":
        H, N, P = case["heads"], case["frames"], case["per_frame"]
        np_, T = N * (P - SPECIAL), N * P
        qb, kb = -(-np_ // 128), -(-np_ // 64)
        pairs = _sparse_pairs(np_, N * SPECIAL, case["sparsity"]) - N * SPECIAL * T
        return {"bytes": H * HEAD_DIM * 2 * (2 * np_ + 2 * T) + H * qb * kb * 4, "flops": 4.0 * HEAD_DIM * H * pairs}
    if kind == "attend":
        H, T = case["heads"], case["tokens"]
        qb, kb = -(-T // 128), -(-T // 64)
        return {"bytes": 4 * H * T * HEAD_DIM * 2 + H * qb * kb * case["density"] * 4,
                "flops": 4.0 * HEAD_DIM * H * T * T * case["density"]}
    if kind == "predict":
        H, T = case["heads"], case["tokens"]
        qb, kb = -(-T // 128), -(-T // 64)
        return {"bytes": 2 * H * T * HEAD_DIM * 2 + H * qb * kb * 4,
                "flops": H * (2.0 * T * HEAD_DIM + 2.0 * qb * kb * HEAD_DIM)}
    rows = case["heads"] * case["qblocks"]
    K = case["kblocks"]
    if kind == "mask":
        return {"bytes": rows * (5 * K + case["sink"]), "flops": rows * K * math.log2(max(K, 2))}
    budget = max(1, int(K * case["keep"]))
    return {"bytes": 2 * (rows * (4 * K + 4 * budget)), "flops": 2 * 4.0 * rows * K}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    kind = case["kind"]
    if kind in ("mask", "select"):
        return "exact"  # whole numbers, and a ledger whose sums have a fixed order
    if kind == "predict":
        # float32 sums in another order: 1.1e-7 measured; at most one bf16 step of a logit at single entries
        return {"rel": 1e-5, "max": 0.02}
    # bf16 probabilities and outputs: 2.3e-3 to 3.3e-3 from the float64 result measured for the attention and the
    # dense layer; pooling in another order left the sparse layers' lists as they were
    return {"rel": 0.01, "max": 0.2}


# ------------------------------------------------------------------- exact
def _exact_prob(q, k):
    """The predictor in float64, with the roundings that belong to its definition (means and logits in bf16)."""
    def means(t, n):
        t = t.to(torch.bfloat16)
        full = t.shape[2] // n * n
        m = [t[:, :, :full].double().unflatten(2, (-1, n)).mean(3)] if full else []
        if full < t.shape[2]:
            m.append(t[:, :, full:].double().mean(2, keepdim=True))
        return torch.cat(m, 2).to(torch.bfloat16).double()
    pq, pk = means(q, 128), means(k, 64)
    dots = (pq @ pk.transpose(2, 3).contiguous()).to(torch.bfloat16).double()
    return torch.softmax((dots * 0.125).to(torch.bfloat16).double(), -1)


def _exact_attend(s):
    q, k, v = (s[n].double() for n in ("q", "k", "v"))
    _, H, T, _ = q.shape
    qb, kb = -(-T // 128), -(-T // 64)
    live = torch.arange(s["index"].shape[-1], device="cuda") < s["count"].unsqueeze(-1)
    chosen = torch.zeros(H, qb, kb + 1, dtype=torch.bool, device="cuda")
    chosen.scatter_(2, torch.where(live, s["index"].long(), kb)[0], True)
    chosen = chosen[..., :kb]
    out = torch.empty_like(q)
    step = max(1, min(qb, (1 << 29) // (128 * kb * 64)))  # query blocks at once
    for h in range(H):
        kt = k[0, h].t().contiguous()
        for b0 in range(0, qb, step):
            rows = slice(128 * b0, min(T, 128 * (b0 + step)))
            logits = (q[0, h, rows] @ kt).mul_(0.125)
            keep = chosen[h, b0:b0 + step].repeat_interleave(64, 1)[:, :T].repeat_interleave(128, 0)
            logits.masked_fill_(~keep[:logits.shape[0]], -math.inf)
            out[0, h, rows] = torch.softmax(logits, -1) @ v[0, h]
    return out


def _exact_dense(s):
    x, pos, attn = s["x"].double(), s["pos"].long(), s["attn"]
    B, T, C = x.shape
    H, D = attn.num_heads, attn.head_dim
    qkv = x @ attn.qkv.weight.double().t() + attn.qkv.bias.double()
    q, k, v = qkv.view(B, T, 3, H, D).permute(2, 0, 3, 1, 4)

    def turn(t, norm):
        t = torch.nn.functional.layer_norm(t, (D,), norm.weight.double(), norm.bias.double(), norm.eps)
        freq = 100.0 ** (-torch.arange(0, D // 2, 2, dtype=torch.float64, device=t.device) / (D // 2))
        halves = []
        for i, part in enumerate(t.chunk(2, -1)):
            ang = pos[:, None, :, i, None] * freq
            lo, hi = part.chunk(2, -1)
            halves += [lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin()]
        return torch.cat(halves, -1)
    q, k = turn(q, attn.q_norm), turn(k, attn.k_norm)
    out = torch.empty(B, T, H, D, dtype=torch.float64, device=x.device)
    for b in range(B):
        for h in range(H):
            kt, step = k[b, h].t().contiguous(), max(1, (1 << 29) // T)
            for r in range(0, T, step):
                out[b, r:r + step, h] = torch.softmax((q[b, h, r:r + step] @ kt).mul_(0.125), -1) @ v[b, h]
    return out.view(B, T, C) @ attn.proj.weight.double().t() + attn.proj.bias.double()


def _exact_arrival(score, iota, cap):
    """Mean over the query blocks of the pairs' conservative arrival: the row's value risk capped to mass cap."""
    H, K = score.shape[1], score.shape[3]
    out = torch.empty(H, iota.shape[2], dtype=torch.float64, device=score.device)
    for h in range(H):
        risk = score[0, h].double() * iota[0, h].double().repeat_interleave(2)[:K]
        a = (risk * (cap[h].double().unsqueeze(-1) / risk.sum(-1, keepdim=True))).clamp(0, 1)
        a = torch.nn.functional.pad(a, (0, K % 2)).view(a.shape[0], -1, 2).sum(-1)
        a /= torch.full((a.shape[1],), 2.0, device=a.device).index_fill_(
            0, torch.arange(a.shape[1] - K % 2, a.shape[1], device=a.device), 1.0)
        out[h] = a.mean(0)
    return out.unsqueeze(0)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("layer", "model", "mask"):
        # the output of a sparse layer follows the blocks that rounded scores select: no value in 64 bits
        return None
    if kind == "dense" and 4.0 * HEAD_DIM * 16 * case["batch"] * case["tokens"] ** 2 > 3e12:
        return None
    s = prepare(case, seed)
    if kind == "dense":
        return _exact_dense(s)
    if kind == "attend":
        return _exact_attend(s)
    if kind == "predict":
        return _exact_prob(s["q"], s["k"])
    if kind == "op":  # the output follows the selected blocks, as above
        return {"score": _exact_prob(s["q"], s["k"][:, :, :s["n_patch"]]), "o": None}
    if case["mode"] != "vasc":
        return None
    out = {}
    for i in range(2):
        score = s["score"][i]
        K = score.shape[3]
        cap = torch.full(score.shape[1:3], max(1, int(K * (1 - (1.0 - case["keep"])))), device="cuda")
        if case["force_last"]:  # the last block joins the rows that did not keep it (ties to the lower block)
            beat = (score[0, :, :, :-1] >= score[0, :, :, -1:]).sum(-1)
            cap = cap + (beat >= cap)
        # the lists, the service and the debt follow the selection; the arrival does not
        out.update({"arrival%d" % i: _exact_arrival(score, s["iota"][i], cap), "index%d" % i: None,
                    "count%d" % i: None, "service%d" % i: None, "debt%d" % i: None})
    return out
