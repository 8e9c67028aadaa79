"""Kernel 3 (pack) and kernel 4 (block-sparse / dense attention) vs the oracle.

Tolerance (from the north star): bf16 GPU output vs float64 oracle on the
same bf16 inputs and the same index lists, max-abs <= 2e-2, mean-abs <= 2e-3.
"""
import math

import numpy as np
import pytest
import torch

from oracle import attention as OA
from oracle import selector as OS

pytestmark = pytest.mark.gpu

MAX_ABS = 2e-2
MEAN_ABS = 2e-3


def _rand(shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(torch.bfloat16)


def _lists(B, H, qb, nkb, seed, density=0.3, allow_empty=False):
    rng = np.random.default_rng(seed)
    counts = rng.binomial(nkb, density, size=(B, H, qb)).clip(0 if allow_empty else 1, nkb)
    idx = np.full((B, H, qb, nkb), -1, np.int32)
    for b in range(B):
        for h in range(H):
            for i in range(qb):
                sel = np.sort(rng.choice(nkb, size=counts[b, h, i], replace=False))
                idx[b, h, i, : sel.size] = sel
    return idx, counts.astype(np.int32)


def _check(out, ref):
    err = np.abs(out.float().cpu().numpy().astype(np.float64) - ref)
    assert np.isfinite(out.float().cpu().numpy()).all()
    assert err.max() <= MAX_ABS, f"max-abs {err.max():.3e}"
    assert err.mean() <= MEAN_ABS, f"mean-abs {err.mean():.3e}"
    return err.max(), err.mean()


def test_pack_v_layout_bit_exact():
    from vasc_amd import ops
    B, H, T, D = 1, 3, 200, 64
    v = _rand((B, H, T, D), 1)
    vt = ops.pack_v(v.cuda()).cpu()
    nkb = math.ceil(T / 64)
    vp = torch.zeros(B, H, nkb * 64, D, dtype=torch.bfloat16)
    vp[:, :, :T] = v
    pos = torch.arange(64)
    s, hh, e = pos // 16, (pos % 16) // 8, pos % 8
    key = 16 * s + 8 * (e // 4) + 4 * hh + (e % 4)
    expect = vp.view(B, H, nkb, 64, D)[:, :, :, key, :].transpose(-1, -2)
    assert torch.equal(vt.view(torch.int16), expect.contiguous().view(torch.int16))


@pytest.mark.parametrize("nq,nk,seed,B", [(128, 64, 0, 1), (300, 200, 1, 1), (1000, 1041, 2, 1), (77, 130, 3, 1),
                                         (300, 330, 4, 2)])
def test_block_sparse_matches_oracle(nq, nk, seed, B):
    from vasc_amd import ops
    H, D = 2, 64
    q, k, v = _rand((B, H, nq, D), seed), _rand((B, H, nk, D), seed + 100), _rand((B, H, nk, D), seed + 200)
    qb, nkb = math.ceil(nq / 128), math.ceil(nk / 64)
    idx, cnt = _lists(B, H, qb, nkb, seed)
    qc, kc, vc = q.cuda(), k.cuda(), v.cuda()
    out = ops.block_sparse_attn(qc, kc, ops.pack_v(vc), torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda())
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), idx, cnt)
    _check(out, ref)


def test_dense_matches_oracle_and_full_lists():
    from vasc_amd import ops
    B, H, nq, nk, D = 1, 2, 520, 777, 64
    q, k, v = _rand((B, H, nq, D), 5), _rand((B, H, nk, D), 6), _rand((B, H, nk, D), 7)
    qc, kc, vt = q.cuda(), k.cuda(), ops.pack_v(v.cuda())
    dense = ops.dense_attn(qc, kc, vt)
    idx, cnt = OA.dense_lists(B, H, nq, nk)
    sparse = ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda())
    assert torch.equal(dense.view(torch.int16), sparse.view(torch.int16))
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), idx, cnt)
    _check(dense, ref)
    sdpa = torch.nn.functional.scaled_dot_product_attention(q.double(), k.double(), v.double())
    assert np.abs(sdpa.numpy() - ref).max() < 1e-9


def test_delta_lut_equals_index_lists():
    from vasc_amd import ops
    from oracle import lut as OL
    B, H, nq, nk = 1, 2, 400, 650
    q, k, v = _rand((B, H, nq, 64), 8), _rand((B, H, nk, 64), 9), _rand((B, H, nk, 64), 10)
    qb, nkb = math.ceil(nq / 128), math.ceil(nk / 64)
    idx, cnt = _lists(B, H, qb, nkb, 11)
    mask = np.zeros((B, H, qb, nkb), bool)
    for b in range(B):
        for h in range(H):
            for i in range(qb):
                mask[b, h, i, idx[b, h, i, : cnt[b, h, i]]] = True
    lut, vcnt = OL.encode(mask)
    assert (vcnt == cnt).all()
    qc, kc, vt = q.cuda(), k.cuda(), ops.pack_v(v.cuda())
    a = ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda())
    b = ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(lut).cuda(), torch.from_numpy(vcnt).cuda(), delta=True)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_empty_rows_and_out_of_range_blocks():
    from vasc_amd import ops
    B, H, nq, nk = 1, 1, 256, 256
    q, k, v = _rand((B, H, nq, 64), 12), _rand((B, H, nk, 64), 13), _rand((B, H, nk, 64), 14)
    idx = np.array([[[[1, 3, -1, 99], [0, 0, 0, 0]]]], np.int32)  # row 0: blocks 1,3 + two invalid
    cnt = np.array([[[4, 0]]], np.int32)
    qc, kc, vt = q.cuda(), k.cuda(), ops.pack_v(v.cuda())
    out = ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda()).float().cpu()
    assert torch.count_nonzero(out[0, 0, 128:]) == 0
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(),
                                    np.array([[[[1, 3], [0, 0]]]], np.int32), np.array([[[2, 0]]], np.int32))
    err = np.abs(out.numpy() - ref)
    assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS


def test_strided_inputs_match_contiguous():
    from vasc_amd import ops
    B, H, T, D = 1, 4, 333, 64
    qkv = _rand((B, T, 3, H, D), 15).cuda()
    q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))  # [B,H,T,D] strided views
    vt = ops.pack_v(v)
    a = ops.dense_attn(q, k, vt)
    b = ops.dense_attn(q.contiguous(), k.contiguous(), ops.pack_v(v.contiguous()))
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_c1_layer_topk_lists():
    """Config 1 shape (8 frames x 1041 tokens, H=16) with Top-K lists + sink."""
    from vasc_amd import ops
    N, P, S, H, D = 8, 1041, 5, 16, 64
    Np, Tk = N * (P - S), N * P
    g = torch.Generator().manual_seed(0)
    q = torch.randn(1, H, Np, D, generator=g).to(torch.bfloat16)
    k = torch.randn(1, H, Tk, D, generator=g).to(torch.bfloat16)
    v = torch.randn(1, H, Tk, D, generator=g).to(torch.bfloat16)
    qb, kb = math.ceil(Np / 128), math.ceil(Np / 64)
    score = np.random.default_rng(0).random((1, H, qb, kb)).astype(np.float32)
    final = OS.topk_block_mask(score, math.ceil(Tk / 64) - kb, sparse_ratio=0.75)
    idx, cnt = OS.index_lists(final)
    out = ops.block_sparse_attn(q.cuda(), k.cuda(), ops.pack_v(v.cuda()), torch.from_numpy(idx).cuda(),
                                torch.from_numpy(cnt).cuda())
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), idx, cnt)
    _check(out, ref)


@pytest.mark.parametrize("case", ["high", "low", "mixed"])
def test_extreme_logits_take_the_exact_path(case):
    """Logits far outside the fast path's range: row sums above 2^120 (the
    largest of them above 2^130) or all logits below -126 in log2 units (every
    probability would underflow). The kernel must move its exponent offset and
    still match the float64 softmax."""
    from vasc_amd import ops
    B, H, nq, nk, D = 1, 2, 256, 640, 64
    g = torch.Generator().manual_seed(21)
    q = torch.randn(B, H, nq, D, generator=g)
    k = torch.randn(B, H, nk, D, generator=g)
    v = torch.randn(B, H, nk, D, generator=g)
    u = torch.randn(D, generator=g)
    u = u / u.norm() * 8.0
    if case == "high":
        # log2 logit std ~ 0.18 * 6 * 6 * 8 = 52: row maxima 100..220
        q, k = q * 6.0, k * 6.0
    else:
        # every key ~ -4u: rows ~ +4u sit near -185 (all below -126), rows
        # ~ -4u near +185; "mixed" interleaves those with ordinary rows
        k = -4.0 * u + 0.5 * torch.randn(B, H, nk, D, generator=g)
        low = 4.0 * u + 0.5 * torch.randn(B, H, nq, D, generator=g)
        if case == "low":
            q = low
        else:
            high = -4.0 * u + 0.5 * torch.randn(B, H, nq, D, generator=g)
            r = torch.arange(nq) % 3
            q = torch.where((r == 0).view(1, 1, nq, 1), low, torch.where((r == 1).view(1, 1, nq, 1), high, q))
    q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)
    qb, nkb = math.ceil(nq / 128), math.ceil(nk / 64)
    idx, cnt = _lists(B, H, qb, nkb, 22, density=0.6)
    sums = _log2_sums(q, k, idx, cnt)
    assert {"high": sums.max() > 130, "low": sums.max() < -100, "mixed": sums.max() > 130 and sums.min() < -100}[case]
    out = ops.block_sparse_attn(q.cuda(), k.cuda(), ops.pack_v(v.cuda()), torch.from_numpy(idx).cuda(),
                                torch.from_numpy(cnt).cuda())
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), idx, cnt)
    _check(out, ref)
    dense = ops.dense_attn(q.cuda(), k.cuda(), ops.pack_v(v.cuda()))
    dl = OA.dense_lists(B, H, nq, nk)
    _check(dense, OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), *dl))


def _log2_sums(q, k, idx, cnt):
    """Row sums of the listed keys' exponentials, log2, in float64."""
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * (q.shape[-1] ** -0.5 * math.log2(math.e))
    keep = torch.zeros(*idx.shape[:3], math.ceil(k.shape[2] / 64), dtype=torch.bool)
    for at in np.ndindex(*cnt.shape):
        keep[at][torch.from_numpy(idx[at][:cnt[at]]).long()] = True
    keep = keep.repeat_interleave(64, -1)[..., :k.shape[2]].repeat_interleave(128, 2)[:, :, :q.shape[2]]
    return torch.logsumexp(s.masked_fill(~keep, -math.inf) * math.log(2), -1) / math.log(2)


@pytest.mark.parametrize("hot", [None, "peak", "ramp", "low"])
@pytest.mark.parametrize("nblk,at,reverse", [(1, 0, False), (2, 1, False), (7, 6, False), (8, 7, True), (9, 8, False),
                                             (9, 0, True), (10, 9, False), (20, 7, False), (20, 8, True), (20, 9, False),
                                             (20, 19, False), (27, 24, False), (27, 25, True), (60, 56, False),
                                             (60, 57, False)])
def test_range_exit_at_every_point_of_the_walk(nblk, at, reverse, hot):
    """Rows whose sums leave the range of exponent offset 0, before, at and after
    the points where the kernel looks at them (after blocks 0, 8, 24, 56 and the
    last), in lists of either order that hold the partial last block, with waves
    that own no rows (nq = 130). Every third row is out: "peak": block ``at`` near
    2^180; "ramp": each block 2^70 above the one before, so that the second walk
    moves its offset in every block; "low": every logit near 2^-180. Same
    tolerance as the other extreme-logit cases: bf16 probabilities of a float64
    softmax."""
    from vasc_amd import ops
    B, H, nq, nk, D = 1, 2, 130, 64 * nblk - 31, 64
    q, k, v = (_rand((B, H, n, D), 30 + i) for i, n in enumerate((nq, nk, nk)))
    q[..., 0] = 0.0
    order = np.arange(nblk)[::-1] if reverse else np.arange(nblk)
    idx = np.ascontiguousarray(np.broadcast_to(order.astype(np.int32), (B, H, 2, nblk)))
    cnt = np.full((B, H, 2), nblk, np.int32)
    if hot:
        q[:, :, ::3, 0] = 8.0  # log2 logit: q0 * k0 / 8 * log2(e)
        level = {"peak": torch.where(torch.arange(nblk) == at, 180.0, 0.0), "ramp": 70.0 * (torch.arange(nblk) + 2),
                 "low": torch.full((nblk,), -180.0)}[hot]
        k[..., 0] = (level / math.log2(math.e)).to(torch.bfloat16).repeat_interleave(64)[:nk]
        sums = _log2_sums(q, k, idx, cnt)
        assert ((sums[:, :, ::3] < -150) if hot == "low" else (sums[:, :, ::3] > 125)).all()
        assert (sums[:, :, 1::3].abs() < 30).all()
    qc, kc, vt = q.cuda(), k.cuda(), ops.pack_v(v.cuda())
    out = ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda())
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), idx, cnt)
    _check(out, ref)
    _check(ops.dense_attn(qc, kc, vt), ref)


@pytest.mark.parametrize("form", ["listed", "delta", "special"])
@pytest.mark.parametrize("later", [0.0, 60.0, 200.0])
@pytest.mark.parametrize("nblk,at", [(2, 0), (3, 0), (4, 0), (10, 8), (11, 8), (28, 24), (70, 0), (70, 56)])
def test_walk_goes_on_with_good_sums(nblk, at, later, form):
    """Row sums near 2^100 (block 0) or 2^110 (later blocks) after a look at them:
    the walk is left two blocks on with sums that are good at exponent offset 0,
    and the rest of the list, the partial last block in it, is added to them; its
    last block lies at 2^``later``, up to a move of the offset. Special queries:
    70 blocks go in two parts, beside a patch block of the same list."""
    from vasc_amd import _lib, ops
    from oracle import lut as OL
    B, H, nq, nk, D = 1, 2, 130, 64 * nblk - 31, 64
    q, k, v = (_rand((B, H, n, D), 33 + i) for i, n in enumerate((nq, nk, nk)))
    level = torch.zeros(nblk)
    level[at] = 110.0 if at else 100.0
    if at + 2 < nblk:
        level[-1] = later
    q[..., 0] = 0.0
    q[:, :, ::3, 0] = 8.0  # log2 logit: q0 * k0 / 8 * log2(e)
    k[..., 0] = (level / math.log2(math.e)).to(torch.bfloat16).repeat_interleave(64)[:nk]
    idx = np.ascontiguousarray(np.broadcast_to(np.arange(nblk, dtype=np.int32), (B, H, 2, nblk)))
    cnt = np.full((B, H, 2), nblk, np.int32)
    left = _log2_sums(q, k, idx, np.full((B, H, 2), min(at + 2, nblk), np.int32))[:, :, ::3]
    assert (left > (104 if at else 72)).all() and (left < 119).all()
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), idx, cnt)
    qc, kc, vt = q.cuda(), k.cuda(), ops.pack_v(v.cuda())
    ic, cc = torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda()
    if form == "special":
        qp, one = qc[:, :, :128], torch.ones_like(cc[:, :, :1])
        assert (_lib.fn("vasc_global_attn_workspace_size")(B, H, 128, nq, nk, 1) > 0) == (nblk == 70)
        _check(ops.global_attn(qp, qc, kc, vt, ic[:, :, :1, :1].contiguous(), one)[1], ref)
    elif form == "delta":
        lut, n = OL.encode(np.ones((B, H, 2, nblk), bool))
        assert (n == cnt).all()
        _check(ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(lut).cuda(), cc, delta=True), ref)
    else:
        _check(ops.block_sparse_attn(qc, kc, vt, ic, cc), ref)
        _check(ops.dense_attn(qc, kc, vt), ref)


@pytest.mark.parametrize("N,P,S,H", [(1, 129, 1, 1), (3, 47, 5, 3), (2, 130, 0, 9)])
def test_prescaled_queries_match_the_oracle(N, P, S, H):
    """Queries packed with the softmax scale: the layout differs in q only, the
    pooled means not at all, and the attention of patch and special queries stays
    within the file's tolerance of the float64 softmax of the unscaled queries
    (which have no norm here, so that the scaled copy is a rounding more)."""
    from vasc_amd import ops
    T = N * P
    qkv = _rand((1, T, 3, H, 64), 40).cuda()
    q, k, v = (qkv[:, :, i] for i in range(3))
    c = ops.LOG2E / 8.0
    ref = ops.pack_global(q, k, v, N, P, S)
    got = ops.pack_global(q, k, v, N, P, S, q_scale=c)
    for i, (a, b) in enumerate(zip(ref, got)):
        if a is None:
            assert b is None
        elif i < 2:  # q_patch, q_special
            assert torch.equal(b, (a.float() * torch.tensor(c, dtype=torch.float32, device="cuda")).to(torch.bfloat16))
        else:
            assert torch.equal(a, b)
    qp, qs, ko, vt = got[:4]
    np_, qb, nkb = N * (P - S), math.ceil(N * (P - S) / 128), math.ceil(T / 64)
    idx, cnt = _lists(1, H, qb, nkb, 41, density=0.6)
    rows = OA.block_sparse_attention(ref[0].float().cpu().numpy(), ko.float().cpu().numpy(),
                                     ops.pack_qkv(q, k, v, N, P, S)[3].float().cpu().numpy(), idx, cnt)
    out = ops.global_attn_tokens(qp, qs, ko, vt, torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda(), N, P, S,
                                 scale=ops.LN2)
    patch = out.view(1, N, P, H, 64)[:, :, S:].reshape(1, np_, H, 64).transpose(1, 2)
    _check(patch, rows)
    if S:
        n_sp = N * S
        full = np.broadcast_to(np.arange(nkb, dtype=np.int32), (1, H, math.ceil(n_sp / 128), nkb))
        _check(out.view(1, N, P, H, 64)[:, :, :S].reshape(1, n_sp, H, 64).transpose(1, 2),
               OA.block_sparse_attention(ref[1].float().cpu().numpy(), ko.float().cpu().numpy(),
                                         ops.pack_qkv(q, k, v, N, P, S)[3].float().cpu().numpy(), full,
                                         np.full(full.shape[:3], nkb)))


@pytest.mark.parametrize("level", [None, "high", "low"])
@pytest.mark.parametrize("N,P,S,parts", [(1, 4032, 1, 1), (1, 4033, 5, 2), (3, 1409, 45, 2), (2, 4099, 65, 4),
                                         (1, 16391, 129, 8)])
def test_split_special_queries_match_the_oracle(N, P, S, parts, level):
    """Special queries whose keys are split over workgroups, at part counts 1,
    2, 4 and 8, ragged last parts and a second query block. "high": the first
    key block's logits near 2^150, "low": the last part's all near 2^-160; both
    are out of the sums' range and take the second walk. The file's tolerance:
    the parts only change the order of a float32 addition."""
    from vasc_amd import _lib, ops
    H, nk, n_patch, n_sp = 2, N * P, N * (P - S), N * S
    nkb = math.ceil(nk / 64)
    q, k, v = _rand((1, H, nk, 64), 50), _rand((1, H, nk, 64), 51), _rand((1, H, nk, 64), 52)
    if level is not None:  # q0 * k0 / 8 * log2(e) = 150 or -160
        q[..., 0] = 8.0
        k[..., 0] = 0.0
        if level == "high":
            k[:, :, :64, 0] = 150.0 / math.log2(math.e)
        else:
            k[:, :, (parts - 1) * math.ceil(nkb / parts) * 64:, 0] = -160.0 / math.log2(math.e)
    qp, qs, kc, vt = q[:, :, :n_patch].cuda(), q[:, :, n_patch:].cuda(), k.cuda(), ops.pack_v(v.cuda())
    idx = torch.zeros(1, H, math.ceil(n_patch / 128), 1, dtype=torch.int32)
    cnt = torch.ones(1, H, math.ceil(n_patch / 128), dtype=torch.int32)
    size = _lib.fn("vasc_global_attn_workspace_size")(1, H, n_patch, n_sp, nk, 1)
    assert size == (0 if parts == 1 else H * math.ceil(n_sp / 128) * parts * 128 * 65 * 4)
    full = torch.arange(nkb, dtype=torch.int32).expand(1, H, math.ceil(n_sp / 128), nkb).contiguous()
    ref = OA.block_sparse_attention(q[:, :, n_patch:].float().numpy(), k.float().numpy(), v.float().numpy(), full.numpy(),
                                    torch.full(full.shape[:3], nkb, dtype=torch.int32).numpy())
    refp = OA.block_sparse_attention(q[:, :, :n_patch].float().numpy(), k.float().numpy(), v.float().numpy(), idx.numpy(),
                                     cnt.numpy())
    op, os_ = ops.global_attn(qp, qs, kc, vt, idx.cuda(), cnt.cuda())
    _check(os_, ref)
    _check(op, refp)
    out = ops.global_attn_tokens(qp, qs, kc, vt, idx.cuda(), cnt.cuda(), N, P, S).view(1, N, P, H, 64)
    assert torch.equal(out[:, :, :S].reshape(1, n_sp, H, 64).transpose(1, 2), os_)
    assert torch.equal(out[:, :, S:].reshape(1, n_patch, H, 64).transpose(1, 2), op)


@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("level", [None, "high", "low", "parts"])
def test_split_special_queries_in_batches(level, unit):
    """The key split with two batch entries, strided queries and both forms of
    the kernel (the plain scale; queries that hold the scale, sm_scale = ln 2).
    "high" and "low" as above; "parts": the last two of three parts near 2^180 with
    comparable weights, the first at 2^0, so that parts of different offsets meet
    in the combination."""
    from vasc_amd import _lib, ops
    B, H, N, P, S = 2, 2, 2, 3201, 3
    nk, n_patch, n_sp = N * P, N * (P - S), N * S
    nkb, qb, parts = math.ceil(nk / 64), math.ceil(n_patch / 128), 3
    k, v = _rand((B, nk, H, 64), 71), _rand((B, H, nk, 64), 72)
    q = _rand((B, nk, H, 64), 70)
    if level is not None:
        q[..., 0] = 8.0
        k[..., 0] = 0.0
        if level == "high":
            k[:, :64, :, 0] = 150.0 / math.log2(math.e)
        elif level == "low":
            k[..., 0] = -160.0 / math.log2(math.e)
        else:
            k[:, math.ceil(nkb / parts) * 64:, :, 0] = 180.0 / math.log2(math.e)
    scale = None
    if unit:
        q, scale = (q.float() * (ops.LOG2E / 8)).to(torch.bfloat16), ops.LN2
    q, k = q.cuda().transpose(1, 2), k.cuda().transpose(1, 2)
    qp, qs, vt = q[:, :, :n_patch], q[:, :, n_patch:], ops.pack_v(v.cuda())
    W = 40  # lists of 40 blocks: 100 key blocks in parts of at least 32 blocks, about as long as the lists
    idx = (torch.arange(W, dtype=torch.int32) * 2 + 1).expand(B, H, qb, W).contiguous()
    cnt = torch.full((B, H, qb), W, dtype=torch.int32)
    size = _lib.fn("vasc_global_attn_workspace_size")(B, H, n_patch, n_sp, nk, W)
    assert size == B * H * math.ceil(n_sp / 128) * parts * 128 * 65 * 4
    op, os_ = ops.global_attn(qp, qs, k, vt, idx.cuda(), cnt.cuda(), scale=scale)
    out = ops.global_attn_tokens(qp, qs, k, vt, idx.cuda(), cnt.cuda(), N, P, S, scale=scale).view(B, N, P, H, 64)
    assert torch.equal(out[:, :, :S].reshape(B, n_sp, H, 64).transpose(1, 2), os_)
    assert torch.equal(out[:, :, S:].reshape(B, n_patch, H, 64).transpose(1, 2), op)
    kn, vn = k.cpu().float().numpy(), v.float().numpy()
    full = np.broadcast_to(np.arange(nkb, dtype=np.int32), (B, H, 1, nkb))
    _check(os_, OA.block_sparse_attention(qs.cpu().float().numpy(), kn, vn, full, np.full((B, H, 1), nkb), scale=scale))
    some = [0, qb - 1]
    ref = OA.block_sparse_attention(qp.cpu().float().numpy(), kn, vn, idx.numpy(), cnt.numpy(), scale=scale, q_blocks=some)
    for i in some:
        _check(op[:, :, 128 * i:128 * i + 128], ref[:, :, 128 * i:128 * i + 128])


@pytest.mark.parametrize("form", ["half", "delta", "unit", "tokens", "outside"])
def test_second_walk_in_every_form_of_call(form):
    """Every third row near 2^180 in one block, so that every workgroup walks
    twice: float16 queries and results, delta lists, queries that hold the scale,
    token-major results, and lists that name blocks outside the sequence (first,
    amid and last) beside the same lists without them."""
    from vasc_amd import ops
    from oracle import lut as OL
    B, H, N, P, S = 2, 3, 2, 350, 3
    nk, nq = N * P, N * (P - S)
    qb, nkb = math.ceil(nq / 128), math.ceil(nk / 64)
    q, k, v = (_rand((B, H, nk, 64), 80 + i).to(torch.float16).to(torch.bfloat16) for i in range(3))  # exact in both
    q[..., 0], k[..., 0] = 0.0, 0.0
    q[:, :, ::3, 0] = 8.0
    k[:, :, 256:320, 0] = 180.0 / math.log2(math.e)
    mask = np.random.default_rng(83).random((B, H, qb, nkb)) < 0.5
    mask[..., 4] = True
    idx, cnt = OS.index_lists(mask)
    idx, cnt = np.ascontiguousarray(idx), np.ascontiguousarray(cnt)
    scale = None
    if form == "unit":
        q, scale = (q.float() * (ops.LOG2E / 8)).to(torch.bfloat16), ops.LN2
    qp, qs = q[:, :, :nq].contiguous(), q[:, :, nq:].contiguous()
    qc, kc, vt = qp.cuda(), k.cuda(), ops.pack_v(v.cuda())
    ic, cc = torch.from_numpy(idx).cuda(), torch.from_numpy(cnt).cuda()
    ref = OA.block_sparse_attention(qp.float().numpy(), k.float().numpy(), v.float().numpy(), idx, cnt, scale=scale)
    out = ops.block_sparse_attn(qc, kc, vt, ic, cc, scale=scale)
    _check(out, ref)
    if form == "half":
        qh, kh, vh = (t.to(torch.float16) for t in (qp, k, v))
        kb, vth = ops.pack_kv_half(kh.cuda(), vh.cuda())
        assert torch.equal(kb, kc) and torch.equal(vth, vt)
        assert torch.equal(ops.block_sparse_attn(qh.cuda(), kb, vth, ic, cc, half_out=True), out.to(torch.float16))
    elif form == "delta":
        lut, n = OL.encode(mask)
        assert (n == cnt).all()
        assert torch.equal(ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(lut).cuda(), cc, delta=True), out)
    elif form == "tokens":
        tok = ops.global_attn_tokens(qc, qs.cuda(), kc, vt, ic, cc, N, P, S).view(B, N, P, H, 64)
        assert torch.equal(tok[:, :, S:].reshape(B, nq, H, 64).transpose(1, 2), out)
        full = np.broadcast_to(np.arange(nkb, dtype=np.int32), (B, H, 1, nkb))
        _check(tok[:, :, :S].reshape(B, N * S, H, 64).transpose(1, 2),
               OA.block_sparse_attention(qs.float().numpy(), k.float().numpy(), v.float().numpy(), full,
                                         np.full((B, H, 1), nkb)))
    elif form == "outside":
        wide = np.full((B, H, qb, nkb + 4), 7, np.int32)
        for at in np.ndindex(B, H, qb):
            n = cnt[at]
            wide[at][:n + 4] = np.concatenate([[-1, nkb], idx[at][:n // 2], [1 << 30], idx[at][n // 2:n], [-5]])
        assert torch.equal(ops.block_sparse_attn(qc, kc, vt, torch.from_numpy(wide).cuda(),
                                                 torch.from_numpy(cnt + 4).cuda()), out)


@pytest.mark.parametrize("gain,rope", [(1.0, False), (1.0, True), (2.0, False), (2.0, True)])
def test_scale_in_normed_queries_costs_no_precision(gain, rope):
    """Normed queries are float32 before their one rounding to bf16, with the
    softmax scale in it or without: against the float64 softmax of the unrounded
    queries (keys and values as packed) the attention's error is the same, 0.99 to
    1.02 of it over gains 0.5 to 3 and 6 seeds; asserted below 1.1."""
    from vasc_amd import ops
    from vasc_amd.aggregator import RotaryPositionEmbedding2D
    N, Hp, S, H = 3, 20, 5, 4
    P = Hp * Hp + S
    g = torch.Generator().manual_seed(90)
    q, k, v = (torch.randn(1, N * P, 3, H, 64, generator=g).to(torch.bfloat16).cuda().unbind(2))
    w, b = gain * (1 + 0.1 * torch.randn(64, generator=g)).cuda(), 0.02 * torch.randn(64, generator=g).cuda()
    i = torch.arange(Hp * Hp)
    pos = torch.cat([torch.zeros(S, 2, dtype=torch.long), torch.stack([i // Hp + 1, i % Hp + 1], -1)])
    pos = pos.repeat(N, 1).unsqueeze(0).cuda()
    tables = RotaryPositionEmbedding2D().tables(64, q.device) if rope else None
    x = torch.nn.functional.layer_norm(q.double(), (64,), w.double(), b.double(), 1e-5)
    if rope:
        freq = 100.0 ** (-torch.arange(0, 32, 2, dtype=torch.float64, device="cuda") / 32)
        halves = []
        for j, part in enumerate(x.chunk(2, -1)):
            ang = pos[:, :, j, None, None].double() * freq
            lo, hi = part.chunk(2, -1)
            halves += [lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin()]
        x = torch.cat(halves, -1)
    x = x.view(1, N, P, H, 64)[:, :, S:].reshape(1, -1, H, 64).transpose(1, 2)
    values = ops.pack_qkv(q, k, v, N, P, S)[3].double()
    err = []
    for q_scale, scale in ((1.0, None), (ops.LOG2E / 8, ops.LN2)):
        qp, _, ko, vt = ops.pack_global(q, k, v, N, P, S, q_norm=(w, b, 1e-5), k_norm=(w, b, 1e-5),
                                        pos=pos if rope else None, rope_tables=tables, q_scale=q_scale)[:4]
        ref = torch.softmax(x @ ko.double().transpose(-1, -2).contiguous() / 8, -1) @ values
        err.append(((ops.dense_attn(qp, ko, vt, scale=scale).double() - ref).norm() / ref.norm()).item())
    assert err[1] < 1.1 * err[0], err


@pytest.mark.parametrize("split", [False, True])
def test_differences_of_huge_logits_are_not_rounded_away(split):
    """Logits of 2^20 whose differences of 0, 1 and 2 decide the weights: every
    score is a whole number below 2^24, exact in float32, while its product with
    log2(e) / 8 alone would be rounded to a multiple of 1/8 (4 percent of a weight)."""
    from vasc_amd import ops
    H, nk, nq = 1, 4225, 130
    q, k, v = torch.zeros(1, H, nq, 64), torch.zeros(1, H, nk, 64), _rand((1, H, nk, 64), 65)
    q[..., 0], q[..., 1] = 2048.0, 1.0
    k[..., 0] = 4096.0
    k[..., 1] = -8.0 * (torch.arange(nk) % 3)
    k[:, :, 12:, 1] -= 4096.0  # twelve keys carry the weight
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    nkb, qb = math.ceil(nk / 64), math.ceil(nq / 128)
    full = torch.arange(nkb, dtype=torch.int32).expand(1, H, qb, nkb).contiguous()
    cnt = torch.full((1, H, qb), nkb, dtype=torch.int32)
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), full.numpy(), cnt.numpy())
    qc, kc, vt = q.cuda(), k.cuda(), ops.pack_v(v.cuda())
    if split:  # as special queries, beside one patch query block with one listed block
        _check(ops.global_attn(qc[:, :, :128], qc, kc, vt, full[:, :, :1, :1].cuda(), torch.ones_like(cnt[:, :, :1]).cuda())[1],
               ref)
    else:
        _check(ops.block_sparse_attn(qc, kc, vt, full.cuda(), cnt.cuda()), ref)
        _check(ops.dense_attn(qc, kc, vt), ref)


@pytest.mark.parametrize("kind", ["listed", "dense", "split"])
@pytest.mark.parametrize("log2_peak", [None, 150.0])
def test_output_may_lie_on_the_queries(kind, log2_peak):
    """The attention written over its own queries gives, bit for bit, what it
    gives beside them, also where the rows' sums leave the range of exponent
    offset 0 (the first key block's logits near 2^150) and are walked again."""
    from vasc_amd import _lib, ops
    H, nq, nk = 2, 300, 4225
    q, k, v = _rand((1, H, nq, 64), 60), _rand((1, H, nk, 64), 61), _rand((1, H, nk, 64), 62)
    if log2_peak is not None:  # q0 * k0 / 8 * log2(e)
        q[..., 0], k[..., 0] = 8.0, 0.0
        k[:, :, :64, 0] = log2_peak / math.log2(math.e)
        assert ((q.double() @ k.double().transpose(-1, -2) / 8 * math.log2(math.e)).amax(-1) > 125).all()
    qc, kc, vt = q.cuda(), k.cuda(), ops.pack_v(v.cuda())
    qb, nkb = math.ceil(nq / 128), math.ceil(nk / 64)
    idx = torch.arange(nkb, dtype=torch.int32, device="cuda").expand(1, H, qb, nkb).contiguous()
    cnt = torch.full((1, H, qb), nkb, dtype=torch.int32, device="cuda")
    over = qc.clone()
    if kind == "listed":
        beside = ops.block_sparse_attn(qc, kc, vt, idx, cnt)
        ops.block_sparse_attn(over, kc, vt, idx, cnt, out=over)
    elif kind == "dense":
        beside = ops.dense_attn(qc, kc, vt)
        ops.dense_attn(over, kc, vt, out=over)
    else:  # as the special queries, whose keys are split; one patch query block with one listed block
        ws_size = _lib.fn("vasc_global_attn_workspace_size")(1, H, 128, nq, nk, 1)
        assert ws_size > 0
        qp, op = _rand((1, H, 128, 64), 63).cuda(), torch.empty(1, H, 128, 64, device="cuda", dtype=torch.bfloat16)
        ws = torch.empty(ws_size, device="cuda", dtype=torch.uint8)
        first, one = idx[:, :, :1, :1].contiguous(), torch.ones_like(cnt[:, :, :1]).contiguous()

        def special(qs, os_):
            _lib.call("vasc_global_attn_ws_fwd", qp.data_ptr(), *qp.stride()[:3], qs.data_ptr(), *qs.stride()[:3],
                      kc.data_ptr(), *kc.stride()[:3], vt.data_ptr(), op.data_ptr(), *op.stride()[:3],
                      os_.data_ptr(), *os_.stride()[:3], 1, H, 128, nq, nk, 64, first.data_ptr(), 1,
                      one.data_ptr(), 0.125, ws.data_ptr(), ws_size, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
        beside = torch.empty_like(qc)
        special(qc, beside)
        special(over, over)
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), idx.cpu().numpy(),
                                    cnt.cpu().numpy())
    _check(beside, ref)
    assert torch.equal(over, beside)


# ---------------------------------------------------------------- PV post-cut
def _graded_blocks(nq, nk, levels, seed):
    """Query rows a*e0 (+ small noise) and key block j = levels[j] / c * e0
    (+ small noise): block j's logits sit at levels[j] in log2 units, so the
    post-cut decisions have margins of whole log2 units."""
    D = 64
    c = D ** -0.5 * math.log2(math.e)
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(1, 2, nq, D, generator=g) * 0.01
    q[..., 0] += 1.0
    k = torch.randn(1, 2, nk, D, generator=g) * 0.01
    for j in range(math.ceil(nk / 64)):
        k[:, :, 64 * j:64 * (j + 1), 0] += float(levels[j % len(levels)]) / c
    v = torch.randn(1, 2, nk, D, generator=g)
    return q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)


@pytest.mark.parametrize("nq,nk,thr", [(512, 1000, 6.0), (300, 1041, 6.0), (256, 640, [6.0, 1e10])])
def test_pv_post_cut_matches_oracle(nq, nk, thr):
    """Execution map bit-exact with the oracle's decisions; output within
    tolerance of float64 attention over the executed blocks."""
    from vasc_amd import ops
    levels = [0, 8, 4, 12, 0, 4, 8, 0]  # log2 units; with threshold 6 every gap + 6 is >= 2 away from 0
    q, k, v = _graded_blocks(nq, nk, levels, seed=nq)
    qb, nkb = math.ceil(nq / 128), math.ceil(nk / 64)
    idx, cnt = _lists(1, 2, qb, nkb, seed=nk, density=0.6)
    o, pv_map = ops.block_sparse_attn_pv(q.cuda(), k.cuda(), ops.pack_v(v.cuda()), torch.from_numpy(idx).cuda(),
                                         torch.from_numpy(cnt).cuda(), thr)
    ex_idx, ex_cnt, ref_map = OA.pv_post_cut(q.float().numpy(), k.float().numpy(), idx, cnt, thr)
    assert ref_map.sum() < 4 * cnt.sum()  # the cut removed blocks
    assert np.array_equal(pv_map.cpu().numpy(), ref_map)
    ref = OA.block_sparse_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), ex_idx, ex_cnt)
    _check(o, ref)


# ------------------------------------------------------------- float16 inputs
@pytest.mark.parametrize("nq,nk,strided", [(1, 1, False), (127, 63, True), (128, 64, False), (129, 65, True),
                                           (333, 700, True)])
def test_half_inputs_equal_their_bf16_casts(nq, nk, strided):
    """float16 q, k, v read by the kernels give, bit for bit, what their bf16
    casts give: the pooled means and the innovation, K and the V tiles, the
    attention (its bf16 result as float16). Values over the whole half range,
    halves that round up to the next bf16, subnormals and infinities among K
    and V's casts."""
    from vasc_amd import ops
    B, H, D = 1, 3, 64
    def half(n, seed):
        t = _rand((B, n, H, D), seed).to(torch.float16).cuda()
        t[:, :, 0, 1::7] = 1.00390625  # between two bf16 values: ties to even
        return t.transpose(1, 2) if strided else t.transpose(1, 2).contiguous()
    q, k, v = half(nq, 50), half(nk, 51), half(nk, 52)
    qc, kc, vc = (t.to(torch.bfloat16) for t in (q, k, v))
    edge = torch.tensor([65504.0, -65504.0, 6.1e-5, 5.96e-8, -5.96e-8, 0.0, -0.0, float("inf")], dtype=torch.float16)
    w = k.clone()
    w[..., :8] = edge.cuda()
    wk, wt = ops.pack_kv_half(w, w)
    assert torch.equal(wk.view(torch.int16), w.to(torch.bfloat16).contiguous().view(torch.int16))
    assert torch.equal(wt.view(torch.int16), ops.pack_v(w.to(torch.bfloat16)).view(torch.int16))
    for a, b in zip(ops.pool_qkv(q, k, v), ops.pool_qkv(qc, kc, vc)):
        assert torch.equal(a, b)
    kb, vt = ops.pack_kv_half(k, v)
    assert torch.equal(kb, kc) and torch.equal(vt, ops.pack_v(vc)) and torch.equal(vt, ops.pack_v(v))
    idx, cnt = (torch.from_numpy(t).cuda() for t in _lists(B, H, math.ceil(nq / 128), math.ceil(nk / 64), 53, 0.6))
    ref = ops.block_sparse_attn(qc, kc, vt, idx, cnt)
    assert torch.equal(ops.block_sparse_attn(q, kb, vt, idx, cnt), ref)
    assert torch.equal(ops.block_sparse_attn(q, kb, vt, idx, cnt, half_out=True), ref.to(torch.float16))


@pytest.mark.parametrize("nq,nk", [(130, 193), (257, 64)])
def test_half_inputs_in_batches(nq, nk):
    """Two batch entries and heads in either order of strides: the float16 pooling,
    packing and attention read every (batch, head) row of strided tensors as they
    read contiguous ones, and as the bf16 kernels read the casts."""
    from vasc_amd import ops
    B, H, D = 2, 3, 64
    q, k, v = (_rand((B, n, H, D), 95 + i).to(torch.float16).cuda().transpose(1, 2) for i, n in enumerate((nq, nk, nk)))
    dense = [t.contiguous() for t in (q, k, v)]
    casts = [t.to(torch.bfloat16) for t in dense]
    for a, b, c in zip(ops.pool_qkv(q, k, v), ops.pool_qkv(*dense), ops.pool_qkv(*casts)):
        assert torch.equal(a, b) and torch.equal(a, c)
    kb, vt = ops.pack_kv_half(k, v)
    assert torch.equal(kb, casts[1]) and torch.equal(vt, ops.pack_v(casts[2]))
    idx, cnt = (torch.from_numpy(t).cuda() for t in _lists(B, H, math.ceil(nq / 128), math.ceil(nk / 64), 96, 0.6))
    ref = ops.block_sparse_attn(casts[0], kb, vt, idx, cnt)
    assert torch.equal(ops.block_sparse_attn(q, kb, vt, idx, cnt, half_out=True), ref.to(torch.float16))
    _check(ref, OA.block_sparse_attention(*(t.float().cpu().numpy() for t in casts), idx.cpu().numpy(), cnt.cpu().numpy()))
