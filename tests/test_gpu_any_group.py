"""The run-time-geometry variants of the attention kernels: any group up to 16
query heads per kv head and any head_dim up to 128, against the f64 reference
(CpuReferenceBackend::decode, portable.rs:575-646).

Bound per output: half a BF16 step of the value (2^-8 |ref|), plus 2^-13 of
the largest |v|: probabilities enter P.V as two BF16 parts (relative error
2^-17 of each, and of their sum), scores are f32 sums of exact BF16 products
(for |score| < 32 an error below 2^-15, so p moves by less than 2^-14).  One
BF16 part per probability (2^-9) does not fit it.
"""
import numpy as np
import pytest
import torch

import mslim_attn
import oracle
from _data import from_torch, normal_bf16, to_torch

pytestmark = pytest.mark.gpu


def _check(got_bits, ref, v_bits, label):
    got = oracle.read_bf16(np.asarray(got_bits, np.uint16).reshape(-1)).astype(np.float64)
    ref = np.asarray(ref, np.float64).reshape(-1)
    bound = np.abs(ref) * 2.0 ** -8 + np.abs(oracle.read_bf16(v_bits.reshape(-1))).max() * 2.0 ** -13
    over = np.abs(got - ref) > bound
    assert not over.any(), (label, int(over.sum()), float((np.abs(got - ref) / bound).max()))


def _unaligned(t):
    """The same values two bytes past a 16-byte boundary."""
    room = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    room[1:].copy_(t.reshape(-1))
    return room[1:].view(t.shape)


# (q heads, kv heads, head_dim): groups without a variant of their own, the
# largest and smallest head_dim of both run-time variants and odd pieces of 8.
DECODE = [(3, 1, 128), (10, 2, 128), (36, 3, 120), (16, 1, 72), (15, 1, 64), (12, 4, 64), (7, 7, 40), (6, 2, 8)]


@pytest.mark.parametrize("qh,kvh,d", DECODE)
def test_decode_any_group(ctx, qh, kvh, d):
    rng = np.random.default_rng(qh * 1000 + d)
    lens = [1, 15, 33, 64, 257, 1025]
    b, stride = len(lens), max(lens)
    qb, kb, vb = (normal_bf16(rng, s) for s in ((b, qh, d), (b, stride, kvh, d), (b, stride, kvh, d)))
    q, k, v = to_torch(qb), to_torch(kb), to_torch(vb)
    pages = [-(-t // 16) for t in lens]
    table = np.zeros((b, max(pages)), np.int32)
    order = rng.permutation(sum(pages)).astype(np.int32)
    for i, n in enumerate(pages):
        table[i, :n] = order[sum(pages[:i]):sum(pages[:i]) + n]
    table = torch.from_numpy(table).cuda()
    k_pool = torch.zeros((sum(pages), kvh, 16, d), dtype=torch.int16, device="cuda")
    v_pool = torch.zeros_like(k_pool)
    for i, t in enumerate(lens):
        ctx.pages_write(k_pool, v_pool, table[i], 16, kvh, d, 0, t, k[i, :t].contiguous(), v[i, :t].contiguous())
    ref = [oracle.cpu_reference_decode(oracle.read_bf16(qb[i]), kb[i, :t], vb[i, :t], 1, qh, kvh, d)[1]
           for i, t in enumerate(lens)]
    for split in (0, 64):
        dense, paged, noalloc, plain = (torch.empty_like(q) for _ in range(4))
        ctx.decode_dense(q, k, v, dense, lens, qh, kvh, d, seq_stride_tokens=stride, split_tokens=split)
        ctx.decode_paged(q, k_pool, v_pool, paged, lens, table, max(pages), 16, qh, kvh, d, split_tokens=split)
        ctx.decode_paged_noalloc(q, k_pool, v_pool, noalloc, lens, table, max(pages), 16, qh, kvh, d,
                                 split_tokens=split)
        # unaligned queries take the any-geometry kernel
        ctx.decode_dense(_unaligned(q), k, v, plain, lens, qh, kvh, d, seq_stride_tokens=stride, split_tokens=split)
        torch.cuda.synchronize()
        assert torch.equal(dense, paged) and torch.equal(dense, noalloc)
        for i in range(b):
            _check(from_torch(dense[i]), ref[i], vb[i], f"split {split} sequence {i}")
            _check(from_torch(plain[i]), ref[i], vb[i], f"unaligned, split {split} sequence {i}")


# (queries, prior): one row, tile and row-block edges, a remainder after a
# prior, and lengths whose launches split their row blocks.
PREFILL = [(1, 0), (33, 0), (257, 130), (600, 1500)]


@pytest.mark.parametrize("queries,prior", PREFILL)
@pytest.mark.parametrize("qh,kvh,d", [(3, 1, 128), (10, 2, 64), (6, 1, 128), (18, 3, 64), (14, 2, 128)])
def test_prefill_any_group(ctx, qh, kvh, d, queries, prior):
    rng = np.random.default_rng(queries * 100 + qh)
    t = queries + prior
    qb, kb, vb = (normal_bf16(rng, s) for s in ((queries, qh, d), (t, kvh, d), (t, kvh, d)))
    _check_prefill(ctx, rng, qb, kb, vb, queries, prior, qh, kvh, d)


@pytest.mark.parametrize("qh,kvh,d", [(3, 1, 128), (6, 1, 64)])
def test_prefill_any_group_moving_reference(ctx, qh, kvh, d):
    # scores that climb past the lazy bound tile after tile, then one so far
    # above the reference that its first p overflows
    rng = np.random.default_rng(d)
    queries = 400
    k = 0.4 * (128.0 / d) ** 0.5 * np.arange(queries, dtype=np.float32) / 64.0
    k[330] = 20.0 * (128.0 / d) ** 0.5
    qb = oracle.write_bf16(np.ones((queries, qh, d), np.float32)).reshape(queries, qh, d)
    kb = oracle.write_bf16(np.broadcast_to(k[:, None, None], (queries, kvh, d))).reshape(queries, kvh, d)
    _check_prefill(ctx, rng, qb, kb, normal_bf16(rng, (queries, kvh, d)), queries, 0, qh, kvh, d)


def _check_prefill(ctx, rng, qb, kb, vb, queries, prior, qh, kvh, d):
    q, k, v = to_torch(qb), to_torch(kb), to_torch(vb)
    whole, unsplit, plain = (torch.empty_like(q) for _ in range(3))
    ctx.prefill_causal(q, k, v, whole, queries, prior, qh, kvh, d)
    try:
        ctx.set_prefill_split(False)
        ctx.prefill_causal(q, k, v, unsplit, queries, prior, qh, kvh, d)
    finally:
        ctx.set_prefill_split(True)
    ctx.prefill_causal(_unaligned(q), k, v, plain, queries, prior, qh, kvh, d)  # the any-geometry kernel
    torch.cuda.synchronize()
    rows = sorted({0, queries // 2, queries - 1} | {int(r) for r in rng.integers(0, queries, 12)})
    outs = [from_torch(x) for x in (whole, unsplit, plain)]
    for r in rows:
        n = prior + r + 1
        ref = oracle.cpu_reference_decode(oracle.read_bf16(qb[r]), kb[:n], vb[:n], 1, qh, kvh, d)[1]
        for name, got in zip(("split", "unsplit", "unaligned"), outs):
            _check(got[r], ref, vb[:n], f"{name} row {r}")


def test_prefill_first_call_under_capture():
    # A shape that splits when run eagerly: a new context has no memory for the
    # partials and can allocate none during capture, so it runs unsplit there.
    queries, prior, qh, kvh, d = 600, 1500, 14, 2, 128
    assert mslim_attn.prefill_split_tiles(queries, prior, qh, kvh, d) > 0
    rng = np.random.default_rng(11)
    q, k, v = (to_torch(normal_bf16(rng, s)) for s in ((queries, qh, d), (queries + prior, kvh, d),
                                                       (queries + prior, kvh, d)))
    got, want = torch.zeros_like(q), torch.zeros_like(q)
    fresh = mslim_attn.Context()
    try:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        fresh.set_stream(stream.cuda_stream)
        with torch.cuda.graph(graph, stream=stream):
            fresh.prefill_causal(q, k, v, got, queries, prior, qh, kvh, d)
        fresh.use_torch_stream()
        fresh.set_prefill_split(False)
        fresh.prefill_causal(q, k, v, want, queries, prior, qh, kvh, d)
        torch.cuda.synchronize()
        for _ in range(3):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)
            fresh.prefill_causal(q, k, v, want, queries, prior, qh, kvh, d)
        torch.cuda.synchronize()
        del graph
    finally:
        fresh.close()


def _attend64(q, k, v, group):
    """q [n][qh][d] attends k, v [t][kvh][d], causal at the end, in float64.
    A key whose score is -inf weighs nothing."""
    n, t = q.shape[0], k.shape[0]
    kl, vl = (x.double().repeat_interleave(group, dim=1) for x in (k, v))
    score = torch.einsum("nhd,thd->nht", q.double().cpu(), kl.cpu()) * q.shape[2] ** -0.5
    seen = torch.arange(t)[None, :] <= torch.arange(n)[:, None] + (t - n)
    score.masked_fill_(~seen[:, None, :], -float("inf"))
    p = torch.softmax(score, dim=2)
    out = torch.zeros(q.shape, dtype=torch.float64)
    for i in range(n):  # only the keys that the row sees and weighs
        for h in range(q.shape[1]):
            keys = (p[i, h] > 0).nonzero()[:, 0]
            out[i, h] = (p[i, h, keys, None] * vl[keys, h].cpu()).sum(dim=0) if len(keys) else float("nan")
    return out


def _check64(got, ref, label):
    # the bound above with |v| < 6, where the reference is finite; elsewhere
    # the same infinity or NaN
    got, finite = got.double().cpu(), torch.isfinite(ref)
    assert torch.equal(torch.nan_to_num(got[~finite], nan=7.0), torch.nan_to_num(ref[~finite], nan=7.0)), label
    over = (got - ref).abs()[finite] > ref.abs()[finite] * 2.0 ** -8 + 6 * 2.0 ** -13
    assert not over.any(), (label, int(over.sum()))


@pytest.mark.parametrize("qh,kvh,d", [(3, 1, 128), (10, 2, 72), (12, 4, 64)])
@pytest.mark.parametrize("t,values,dead", [(33, [32], []), (300, [0, 150], []), (257, [256], [255]), (33, [], [32]),
                                           (300, [7], list(range(64, 128)))])
def test_decode_any_group_values_that_are_not_finite(ctx, qh, kvh, d, t, values, dead):
    # values: tokens whose V row holds +Inf, -Inf and NaN in three dimensions;
    # dead: keys at -inf, alone in a wavefront's tile or filling a partition.
    # Rows past the sequence hold NaN and must not be read into the result.
    gen = torch.Generator(device="cuda").manual_seed(t + d)
    q = (torch.rand((1, qh, d), generator=gen, device="cuda") + 0.25).to(torch.bfloat16)
    k, v = (torch.randn((t + 64, kvh, d), generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    k[dead] = -float("inf")
    for i in values:
        v[i, :, 3], v[i, :, 17], v[i, :, d - 1] = float("inf"), -float("inf"), float("nan")
    k[t:], v[t:] = float("nan"), float("nan")
    ref = _attend64(q, k[:t], v[:t], qh // kvh)
    for split in (0, 64):
        out = torch.empty_like(q)
        ctx.decode_dense(q, k, v, out, [t], qh, kvh, d, seq_stride_tokens=t + 64, split_tokens=split)
        _check64(out, ref, f"split {split}")


@pytest.mark.parametrize("qh,kvh,d", [(3, 1, 128), (10, 2, 64), (14, 2, 128)])
@pytest.mark.parametrize("queries,prior,values,dead", [(90, 0, [40, 89], []), (300, 0, [130, 299], [64]),
                                                       (64, 1500, [1530], [1500]), (65, 0, [], [0, 64])])
def test_prefill_any_group_values_that_are_not_finite(ctx, qh, kvh, d, queries, prior, values, dead):
    # An infinity or NaN of V reaches the rows that see its key, in its own
    # dimension, and no earlier row; a key at -inf weighs nothing.
    gen = torch.Generator(device="cuda").manual_seed(queries + d)
    t = queries + prior
    q = (torch.rand((queries, qh, d), generator=gen, device="cuda") + 0.25).to(torch.bfloat16)
    k, v = (torch.randn((t, kvh, d), generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    k[dead] = -float("inf")
    for i in values:
        v[i, :, 3], v[i, :, 17], v[i, :, d - 1] = float("inf"), -float("inf"), float("nan")
    ref = _attend64(q, k, v, qh // kvh)
    split, unsplit = torch.empty_like(q), torch.empty_like(q)
    ctx.prefill_causal(q, k, v, split, queries, prior, qh, kvh, d)
    try:
        ctx.set_prefill_split(False)
        ctx.prefill_causal(q, k, v, unsplit, queries, prior, qh, kvh, d)
    finally:
        ctx.set_prefill_split(True)
    _check64(split, ref, "split")
    _check64(unsplit, ref, "unsplit")
