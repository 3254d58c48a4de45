"""The frames decode that shares K and V over a query-head group, at the edges
of its lane layouts (rows of 8, 16 and 32 lanes, partly used), head chunks and
splits, against the f64 reference (CpuReferenceBackend::decode,
portable.rs:575-646), and against the kernel for unaligned rows.

Bound, eps = 2^-24: a score is a chain of 8 FMAs, up to five lane additions and
two scalings, so its error is at most 15 eps of A = max sum |q k| scale, plus
2 eps of the largest |score| from the log2 units.  A probability moves by that
much relatively, numerator and denominator alike, and each sum adds an eps per
term of its chain (a part's tokens, 16 to 32 parts, 64 splits).
"""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

BF16, F16, F32 = 1, 2, 3


def _encode(x, fmt):
    if fmt == BF16:
        return oracle.write_bf16(x)
    return x.astype(np.float16).view(np.uint16) if fmt == F16 else x


def _decode(x, fmt):
    return oracle.read_bf16(x) if fmt == BF16 else x.view(np.float16).astype(np.float32) if fmt == F16 else x


@pytest.mark.parametrize("tokens", [1, 15, 64, 65, 700])
@pytest.mark.parametrize("qh,kvh,d,kf,vf", [(1, 1, 8, F16, F32), (6, 2, 64, BF16, F16), (4, 4, 72, F32, BF16),
                                            (32, 8, 128, F16, F16), (10, 2, 136, BF16, BF16), (13, 1, 256, F32, F32),
                                            (40, 2, 104, F16, BF16)])
def test_group_kernel(ctx, qh, kvh, d, kf, vf, tokens):
    rng = np.random.default_rng(tokens * 100 + d)
    q = rng.standard_normal(qh * d, dtype=np.float32)
    k = _encode(rng.standard_normal(tokens * kvh * d, dtype=np.float32), kf)
    v = _encode(rng.standard_normal(tokens * kvh * d, dtype=np.float32), vf)
    rc, ref = oracle.cpu_reference_decode_formats(q, k, kf, v, vf, qh, kvh, d)
    assert rc == 0

    def device(x, shift):
        raw = np.ascontiguousarray(x).view(np.uint8).reshape(-1)
        room = torch.zeros(raw.size + 16, dtype=torch.uint8, device="cuda")
        room[shift:shift + raw.size] = torch.from_numpy(raw.copy()).cuda()
        return room[shift:shift + raw.size]

    k64 = _decode(k, kf).reshape(tokens, kvh, d).astype(np.float64)
    q64 = q.reshape(kvh, qh // kvh, d).astype(np.float64)
    scores = np.einsum("hgd,thd->hgt", q64, k64) / np.sqrt(d)
    a = np.einsum("hgd,thd->hgt", np.abs(q64), np.abs(k64)).max() / np.sqrt(d)
    eps, vmax = 2.0 ** -24, np.abs(_decode(v, vf)).max()
    bound = eps * vmax * (2 * (15 * a + 2 * np.abs(scores).max() + 4) + 2 * (tokens / 16 + 32 + 64 + 8))
    for shift in (0, 4):  # 4: rows not 16-byte aligned take the per-head kernel
        outs = []
        for _ in range(2):
            out = torch.full((qh * d + 4,), float("nan"), dtype=torch.float32, device="cuda")[:qh * d]
            ctx.frames_decode(device(q, shift), device(k, shift), kf, device(v, shift), vf, out, tokens, qh, kvh, d)
            torch.cuda.synchronize()
            outs.append(out.cpu().numpy())
        assert np.array_equal(outs[0], outs[1])
        err = np.abs(outs[0].astype(np.float64) - ref).max()
        assert err <= bound, (shift, err, bound)


@pytest.mark.parametrize("qh,kvh,d,tokens", [(2, 1, 8, 2048), (2, 1, 8, 2049), (16, 1, 16, 512), (16, 1, 16, 513)])
def test_rows_of_few_pieces(ctx, qh, kvh, d, tokens):
    # either side of the token count from which they take the group kernel
    test_group_kernel(ctx, qh, kvh, d, F16, BF16, tokens)


def test_group_kernel_ignores_what_follows_the_last_token(ctx):
    # rows past the token count hold infinities: lanes past the last token
    # must not read them into the result
    qh, kvh, d, tokens = 8, 2, 128, 37
    gen = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn((qh, d), generator=gen, device="cuda")
    kv = torch.randn((2, tokens + 64, kvh, d), generator=gen, device="cuda").to(torch.float16)
    clean, out = torch.empty_like(q), torch.empty_like(q)
    ctx.frames_decode(q, kv[0, :tokens].clone(), F16, kv[1, :tokens].clone(), F16, clean, tokens, qh, kvh, d)
    kv[:, tokens:] = float("inf")
    ctx.frames_decode(q, kv[0], F16, kv[1], F16, out, tokens, qh, kvh, d)
    torch.cuda.synchronize()
    assert torch.equal(clean, out) and torch.isfinite(out).all()


@pytest.mark.parametrize("tokens,dead", [(65, [64]), (65, list(range(64))), (300, [0, 5, 130, 299]), (9, [3])])
@pytest.mark.parametrize("qh,kvh,d", [(32, 8, 128), (3, 3, 64), (8, 1, 136)])
def test_keys_at_minus_infinity_weigh_nothing(ctx, qh, kvh, d, tokens, dead):
    # A key whose scores are all -inf has probability zero, also where it is
    # the first or only key that a lane group, a wavefront or a split meets:
    # the output is that of the other keys.  With fewer than 300 keys left,
    # |score| < 16 and |v| < 6, test_group_kernel's bound is below 6e-4.
    gen = torch.Generator(device="cuda").manual_seed(tokens + d)
    q = torch.rand((qh, d), generator=gen, device="cuda") + 0.25
    k, v = (torch.randn((tokens, kvh, d), generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    live = [t for t in range(tokens) if t not in dead]
    k[dead] = -float("inf")
    out = torch.empty_like(q)
    ctx.frames_decode(q, k, BF16, v, BF16, out, tokens, qh, kvh, d)
    group = qh // kvh
    kl, vl = (x[live].double().repeat_interleave(group, dim=1) for x in (k, v))
    p = torch.softmax((kl * q.double()).sum(dim=2) * d ** -0.5, dim=0)
    ref = (p[:, :, None] * vl).sum(dim=0)
    assert (out.double() - ref).abs().max() <= 6e-4
