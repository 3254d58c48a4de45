"""The tiled projection kernel at the edges of its tiles, k splits and shapes:
every configuration (64 x 64 to 128 x 256 outputs), split and unsplit, with
partial tiles on both sides, against a float64 product, and its fused forms
against the plain one, bit for bit.

Bound per output of the float64 comparison: half a BF16 step (2^-8 |ref|) plus
the f32 accumulation, 2^-24 per step of a chain of inner / 16 MFMA results on
a running sum no larger than sum |x w|.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (inner, rows of Q, rows of K and V, tokens): one k-step; 64 x 64 tiles split
# and not; one past a tile in either direction; 64 x 128, 128 x 128 and
# 128 x 256 tiles; a long inner dimension with a split per product.
SHAPES = [(64, 17, 5, 17), (4096, 4100, 1000, 20), (4096, 15000, 70, 64), (4096, 4160, 1024, 65),
          (2048, 2048, 513, 128), (4096, 4096, 129, 129), (4096, 4096, 1024, 257), (1024, 7000, 300, 512),
          (4096, 14336, 64, 300), (14336, 4096, 512, 20), (14336, 4097, 200, 130), (8192, 1030, 1030, 511)]


@pytest.mark.parametrize("inner,rows,kv_rows,tokens", SHAPES)
def test_projection_tiles(ctx, inner, rows, kv_rows, tokens):
    gen = torch.Generator(device="cuda").manual_seed(inner + rows + tokens)

    def normal(shape, scale):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(torch.bfloat16)

    def out(n):
        return torch.full((tokens, n), float("nan"), dtype=torch.bfloat16, device="cuda")

    x, wq = normal((tokens, inner), 1.0), normal((rows, inner), 0.02)
    wk, wv = normal((kv_rows, inner), 0.02), normal((kv_rows, inner), 0.02)
    y, q, k, v, k1, v1 = out(rows), out(rows), out(kv_rows), out(kv_rows), out(kv_rows), out(kv_rows)
    ctx.gemm_bf16(wq, x, y, inner, rows, tokens)
    ctx.gemm_bf16(wk, x, k1, inner, kv_rows, tokens)
    ctx.gemm_bf16(wv, x, v1, inner, kv_rows, tokens)
    ctx.gemm_qkv(wq, wk, wv, x, q, k, v, inner, rows, kv_rows, tokens)
    for w, got in ((wq, y), (wk, k1), (wv, v1)):
        ref = x.double() @ w.double().t().contiguous()
        magnitude = x.double().abs() @ w.double().abs().t().contiguous()
        bound = ref.abs() * 2.0 ** -8 + magnitude * (inner / 16 * 2.0 ** -24)
        over = ~((got.double() - ref).abs() <= bound)
        assert not over.any(), (int(over.sum()), over.nonzero()[0].tolist())

    def same(a, b):
        return torch.equal(a.view(torch.int16), b.view(torch.int16))

    assert same(q, y) and same(k, k1) and same(v, v1)
    resid, add, fused = normal((tokens, rows), 1.0), out(rows), normal((tokens, rows), 1.0)
    ctx.add(resid, y, add, tokens * rows)
    fused.copy_(resid)
    ctx.gemm_bf16_add(wq, x, fused, fused, inner, rows, tokens)  # in place
    assert same(fused, add)
    up, act, swiglu = out(kv_rows), out(kv_rows), out(kv_rows)
    ctx.gemm_bf16(wv, x, up, inner, kv_rows, tokens)
    ctx.swiglu(k1, up, act, tokens * kv_rows)
    ctx.gemm_swiglu(wk, wv, x, swiglu, inner, kv_rows, tokens)
    assert same(swiglu, act)


# (inner, rows of Q, rows of K and V): one, two, four and eight k segments, and
# K and V with other counts than their Q.
@pytest.mark.parametrize("inner,rows,kv_rows", [(4096, 4096, 1024), (14336, 4096, 4096), (8192, 2048, 512),
                                                (2048, 9000, 2048), (1024, 4096, 256), (8192, 8192, 1024)])
def test_a_rows_bits_do_not_depend_on_its_launch(ctx, inner, rows, kv_rows):
    # every row count of more than 16 gives a token row the bits it has among
    # 512 rows, in the plain, residual, SwiGLU and Q-K-V products
    gen = torch.Generator(device="cuda").manual_seed(inner + rows)

    def normal(shape, scale):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(torch.bfloat16)

    x, wq, wk, wv = (normal(s, c) for s, c in (((512, inner), 1.0), ((rows, inner), 0.02), ((kv_rows, inner), 0.02),
                                               ((kv_rows, inner), 0.02)))

    def products(t):
        plain, add, swiglu, q, k, v = (torch.full((t, n), float("nan"), dtype=torch.bfloat16, device="cuda")
                                       for n in (rows, rows, kv_rows, rows, kv_rows, kv_rows))
        ctx.gemm_bf16(wq, x, plain, inner, rows, t)
        ctx.gemm_bf16_add(wq, x, plain, add, inner, rows, t)
        ctx.gemm_swiglu(wk, wv, x, swiglu, inner, kv_rows, t)
        ctx.gemm_qkv(wq, wk, wv, x, q, k, v, inner, rows, kv_rows, t)
        return [y.view(torch.int16) for y in (plain, add, swiglu, q, k, v)]

    want = products(512)
    for t in (17, 32, 64, 65, 100, 120, 128, 129, 200, 250, 256, 257, 300, 400, 511):
        for got, ref in zip(products(t), want):
            assert torch.equal(got, ref[:t]), t
