"""Calls recorded into a graph: the first one a context makes, and replays
after later calls have needed larger buffers.  Every replay is compared with
the eager result, with eager work and synchronisations between them.
"""
import pytest
import torch

import mslim_attn

pytestmark = pytest.mark.gpu


def _normal(shape, dtype=torch.bfloat16, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


@pytest.fixture
def fresh():
    c = mslim_attn.Context()
    c.use_torch_stream()
    yield c
    torch.cuda.synchronize()
    c.close()


def _record(c, call):
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    c.set_stream(stream.cuda_stream)
    with torch.cuda.graph(graph, stream=stream):
        call()
    c.use_torch_stream()
    return graph


@pytest.mark.parametrize("tokens", [65, 200, 256, 1000])
@pytest.mark.parametrize("qh,kvh,d", [(32, 8, 128), (3, 1, 64)])
def test_portable_decode_first_call_under_capture(fresh, qh, kvh, d, tokens):
    # Run eagerly these lengths split; a new context has no memory for the
    # partials, so the recorded call runs as one split.  It differs from the
    # eager one in the order of its sums only: eps = 2^-24 per term of a chain
    # of tokens / 16 weighted values below 6, both ways, and 64 merges.
    q = _normal((qh, d), torch.float32)
    k, v = _normal((tokens, kvh, d), torch.float16, 1), _normal((tokens, kvh, d), torch.float16, 2)
    got, want = torch.zeros_like(q), torch.zeros_like(q)
    fmt = mslim_attn.FORMAT_F16
    graph = _record(fresh, lambda: fresh.frames_decode(q, k, fmt, v, fmt, got, tokens, qh, kvh, d))
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        fresh.frames_decode(q, k, fmt, v, fmt, want, tokens, qh, kvh, d)
        assert (got - want).abs().max() <= 6 * 2.0 ** -24 * (2 * tokens / 16 + 64)
    torch.cuda.synchronize()


def _prefill(c, queries, prior, qh, kvh, d):
    assert mslim_attn.prefill_split_tiles(queries, prior, qh, kvh, d) > 0
    q, k, v = _normal((queries, qh, d)), _normal((queries + prior, kvh, d), seed=1), _normal((queries + prior, kvh, d), seed=2)
    return lambda out: c.prefill_causal(q, k, v, out, queries, prior, qh, kvh, d), torch.zeros_like(q)


def _decode(c, lens, qh, kvh, d):
    b, stride = len(lens), max(lens)
    q, k, v = _normal((b, qh, d)), _normal((b, stride, kvh, d), seed=1), _normal((b, stride, kvh, d), seed=2)
    return lambda out: c.decode_dense(q, k, v, out, lens, qh, kvh, d, seq_stride_tokens=stride), torch.zeros_like(q)


def _frames(c, tokens, qh, kvh, d):
    q = _normal((qh, d), torch.float32)
    k, v = _normal((tokens, kvh, d), seed=1), _normal((tokens, kvh, d), seed=2)
    fmt = mslim_attn.FORMAT_BF16
    return lambda out: c.frames_decode(q, k, fmt, v, fmt, out, tokens, qh, kvh, d), torch.zeros_like(q)


def _product(c, inner, rows, tokens):
    w, x = _normal((rows, inner)), _normal((tokens, inner))
    return lambda out: c.gemm_bf16(w, x, out, inner, rows, tokens), torch.zeros_like(x[:, :1]).repeat(1, rows)


def _norm_mlp(c, inner, rows, tokens):
    n, g, u, x = _normal((inner,)), _normal((rows, inner)), _normal((rows, inner), seed=1), _normal((tokens, inner))
    return (lambda out: c.rmsnorm_gemm_swiglu(n, 1e-5, g, u, x, out, inner, rows, tokens),
            torch.zeros_like(x[:, :1]).repeat(1, rows))


def _rope(c, start, tokens):
    x = _normal((tokens, 8, 128))
    return lambda out: c.rope(x, out, tokens, 8, 128, start, 500000.0), torch.zeros_like(x)


# Each: a call, and one that needs more of the same context buffers.
GROWTH = {
    "prefill group 7": (_prefill, (600, 1500, 14, 2, 128), (600, 1500, 56, 8, 128)),
    "prefill group 4": (_prefill, (512, 512, 32, 8, 128), (512, 3584, 32, 8, 128)),
    "decode group 3": (_decode, ([300, 700], 6, 2, 128), ([4000] * 32, 24, 8, 128)),
    "decode group 4": (_decode, ([300, 700], 8, 2, 128), ([4000] * 32, 32, 8, 128)),
    "portable decode": (_frames, (200, 8, 2, 128), (16384, 32, 8, 128)),
    "32-row product": (_product, (4096, 4096, 32), (14336, 4096, 512)),
    "32-row product, more rows": (_product, (4096, 4096, 32), (14336, 12288, 512)),
    "long product": (_product, (14336, 1024, 32), (14336, 12288, 512)),
    "norm and SwiGLU": (_norm_mlp, (1024, 2048, 32), (4096, 2048, 512)),
    "RoPE": (_rope, (0, 32), (60000, 32)),
}


@pytest.mark.parametrize("name", GROWTH)
def test_replay_after_a_larger_call(fresh, name):
    make, small, large = GROWTH[name]
    call, want = make(fresh, *small)
    call(want)
    torch.cuda.synchronize()
    got = torch.zeros_like(want)
    graph = _record(fresh, lambda: call(got))
    big_call, big = make(fresh, *large)
    for _ in range(3):
        big_call(big)
        again = torch.zeros_like(want)
        call(again)  # the eager call now uses the larger buffers
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(again, want)
    big_again = torch.zeros_like(big)
    big_call(big_again)
    torch.cuda.synchronize()
    assert torch.equal(big, big_again)


@pytest.mark.parametrize("inner,rows,tokens", [(4096, 4096, 32), (14336, 4096, 64), (8192, 2048, 300)])
def test_product_first_call_under_capture(fresh, inner, rows, tokens):
    # Run eagerly these split along k; with nothing allocated for the partials
    # the recorded call adds its segments in registers, to the same bits.
    call, want = _product(fresh, inner, rows, tokens)
    got = torch.zeros_like(want)
    graph = _record(fresh, lambda: call(got))
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        call(want)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
