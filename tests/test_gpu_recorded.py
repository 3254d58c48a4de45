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
