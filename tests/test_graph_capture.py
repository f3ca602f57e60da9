"""The entry points under HIP graph capture (torch.cuda.CUDAGraph), as a serving
loop runs decode: each graph is replayed several times with the program's own
eager work and synchronisations in between, and every replay must equal the
eager call bit for bit.  The captured paths record only kernel launches (no
memset nodes): outputs and split partials come from the caching allocator
uninitialised, and the kernels write every element they read back."""
import numpy as np
import pytest
import torch

import attnkernels as ak
import oracle

pytestmark = pytest.mark.gpu


def _capture(fn):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # warm the allocator off the capture
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _replays_match(fn, replays=4):
    want = fn().clone()
    torch.cuda.synchronize()
    g, out = _capture(fn)
    for i in range(replays):
        out.fill_(float("nan"))  # a replay must rewrite every element
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        junk = torch.randn(1 << 20, device="cuda").sum()  # eager work between replays
        torch.cuda.synchronize()
        del junk


@pytest.mark.parametrize("hq,hkv,part", [(32, 8, None), (16, 16, 256), (64, 8, 1024)])
def test_paged_decode_replays(hq, hkv, part):
    lens = [1, 700, 4096, 2500]
    kc, vc, bt, cl = oracle.make_paged_cache(lens, hkv, 128, block_size=16, extra_blocks=3, seed=3)
    q = np.random.default_rng(4).standard_normal((len(lens), hq, 128), dtype=np.float32).astype(np.float16)
    q, kc, vc, bt, cl = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vc, bt, cl))
    _replays_match(lambda: ak.paged_decode(q, kc, vc, bt, cl, max(lens), partition_size=part))


@pytest.mark.parametrize("d,causal", [(64, False), (128, True)])
def test_flash_attention_replays(d, causal):
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn(2, 4, 1000, d, generator=g, device="cuda", dtype=torch.float16) for _ in range(3))
    _replays_match(lambda: ak.flash_attention(q, k, v, causal=causal))


def test_graphs_in_one_pool_have_split_counters_of_their_own():
    """Three graphs in one memory pool: the first leaves other values where the next
    ones' memory lies, and is replayed between them; the third never relies on the
    second having run."""
    lens = [8000] * 4 + [300] * 12
    kc, vc, bt, cl = oracle.make_paged_cache(lens, 8, 128, block_size=16, extra_blocks=3, seed=3)
    q = np.random.default_rng(4).standard_normal((len(lens), 32, 128), dtype=np.float32).astype(np.float16)
    q, kc, vc, bt, cl = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vc, bt, cl))
    fn = lambda: ak.paged_decode(q, kc, vc, bt, cl, max(lens))  # noqa: E731
    want = fn().clone()
    torch.cuda.synchronize()
    junk, first, second = (torch.cuda.CUDAGraph() for _ in range(3))
    with torch.cuda.graph(junk):
        x = [torch.full((1 << 17,), 0x01010101, dtype=torch.int32, device="cuda") for _ in range(8)]
        del x
    outs = {}
    for g in (first, second):
        with torch.cuda.graph(g, pool=junk.pool()):
            outs[g] = fn()
    for g in (junk, second, first, junk, second, second, first):
        if g in outs:
            outs[g].fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        if g in outs:
            assert torch.equal(outs[g], want)
        assert torch.equal(fn(), want)  # the stream's own counters


def test_calls_after_a_capture_on_their_stream():
    """The first split decode on a stream is recorded, not run: the calls that follow it
    there do not take its counters, which nothing has zeroed yet."""
    lens = [8000] * 4 + [300] * 12
    kc, vc, bt, cl = oracle.make_paged_cache(lens, 8, 128, block_size=16, extra_blocks=3, seed=5)
    q = np.random.default_rng(6).standard_normal((len(lens), 32, 128), dtype=np.float32).astype(np.float16)
    q, kc, vc, bt, cl = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vc, bt, cl))
    fn = lambda: ak.paged_decode(q, kc, vc, bt, cl, max(lens))  # noqa: E731
    want = fn().clone()
    side = torch.cuda.Stream()
    junk, g = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(junk):
        x = [torch.full((1 << 17,), 0x01010101, dtype=torch.int32, device="cuda") for _ in range(8)]
        del x
    with torch.cuda.graph(g, pool=junk.pool(), stream=side):
        out = fn()
    junk.replay()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        assert torch.equal(fn(), want)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
