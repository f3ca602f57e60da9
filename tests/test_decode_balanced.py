"""Decode with splits cut evenly over the batch (no partition given): every
kernel, at the edges of the cut, against the oracle; the counters are back at
zero after each call (the next one, with other lengths, would merge too early)."""
import ctypes

import numpy as np
import pytest
import torch

import attnkernels as ak
import oracle
from conftest import PKG_DIR, TOL, max_err

pytestmark = pytest.mark.gpu

BATCHES = {
    "edges": [1, 255, 256, 257, 1279, 1280, 1281, 2048],
    "skewed": [20000] + [3] * 15,
    "full": [1100 + 7 * i for i in range(64)],       # the most sequences, a lane each
    "few": [1, 4099, 2, 5000, 1, 1, 300, 17, 1],
    "one long": [40000] + [30] * 7,                  # as many splits as one workgroup merges
    "empty": [0, 1500, 0, 2049, 0],                  # outside the >= 1 contract: zero rows
}
LONGEST = 1 << 16  # max_context_len given, so that even the small batches are cut by the kernel


def workers(batch, hq, hkv, d, longest):
    """Workgroups per kv head of a balanced launch for these sizes, 0: fixed splits serve them."""
    size = ctypes.CDLL(str(PKG_DIR / "attnkernels" / "libattnkernels.so")).ak_paged_decode_balanced_workspace_size
    size.argtypes, size.restype = [ctypes.c_int64] * 6, ctypes.c_size_t
    return size(batch, hq, hkv, d, longest, ak.decode_partition(batch, hkv, longest)) // (hq * (d + 2) * 4)


@pytest.mark.parametrize("name", BATCHES)
@pytest.mark.parametrize("g,hkv,d,bs", [(1, 4, 128, 16), (1, 2, 64, 8), (2, 2, 128, 16), (4, 8, 128, 16),
                                        (4, 2, 64, 32), (8, 4, 128, 16), (8, 2, 64, 12), (8, 2, 128, 64), (4, 2, 128, 256)])
def test_matches_oracle(name, g, hkv, d, bs):
    check_against_oracle(BATCHES[name], g, hkv, d, bs)


@pytest.mark.parametrize("g,hkv,d,bs", [(1, 16, 128, 16), (1, 8, 64, 16), (2, 8, 128, 32), (4, 8, 128, 16), (8, 4, 128, 16),
                                        (8, 8, 64, 16)])
def test_two_sequences(g, hkv, d, bs):
    """Enough kv heads that two sequences have no more than 32 workgroups each."""
    check_against_oracle([1, 4099], g, hkv, d, bs)


def check_against_oracle(lens, g, hkv, d, bs):
    assert workers(len(lens), g * hkv, hkv, d, LONGEST) >= len(lens)
    kc, vc, bt, cl = oracle.make_paged_cache([max(1, n) for n in lens], hkv, d, block_size=bs, extra_blocks=3, seed=g)
    cl[:] = lens
    q = np.random.default_rng(g + d).standard_normal((len(lens), g * hkv, d), dtype=np.float32).astype(np.float16)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vc, bt, cl)]
    rows = [b for b, n in enumerate(lens) if n > 0]
    ref = np.zeros(q.shape, np.float32)
    ref[rows] = oracle.paged_decode_fp32(q[rows], kc, vc, bt[rows], cl[rows])
    for _ in range(2):
        assert max_err(ak.paged_decode(*dev, LONGEST), ref) < TOL[d]
    # other lengths right after, on the same counters
    dev[4] = torch.clamp(dev[4] // 2, min=1)
    short = cl // 2
    short[short < 1] = 1
    assert max_err(ak.paged_decode(*dev, LONGEST), oracle.paged_decode_fp32(q, kc, vc, bt, short)) < TOL[d]


@pytest.mark.parametrize("g,hkv,d", [(1, 16, 128), (1, 8, 64), (2, 8, 128), (8, 8, 64)])
def test_longest_first(g, hkv, d):
    """More workgroups than one round, lengths in all four classes, at their edges and empty."""
    lens = [0, 1, 4096, 1024, 1023, 1025, 2048, 2049, 3072, 3071] + [1 + 37 * i * i % 4096 for i in range(38)]
    assert workers(len(lens), g * hkv, hkv, d, 8192) * hkv > 512  # past it the longest run first
    kc, vc, bt, cl = oracle.make_paged_cache([max(1, n) for n in lens], hkv, d, block_size=16, extra_blocks=3, seed=d)
    cl[0] = 0
    q = np.random.default_rng(g + d).standard_normal((len(lens), g * hkv, d), dtype=np.float32).astype(np.float16)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vc, bt, cl)]
    ref = np.zeros(q.shape, np.float32)
    ref[1:] = oracle.paged_decode_fp32(q[1:], kc, vc, bt[1:], cl[1:])
    for _ in range(2):
        assert max_err(ak.paged_decode(*dev, 8192), ref) < TOL[d]


@pytest.mark.parametrize("g,d", [(4, 128), (8, 128), (2, 64)])
@pytest.mark.parametrize("shortest", [1792, 1791])  # within an eighth of the longest: whole; a token less: cut
def test_about_equal_sequences(g, d, shortest):
    lens = [2048, shortest] + [1800 + 13 * i % 249 for i in range(62)]
    assert workers(64, g * 8, 8, d, 2048) > 64 and 64 * 8 % 512 == 0  # whole rounds of sequences times kv heads
    kc, vc, bt, cl = oracle.make_paged_cache(lens, 8, d, block_size=16, extra_blocks=3, seed=d)
    q = np.random.default_rng(g + d).standard_normal((len(lens), g * 8, d), dtype=np.float32).astype(np.float16)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vc, bt, cl)]
    ref = oracle.paged_decode_fp32(q, kc, vc, bt, cl)
    for _ in range(2):
        assert max_err(ak.paged_decode(*dev, 2048), ref) < TOL[d]


def test_tokens_past_the_longest_context_given_are_cut_as_with_fixed_splits():
    """A length above max_context_len (outside the contract) reads up to the end of the last fixed split."""
    kc, vc, bt, cl = oracle.make_paged_cache([20000, 300], 4, 128, block_size=16, extra_blocks=1, seed=1)
    q = np.random.default_rng(2).standard_normal((2, 8, 128), dtype=np.float32).astype(np.float16)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vc, bt, cl)]
    part = ak.decode_partition(2, 4, 16500)
    assert workers(2, 8, 4, 128, 16500) > 0
    a = ak.paged_decode(*dev, 16500)
    b = ak.paged_decode(*dev, 16500, partition_size=part)
    assert max_err(a, b.float().cpu().numpy()) < 1e-3
