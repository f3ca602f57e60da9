"""The cut of a batch's contexts into splits that the decode kernels make when
no partition is given (balanced_segment in decode.hip), replayed lane by lane in
float32 and int32, and the rule that picks that path (decode_balanced_plan).

Every split must hold a token, the splits of a sequence must tile its context,
and no kv head may need more splits than the launch has workgroups: a split
that is never run, or that holds nothing and so never arrives at the merge,
would leave its sequence without an output."""
import ctypes

import numpy as np
import pytest

from conftest import PKG_DIR

F = np.float32
MIN_SPLIT, MAX_BATCH = 256, 64


def rcp(x, ulp):
    """1 / x as a hardware reciprocal may return it: off by one unit in the last place."""
    r = F(1) / F(x)
    return np.nextafter(r, F(np.inf if ulp > 0 else -np.inf)) if ulp else r


def split_count(c, size, reciprocal):
    n = (c.astype(F) * reciprocal).astype(np.int64)
    r = c - n * size
    return n + (r > 0) + (r > size) - (r <= -size)


def rounded_up_count(c, size, reciprocal):
    """The planted mistake: a float ceiling with no correction."""
    return np.ceil(c.astype(F) * reciprocal).astype(np.int64)


def cut(lens, workers, cap, gran, ulp=0, most=96, equal_uncut=False, count_splits=split_count):
    c = np.minimum(np.maximum(np.asarray(lens, np.int64), 0), cap)
    if equal_uncut and (c * 8 >= c.max() * 7).all():
        return [(b, 0, 1, 0, int(n)) for b, n in enumerate(c)], len(lens), max(MIN_SPLIT, int(c.max()))

    def up(x):
        return (int(x) + gran - 1) // gran * gran

    size = max(MIN_SPLIT, up(1 + int(F(c.sum() - 1) * rcp(workers, ulp))), up(-(-int(c.max()) // most)))
    for it in range(9):
        n = np.maximum(1, count_splits(c, size, rcp(size, ulp)))
        count = int(n.sum())
        if count <= workers:
            break
        if it == 0:
            more = int(F(c.sum()) * rcp(max(1, workers - len(lens) // 2), ulp))
        else:
            more = size + int(F(size) * F(count - workers) * rcp(workers, ulp))
        size = up(max(size, more) + 1) if it < 6 else up(cap)
    segs = []
    for b, (ctx, ns) in enumerate(zip(c, n)):
        length = up((ctx + ns - 1) // ns)
        segs += [(b, s, int(ns), s * length, min(int(ctx), (s + 1) * length)) for s in range(ns)]
    return segs, count, size


def batches():
    rng = np.random.default_rng(0)
    yield [0, 1, 256, 257, 1025]
    yield [1025] * MAX_BATCH
    yield [32768] + [1] * 31
    yield [0] * 7 + [5000]
    yield [(1 << 24) - 257, 1]
    yield [14697473] + [1] * 15
    for _ in range(400):
        batch, high = int(rng.integers(2, MAX_BATCH + 1)), int(2 ** rng.uniform(10, 17))
        yield rng.integers(0 if rng.random() < 0.3 else 1, high + 1, batch).tolist()


@pytest.mark.parametrize("gran", [32, 64, 128])  # 32 and 64 in the kernels
@pytest.mark.parametrize("ulp", [-1, 0, 1])
def test_every_token_is_in_one_split(gran, ulp):
    for lens in batches():
        cap = -(-max(lens) // 256) * 256
        for workers in (len(lens), len(lens) + 1, 2 * len(lens), 300, 512):
            segs, count, size = cut(lens, workers, cap, gran, ulp)
            assert count <= workers and size % gran == 0, (lens, workers)
            assert tiles(lens, segs), (lens, workers)


def tiles(lens, segs):
    """Whether the splits tile every context, and each holds a token (or its sequence none)."""
    at = {}
    for b, s, ns, start, end in segs:
        if start != at.get(b, 0) or (end <= start and lens[b] > 0):
            return False
        at[b] = end
    return [at[b] for b in range(len(lens))] == list(lens)


def test_about_equal_sequences_stay_whole_where_the_launch_says_so():
    for lens, whole in (([2048, 1792] + [1900] * 62, True), ([2048, 1791] + [1900] * 62, False), ([0] * 64, True),
                        ([0] + [5] * 63, False), ([4096] * 32, True)):
        segs, count, _ = cut(lens, 2 * len(lens), 4096, 32, equal_uncut=True)
        assert tiles(lens, segs) and count <= 2 * len(lens)
        assert (all(ns == 1 for _, _, ns, _, _ in segs) and count == len(lens)) == (whole or max(lens) <= MIN_SPLIT)


@pytest.mark.parametrize("most", [96, 256])  # grouped-query heads, one head
@pytest.mark.parametrize("gran", [32, 64])
def test_no_sequence_has_more_splits_than_one_workgroup_merges(gran, most):
    """One long sequence among short ones may take nearly every workgroup of a kv head."""
    skewed = [([100000] + [500] * 7, 256), ([32768] + [500] * 7, 256), ([100000] + [500] * 15, 128),
              ([100000] + [500] * 63, 512), ([32768] + [500] * 63, 1024), ([100000, 90000] + [1] * 14, 512)]
    for lens, workers in [*skewed, *((b, 32 * len(b)) for b in batches())]:
        segs, count, _ = cut(lens, workers, -(-max(lens) // 256) * 256, gran, most=most)
        assert count <= workers and max(ns for _, _, ns, _, _ in segs) <= most, (lens, workers)
    assert max(ns for _, _, ns, _, _ in cut(skewed[0][0], 256, 100352, gran, most=1 << 24)[0]) > 200


@pytest.mark.parametrize("ulp", [-1, 0, 1])
def test_longest_first_order_is_a_permutation(ulp):
    """The workgroups of the sequences, in classes by the quarters of the longest split: no gap, no overlap."""
    for lens in batches():
        c, n = np.asarray(lens, np.int64), None
        segs, count, _ = cut(lens, 2 * len(lens), -(-max(lens) // 256) * 256, 128, ulp)
        n = np.array([sum(1 for s in segs if s[0] == b) for b in range(len(lens))])
        length = c.astype(F) * np.array([rcp(x, ulp) for x in n])
        quarter = np.minimum(3, (F(4) * length * rcp(max(length.max(), F(1)), ulp)).astype(np.int64))
        first, before = np.zeros(len(lens), np.int64), 0
        for k in (3, 2, 1, 0):
            nk = np.where(quarter == k, n, 0)
            first = np.where(quarter == k, before + nk.cumsum() - nk, first)
            before += nk.sum()
        assert sorted(int(f) + i for f, m in zip(first, n) for i in range(m)) == list(range(count))
        assert all(length[a] >= length[b] or quarter[a] == quarter[b]
                   for a in range(len(lens)) for b in range(len(lens)) if first[a] < first[b])


def test_even_batches_are_cut_evenly():
    for batch, workers, ctx in ((16, 32, 8192), (8, 32, 8192), (4, 64, 30000), (10, 32, 22420)):
        segs, _, _ = cut([ctx] * batch, workers, ctx + 255, 128)
        assert len(segs) == workers // batch * batch
        assert max(e - s for _, _, _, s, e in segs) <= ctx // (workers // batch) + 128


def test_a_cut_that_rounds_up_its_count_is_caught():
    """With a float ceiling alone 2 * size tokens can count as 3 splits, one of them empty."""
    lens = [2 * MIN_SPLIT] * 2
    assert tiles(lens, cut(lens, 8, 512, 128, ulp=1)[0])
    assert not tiles(lens, cut(lens, 8, 512, 128, ulp=1, count_splits=rounded_up_count)[0])


@pytest.fixture(scope="module")
def lib():
    L = ctypes.CDLL(str(PKG_DIR / "attnkernels" / "libattnkernels.so"))
    vp, i64, f64 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_double
    L.ak_last_error.restype = ctypes.c_char_p
    L.ak_paged_decode_balanced_workspace_size.argtypes = [i64] * 6
    L.ak_paged_decode_balanced_workspace_size.restype = ctypes.c_size_t
    L.ak_paged_decode_balanced.argtypes = [vp] * 6 + [i64] * 8 + [f64, i64, vp, ctypes.c_size_t, vp, i64, vp]
    return L


def workers(lib, batch, hq, hkv, d, max_ctx, partition=1024):
    size = lib.ak_paged_decode_balanced_workspace_size(batch, hq, hkv, d, max_ctx, partition)
    assert size % (hq * (d + 2) * 4) == 0
    return size // (hq * (d + 2) * 4)


def test_rule(lib):
    # fixed splits: one sequence, more than 64, short contexts, little K and V, lengths past 2^24, invalid sizes
    for args in ((1, 32, 8, 128, 8192), (65, 32, 8, 128, 8192), (16, 32, 8, 128, 1024), (16, 32, 8, 128, 1 << 24), (3, 16, 4, 128, 8100),
                 (16, 32, 0, 128, 8192), (16, 30, 8, 128, 8192), (0, 32, 8, 128, 8192)):
        assert workers(lib, *args) == 0, args
    assert workers(lib, 16, 32, 8, 128, 8192, 0) == 0
    # every sequence has a workgroup, and whole rounds of 256 CUs (512 slots for one head at D = 128) of them
    for batch in (2, 3, 16, 33, 64):
        for hq, hkv in ((32, 32), (32, 8), (64, 8), (4, 4), (40, 5), (600, 600)):
            for d in (64, 128):
                for ctx in (1025, 8192, 8193, 100000):
                    w = workers(lib, batch, hq, hkv, d, ctx)
                    if batch * hkv * ctx * d * 4 < 64 << 20:
                        assert w == 0
                        continue
                    if batch * 32 * hkv < (512 if hq == hkv and d == 128 else 256):  # more splits than the decode kernel merges
                        assert w == 0
                        continue
                    if w == 0:  # no room to cut in one round: about one workgroup per sequence
                        assert hq == hkv and d == 128 and ctx <= 8192 and batch * hkv <= 512
                        continue
                    assert w >= batch + (batch // 2 if ctx > 8192 else 0) and w <= 65535
                    unit = 512 if hq == hkv and d == 128 else 256
                    assert w * hkv % unit > unit - hkv or w * hkv % unit == 0
    assert workers(lib, 2, 8, 1, 128, 100000) == 0 and workers(lib, 8, 8, 1, 128, 100000) == 256
    assert workers(lib, 8, 64, 8, 128, 8192) == 32 and workers(lib, 12, 64, 8, 128, 8192) == 64
    assert workers(lib, 16, 32, 8, 128, 8192) == 32 and workers(lib, 16, 32, 32, 128, 8192) == 0 and workers(lib, 8, 32, 32, 128, 8192) == 16


@pytest.mark.parametrize("batch,hq,hkv,d,max_ctx,per_cu", [
    # the first size that equal sequences keep three quarters busy, cut or whole
    (16, 32, 8, 128, 8192, 1), (22, 32, 8, 128, 4096, 3), (33, 64, 8, 128, 4096, 4), (40, 32, 8, 128, 4096, 3),
    (52, 64, 8, 128, 3000, 3), (56, 64, 8, 128, 2048, 3), (57, 64, 8, 128, 2048, 4), (64, 32, 8, 128, 4096, 4),
    # a lone long sequence, and just not
    (16, 8, 8, 64, 32768, 2), (16, 8, 8, 64, 32767, 1), (8, 128, 32, 128, 16384, 4), (8, 128, 32, 128, 16383, 2),
    (7, 128, 32, 128, 100000, 2),
    # one head at D = 128: from two, the best filled size, fewer for short contexts, fixed when nearly full
    (12, 8, 8, 128, 4096, 2), (22, 8, 8, 128, 4096, 3), (24, 8, 8, 128, 8192, 2), (33, 8, 8, 128, 4096, 4), (40, 8, 8, 128, 4096, 4),
    (24, 16, 16, 128, 2048, 2), (24, 16, 16, 128, 2049, 3), (56, 8, 8, 128, 4096, 3), (56, 8, 8, 128, 4097, 4),
    (56, 8, 8, 128, 8192, 4), (57, 8, 8, 128, 8192, 0), (57, 8, 8, 128, 8193, 4), (16, 16, 16, 128, 65536, 6), (16, 16, 16, 128, 65535, 2),
    # past 512 sequences times kv heads
    (64, 64, 16, 128, 4096, 5), (64, 64, 16, 128, 8193, 6), (33, 16, 16, 128, 4096, 4), (64, 32, 32, 128, 8193, 12)])
def test_sizes_of_the_rule(lib, batch, hq, hkv, d, max_ctx, per_cu):
    """Workgroups per CU (256 of them) that the rule launches for sizes on both sides of its lines."""
    assert workers(lib, batch, hq, hkv, d, max_ctx) == per_cu * 256 // hkv


def test_every_sequence_has_a_workgroup_and_a_long_one_is_cut(lib):
    for batch in range(2, MAX_BATCH + 1):
        for hkv in (1, 2, 3, 4, 5, 7, 8, 12, 16, 32, 40, 100, 256, 300, 513):
            for g in (1, 4, 8):
                for d in (64, 128):
                    for ctx in (1025, 4096, 8193, 200000):
                        w = workers(lib, batch, g * hkv, hkv, d, ctx)
                        if w and batch * hkv <= 512:
                            lens = [ctx] + [500] * (batch - 1)
                            segs, count, _ = cut(lens, w, ctx + 255, 64)
                            assert count <= w
                            if ctx > 4096:
                                assert segs[0][2] >= 2, (batch, hkv, g, d, ctx, w)
                        assert w == 0 or w >= batch


def test_refused_calls(lib):
    fake = ctypes.c_void_p(4096)

    def call(batch=4, hq=32, hkv=8, max_ctx=4096, partition=1024, ws=fake, ws_bytes=1 << 30, counters=fake, n=1 << 20):
        return lib.ak_paged_decode_balanced(fake, fake, fake, fake, fake, fake, batch, hq, hkv, 128, 10, 16, 512,
                                            max_ctx, 0.1, partition, ws, ws_bytes, counters, n, None)

    assert call(batch=1) == 2 and b"fixed splits" in lib.ak_last_error()
    assert call(partition=100) == 1 and lib.ak_last_error() == b"partition size must be a positive multiple of 256"
    assert call(hq=30) == 1 and call(max_ctx=0) == 1
    assert call(counters=None) == 1 and call(n=31) == 1 and b"counters" in lib.ak_last_error()
    assert call(ws=None) == 3 and call(ws_bytes=100) == 3 and call(ws=ctypes.c_void_p(4100)) == 1
