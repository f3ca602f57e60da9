"""The one-pass route of the Python wrappers (the extension's plain_* functions)
against the checked route: the same answers and the same errors, and None for
whatever is not the plain case."""
import numpy as np
import pytest
import torch

import attnkernels as ak
import oracle

pytestmark = pytest.mark.gpu


def rand(*shape, dtype=torch.float16):
    return torch.randn(*shape, device="cuda", dtype=dtype, generator=torch.Generator("cuda").manual_seed(len(shape)))


def checked(monkeypatch, fn):
    """fn's answer or error by the checked route."""
    with monkeypatch.context() as m:
        m.setattr(ak, "_on_gpu", lambda x: False)
        return outcome(fn)


def outcome(fn):
    try:
        return fn()
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)


def same(a, b):
    if isinstance(a, torch.Tensor) and isinstance(b, torch.Tensor):
        return a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    return a == b


def prefill_calls():
    q, k, v = rand(2, 4, 33, 64), rand(2, 4, 33, 64), rand(2, 4, 33, 64)
    kg = k[:, :2].contiguous()
    for causal in (True, False, 1, None, np.bool_(True)):
        yield lambda c=causal: ak.flash_attention(q, k, v, causal=c)
    for scale in (None, 0.3, 1, np.float64(0.2), -0.5):
        yield lambda s=scale: ak.flash_attention(q, k, v, scale=s)
        yield lambda s=scale: ak.flash_attention_gqa(q, kg, kg, scale=s)
    qt = q.transpose(1, 2).contiguous().transpose(1, 2)
    for bad in ((qt, k, v), (q, k[:, :2], v[:, :2]), (q, k, v[:, :, :5]), (q.float(), k, v), (q[0], k[0], v[0]),
                (q, k.cpu(), v), (q[..., :40],) * 3, (q[:, :, :0],) * 3, (q, None, v)):
        yield lambda b=bad: ak.flash_attention(*b)
        yield lambda b=bad: ak.flash_attention_gqa(*b)
    yield lambda: ak.flash_attention_gqa(q[:, :3].contiguous(), kg, kg)
    x = rand(20, 4, 64)
    for cu in (torch.tensor([0, 7, 20], dtype=torch.int32, device="cuda"), torch.tensor([0, 20], device="cuda"),
               torch.tensor([0, 9, 20]), torch.tensor([[0, 20]], device="cuda"),
               torch.tensor([9, 0, 7, 20], dtype=torch.int32, device="cuda")[1:]):
        for longest in (20, 13, np.int64(20)):
            yield lambda c=cu, n=longest: ak.flash_attention_varlen(x, x, x, c, n, causal=True)


def decode_calls():
    kc, vc, bt, cl = oracle.make_paged_cache([40, 300], 2, 64, block_size=16, extra_blocks=1, seed=0)
    kc, vc, bt, cl = (torch.from_numpy(a).cuda() for a in (kc, vc, bt, cl))
    q = rand(2, 4, 64)
    for part in (None, 256, 100, 0, -256, 1 << 40, 256.0):
        yield lambda p=part: ak.paged_decode(q, kc, vc, bt, cl, 300, partition_size=p)
    for longest in (300, 300.0, np.int64(300), 0, -5, 1 << 40):
        yield lambda n=longest: ak.paged_decode(q, kc, vc, bt, cl, n)
    for bad in ((q, kc, vc, bt.long(), cl), (q, kc, vc, bt, cl.long()), (q.bfloat16(), kc, vc, bt, cl),
                (q, kc, vc[:-1], bt, cl), (q[:1], kc, vc, bt, cl), (q[:, :3], kc, vc, bt, cl), (q[:0], kc, vc, bt[:0], cl[:0]),
                (q, kc.transpose(2, 3).contiguous().transpose(2, 3), vc, bt, cl), (q, kc, vc, bt, cl.cpu()),
                (q, kc, vc, bt[:, ::2], cl), (q[0], kc, vc, bt, cl)):
        yield lambda b=bad: ak.paged_decode(*b, 300)


def balanced_calls():
    """Large enough at the longest context given that the splits are balanced, as each route reaches them."""
    kc, vc, bt, cl = oracle.make_paged_cache([3000, 40, 1700, 1], 8, 128, block_size=16, extra_blocks=1, seed=0)
    kc, vc, bt, cl = (torch.from_numpy(a).cuda() for a in (kc, vc, bt, cl))
    q = rand(4, 16, 128)
    for args in ((bt, cl), (bt.long(), cl), (bt, cl.long())):
        yield lambda a=args: ak.paged_decode(q, kc, vc, *a, 16000)


def test_balanced_routes_agree(monkeypatch):
    """One answer for tables and lengths of either integer type, by either route."""
    answers = [f() for f in balanced_calls()] + [checked(monkeypatch, f) for f in balanced_calls()]
    assert all(same(a, answers[0]) for a in answers)
    fixed = ak.load_extension().paged_decode  # other sums: the default did take balanced splits
    kc, vc, bt, cl = (torch.from_numpy(a).cuda() for a in oracle.make_paged_cache([3000, 40, 1700, 1], 8, 128, block_size=16,
                                                                                 extra_blocks=1, seed=0))
    part = ak.decode_partition(4, 8, 16000)
    other = fixed(rand(4, 16, 128), kc, vc, bt, cl, 16000, 128 ** -0.5, part)
    assert not torch.equal(other, answers[0]) and (other - answers[0]).abs().max() < 1e-3


@pytest.mark.parametrize("calls", [prefill_calls, decode_calls])
def test_answers_and_errors_are_those_of_the_checked_route(calls, monkeypatch):
    for i, fn in enumerate(calls()):
        a, b = outcome(fn), checked(monkeypatch, fn)
        assert same(a, b), (i, a, b)


def test_writes_are_those_of_the_checked_route(monkeypatch):
    tokens, hkv, d, bs = 5, 2, 64, 8
    qkv = rand(tokens, 6 * d)
    key, value = qkv[:, 2 * d:4 * d].view(tokens, hkv, d), qkv[:, 4 * d:].view(tokens, hkv, d)
    slots = torch.tensor([3, 17, -1, 30, 9], device="cuda")
    odd = rand(tokens * hkv * d + 4)[4:].view(tokens, hkv, d)  # 8 bytes off
    cases = [(key, value, slots), (key[:1], value[:1], slots[:1]), (key[:0], value[:0], slots[:0]),
             (key, value, slots.int()), (key, value, slots.cpu()), (odd, value, slots), (key, odd, slots),
             (key.transpose(1, 2).contiguous().transpose(1, 2), value, slots), (key.float(), value, slots),
             (key.bfloat16(), value.bfloat16(), slots), (key, value, slots[:3]), (key[..., :60], value[..., :60], slots)]
    for i, (k, v, s) in enumerate(cases):
        got = []
        for route in (outcome, lambda f: checked(monkeypatch, f)):
            kc, vc = (torch.zeros(4, hkv, bs, d, device="cuda", dtype=torch.float16) for _ in range(2))
            answer = route(lambda: ak.reshape_and_cache(k, v, kc, vc, s))
            got.append((answer, kc, vc))
        assert got[0][0] == got[1][0], (i, got[0][0], got[1][0])
        assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][2], got[1][2]), i


def test_only_plain_tensors_take_it():
    ext = ak.load_extension()
    q = rand(1, 2, 16, 64)
    assert isinstance(ext.plain_prefill(q, q, q, False, None, False), torch.Tensor)
    assert isinstance(ext.plain_prefill(q, q[:, :1], q[:, :1], True, 0.5, True), torch.Tensor)
    x, cu = rand(20, 4, 64), torch.tensor([0, 7, 20], dtype=torch.int32, device="cuda")
    assert isinstance(ext.plain_varlen(x, x, x, cu, 13, True, None), torch.Tensor)
    assert ext.plain_varlen(x, x, x, cu.long(), 13, True, None) is None
    kc, vc, bt, cl = (torch.from_numpy(a).cuda() for a in oracle.make_paged_cache([40, 300], 2, 64, block_size=16, seed=0))
    qd = rand(2, 4, 64)
    for part in (None, 256):
        assert isinstance(ext.plain_decode(qd, kc, vc, bt, cl, 300, None, part, ak.decode_partition), torch.Tensor)
        assert ext.plain_decode(qd, kc, vc, bt.long(), cl, 300, None, part, ak.decode_partition) is None
    key, slots = rand(5, 2, 64), torch.arange(5, device="cuda")
    assert ext.plain_write(key, key, kc, vc, slots) is True
    assert ext.plain_write(key, key, kc, vc, slots.int()) is False
    assert ext.plain_prefill(q.cpu(), q, q, False, None, False) is None
    assert ext.plain_prefill(q, q, q, 1, None, False) is None

    class Sub(torch.Tensor):
        pass

    assert ext.plain_prefill(q.as_subclass(Sub), q, q, False, None, False) is None
    seen = []
    torch.vmap(lambda x: seen.append(ext.plain_prefill(x, x, x, False, None, False)) or x)(torch.stack([q, q]))
    assert seen == [None]
