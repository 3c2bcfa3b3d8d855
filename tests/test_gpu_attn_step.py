"""Attention of one query over a caller's cache (attn_step.hip): both sides of every line between one workgroup per KV head, parts and
the pair of kernels, of a wave's 32 keys and of a part, against float64.

Limit: a score of up to 5 is rounded to 2^-22 a few times, a weight follows it, and a result is weights that add up to 1 times values of
up to 4: 4 * 4 * 2^-22 = 4e-6."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(32, 8, 64), (9, 3, 64), (14, 2, 64), (5, 5, 64), (48, 16, 64), (257, 257, 64), (32, 32, 96), (4, 2, 96), (12, 2, 128), (3, 3, 128)]
EDGES = [1, 16, 31, 33, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1000, 4100]


def _case(torch, heads, kv_heads, hd, seq, seed):
    gen = torch.Generator().manual_seed(seed)
    q = torch.randn(heads * hd, generator=gen)
    k, v = (torch.randn(seq, kv_heads * hd, generator=gen).half() for _ in range(2))
    return q, k, v


def _want(q, k, v, heads, kv_heads, hd, start=0):
    q, (k, v) = q.double().view(kv_heads, heads // kv_heads, hd), (x.double()[start:].view(-1, kv_heads, hd).transpose(0, 1).contiguous() for x in (k, v))
    return ((q @ k.transpose(1, 2).contiguous() * hd ** -0.5).softmax(-1) @ v).reshape(-1).numpy()


def _dev(*a):
    import torch
    return [x.cuda() if x.dtype.itemsize == 4 else x.cuda().view(torch.int16) for x in a]


@pytest.mark.parametrize("heads,kv_heads,hd", SHAPES)
def test_every_form_at_its_edges(fh, torch_gpu, heads, kv_heads, hd):
    for seq in EDGES:
        q, k, v = _case(torch_gpu, heads, kv_heads, hd, seq, seq + heads)
        dev = _dev(q, k, v)
        got = fh.ops.attention_flash(*dev, seq, heads, kv_heads, hd, 0).cpu().numpy()
        assert np.abs(got - _want(q, k, v, heads, kv_heads, hd)).max() <= 4e-6, seq
        for window in (1, 32, 100, 600):
            if window < seq:
                got = fh.ops.attention_sliding(*dev, seq, window, heads, kv_heads, hd, 0).cpu().numpy()
                assert np.abs(got - _want(q, k, v, heads, kv_heads, hd, seq - window)).max() <= 4e-6, (seq, window)


@pytest.mark.parametrize("heads,kv_heads,hd,seq", [(32, 8, 64, 40), (32, 8, 64, 700), (32, 32, 96, 200), (12, 2, 128, 100)])
def test_queries_of_any_size(fh, torch_gpu, heads, kv_heads, hd, seq):
    """Zero, tiny, huge, and elements far apart in size: scores to within their rounding (the one largest weight where they overflow a weight's range)."""
    torch = torch_gpu
    q, k, v = _case(torch, heads, kv_heads, hd, seq, 3)
    spread = q * torch.logspace(-6, 0, hd).repeat(heads)
    for query, limit in ((q * 0, 4e-6), (q * 1e-30, 4e-6), (q * 1e-4, 4e-6), (spread, 4e-6), (q * 8, 3e-4)):
        got = fh.ops.attention_flash(*_dev(query, k, v), seq, heads, kv_heads, hd, 0).cpu().numpy()
        # q * 8: |score| up to 50, a rounding of 2^-19 each of them, which a weight shows and a value of 4 multiplies
        assert np.abs(got - _want(query, k, v, heads, kv_heads, hd)).max() <= limit
    got = fh.ops.attention_flash(*_dev(q * 1e30, k, v), seq, heads, kv_heads, hd, 0).cpu().numpy()
    assert np.abs(got - _want(q * 1e30, k, v, heads, kv_heads, hd)).max() <= 1e-3


@pytest.mark.parametrize("heads,kv_heads,hd,seq", [(32, 8, 64, 40), (32, 8, 64, 700), (32, 32, 96, 200), (12, 2, 128, 100)])
def test_infinities_and_no_number(fh, torch_gpu, heads, kv_heads, hd, seq):
    """A key that scores -inf has no weight; an infinite value makes its column infinite; NaN spreads to its heads only; rows beyond the end are not read for arithmetic."""
    torch = torch_gpu
    q, k, v = _case(torch, heads, kv_heads, hd, seq, 4)
    at = seq // 2
    k2 = k.clone()
    k2[at, :hd] = -torch.inf * q[:hd].sign()          # KV head 0: -inf for query head 0 (other heads of it: no number)
    got = fh.ops.attention_flash(*_dev(q, k2, v), seq, heads, kv_heads, hd, 0).cpu().numpy().reshape(heads, hd)
    keep = [i for i in range(seq) if i != at]
    assert np.abs(got[0] - _want(q, k[keep], v[keep], heads, kv_heads, hd).reshape(heads, hd)[0]).max() <= 4e-6
    rest = heads // kv_heads
    assert np.abs(got[rest:] - _want(q, k, v, heads, kv_heads, hd).reshape(heads, hd)[rest:]).max(initial=0) <= 4e-6
    for first in (0, at):                             # ... but 0 times an infinite value is no number, as in 64 bits
        k3, v3 = k.clone(), v.clone()
        k3[first, :hd], v3[first, 7] = -torch.inf * q[:hd].sign(), torch.inf
        got = fh.ops.attention_flash(*_dev(q, k3, v3), seq, heads, kv_heads, hd, 0).cpu().numpy().reshape(heads, hd)
        assert np.isnan(got[0, 7]) and np.isfinite(got[0, np.arange(hd) != 7]).all()
    v2 = v.clone()
    v2[at, 3], v2[at, 5] = torch.inf, torch.nan
    got = fh.ops.attention_flash(*_dev(q, k, v2), seq, heads, kv_heads, hd, 0).cpu().numpy().reshape(heads, hd)
    want = _want(q, k, v, heads, kv_heads, hd).reshape(heads, hd)
    assert (got[:rest, 3] == np.inf).all() and np.isnan(got[:rest, 5]).all()
    want[:rest, [3, 5]] = got[:rest, [3, 5]] = 0
    assert np.abs(got - want).max() <= 4e-6
    tail = _dev(q, *(torch.cat([x, torch.full_like(x[:64], torch.nan)]) for x in (k, v)))
    assert np.abs(fh.ops.attention_flash(*tail, seq, heads, kv_heads, hd, 0).cpu().numpy() - _want(q, k, v, heads, kv_heads, hd)).max() <= 4e-6


@pytest.mark.parametrize("heads,kv_heads,hd,seq", [(32, 8, 64, 40), (32, 8, 64, 700), (32, 32, 96, 200), (12, 2, 128, 100), (3, 3, 128, 1)])
def test_a_key_without_a_number(fh, torch_gpu, heads, kv_heads, hd, seq):
    """NaN in a key makes every result of its heads NaN wherever the key stands: the first a wave sees, the last, behind one that scores -inf."""
    torch = torch_gpu
    q, k, v = _case(torch, heads, kv_heads, hd, seq, 6)
    want, rest = _want(q, k, v, heads, kv_heads, hd).reshape(heads, hd), heads // kv_heads
    for at in sorted({0, min(32, seq - 1), seq // 2, seq - 1}):
        for behind in (False, True):
            k2 = k.clone()
            if behind and at:
                k2[at // 32 * 32:at, :hd] = -torch.inf * q[:hd].sign()
            k2[at, 3] = torch.nan
            got = fh.ops.attention_flash(*_dev(q, k2, v), seq, heads, kv_heads, hd, 0).cpu().numpy().reshape(heads, hd)
            assert np.isnan(got[:rest]).all(), (at, behind)
            assert np.abs(got[rest:] - want[rest:]).max(initial=0) <= 4e-6


@pytest.mark.parametrize("heads,kv_heads,hd,seq", [(64, 16, 64, 300), (300, 100, 64, 40), (96, 96, 96, 200), (12, 2, 128, 100)])
def test_result_over_the_inputs(fh, torch_gpu, heads, kv_heads, hd, seq):
    """A result in place of the query, over a part of it or over a part of the cache has the bits of one with a buffer of its own."""
    torch = torch_gpu
    n, cache = heads * hd, seq * kv_heads * hd // 2                         # cache in floats
    src = dict(zip("qkv", _dev(*_case(torch, heads, kv_heads, hd, seq, 5))))
    want = fh.ops.attention_flash(src["q"], src["k"], src["v"], seq, heads, kv_heads, hd, 0).cpu().numpy()
    for name, at in (("q", 0), ("q", hd), ("q", n - 1), ("k", 0), ("v", max(0, cache - hd))):
        buf = {c: torch.cat([x.view(-1).view(torch.float32), torch.zeros(n, device="cuda")]) for c, x in src.items()}
        p = {c: C.c_void_p(x.data_ptr()) for c, x in buf.items()}
        fh.check(fh.lib().forge_hip_attn_decode_f16kv(p["q"], p["k"], p["v"], C.c_void_p(buf[name].data_ptr() + 4 * at), seq, heads, kv_heads, hd, 0, None))
        torch.cuda.synchronize()
        assert np.array_equal(buf[name][at:at + n].cpu().numpy().view(np.uint32), want.view(np.uint32)), (name, at)


def test_paged_contexts_have_the_flat_bits(fh, torch_gpu):
    """Pages of one row: a part's table entries within what LDS holds, and beyond (few, long parts)."""
    torch = torch_gpu
    for heads, kv_heads, seq in ((32, 8, 512), (32, 8, 33000), (256, 64, 9000)):
        q, k, v = _case(torch, heads, kv_heads, 64, seq, seq)
        order = torch.randperm(seq, generator=torch.Generator().manual_seed(1))
        pools = [torch.empty_like(x).index_copy_(0, order, x) for x in (k, v)]
        paged = fh.ops.attention_flash_paged(*_dev(q, *pools), order.int().cuda(), 1, seq, heads, kv_heads, 64).cpu().numpy()
        flat = fh.ops.attention_flash(*_dev(q, k, v), seq, heads, kv_heads, 64, 0).cpu().numpy()
        assert np.array_equal(paged.view(np.uint32), flat.view(np.uint32)), (heads, seq)
