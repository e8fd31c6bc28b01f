"""The rounding of fp32 sums to bf16 where the kernels store them (a hardware conversion, two values at once) against
round-to-nearest-even written out in integers: ties, subnormals, overflow to infinity, infinities and NaN."""
import numpy as np
import pytest
import torch

from valora_amd import _lib, workloads as W
from valora_amd.plan import LoraPlan

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def rne_bits(f):
    """fp32 -> bf16 bits, to nearest, ties to even; NaN stays NaN."""
    x = f.view(np.uint32).astype(np.uint64)
    out = ((x + 0x7FFF + ((x >> 16) & 1)) >> 16) & 0xFFFF
    nan = (x & 0x7FFFFFFF) > 0x7F800000
    return np.where(nan, (x >> 16) | 0x40, out).astype(np.uint16)


def patterns(lo_exp, hi_exp, n, seed):
    """fp32 values with biased exponents in [lo_exp, hi_exp]: random ones, ties, their neighbours, all-ones mantissas."""
    rng = np.random.RandomState(seed)
    sign, exp = rng.randint(0, 2, n).astype(np.uint32) << 31, rng.randint(lo_exp, hi_exp + 1, n).astype(np.uint32) << 23
    top = rng.randint(0, 128, n).astype(np.uint32) << 16
    low = rng.randint(0, 1 << 16, n).astype(np.uint32)
    kind = np.arange(n) % 8
    for k, v in ((0, 0x8000), (1, 0x8001), (2, 0x7FFF), (3, 0), (4, 0xFFFF)):
        low[kind == k] = v
    top[kind == 5] = 127 << 16                       # rounds into the next exponent
    low[kind == 5] |= 0x8000
    return (sign | exp | top | low).view(np.float32)


def parts(f, n):
    """f as n bf16 values that add up to it exactly, cut from the top."""
    out = []
    for _ in range(n):
        p = (f.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
        out.append(p)
        f = f - p
    assert not f.any()
    return out


def as_bf16(a):
    return torch.from_numpy((np.ascontiguousarray(a).view(np.uint32) >> 16).astype(np.int16)).view(BF)


def bits(t):
    return t.view(torch.int16).numpy().view(np.uint16)


def expand(dev, y, v, scale, bm, h_out=264):
    """y + scale * (sum of v's columns), through the expand: B is ones."""
    T = y.numel()
    pool = W.make_pool([8], h_out, h_out, BF, torch.Generator().manual_seed(0), True, heads=1, scalings=[scale])
    pool.value_buffer.fill_(1.0)
    pd = pool.to(dev)
    ids = torch.zeros(T, dtype=torch.long, device=dev)
    plan = LoraPlan(ids, pd.a_start, pd.a_len, 8, hidden=h_out, bm_shrink=16, bm_expand=bm, ksplit=1, one_launch=False)
    yd = y[:, None].expand(T, h_out).contiguous().to(dev)
    vd = torch.zeros(T, 8, dtype=BF)
    for j, col in enumerate(v):
        vd[:, j] = col
    vd = vd.to(dev)
    pb = _lib.make_pool(pd.value_buffer, pd.a_start, pd.a_len, pd.a_loc, h_out)
    _lib.check(_lib.lib().mlora_expand(_lib.current_stream(dev), plan.handle, _lib.ptr(yd), T, h_out, None, _lib.ptr(vd), 8, 8,
                                       pb, 0, _lib.ptr(pd.a_scaling), 1, 0, _lib.dtype_code(BF)))
    out = yd.cpu()
    assert torch.equal(out.view(torch.int16), out.view(torch.int16)[:, :1].expand(T, h_out))
    return bits(out[:, 0].contiguous())


@pytest.mark.parametrize("bm", [16, 32])
def test_expand_rounds_to_nearest_even(dev, bm):
    # the sum is put together exactly: y holds the value's upper part, the product the rest
    f = np.concatenate([patterns(30, 254, 8000, 1), np.array([3.3895314e38, 3.3961775e38, -3.3961776e38, 3.4028235e38], np.float32)])
    hi, mid, lo = parts(f, 3)
    got = expand(dev, as_bf16(hi), [as_bf16(mid), as_bf16(lo)], 1.0, bm)
    want = rne_bits(f)
    assert (got == want).all(), [(hex(a), hex(b), float(v)) for a, b, v in zip(got, want, f) if a != b][:5]


@pytest.mark.parametrize("bm", [16, 32])
def test_expand_rounds_subnormal_sums(dev, bm):
    # down to the last bit of fp32: the product is scaled into the range, y is zero
    f = np.concatenate([patterns(0, 20, 8000, 2), np.arange(1, 1 << 17, 37).astype(np.uint32).view(np.float32)])
    f = f[f != 0]
    acc = (f.astype(np.float64) * 2.0 ** 100).astype(np.float32)
    got = expand(dev, torch.zeros(len(f), dtype=BF), [as_bf16(p) for p in parts(acc, 3)], 2.0 ** -100, bm)
    want = rne_bits(f)
    assert (got == want).all(), [(hex(a), hex(b), float(v)) for a, b, v in zip(got, want, f) if a != b][:5]


@pytest.mark.parametrize("bm", [16, 32])
def test_expand_keeps_infinities_and_nan(dev, bm):
    y = np.array([0x7F80, 0xFF80, 0x7F81, 0x7FC0, 0xFFC1, 0xFFFF, 0x7FFF], np.uint16)
    yt = torch.from_numpy(y.view(np.int16)).view(BF)
    got = expand(dev, yt, [torch.full((len(y),), 0.5, dtype=BF)], 1.0, bm)
    want = np.where((y & 0x7FFF) > 0x7F80, y | 0x40, y)
    assert (got == want).all()


@pytest.mark.parametrize("bm,ksplit", [(16, 1), (16, 4), (128, 1), (128, 2)])
def test_shrink_rounds_to_nearest_even(dev, bm, ksplit):
    f = patterns(30, 250, 4000, 3)
    T, h_in = len(f), 512
    pool = W.make_pool([8], h_in, h_in, BF, torch.Generator().manual_seed(0), True, heads=1)
    pool.key_buffer.fill_(1.0)
    pd = pool.to(dev)
    x = torch.zeros(T, h_in, dtype=BF)
    # the parts lie in K steps (and with several, K chunks) of their own
    for at, p in zip((5, 70, 400), parts(f, 3)):
        x[:, at] = as_bf16(p)
    ids = torch.zeros(T, dtype=torch.long, device=dev)
    plan = LoraPlan(ids, pd.a_start, pd.a_len, 8, hidden=h_in, bm_shrink=bm, bm_expand=16, ksplit=ksplit,
                    reduce_in_expand=False, one_launch=False)
    xd, v = x.to(dev), torch.zeros(T, 8, dtype=BF, device=dev)
    pa = _lib.make_pool(pd.key_buffer, pd.a_start, pd.a_len, pd.a_loc, h_in)
    _lib.check(_lib.lib().mlora_shrink(_lib.current_stream(dev), plan.handle, _lib.ptr(plan.scratch), plan.scratch.numel(),
                                       _lib.ptr(xd), T, h_in, 8, pa, 0, ksplit, _lib.ptr(v), 8, 0, 0, 0, _lib.dtype_code(BF)))
    got, want = v.cpu(), rne_bits(f)
    for j in range(8):
        g = bits(got[:, j].contiguous())
        assert (g == want).all(), [(hex(a), hex(b), float(v)) for a, b, v in zip(g, want, f) if a != b][:5]
