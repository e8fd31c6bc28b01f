"""The expand of tiles of 32 tokens and more against the oracle: remainders of the 16- and 32-token blocks and of the column
chunks, widths on either side of the one from which a lane's units lie in two pool rows, v rows that take one and several
batches of requests, by position (finished and partial) and by token, and two operand sets (compensation)."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import _lib
from valora_amd import workloads as W
from valora_amd.merge import DeLoraPlan
from valora_amd.plan import LoraPlan

from _util import REL_L2

pytestmark = pytest.mark.gpu
COUNTS = (1, 15, 17, 31, 33, 95, 97, 255, 257)   # tokens of one adapter each
H_IN = 264


def _case(dev, counts, h_out, ranks, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    pool = W.make_pool([ranks[i % len(ranks)] for i in range(len(counts))], H_IN, h_out, dtype, g, True, n_slots=2, std=0.05,
                       scalings=[0.5 + 0.25 * (i % 3) for i in range(len(counts))], heads=1, extra_rows=2)
    ids = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    ids = torch.cat([ids, torch.full((5,), -1)])[torch.randperm(len(ids) + 5, generator=g)]
    x, y = torch.randn(len(ids), H_IN, generator=g).to(dtype), torch.randn(len(ids), h_out, generator=g).to(dtype)
    return pool, ids, x, y


def _close(got, want, dtype):
    """One rounding of y and one of v on top of sums of 32 bits: half a unit of the type each, relative to y, and v's error passes
    through B (a fraction of y here)."""
    eps = 2.0 ** -11 if dtype is torch.float16 else 2.0 ** -8
    err = (got.cpu().double() - want.double()).abs()
    assert float((err / want.double().abs().clamp_min(1.0)).max()) <= 2.5 * eps
    assert O.rel_l2(got.cpu(), want) <= (REL_L2 if dtype is torch.float16 else 8 * REL_L2)


@pytest.mark.parametrize("h_out", [72, 264, 1624, 1640, 4104])
@pytest.mark.parametrize("ranks", [[8], [32, 16], [64, 8, 40], [128, 24, 72]])
def test_tall_tiles(dev, h_out, ranks):
    dtype = torch.bfloat16 if h_out == 264 else torch.float16
    pool, ids, x, y0 = _case(dev, COUNTS, h_out, ranks, dtype, h_out + ranks[0])
    want = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1, pool.a_scaling, n_slots=2)
    p, ids, x, y0 = pool.to(dev), ids.to(dev), x.to(dev), y0.to(dev)
    idx, R, T = (p.a_start, p.a_len, p.a_loc), max(ranks), len(ids)
    for bm in (32, 96, 256):
        print(h_out, ranks, bm, flush=True)
        outs = []
        for kw in (dict(ksplit=1), dict(ksplit=5, reduce_in_expand=True)):
            plan = LoraPlan(ids, *idx[:2], R, n_slots=2, hidden=H_IN, bm_shrink=16, bm_expand=bm, one_launch=False, **kw)
            y = y0.clone()
            plan.apply(y, x, p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling)
            outs.append(y)
        # the same v, handed over as a caller's matrix of one row per token, wider than the rank
        plan = LoraPlan(ids, *idx[:2], R, n_slots=2, hidden=H_IN, bm_shrink=16, bm_expand=bm, one_launch=False, ksplit=1)
        plan.shrink(x, p.key_buffer, *idx, 1)
        perm = plan.perm().long()
        rp = (R + 15) // 16 * 16
        v = torch.full((T, rp + 8), float("nan"), dtype=dtype, device=dev)
        v[perm, :rp] = plan.scratch.view(dtype)[:T * rp].view(T, rp)[:len(perm)]
        y = y0.clone()
        pb = _lib.make_pool(p.value_buffer, *idx, h_out, 2)
        _lib.check(_lib.lib().mlora_expand(_lib.current_stream(dev), plan.handle, _lib.ptr(y), T, h_out, None, _lib.ptr(v), rp + 8, R, pb, 1,
                                           _lib.ptr(p.a_scaling), 1, 0, _lib.dtype_code(dtype)))
        outs.append(y)
        for y in outs:
            _close(y, want, dtype)
        assert torch.equal(outs[0], outs[2])   # the same sums of the same v


@pytest.mark.parametrize("h_out", [264, 1640])
@pytest.mark.parametrize("ranks", [[16, 32], [64, 8], [128, 40, 24]])
@pytest.mark.parametrize("bm", [48, 256])
def test_tall_tiles_of_a_compensation(dev, h_out, ranks, bm):
    pool, ids, x, y0 = _case(dev, COUNTS, h_out, ranks, torch.float16, h_out + bm)
    want = O.delora_compensate(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 2, 1, pool.a_scaling,
                               n_slots=2)
    p = pool.to(dev)
    plan = DeLoraPlan(ids.to(dev), 2, p.a_start, p.a_len, max(ranks), H_IN, n_slots=2, bm_shrink=16, bm_expand=bm, ksplit=1)
    y = y0.to(dev)
    plan.apply(y, x.to(dev), p.key_buffer, p.value_buffer, p.a_start, p.a_len, p.a_loc, 1, p.a_scaling)
    _close(y, want, torch.float16)
