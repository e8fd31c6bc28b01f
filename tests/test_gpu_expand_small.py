"""The expand of 16-token tiles against the expand of taller ones: another kernel, the same sums in the same order, so the
same bits -- over rank classes, widths on either side of the one from which a lane's units lie in two pool rows, remainders
of the column chunks, tile remainders, finished and partial narrow operands, infinities, and more tiles than a grid
dimension takes."""
import pytest
import torch

from valora_amd import workloads as W
from valora_amd.merge import DeLoraPlan
from valora_amd.plan import LoraPlan

pytestmark = pytest.mark.gpu


def _same(a, b):
    return bool(torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num()))


def _case(dev, T, h_in, h_out, ranks, dtype, seed, inf=False, hole=True):
    g = torch.Generator().manual_seed(seed)
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, n_slots=2, std=0.05, scalings=[0.5 + 0.25 * i for i in range(len(ranks))],
                       heads=1, extra_rows=2)
    if inf:
        pool.value_buffer.view(-1)[7::997] = float("inf")
    ids = torch.randint(-1 if hole else 0, len(ranks), (T,), generator=g)
    x, y = torch.randn(T, h_in, generator=g).to(dtype), torch.randn(T, h_out, generator=g).to(dtype)
    return pool.to(dev), ids.to(dev), x.to(dev), y.to(dev)


@pytest.mark.parametrize("T", [1, 17, 50])
@pytest.mark.parametrize("h_out", [24, 136, 520, 1624, 1632, 2056, 4104])
@pytest.mark.parametrize("ranks", [[8], [16, 8], [24, 8, 32], [64, 40, 8], [128, 72, 16]])
def test_same_bits_as_taller_tiles(dev, T, h_out, ranks):
    dtype = torch.bfloat16 if (T + h_out) % 3 == 0 else torch.float16
    print(T, h_out, ranks, dtype, flush=True)
    p, ids, x, y0 = _case(dev, T, 264, h_out, ranks, dtype, T + h_out, inf=h_out == 520)
    idx = (p.a_start, p.a_len, p.a_loc)
    for kw in (dict(ksplit=1), dict(ksplit=2, reduce_in_expand=True)):
        got = []
        for bm in (16, 32):
            plan = LoraPlan(ids, *idx[:2], max(ranks), n_slots=2, hidden=264, bm_shrink=16, bm_expand=bm, one_launch=False, **kw)
            ys = [y0.clone(), y0.clone()]
            plan.apply_multi(ys, x, p.key_buffer, p.value_buffer, *idx, [1, 0], p.a_scaling)
            got.append(ys)
        for a, b in zip(*got):
            assert _same(a, b), kw


@pytest.mark.parametrize("h_out", [520, 1632, 4104])
@pytest.mark.parametrize("ranks", [[16, 8], [32, 24, 8], [64, 16, 40], [128, 8, 96], [16, 12, 8]])
def test_compensation_same_bits_as_taller_tiles(dev, h_out, ranks):
    # (a length that is no multiple of 8 ranks has no product of its own: the merged adapter comes off all the same)
    p, ids, x, y0 = _case(dev, 70, 264, h_out, ranks, torch.float16, h_out + ranks[0])
    idx = (p.a_start, p.a_len, p.a_loc)
    got = []
    for bm in (16, 32):
        plan = DeLoraPlan(ids, 0, *idx[:2], max(ranks), 264, n_slots=2, bm_shrink=16, bm_expand=bm, ksplit=2)
        y = y0.clone()
        plan.apply(y, x, p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling)
        got.append(y)
    assert torch.equal(*got)
    assert not torch.equal(got[0], y0)


def test_the_column_loop_flag_is_accepted(dev):
    p, ids, x, y0 = _case(dev, 50, 264, 520, [16, 8], torch.float16, 3)
    got = []
    for flag in (False, True):
        plan = LoraPlan(ids, p.a_start, p.a_len, 16, n_slots=2, hidden=264, bm_shrink=16, bm_expand=16, ksplit=2, one_launch=False,
                        expand_column_loop=flag)
        y = y0.clone()
        plan.apply(y, x, p.key_buffer, p.value_buffer, p.a_start, p.a_len, p.a_loc, 1, p.a_scaling)
        got.append(y)
    assert torch.equal(*got) and not torch.equal(got[0], y0)


def test_more_tiles_than_a_grid_dimension(dev):
    T = 16 * 65535 + 40
    p, ids, x, y0 = _case(dev, T, 8, 72, [16, 8], torch.float16, 5, hole=False)
    idx = (p.a_start, p.a_len, p.a_loc)
    got = []
    for bm in (16, 128):
        plan = LoraPlan(ids, *idx[:2], 16, n_slots=2, hidden=8, bm_shrink=256, bm_expand=bm, ksplit=1, one_launch=False)
        y = y0.clone()
        plan.apply(y, x, p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling)
        got.append(y)
    assert torch.equal(*got)



@pytest.mark.parametrize("T", [16 * 65533, 16 * 65534, 16 * 65535 + 40])
def test_tiles_around_a_grid_dimension_on_a_used_plan(dev, T):
    """65535, 65536 and 65540 tile records.  The words behind them number the one-launch calls on the plan: after such a
    call they are no longer zero, and a two-launch call on the same plan must not take them for records."""
    p, ids, x, y0 = _case(dev, T, 8, 72, [16, 8], torch.float16, 6, hole=False)
    idx = (p.a_start, p.a_len, p.a_loc)
    pools = (p.key_buffer, p.value_buffer, *idx, 1)
    used = LoraPlan(ids, *idx[:2], 16, n_slots=2, hidden=8, ksplit=2, one_launch=True)
    print(T, "one launch", flush=True)
    first = y0.clone()
    used.apply(first, x, *pools, p.a_scaling)
    print(T, "two launches on the same plan", flush=True)
    got = y0.clone()
    used.shrink(x, p.key_buffer, *idx, 1)
    used.expand(got, p.value_buffer, *idx, 1, p.a_scaling)
    tall = LoraPlan(ids, *idx[:2], 16, n_slots=2, hidden=8, bm_shrink=16, bm_expand=128, ksplit=2, reduce_in_expand=True, one_launch=False)
    want = y0.clone()
    tall.apply(want, x, *pools, p.a_scaling)
    assert torch.equal(first, want) and torch.equal(got, want)
