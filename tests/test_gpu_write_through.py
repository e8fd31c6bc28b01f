"""Launches that write y on to memory at once (from 2 MB of y on, 3 MB where the op is one launch) against the same tokens in
batches below that size: the same bits, for tiles of odd and even token counts, widths that end inside a chunk, tokens without an
adapter, and nothing written beside the rows.  16-token tiles above rank 64 and tall ones of compensations are never written through:
their cases hold that large batches give the bits of small ones all the same."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import workloads as W
from valora_amd.merge import DeLoraPlan
from valora_amd.plan import LoraPlan

from _util import REL_L2

pytestmark = pytest.mark.gpu
H_IN = 264


def _case(T, h_out, ranks, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    pool = W.make_pool(ranks, H_IN, h_out, dtype, g, True, n_slots=2, std=0.05, scalings=[0.5 + 0.25 * i for i in range(len(ranks))],
                       heads=1, extra_rows=2)
    ids = torch.randint(-1, len(ranks), (T,), generator=g)
    x, y = torch.randn(T, H_IN, generator=g).to(dtype), torch.randn(T, h_out, generator=g).to(dtype)
    return pool, ids, x, y


def _framed(y):
    frame = torch.full((y.size(0) + 2, y.size(1)), 7.0, dtype=y.dtype, device=y.device)
    frame[1:-1] = y
    return frame


def _both(dev, make_plan, call, pool, ids, x, y0, least):
    """The whole batch, and its two halves; the former is above the size from which y is written through, the latter are below."""
    T, h_out = y0.shape
    assert T * h_out * 2 >= least > (T + 1) // 2 * h_out * 2
    whole, parts = _framed(y0), _framed(y0)
    call(make_plan(ids), whole[1:-1], x)
    for a, b in ((0, T // 2), (T // 2, T)):
        call(make_plan(ids[a:b].contiguous()), parts[1 + a:1 + b], x[a:b])
    assert torch.equal(whole, parts)
    assert bool((whole[0] == 7).all() and (whole[-1] == 7).all())
    none = ids < 0
    assert torch.equal(whole[1:-1][none], y0[none])
    return whole[1:-1]


@pytest.mark.parametrize("h_out", [1600, 4160, 4288])   # rows of whole lines: others are not written through
@pytest.mark.parametrize("ranks,bm,one", [(r, bm, one) for r in ([16, 8], [32, 24, 8], [64, 40, 8], [128, 72, 16])
                                          for bm, one in ((16, False), (48, False), (16, True)) if not one or max(r) <= 64])
def test_same_bits_as_smaller_batches(dev, h_out, ranks, bm, one):
    least = (3 if one and max(ranks) <= 32 else 2) << 20
    T = least // (2 * h_out) + 3
    dtype = torch.bfloat16 if h_out == 4160 else torch.float16
    print(T, h_out, ranks, bm, one, flush=True)
    pool, ids, x, y0 = _case(T, h_out, ranks, dtype, h_out + ranks[0])
    p = pool.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    got = _both(dev, lambda i: LoraPlan(i, *idx[:2], max(ranks), n_slots=2, hidden=H_IN, bm_shrink=16, bm_expand=bm, one_launch=one, ksplit=2),
                lambda plan, y, xs: plan.apply(y, xs, p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling),
                p, ids.to(dev), x.to(dev), y0.to(dev), least)
    want = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1, pool.a_scaling, n_slots=2)
    # one rounding of y, and one of v on its way through B
    assert O.rel_l2(got.cpu(), want) <= (REL_L2 if dtype is torch.float16 else 8 * REL_L2)


@pytest.mark.parametrize("ranks", [[16, 8], [32, 24, 8], [64, 40, 8], [128, 72, 16]])
@pytest.mark.parametrize("bm", [16, 48])
def test_compensation_same_bits_as_smaller_batches(dev, ranks, bm):
    h_out = 4160
    T = (2 << 20) // (2 * h_out) + 3
    pool, ids, x, y0 = _case(T, h_out, ranks, torch.float16, ranks[0] + bm)
    p = pool.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    got = _both(dev, lambda i: DeLoraPlan(i, 1, *idx[:2], max(ranks), H_IN, n_slots=2, bm_shrink=16, bm_expand=bm, ksplit=2),
                lambda plan, y, xs: plan.apply(y, xs, p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling),
                p, ids.to(dev), x.to(dev), y0.to(dev), 2 << 20)
    want = O.delora_compensate(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1, 1, pool.a_scaling,
                               n_slots=2)
    assert O.rel_l2(got.cpu(), want) <= REL_L2


@pytest.mark.parametrize("ranks", [[16, 8], [32, 24, 8], [64, 40, 8]])
@pytest.mark.parametrize("h_out,odd", [(1600, 2), (4160, 3), (4288, 5)])
@pytest.mark.parametrize("own", [0.03, 0.6])   # of the tokens, not the merged adapter's
def test_compensation_of_small_tiles(dev, ranks, h_out, odd, own):
    """4 MB of y and more, of which half counts; with some tokens of no rank of their own."""
    T = (4 << 20) // (2 * h_out) + odd
    g = torch.Generator().manual_seed(h_out + ranks[0])
    ranks = ranks + [0]
    pool, _, x, y0 = _case(T, h_out, ranks, torch.float16, h_out)
    ids = torch.where(torch.rand(T, generator=g) < own, torch.randint(-1, len(ranks), (T,), generator=g), torch.tensor(1))
    print(T, h_out, ranks, own, flush=True)
    p = pool.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    got = _both(dev, lambda i: DeLoraPlan(i, 1, *idx[:2], max(ranks), H_IN, n_slots=2, bm_shrink=16, bm_expand=16, ksplit=2),
                lambda plan, y, xs: plan.apply(y, xs, p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling),
                p, ids.to(dev), x.to(dev), y0.to(dev), 4 << 20)
    want = O.delora_compensate(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1, 1, pool.a_scaling,
                               n_slots=2)
    assert O.rel_l2(got.cpu(), want) <= REL_L2


@pytest.mark.parametrize("h_out", [1600, 4128])   # the latter's rows are no whole lines: never written through
@pytest.mark.parametrize("targets", [2, 3])
@pytest.mark.parametrize("ranks,bm,one", [([16, 8], 16, True), ([32, 24, 8], 16, True), ([32, 24, 8], 16, False), ([64, 40, 8], 16, False),
                                          ([16, 8], 48, False), ([64, 40, 8], 48, False), ([128, 72, 16], 48, False)])
def test_targets_count_together_and_one_beside_lines(dev, h_out, targets, ranks, bm, one):
    """Targets that reach the size only together, all on 128-byte lines; the same with the last one beside them, which is written, with the
    others, the plain way; and the targets one by one, below the size.  Nothing beside the rows."""
    least = (3 if one else 2) << 20
    T = least // (2 * h_out * targets) + 5
    assert T * h_out * 2 * targets >= least > T * h_out * 2
    pool, ids, x, y0 = _case(T, h_out, ranks, torch.float16, targets + ranks[0])
    print(T, h_out, targets, ranks, bm, one, flush=True)
    p, xd = pool.to(dev), x.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    plan = LoraPlan(ids.to(dev), *idx[:2], max(ranks), n_slots=2, hidden=H_IN, bm_shrink=16, bm_expand=bm, one_launch=one, ksplit=2)
    slots = [z % 2 for z in range(targets)]

    def run(offs, calls):
        rooms = [torch.full(((T + 2) * h_out + 64,), 7.0, dtype=torch.float16, device=dev) for _ in offs]
        rows = [room[off:off + (T + 2) * h_out].view(T + 2, h_out) for room, off in zip(rooms, offs)]
        ys = [r[1:-1].copy_(y0.to(dev)) for r in rows]
        if h_out % 64 == 0:
            assert [y.data_ptr() % 128 == 0 for y in ys] == [off % 64 == 0 for off in offs]
        for zs in calls:
            plan.apply_multi([ys[z] for z in zs], xd, p.key_buffer, p.value_buffer, *idx, [slots[z] for z in zs], p.a_scaling)
        for y, room, off in zip(ys, rooms, offs):
            a = off + h_out
            assert bool((room[:a] == 7).all() and (room[a + T * h_out:] == 7).all())
        return torch.stack(ys)

    together = list(range(targets))
    got = run([0] * targets, [together])
    assert torch.equal(got, run([0] * (targets - 1) + [8], [together]))
    assert torch.equal(got, run([0] * targets, [[z] for z in together]))
    for z in together:
        want = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, slots[z], pool.a_scaling, n_slots=2)
        assert O.rel_l2(got[z].cpu(), want) <= REL_L2


@pytest.mark.parametrize("ranks", [[16, 8], [32, 24, 8], [64, 40, 8], [128, 72, 16]])
@pytest.mark.parametrize("bm,h_out", [(48, 4160), (64, 1600)])
def test_more_of_y_than_the_l2s_hold(dev, ranks, bm, h_out):
    """y that is read as lines that nobody reads again as well, against the same y beside 128-byte lines, which is read and written the plain way."""
    T = (32 << 20) // (2 * h_out) + 7
    pool, ids, x, y0 = _case(T, h_out, ranks, torch.bfloat16, ranks[0])
    print(T, h_out, ranks, bm, flush=True)
    p, xd = pool.to(dev), x.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    plan = LoraPlan(ids.to(dev), *idx[:2], max(ranks), n_slots=2, hidden=H_IN, bm_shrink=16, bm_expand=bm, one_launch=False, ksplit=1)
    got = []
    for off in (0, 8):
        room = torch.full(((T + 2) * h_out + 64,), 7.0, dtype=torch.bfloat16, device=dev)
        y = room[off + h_out:off + (T + 1) * h_out].view(T, h_out)
        assert (y.data_ptr() % 128 == 0) == (off == 0)
        y.copy_(y0)
        plan.apply(y, xd, p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling)
        assert bool((room[:off + h_out] == 7).all() and (room[off + (T + 1) * h_out:] == 7).all())
        got.append(y)
    assert torch.equal(got[0], got[1])
    want = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1, pool.a_scaling, n_slots=2)
    assert O.rel_l2(got[0].cpu(), want) <= 8 * REL_L2
