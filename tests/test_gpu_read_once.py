"""Launches whose operands are read as lines that nobody reads again (the rules stand beside the kernels) against the same tokens
in calls that the rules leave out: the same bits, and the oracle's result."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import _lib
from valora_amd import workloads as W
from valora_amd.plan import LoraPlan

from _util import REL_L2

pytestmark = pytest.mark.gpu


def _case(T, n, rank, h_in, h_out, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    ranks = [max(8, rank - 8 * (i % 3)) for i in range(n)]
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, n_slots=2, std=0.05, scalings=[0.5 + 0.25 * (i % 4) for i in range(n)],
                       heads=1, extra_rows=2)
    ids = torch.randint(-1, n, (T,), generator=g)
    return pool, ids, torch.randn(T, h_in, generator=g).to(dtype), torch.randn(T, h_out, generator=g).to(dtype)


def _oracle(pool, ids, x, y):
    return O.lora_op(y, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1, pool.a_scaling, n_slots=2)


def _bound(dtype):
    return REL_L2 if dtype is torch.float16 else 8 * REL_L2   # one rounding of y, and one of v on its way through B


@pytest.mark.parametrize("rank,one,ksplit", [(r, one, k) for r in (16, 32, 64, 128) for one in (False, True) for k in (1, 4)
                                             if not one or (r <= 32 and k > 1)])
@pytest.mark.parametrize("odd", [0, 64, -128])   # K ranges that are whole batches of steps, or end in the middle of one
def test_rows_of_a_in_small_tiles(dev, rank, one, ksplit, odd):
    """4 MB of A and more by the bound over the adapters of the index in the whole batch, less in each half."""
    n, T = 40, 43
    h_in = 65536 // rank + odd
    dtype = torch.bfloat16 if odd else torch.float16
    print(rank, one, ksplit, h_in, flush=True)
    rp = rank
    assert ((T + 15) // 16 + n) * rp * h_in * 2 >= 4 << 20 > ((T + 31) // 32 + (T + 1) // 2) * rp * h_in * 2
    pool, ids, x, y0 = _case(T, n, rank, h_in, 264, dtype, rank + odd)
    p, xd = pool.to(dev), x.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)

    def call(a, b, y):
        plan = LoraPlan(ids[a:b].to(dev).contiguous(), *idx[:2], rank, n_slots=2, hidden=h_in, bm_shrink=16, bm_expand=16, one_launch=one,
                        ksplit=ksplit)
        plan.apply(y, xd[a:b], p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling)

    whole, halves = y0.to(dev), y0.to(dev)
    call(0, T, whole)
    call(0, T // 2, halves[: T // 2])
    call(T // 2, T, halves[T // 2:])
    assert torch.equal(whole, halves)
    assert O.rel_l2(whole.cpu(), _oracle(pool, ids, x, y0)) <= _bound(dtype)


@pytest.mark.parametrize("rank", [16, 32, 64, 128])
@pytest.mark.parametrize("ksplit", [1, 4])
@pytest.mark.parametrize("odd", [0, 64, -128])   # K ranges that are whole batches of steps, or end in the middle of one
def test_rows_of_a_in_tiles_alone_with_their_adapter(dev, rank, ksplit, odd):
    """4 MB of A and more in the whole batch, less in each half; every adapter has one tile."""
    n, T = 44, 47
    h_in = 65536 // rank + odd
    dtype = torch.bfloat16 if odd else torch.float16
    print(rank, ksplit, h_in, flush=True)
    rp = rank
    pool, _, x, y0 = _case(T, n, rank, h_in, 264, dtype, rank + odd)
    ids = torch.arange(T) * 7 % n
    ids[5] = -1
    tiles = [len(set(part.tolist()) - {-1}) for part in (ids, ids[:T // 2], ids[T // 2:])]
    assert tiles[0] * rp * h_in * 2 >= 4 << 20 > max(tiles[1:]) * rp * h_in * 2
    p, xd = pool.to(dev), x.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)

    def call(a, b, y):
        plan = LoraPlan(ids[a:b].to(dev).contiguous(), *idx[:2], rank, n_slots=2, hidden=h_in, bm_shrink=16, bm_expand=16, one_launch=False,
                        ksplit=ksplit)
        plan.apply(y, xd[a:b], p.key_buffer, p.value_buffer, *idx, 1, p.a_scaling)

    whole, halves = y0.to(dev), y0.to(dev)
    call(0, T, whole)
    call(0, T // 2, halves[: T // 2])
    call(T // 2, T, halves[T // 2:])
    assert torch.equal(whole, halves)
    assert O.rel_l2(whole.cpu(), _oracle(pool, ids, x, y0)) <= _bound(dtype)


@pytest.mark.parametrize("ranks,bm,targets", [(r, bm, t) for r in ([16, 8], [32, 24, 8], [48, 16], [64, 40, 8], [128, 72, 16])
                                              for bm in (128, 256) for t in (1, 2, 3) if bm == 128 or (max(r) <= 64 and t == 1)])
@pytest.mark.parametrize("ksplit", [1, 2, 4])
def test_tall_tiles(dev, ranks, bm, targets, ksplit):
    """x on 128-byte lines against the same x beside them."""
    T, h_in, h_out = 5861, 576, 72       # two and three targets in four chunks share a workgroup
    g = torch.Generator().manual_seed(ranks[0] + bm + targets)
    dtype = torch.bfloat16 if ranks[0] == 64 else torch.float16
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, n_slots=3, std=0.05, scalings=[0.5 + 0.25 * i for i in range(len(ranks))],
                       heads=1, extra_rows=2)
    ids = torch.randint(-1, len(ranks), (T,), generator=g)
    x, y0 = torch.randn(T, h_in, generator=g).to(dtype), torch.randn(targets, T, h_out, generator=g).to(dtype)
    print(ranks, bm, targets, ksplit, flush=True)
    p, idsd = pool.to(dev), ids.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    plan = LoraPlan(idsd, *idx[:2], max(ranks), n_slots=3, hidden=h_in, bm_shrink=bm, bm_expand=64, one_launch=False, ksplit=ksplit,
                    reduce_in_expand=False)
    got = []
    for off in (0, 8):
        room = torch.empty(T * h_in + off, dtype=dtype, device=dev)
        xd = room[off:].view(T, h_in)
        assert (xd.data_ptr() % 128 == 0) == (off == 0)
        xd.copy_(x)
        y = y0.to(dev)
        plan.apply_multi(list(y.unbind(0)), xd, p.key_buffer, p.value_buffer, *idx, list(range(targets)), p.a_scaling)
        got.append(y)
    assert torch.equal(got[0], got[1])
    for t in range(targets):
        want = O.lora_op(y0[t], x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, t, pool.a_scaling, n_slots=3)
        assert O.rel_l2(got[0][t].cpu(), want) <= _bound(dtype)


@pytest.mark.parametrize("ranks,bm,targets", [(r, bm, t) for r in ([16, 8], [32, 24, 8], [48, 16], [64, 40, 8], [128, 72, 16])
                                              for bm in (128, 256) for t in (1, 2, 3) if bm == 128 or (max(r) <= 64 and t == 1)])
@pytest.mark.parametrize("ksplit", [1, 2, 4])
def test_tall_tiles_of_more_x_than_the_l2s_hold(dev, ranks, bm, targets, ksplit):
    """x and scratch on 128-byte lines; the same with x beside them, which is read the plain way; and with scratch beside them, whose partial
    sums are written and read the plain way."""
    T, h_in, h_out = 5861, 3008, 72      # two and three targets in four chunks share a workgroup; more of x than the L2s hold
    assert T * h_in * 2 >= 32 << 20
    g = torch.Generator().manual_seed(ranks[0] + bm + targets)
    dtype = torch.bfloat16 if ranks[0] == 64 else torch.float16
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, n_slots=3, std=0.05, scalings=[0.5 + 0.25 * i for i in range(len(ranks))],
                       heads=1, extra_rows=2)
    ids = torch.randint(-1, len(ranks), (T,), generator=g)
    x, y0 = torch.randn(T, h_in, generator=g).to(dtype), torch.randn(targets, T, h_out, generator=g).to(dtype)
    print(ranks, bm, targets, ksplit, flush=True)
    p, idsd = pool.to(dev), ids.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    plan = LoraPlan(idsd, *idx[:2], max(ranks), n_slots=3, hidden=h_in, bm_shrink=bm, bm_expand=64, one_launch=False, ksplit=ksplit,
                    reduce_in_expand=False)
    got = []
    for off in (0, 8):
        room = torch.empty(T * h_in + off, dtype=dtype, device=dev)
        xd = room[off:].view(T, h_in)
        assert (xd.data_ptr() % 128 == 0) == (off == 0)
        xd.copy_(x)
        y = y0.to(dev)
        plan.apply_multi(list(y.unbind(0)), xd, p.key_buffer, p.value_buffer, *idx, list(range(targets)), p.a_scaling)
        got.append(y)
    xd, y = x.to(dev), y0.to(dev)
    assert xd.data_ptr() % 128 == plan.scratch.data_ptr() % 128 == 0
    tg = (_lib.Target * targets)(*[_lib.Target(_lib.ptr(y[i]), _lib.ptr(p.value_buffer), p.value_buffer.numel() // h_out, i) for i in range(targets)])
    _lib.check(_lib.lib().mlora_lora_apply_multi(_lib.current_stream(dev), plan.handle, _lib.c_void_p(plan.scratch.data_ptr() + 16),
                                                 plan.scratch.numel() - 16, _lib.ptr(xd), T, h_in, h_out, max(ranks),
                                                 _lib.make_pool(p.key_buffer, *idx, h_in, 3), targets, tg, _lib.ptr(p.a_scaling), plan.ksplit,
                                                 plan.flags, _lib.dtype_code(dtype)))
    torch.cuda.synchronize()
    got.append(y)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    for t in range(targets):
        want = O.lora_op(y0[t], x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, t, pool.a_scaling, n_slots=3)
        assert O.rel_l2(got[0][t].cpu(), want) <= _bound(dtype)


@pytest.mark.parametrize("T,A,bm_s,bm_e,merged", [(1, 5, 16, 16, None), (60, 40, 16, 16, None), (300, 9, 16, 48, None), (900, 64, 16, 32, None),
                                                  (700, 3000, 16, 16, None), (5000, 600, 64, 16, None), (250, 12, 16, 16, 2)])
def test_record_says_which_tile_is_its_adapters_only_one(dev, T, A, bm_s, bm_e, merged):
    from valora_amd.merge import DeLoraPlan
    g = torch.Generator().manual_seed(T + A)
    a_len = (torch.randint(1, 9, (A,), generator=g) * 16)
    a_start = torch.cumsum(a_len, 0) - a_len
    index = (a_start.to(dev), a_len.to(dev))

    def check(plan, ids):
        for tiles, bm in ((plan.tiles_shrink().cpu().tolist(), bm_s), (plan.tiles_expand().cpu().tolist(), bm_e)):
            assert tiles
            for t in tiles:
                assert t[5:] == [len(tiles) if sum(u[0] == t[0] for u in tiles) == 1 else 0, 0, 0], (t, bm)

    hot = torch.where(torch.rand(T, generator=g) < 0.5, torch.tensor(A // 2), torch.randint(0, A, (T,), generator=g))
    one = torch.full((T,), A - 1)
    kw = dict(n_slots=2, bm_shrink=bm_s, bm_expand=bm_e)
    plan = LoraPlan(hot.to(dev), *index, 64, hidden=4096, **kw) if merged is None else DeLoraPlan(hot.to(dev), merged, *index, 64, 4096, **kw).plan
    check(plan, hot)
    plan.rebuild(one.to(dev))
    check(plan, one)


@pytest.mark.parametrize("rank", [16, 32, 64, 128])
@pytest.mark.parametrize("ksplit", [1, 4])
@pytest.mark.parametrize("shared", [0.0, 0.5, 1.0])   # of the tokens on one adapter, whose tiles share its A
def test_adapters_of_one_tile_among_others(dev, rank, ksplit, shared):
    """A on 128-byte lines against the same A beside them, which is read the plain way."""
    n, T, h_in, h_out = 60, 90, 2048 if rank > 16 else 4096, 72
    g = torch.Generator().manual_seed(rank + ksplit)
    pool, _, x, y0 = _case(T, n, rank, h_in, h_out, torch.float16, rank)
    ids = torch.where(torch.rand(T, generator=g) < shared, torch.tensor(7), torch.arange(T) % n)
    print(rank, ksplit, shared, flush=True)
    p, xd, idsd = pool.to(dev), x.to(dev), ids.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    plan = LoraPlan(idsd, *idx[:2], rank, n_slots=2, hidden=h_in, bm_shrink=16, bm_expand=16, one_launch=False, ksplit=ksplit)
    tiles = plan.tiles_shrink().cpu()
    some = shared < 1.0   # (batches that the rule takes: enough tiles, some of which are their adapter's only one)
    assert bool((tiles[:, 5] > 0).any()) == some and tiles.size(0) * rank * h_in * 2 >= (4 << 20 if some else 0)
    got = []
    for off in (0, 8):
        room = torch.empty(p.key_buffer.numel() + off, dtype=torch.float16, device=dev)
        kb = room[off:].view(p.key_buffer.shape)
        assert (kb.data_ptr() % 128 == 0) == (off == 0)
        kb.copy_(p.key_buffer)
        y = y0.to(dev)
        plan.apply(y, xd, kb, p.value_buffer, *idx, 1, p.a_scaling)
        got.append(y)
    assert torch.equal(got[0], got[1])
    assert O.rel_l2(got[0].cpu(), _oracle(pool, ids, x, y0)) <= REL_L2
