"""The shrink of 16- to 64-token tiles where its branches meet: K chunks of less than a batch, a whole batch and a remainder, ranks
that leave blocks of the tile empty, rank rows outside the pool (the masked loop up to rank 32, a line of zeros above), tile counts
that are no multiple of eight with several targets, and up to nine chunks summed by the last workgroup, by the expand or
recomputed.  The same sums in the same order on every route, so the same bits; the oracle has the numbers."""
import copy

import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import _lib, workloads as W
from valora_amd.plan import LoraPlan
from tests._util import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 9, 75])
@pytest.mark.parametrize("h_in, ksplit", [(200, 1), (200, 2), (1096, 1), (2304, 5), (2304, 9), (4096, 3)])
@pytest.mark.parametrize("ranks", [[8], [16, 8], [32, 24, 8], [64, 40, 16], [128, 72, 8]])
def test_routes_and_missing_rows(dev, T, h_in, ksplit, ranks):
    dtype = torch.bfloat16 if (T + ksplit) % 2 else torch.float16
    print(T, h_in, ksplit, ranks, dtype, flush=True)
    g = torch.Generator().manual_seed(T + h_in)
    A, h_out, slots = len(ranks), 264, [1, 0, 2]
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, n_slots=3, std=0.05, scalings=[0.5 + 0.25 * i for i in range(A)], heads=1,
                       extra_rows=2)
    ids = torch.randint(-1, A, (T,), generator=g)
    ids[0] = 0
    x = torch.randn(T, h_in, generator=g).to(dtype)
    ys = [torch.randn(T, h_out, generator=g).to(dtype) for _ in slots]
    # without missing rows, and with one rank row of every slot outside the pool: the oracle sees a row of zeros there
    for missing in (False, True):
        zero = copy.copy(pool)
        loc = pool.a_loc.clone()
        if missing:
            at = [int(pool.a_start[i]) + ranks[i] * s + (ranks[i] - 1) // 2 for i in range(A) for s in range(3)]
            zero.a_loc = pool.a_loc.clone()
            zero.a_loc[at] = zero.key_buffer.shape[0]
            zero.key_buffer = torch.cat([pool.key_buffer, torch.zeros_like(pool.key_buffer[:1])])
            zero.value_buffer = torch.cat([pool.value_buffer, torch.zeros_like(pool.value_buffer[:1])])
            loc[at] = torch.tensor([pool.key_buffer.shape[0] + 7, -3, 1 << 40])[torch.arange(len(at)) % 3]
        p = pool.to(dev)
        idx = (p.a_start, p.a_len, loc.to(dev))
        for bm in (16, 32, 64):
            if bm == 64 and max(ranks) > 64:
                continue
            got = {}
            for name, kw in (("expand", dict(reduce_in_expand=True)), ("shrink", dict(reduce_in_expand=False)),
                             ("recompute", dict(reduce_in_expand=False, shrink_recompute=True))):
                plan = LoraPlan(ids.to(dev), *idx[:2], max(ranks), n_slots=3, hidden=h_in, bm_shrink=bm, bm_expand=16, ksplit=ksplit,
                                one_launch=False, **kw)
                got[name] = [y.to(dev) for y in ys]
                plan.apply_multi(got[name], x.to(dev), p.key_buffer, p.value_buffer, *idx, slots, p.a_scaling)
            for i, s in enumerate(slots):
                what = f"bm={bm} missing={missing} target {i}"
                assert torch.equal(got["shrink"][i], got["expand"][i]), what
                assert torch.equal(got["recompute"][i], got["expand"][i]), what
                if bm == 16:
                    ref = O.lora_op(ys[i], x, zero.key_buffer, zero.value_buffer, zero.a_start, zero.a_len, zero.a_loc, ids, s,
                                    zero.a_scaling, n_slots=3)
                    assert_parity(got["shrink"][i].cpu(), ref, what)
                    first = got["shrink"]
                else:
                    assert torch.equal(got["shrink"][i], first[i]), what + ": the tile height changed the sums"


@pytest.mark.parametrize("rank, ksplit, T, n_targets", [(16, 4, 40, 3), (16, 6, 40, 3), (16, 5, 640, 1), (16, 4, 4, 3), (16, 4, 4, 2),
                                                        (32, 8, 40, 2), (32, 4, 40, 1), (32, 4, 400, 3), (48, 4, 40, 1)])
def test_one_or_two_launches(dev, rank, ksplit, T, n_targets):
    """On either side of the lines from which a one-launch call runs as two, with room for two launches and with just enough
    scratch for one: the bits of the two-launch op with the same split (K chunks x targets are cut to 16)."""
    print(rank, ksplit, T, n_targets, flush=True)
    g = torch.Generator().manual_seed(T)
    h, A = 2304, 20
    pool = W.make_pool([rank] * A, h, h, torch.float16, g, True, n_slots=4, std=0.05, scalings=[0.5] * A, heads=1)
    ids = torch.randint(0, A, (T,), generator=g)
    p = pool.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    x, y0 = torch.randn(T, h, generator=g).half(), torch.randn(T, h, generator=g).half()
    slots = list(range(n_targets))

    def run(plan, short=0):
        ys = [y0.to(dev) for _ in slots]
        if not short:
            plan.apply_multi(ys, x.to(dev), p.key_buffer, p.value_buffer, *idx, slots, p.a_scaling)
            return ys
        pa = _lib.make_pool(p.key_buffer, *idx, h, 4)
        tg = (_lib.Target * n_targets)(*[_lib.Target(_lib.ptr(ys[i]), _lib.ptr(p.value_buffer), p.value_buffer.numel() // h, slots[i])
                                         for i in slots])
        xd = x.to(dev)
        _lib.check(_lib.lib().mlora_lora_apply_multi(_lib.current_stream(dev), plan.handle, _lib.ptr(plan.scratch), short, _lib.ptr(xd), T, h, h,
                                                     rank, pa, n_targets, tg, _lib.ptr(p.a_scaling), plan.ksplit, plan.flags,
                                                     _lib.dtype_code(torch.float16)))
        torch.cuda.synchronize()
        return ys

    kw = dict(n_slots=4, hidden=h, bm_shrink=16, bm_expand=16)
    one = LoraPlan(ids.to(dev), *idx[:2], rank, one_launch=True, ksplit=ksplit, **kw)
    two = LoraPlan(ids.to(dev), *idx[:2], rank, one_launch=False, ksplit=min(ksplit, 16 // n_targets), reduce_in_expand=True, **kw)
    want = run(two)
    for i in slots:
        ref = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, slots[i], pool.a_scaling, n_slots=4)
        assert_parity(want[i].cpu(), ref, f"target {i}")
    for got in (run(one), run(one)):
        for a, b in zip(got, want):
            assert torch.equal(a, b)
    # what one launch needs, the tiles' partials and the narrow operand (at rank 16, whose rows two launches pad, they can need more)
    rp = (rank + 15) // 16 * 16
    tiles = (T + 15) // 16 + min(A, T)
    need = (T * rp * 2 + 255) // 256 * 256 + tiles * n_targets * two.ksplit * 16 * rp * 4
    if rank <= 32 and need < _lib.lib().mlora_scratch_bytes(T, rank, two.ksplit) * n_targets:
        for a, b in zip(run(one, need), want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("T", [1, 22, 300])
@pytest.mark.parametrize("ksplit", [2, 4, 5, 9])
@pytest.mark.parametrize("ranks", [[16], [24, 32], [48, 8], [64, 16], [96, 72], [128, 40]])
def test_sum_in_a_launch_of_its_own(dev, T, ksplit, ranks):
    """The launch that sums the chunks of tall tiles: rows of 4 to 32 quarters (12, 20 and 24 leave threads of a workgroup without
    one), fewer and more chunks than it requests at once -- the bits of the expand that sums them itself -- and the caller's own
    matrix in its three modes."""
    print(T, ksplit, ranks, flush=True)
    g = torch.Generator().manual_seed(T + ksplit)
    A, h_in, h_out, R = len(ranks), 2312, 264, max(ranks)
    pool = W.make_pool(ranks, h_in, h_out, torch.float16, g, True, n_slots=2, std=0.05, scalings=[0.5] * A, heads=1)
    ids = torch.randint(-1, A, (T,), generator=g)
    x, y0 = torch.randn(T, h_in, generator=g).half().to(dev), torch.randn(T, h_out, generator=g).half()
    p = pool.to(dev)
    idx = (p.a_start, p.a_len, p.a_loc)
    got = []
    for rie in (True, False):
        plan = LoraPlan(ids.to(dev), *idx[:2], R, n_slots=2, hidden=h_in, bm_shrink=128, bm_expand=32, ksplit=ksplit, reduce_in_expand=rie,
                        one_launch=False)
        ys = [y0.to(dev), y0.to(dev)]
        plan.apply_multi(ys, x, p.key_buffer, p.value_buffer, *idx, [1, 0], p.a_scaling)
        got.append(ys)
    for a, b in zip(*got):
        assert torch.equal(a, b)
    lib, pa = _lib.lib(), _lib.make_pool(p.key_buffer, *idx, h_in, 2)
    rk = torch.tensor(ranks)[ids.clamp(min=0)] * (ids >= 0)
    inside = (torch.arange(R)[None] < rk[:, None]).to(dev)
    width = R + 8
    before = torch.randn(T, width, generator=g).half().to(dev)
    out = {}
    for mode in (0, 1, 2):
        d = before.clone()
        _lib.check(lib.mlora_shrink(_lib.current_stream(dev), plan.handle, _lib.ptr(plan.scratch), plan.scratch.numel(), _lib.ptr(x), T, h_in, R, pa,
                                    1, ksplit, _lib.ptr(d), width, mode, R, 0, _lib.dtype_code(torch.float16)))
        torch.cuda.synchronize()
        out[mode] = d
    over, pad, acc = out[0], out[1], out[2]
    has = (ids >= 0).to(dev)[:, None]
    assert torch.equal(over[:, R:], before[:, R:])
    # accumulate adds the unrounded sum: within one rounding of (what was there + the rounded sum)
    v = torch.where(inside, over[:, :R], torch.zeros_like(before[:, :R])).float()
    want = torch.where(inside, before[:, :R].float() + v, before[:, :R].float())
    tol = 2.0 ** -11 * (v.abs() + 2 * want.abs()) + 2.0 ** -24
    assert bool(((acc[:, :R].float() - want).abs() <= tol).all())
    assert torch.equal(pad[:, :R], torch.where(has, torch.where(inside, over[:, :R], torch.zeros_like(before[:, :R])),
                                                             before[:, :R]))
    assert torch.equal(torch.where(inside, before[:, :R], over[:, :R]), before[:, :R])
