"""The 128- and 256-token shrink tiles at the edges of their K steps (64 elements; whole steps are loaded without looking
at any lane, a last step that is not whole is masked) and of their tiles and waves (rows past the tile's end read another
row), against the oracle at the tolerance of the whole op."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import _lib, workloads as W
from valora_amd.plan import LoraPlan
from tests._util import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bm,rank", [(128, 8), (128, 32), (128, 64), (128, 128), (256, 16), (256, 64)])
@pytest.mark.parametrize("h_in", [8, 56, 64, 72, 120, 128, 136, 1032])
def test_k_steps_and_rows(dev, h_in, bm, rank):
    g = torch.Generator().manual_seed(h_in * 1000 + bm + rank)
    dtype = torch.bfloat16 if rank == 64 else torch.float16
    lens = [1, 8, 31, 33, bm - 1, bm, bm + 1]
    ids = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens))
    ids = ids[torch.randperm(ids.numel(), generator=g)]
    ranks = [rank if i % 3 else 8 for i in range(len(lens))]
    pool = W.make_pool(ranks, h_in, 64, dtype, g, True, std=0.05, heads=1, extra_rows=3)
    x = torch.randn(ids.numel(), h_in, generator=g).to(dtype)
    y0 = torch.randn(ids.numel(), 64, generator=g).to(dtype)
    pd = pool.to(dev)
    idx = (pd.a_start, pd.a_len, pd.a_loc)
    want = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1, pool.a_scaling)
    for ks in (1, 2, 3):
        plan = LoraPlan(ids.to(dev), pd.a_start, pd.a_len, rank, hidden=h_in, bm_shrink=bm, bm_expand=32, ksplit=ks,
                        reduce_in_expand=False, one_launch=False)
        y = y0.to(dev)
        plan.apply(y, x.to(dev), pd.key_buffer, pd.value_buffer, *idx, 1, pd.a_scaling)
        assert_parity(y.cpu(), want, f"h_in={h_in} bm={bm} rank={rank} ks={ks}")


@pytest.mark.parametrize("bm,rank", [(16, 32), (64, 64), (128, 8), (128, 16), (128, 32), (128, 64), (128, 128), (256, 16),
                                     (256, 32), (256, 64)])
@pytest.mark.parametrize("h_in", [72, 512])
def test_rows_outside_the_pool(dev, h_in, bm, rank):
    """Rank rows whose index entry names no pool row, or that lie beyond the index, count as rows of zeros in every tile
    height: their columns of v are zero and their part of B is skipped."""
    g = torch.Generator().manual_seed(h_in + 10 * bm + rank)
    dtype = torch.bfloat16 if rank == 64 else torch.float16
    T, slot = 2 * bm + 7, 1
    pool = W.make_pool([rank, rank, rank], h_in, 64, dtype, g, True, std=0.05, heads=1, extra_rows=1)
    n_rows = pool.key_buffer.shape[0]
    # the last pool row stands for "no row": zeros for the oracle, out of the pool's bounds for the op
    pool.key_buffer[-1], pool.value_buffer[-1] = 0, 0
    spare = n_rows - 1
    taken = torch.where(pool.a_loc == spare)[0]
    free = next(r for r in range(n_rows) if r not in set(pool.a_loc.tolist()))
    pool.a_loc[taken] = free
    seen, given = pool.a_loc.clone(), pool.a_loc.clone()
    first = [int(s) + rank * slot for s in pool.a_start]
    for k, bad in enumerate((-1, n_rows, 1 << 40, -(1 << 40))):
        for at in (first[0] + (3 * k) % rank, first[1] + rank - 1 - k):
            seen[at], given[at] = spare, bad
    cut = first[2] + rank // 2                   # the last adapter's rows from here on lie beyond the index
    seen[cut:] = spare
    given = given[:cut].contiguous()
    ids = torch.randint(-1, 3, (T,), generator=g)
    x, y0 = torch.randn(T, h_in, generator=g).to(dtype), torch.randn(T, 64, generator=g).to(dtype)
    v0 = torch.zeros(T, rank, dtype=dtype)
    want_v = O.bgmv_shrink(v0, x, pool.key_buffer, pool.a_start, pool.a_len, seen, ids, slot)
    want = O.bgmv_expand(y0, want_v, pool.value_buffer, pool.a_start, pool.a_len, seen, ids, slot, pool.a_scaling)
    pd = pool.to(dev)
    kb, vb = pd.key_buffer[:spare], pd.value_buffer[:spare]
    loc, xd = given.to(dev), x.to(dev)
    none = want_v == 0
    for ks in (1, 2):
        plan = LoraPlan(ids.to(dev), pd.a_start, pd.a_len, rank, hidden=h_in, bm_shrink=bm, bm_expand=32, ksplit=ks,
                        reduce_in_expand=False, one_launch=False)
        y = y0.to(dev)
        plan.apply(y, xd, kb, vb, pd.a_start, pd.a_len, loc, slot, pd.a_scaling)
        assert_parity(y.cpu(), want, f"h_in={h_in} bm={bm} rank={rank} ks={ks}")
        # the same tiles through the entry point that hands v out
        v = v0.to(dev)
        pa = _lib.make_pool(kb, pd.a_start, pd.a_len, loc, h_in)
        _lib.check(_lib.lib().mlora_shrink(_lib.current_stream(dev), plan.handle, _lib.ptr(plan.scratch), plan.scratch.numel(),
                                           _lib.ptr(xd), T, h_in, rank, pa, slot, ks, _lib.ptr(v), rank, 0, 0, 0,
                                           _lib.dtype_code(dtype)))
        v = v.cpu()
        assert not v[none].any(), f"bm={bm} rank={rank} ks={ks}: a row outside the pool has a product"
        assert_parity(v, want_v, f"v h_in={h_in} bm={bm} rank={rank} ks={ks}")


@pytest.mark.parametrize("bm,rank", [(128, 8), (128, 32), (128, 64), (128, 128), (256, 16), (256, 64)])
@pytest.mark.parametrize("h_in", [8, 64, 72, 192, 1032, 4096])
def test_k_steps_same_bits(dev, h_in, bm, rank):
    """Small integers: every product and sum is exact in any order (at most 4096 * 8 < 2^24), so v has one right value per
    element and the tall tiles must give it bit for bit, whole steps and masked ones, as the 16-token tiles do."""
    g = torch.Generator().manual_seed(h_in + bm + rank)
    dtype = torch.bfloat16 if rank == 64 else torch.float16
    lens = [1, 8, 31, 33, bm - 1, bm, bm + 1]
    ids = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens))
    ids = ids[torch.randperm(ids.numel(), generator=g)]
    T = ids.numel()
    pool = W.make_pool([rank if i % 3 else 8 for i in range(len(lens))], h_in, 64, dtype, g, True, heads=1)
    pool.key_buffer.copy_(torch.randint(-2, 3, pool.key_buffer.shape, generator=g))
    x = torch.randint(-4, 5, (T, h_in), generator=g).to(dtype)
    v0 = torch.full((T, rank), 0.5, dtype=dtype)
    want = O.bgmv_shrink(v0, x, pool.key_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 2)
    pd, xd = pool.to(dev), x.to(dev)
    pa = _lib.make_pool(pd.key_buffer, pd.a_start, pd.a_len, pd.a_loc, h_in)
    for tile in (bm, 16):
        for ks in (1, 3):
            plan = LoraPlan(ids.to(dev), pd.a_start, pd.a_len, rank, hidden=h_in, bm_shrink=tile, bm_expand=32, ksplit=ks,
                            reduce_in_expand=False, one_launch=False)
            v = v0.to(dev)
            _lib.check(_lib.lib().mlora_shrink(_lib.current_stream(dev), plan.handle, _lib.ptr(plan.scratch),
                                               plan.scratch.numel(), _lib.ptr(xd), T, h_in, rank, pa, 2, ks, _lib.ptr(v), rank,
                                               0, 0, 0, _lib.dtype_code(dtype)))
            assert torch.equal(v.cpu(), want), f"tile {tile} ks {ks}"


@pytest.mark.parametrize("bm,ranks", [(128, [8, 24, 40, 72, 128, 16]), (128, [16, 8, 32, 24]), (256, [64, 16, 40, 24, 8])])
@pytest.mark.parametrize("h_in", [200, 320])
def test_narrow_adapters_among_wide_ones(dev, h_in, bm, ranks):
    """A tile takes the products of its own adapter's rank class, whatever the batch's widest.  Small integers, as above: one
    right value per element, for every number of chunks and both ways to store it."""
    g = torch.Generator().manual_seed(h_in + bm + len(ranks))
    ids = torch.randint(-1, len(ranks), (3 * bm,), generator=g)
    T, R = ids.numel(), max(ranks)
    pool = W.make_pool(ranks, h_in, 64, torch.float16, g, True, heads=1)
    pool.key_buffer.copy_(torch.randint(-2, 3, pool.key_buffer.shape, generator=g))
    x = torch.randint(-4, 5, (T, h_in), generator=g).to(torch.float16)
    v0 = torch.full((T, R), 0.5, dtype=torch.float16)
    want = O.bgmv_shrink(v0, x, pool.key_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, 1)
    pd, xd = pool.to(dev), x.to(dev)
    pa = _lib.make_pool(pd.key_buffer, pd.a_start, pd.a_len, pd.a_loc, h_in)
    for ks in (1, 2, 3):
        plan = LoraPlan(ids.to(dev), pd.a_start, pd.a_len, R, hidden=h_in, bm_shrink=bm, bm_expand=32, ksplit=ks,
                        reduce_in_expand=False, one_launch=False)
        v = v0.to(dev)
        _lib.check(_lib.lib().mlora_shrink(_lib.current_stream(dev), plan.handle, _lib.ptr(plan.scratch), plan.scratch.numel(), _lib.ptr(xd),
                                           T, h_in, R, pa, 1, ks, _lib.ptr(v), R, 0, 0, 0, _lib.dtype_code(torch.float16)))
        assert torch.equal(v.cpu(), want), ks
        plan.shrink(xd, pd.key_buffer, pd.a_start, pd.a_len, pd.a_loc, 1)
        perm, rp = plan.perm().long().cpu(), (R + 15) // 16 * 16
        held = plan.scratch.view(torch.float16)[:T * rp].view(T, rp)[:len(perm)].cpu()
        for col in range(0, R, 8):
            has = torch.tensor([ranks[int(ids[t])] > col for t in perm])
            assert torch.equal(held[has, col:col + 8], want[perm[has], col:col + 8]), (ks, col)
            assert not held[~has, col:col + 8].any()   # columns past a row's rank are zeros
