"""Two or three targets of 128-token shrink tiles in one workgroup: the bits of separate calls, at the edges of tiles, K steps
and chunks, with adapters of several rank classes and rank rows that are not in the pool, and on both sides of the rule (128 or 160
workgroups)."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import _lib, workloads as W
from valora_amd.plan import LoraPlan
from tests._util import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ranks", [(8, 16), (32, 8, 16, 24), (64, 8, 40, 16, 32, 56), (128, 8, 72, 16, 104, 56)])
@pytest.mark.parametrize("h_in,ksplit", [(1024, 16), (1032, 15), (2048, 32), (4104, 16), (136, 2)])
def test_bits_of_separate_calls(dev, h_in, ksplit, ranks):
    g = torch.Generator().manual_seed(h_in + len(ranks))
    dtype = torch.bfloat16 if len(ranks) == 4 else torch.float16
    A, R, h_out = len(ranks), max(ranks), 72
    for tiles in ((9, 5) if ksplit > 2 else (90, 65, 30)):   # (tiles + tails) * chunks on either side of the rule
        lens = torch.full((A,), tiles * 128 // A)
        lens[0], lens[-1] = lens[0] // 2 + 1, lens[-1] + 130
        ids = torch.repeat_interleave(torch.arange(A), lens)
        ids = ids[torch.randperm(ids.numel(), generator=g)]
        T = ids.numel()
        pool = W.make_pool(list(ranks), h_in, h_out, dtype, g, True, std=0.05, heads=1, extra_rows=1)
        x = torch.randn(T, h_in, generator=g).to(dtype)
        y0 = [torch.randn(T, h_out, generator=g).to(dtype) for _ in range(3)]
        # the last pool row stands for "no row": zeros for the oracle, out of the pool's bounds for the op
        spare = pool.key_buffer.shape[0] - 1
        pool.key_buffer[-1], pool.value_buffer[-1] = 0, 0
        pool.a_loc[torch.where(pool.a_loc == spare)[0]] = next(r for r in range(spare) if r not in set(pool.a_loc.tolist()))
        seen = pool.a_loc.clone()
        for slot in range(3):
            at = int(pool.a_start[-1]) + ranks[-1] * slot + 3 * slot + 1
            seen[at], pool.a_loc[at] = spare, (-1, spare + 1, 1 << 40)[slot]
        pd, xd = pool.to(dev), x.to(dev)
        idx = (pd.a_start, pd.a_len, pd.a_loc)
        plan = LoraPlan(ids.to(dev), pd.a_start, pd.a_len, R, hidden=h_in, bm_shrink=128, bm_expand=32, ksplit=ksplit,
                        reduce_in_expand=False, one_launch=False)
        alone = []
        for z in range(3):
            y = y0[z].to(dev)
            plan.apply(y, xd, pd.key_buffer, pd.value_buffer, *idx, z, pd.a_scaling)
            alone.append(y.cpu())
            want = O.lora_op(y0[z], x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, seen, ids, z, pool.a_scaling)
            assert_parity(alone[-1], want, f"{h_in} {ksplit} {ranks} target {z}")
        for slots in ((0, 1, 2), (2, 0)):
            ys = [y0[z].to(dev) for z in slots]
            plan.apply_multi(ys, xd, pd.key_buffer, pd.value_buffer, *idx, list(slots), pd.a_scaling)
            for z, y in zip(slots, ys):
                assert torch.equal(y.cpu(), alone[z]), f"{h_in} {ksplit} {ranks} targets {slots}, {z}"


@pytest.mark.parametrize("T,h_in,ksplit,rank,n,together", [
    (5249, 1032, 4, 16, 3, 1),     # 42 tiles: the odd block of columns and a K remainder, together
    (5120, 1032, 4, 64, 3, 1), (4992, 1032, 4, 64, 3, 0),       # 160 and 156 workgroups at least
    (4096, 1032, 4, 40, 2, 1), (3968, 1032, 4, 40, 2, 0),       # 128 and 124
    (8064, 1032, 4, 32, 3, 1), (8192, 1032, 4, 32, 3, 0), (10624, 264, 4, 32, 3, 0), (10752, 264, 4, 32, 3, 1),   # 256, 260, 336, 340 usually
    (3968, 2056, 16, 24, 2, 1), (4096, 2056, 16, 24, 2, 0), (5504, 2056, 16, 16, 3, 0), (5632, 2056, 16, 16, 3, 1),   # 512, 528, 704, 720
    (5760, 1032, 4, 128, 3, 1), (5632, 1032, 4, 128, 3, 0), (4736, 1032, 4, 72, 2, 1), (4608, 1032, 4, 72, 2, 0),
])
def test_both_sides_of_the_rule(dev, T, h_in, ksplit, rank, n, together):
    """The route a call takes, and the bits of separate calls on it."""
    ranks = (rank, 8)
    assert _lib.lib().mlora_targets_together(T, len(ranks), rank, 128, ksplit, n) == together
    g = torch.Generator().manual_seed(T + h_in)
    ids = torch.where(torch.arange(T) < T // 3 + 5, 1, 0)[torch.randperm(T, generator=g)]
    pool = W.make_pool(list(ranks), h_in, 72, torch.float16, g, True, std=0.05, heads=1).to(dev)
    x = torch.randn(T, h_in, generator=g).to(torch.float16).to(dev)
    idx = (pool.a_start, pool.a_len, pool.a_loc)
    plan = LoraPlan(ids.to(dev), *idx[:2], rank, hidden=h_in, bm_shrink=128, bm_expand=32, ksplit=ksplit, reduce_in_expand=False, one_launch=False)
    ys = [torch.zeros(T, 72, dtype=torch.float16, device=dev) for _ in range(2 * n)]
    plan.apply_multi(ys[:n], x, pool.key_buffer, pool.value_buffer, *idx, list(range(n)), pool.a_scaling)
    for z in range(n):
        plan.apply(ys[n + z], x, pool.key_buffer, pool.value_buffer, *idx, z, pool.a_scaling)
        assert ys[z].any() and torch.equal(ys[z], ys[n + z]), z


@pytest.mark.parametrize("T,ranks", [(5401, (16, 8, 8, 16)), (5402, (32, 8, 24, 16)), (5403, (64, 8, 40, 16)), (5901, (128, 8, 72, 40))])
@pytest.mark.parametrize("h_in,ksplit", [(1032, 4), (1024, 2), (4104, 4), (520, 3)])
@pytest.mark.parametrize("n", [2, 3])
def test_together(dev, T, ranks, h_in, ksplit, n):
    """Calls that do go together: adapters of several rank classes with short last tiles, K remainders, rank rows outside the index
    or the pool, against separate calls (same bits) and the oracle."""
    T = T if ksplit == 4 else T * 4 // ksplit
    A, R = len(ranks), max(ranks)
    assert _lib.lib().mlora_targets_together(T, A, R, 128, ksplit, n) == 1
    g = torch.Generator().manual_seed(T + h_in)
    dtype = torch.bfloat16 if T % 2 else torch.float16
    lens = torch.tensor([T // 3 + 1, T // 6 + 127, 129, 0])
    lens[3] = T - int(lens.sum()) - 7
    ids = torch.cat([torch.repeat_interleave(torch.arange(A), lens), torch.full((7,), -1)])[torch.randperm(T, generator=g)]
    pool = W.make_pool(list(ranks), h_in, 72, dtype, g, True, std=0.05, heads=1, extra_rows=1)
    spare = pool.key_buffer.shape[0] - 1   # zeros for the oracle, out of the pool's bounds for the op
    pool.key_buffer[-1], pool.value_buffer[-1] = 0, 0
    pool.a_loc[pool.a_loc == spare] = 0
    seen = pool.a_loc.clone()
    for slot in range(3):
        at = int(pool.a_start[slot]) + ranks[slot] * slot + 2 * slot + 1
        seen[at], pool.a_loc[at] = spare, (-1, spare + 1, 1 << 40)[slot]
    x = torch.randn(T, h_in, generator=g).to(dtype)
    y0 = torch.randn(T, 72, generator=g).to(dtype)
    pd, xd = pool.to(dev), x.to(dev)
    idx = (pd.a_start, pd.a_len, pd.a_loc)
    plan = LoraPlan(ids.to(dev), *idx[:2], R, hidden=h_in, bm_shrink=128, bm_expand=32, ksplit=ksplit, reduce_in_expand=False, one_launch=False)
    ys = [y0.to(dev) for _ in range(2 * n)]
    plan.apply_multi(ys[:n], xd, pd.key_buffer, pd.value_buffer, *idx, list(range(n)), pd.a_scaling)
    for z in range(n):
        plan.apply(ys[n + z], xd, pd.key_buffer, pd.value_buffer, *idx, z, pd.a_scaling)
        assert torch.equal(ys[z], ys[n + z]), z
    want = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, seen, ids, n - 1, pool.a_scaling)
    assert_parity(ys[n - 1].cpu(), want, f"{T} {h_in} {ksplit} {ranks}")
