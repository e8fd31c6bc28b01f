"""GPU: the adapter-grouped plan and the run-length encoder.

The run-length encoding must be bit-exact with the reference's count_consecutive_requests
(checked against the CPU oracle).  The grouped tile list is the build's own structure and is
checked by invariants: perm is a permutation of the tokens that have an adapter, every group's
size equals the histogram of ids, order inside a group is the original order (stable), tiles
partition the groups."""
import numpy as np
import pytest
import torch

from oracle import lora_oracle as O

pytestmark = pytest.mark.gpu


def _check_plan(ids_cpu, a_len_cpu, n_slots, bm_s, bm_e, dev):
    from valora_amd.plan import LoraPlan
    A = a_len_cpu.numel()
    a_start = (torch.cumsum(a_len_cpu, 0) - a_len_cpu).to(dev)
    plan = LoraPlan(ids_cpu.to(dev), a_start, a_len_cpu.to(dev), 64, n_slots=n_slots, bm_shrink=bm_s,
                    bm_expand=bm_e, ksplit=1)
    h = plan.header()
    ranks = (a_len_cpu // n_slots).tolist()
    valid = [t for t, a in enumerate(ids_cpu.tolist()) if 0 <= a < A and ranks[a] > 0]
    assert h["magic"] == 0x4d4c5241 and h["T"] == ids_cpu.numel()
    assert h["n_active"] == len(valid)
    perm = plan.perm().cpu().tolist()
    assert sorted(perm) == valid, "perm must be a permutation of the tokens that have an adapter"
    pa = plan.position_adapters().cpu().tolist()
    pr = plan.position_ranks().cpu().tolist()
    assert pa == [int(ids_cpu[t]) for t in perm]
    assert pr == [ranks[a] for a in pa]
    assert pa == sorted(pa), "positions are grouped by ascending adapter"
    for i in range(1, len(perm)):
        if pa[i] == pa[i - 1]:
            assert perm[i] > perm[i - 1], "original order is kept inside a group (stable)"
    hist = np.bincount([int(ids_cpu[t]) for t in valid], minlength=A) if valid else np.zeros(A, int)
    assert h["n_groups"] == int((hist > 0).sum())
    assert h["max_rank"] == max([ranks[a] for a in range(A) if hist[a] > 0], default=0)
    for tiles, bm, key in ((plan.tiles_shrink(), bm_s, "n_tiles_shrink"), (plan.tiles_expand(), bm_e, "n_tiles_expand")):
        tiles = tiles.cpu().tolist()
        assert len(tiles) == h[key] == int(sum(-(-c // bm) for c in hist if c > 0))
        pos = 0
        for (a, r, p0, cnt, st, *_rest) in tiles:
            assert p0 == pos and 1 <= cnt <= bm and r == ranks[a] and st == int(a_start[a])
            assert all(x == a for x in pa[p0:p0 + cnt])
            pos += cnt
        assert pos == len(valid)


@pytest.mark.parametrize("T,A,style", [
    (1, 1, "random"), (256, 64, "zipf"), (1000, 7, "random"), (4416, 32, "runs"), (64, 600, "random"),
    (5000, 5000, "random"), (300, 8192, "random"), (3000, 2048, "random"), (3000, 2049, "random"), (777, 3, "holes"), (20000, 16, "runs"), (0, 4, "random")])
def test_plan_invariants(dev, T, A, style):
    g = torch.Generator().manual_seed(T * 31 + A)
    a_len = torch.randint(1, 9, (A,), generator=g) * 8 * 4
    if style == "zipf":
        from valora_amd.workloads import zipf_ids
        ids = zipf_ids(A, T, 0.6, g)
    elif style == "runs":
        ids = torch.repeat_interleave(torch.randint(0, A, (T,), generator=g),
                                      torch.randint(1, 600, (T,), generator=g))[:T]
    elif style == "holes":
        ids = torch.randint(-2, A + 2, (T,), generator=g)       # out-of-range ids = no adapter
        a_len[1] = 0                                            # rank-0 adapter = no adapter
    else:
        ids = torch.randint(0, A, (T,), generator=g) if T else torch.zeros(0, dtype=torch.long)
    for bm_s, bm_e in ((16, 32), (64, 256)):
        _check_plan(ids, a_len, 4, bm_s, bm_e, dev)


@pytest.mark.parametrize("T,A", [(512, 8), (513, 8), (1024, 512), (1025, 33), (4096, 600), (4097, 3), (16385, 9), (40000, 2047), (2000, 4097)])
def test_plan_in_parts(dev, T, A):
    """Both sides of the sizes at which a plan is written by one, four or eight workgroups, with fewer histogram rows than
    waves, and with rows that take more than one batch of look-ups."""
    g = torch.Generator().manual_seed(T + A)
    a_len = torch.randint(0, 9, (A,), generator=g) * 8 * 4
    a_len[A // 2] = 32
    runs = torch.repeat_interleave(torch.randint(-1, A + 1, (T,), generator=g), torch.randint(1, 300, (T,), generator=g))[:T]
    mixed = torch.where(torch.rand(T, generator=g) < 0.5, runs, torch.randint(0, A, (T,), generator=g))
    for ids in (runs, mixed):
        _check_plan(ids, a_len, 4, 16, 96, dev)


@pytest.mark.parametrize("T,A", [(7, 2048), (7, 2049), (600, 2049), (3000, 2049), (8, 8192)])
def test_compensation_plan_keeps_adapters_without_a_rank(dev, T, A):
    """Their tokens have no product of their own, but the merged adapter's comes off them: on both sides of the number of
    adapters whose tables fit in LDS."""
    from valora_amd.plan import LoraPlan
    g = torch.Generator().manual_seed(T + A)
    rank = torch.randint(0, 3, (A,), generator=g) * 16
    rank[1] = 16
    ids = torch.where(torch.rand(T, generator=g) < 0.3, 1, torch.randint(-1, A + 1, (T,), generator=g))
    plan = LoraPlan(ids.to(dev), (torch.cumsum(rank, 0) * 4 - rank * 4).to(dev), (rank * 4).to(dev), 32, bm_shrink=32, bm_expand=48,
                    ksplit=1, _merged=1)
    want = sorted((t for t in range(T) if 0 <= ids[t] < A and ids[t] != 1), key=lambda t: (int(ids[t]), t))
    assert plan.perm().cpu().tolist() == want
    assert plan.position_ranks().cpu().tolist() == [int(rank[ids[t]]) for t in want]


@pytest.mark.parametrize("T,A", [(256, 512), (257, 512), (64, 513), (900, 2048), (901, 2048), (901, 513), (600, 2049), (601, 2049), (8, 8192)])
@pytest.mark.parametrize("merged", [-1, 1])
def test_plan_forms(dev, T, A, merged):
    """Both sides of the sizes at which the one-part form of the kernel ends, with unusable ranks, ids outside the index and
    several plans in one launch; a compensation plan leaves the merged adapter out and keeps adapters without a rank."""
    from valora_amd.plan import LoraPlan
    g = torch.Generator().manual_seed(T + A)
    rank = torch.randint(0, 3, (A,), generator=g) * 16
    rank[merged] = 16
    ids = torch.where(torch.rand(T, generator=g) < 0.3, 1, torch.randint(-1, A + 1, (T,), generator=g))
    a_len, a_start = rank * 4, torch.cumsum(rank * 4, 0) - rank * 4
    index = (ids.to(dev), a_start.to(dev), a_len.to(dev))
    plans = [LoraPlan(*index, 32, bm_shrink=32, bm_expand=48, ksplit=1, _merged=merged)]
    if merged < 0:
        plans += LoraPlan.of_widths(*index, 32, (4096, 11008))
    kept = [t for t in range(T) if 0 <= ids[t] < A and ids[t] != merged and (merged >= 0 or rank[ids[t]] > 0)]
    want = sorted(kept, key=lambda t: (int(ids[t]), t))   # stable, by adapter
    for p in plans:
        assert p.perm().cpu().tolist() == want
        assert p.position_adapters().cpu().tolist() == [int(ids[t]) for t in want]
        assert p.position_ranks().cpu().tolist() == [int(rank[ids[t]]) for t in want]
        for tiles, bm in ((p.tiles_shrink().cpu(), p.bm_shrink), (p.tiles_expand().cpu(), p.bm_expand)):
            at, seen = 0, []
            while at < len(want):
                a = int(ids[want[at]])
                n = min(bm, sum(1 for t in want[at:at + bm] if int(ids[t]) == a))
                seen.append([a, int(rank[a]), at, n if rank[a] > 0 else -n, int(a_start[a])])
                at += n
            assert tiles[:, :5].tolist() == seen


@pytest.mark.parametrize("T,A", [(1, 1), (700, 40), (5000, 33)])
def test_plans_cut_in_one_launch(dev, T, A):
    from valora_amd.plan import LoraPlan
    g = torch.Generator().manual_seed(T)
    a_len = (torch.randint(1, 9, (A,), generator=g) * 32).to(dev)
    a_start = torch.cumsum(a_len, 0) - a_len
    ids = torch.randint(0, A, (T,), generator=g).to(dev)
    widths = (4096, 11008, 2048, 4096)
    for w, p in zip(widths, LoraPlan.of_widths(ids, a_start, a_len, 64, widths)):
        q = LoraPlan(ids, a_start, a_len, 64, hidden=w)
        assert (p.bm_shrink, p.bm_expand, p.ksplit, p.flags) == (q.bm_shrink, q.bm_expand, q.ksplit, q.flags)
        assert p.header() == q.header()
        for a, b in ((p.perm(), q.perm()), (p.tiles_shrink(), q.tiles_shrink()), (p.tiles_expand(), q.tiles_expand()),
                     (p.position_adapters(), q.position_adapters()), (p.position_ranks(), q.position_ranks())):
            assert torch.equal(a, b)
        p.rebuild(ids.flip(0))
        q.rebuild(ids.flip(0))
        assert torch.equal(p.perm(), q.perm())
    with pytest.raises(RuntimeError):
        LoraPlan.of_widths(ids, a_start, a_len, 64, (4096,) * 5)


@pytest.mark.parametrize("T", [1, 2, 63, 64, 65, 1024, 1025, 5000])
@pytest.mark.parametrize("style", ["random", "runs", "equal", "distinct"])
def test_count_consecutive_bit_exact(dev, T, style):
    from valora_amd.segments import count_consecutive_requests
    g = torch.Generator().manual_seed(T)
    lora_rank = torch.tensor([32, 64, 128, 256, 32, 96])
    if style == "random":
        ids = torch.randint(0, 6, (T,), generator=g)
    elif style == "runs":
        ids = torch.repeat_interleave(torch.randint(0, 6, (T,), generator=g),
                                      torch.randint(1, 40, (T,), generator=g))[:T]
    elif style == "equal":
        ids = torch.full((T,), 4)
    else:
        ids = torch.arange(T) % 6
    oc, rc, li, st, num = count_consecutive_requests(lora_rank.to(dev), ids.to(dev))
    want = O.count_consecutive_requests(lora_rank, ids)
    P = int(num.item())
    assert P == len(want[0])
    for got, w in zip((oc, rc, li, st), want):
        assert got.dtype == torch.long and got[:P].cpu().tolist() == w


def test_planned_calls_give_the_interpreter_lock_back(dev):
    """With a switch interval no test outlasts, a thread that waits for the interpreter lock only gets it where the
    thread that holds it gives it back of its own accord.  Every planned call does, around its launches."""
    import sys
    import threading
    import time
    from valora_amd import workloads as W
    from valora_amd.merge import DeLoraPlan
    from valora_amd.plan import LoraPlan
    g = torch.Generator().manual_seed(1)
    pool = W.make_pool([8, 8], 64, 64, torch.float16, g, True, heads=1).to(dev)
    idx = (pool.a_start, pool.a_len, pool.a_loc)
    ids = torch.zeros(4, dtype=torch.long, device=dev)
    x, y, z = (torch.zeros(4, 64, dtype=torch.float16, device=dev) for _ in range(3))
    plan, de = LoraPlan(ids, idx[0], idx[1], 8, hidden=64), DeLoraPlan(ids, 1, idx[0], idx[1], 8, hidden=64)
    kb, vb, sc = pool.key_buffer, pool.value_buffer, pool.a_scaling
    calls = {"apply": lambda: plan.apply(y, x, kb, vb, *idx, 0, sc),
             "apply_multi": lambda: plan.apply_multi([y, z], x, kb, vb, *idx, [0, 1], sc),
             "compensate": lambda: de.apply(y, x, kb, vb, *idx, 0, sc), "rebuild": lambda: plan.rebuild(ids)}
    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)

    thread = threading.Thread(target=other)
    was = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        thread.start()
        seen = {}
        for name, call in calls.items():
            before = turns[0]
            for _ in range(200):
                call()
            seen[name] = turns[0] - before
    finally:
        stop.set()
        sys.setswitchinterval(was)
        thread.join()
    torch.cuda.synchronize()
    assert all(n > 0 for n in seen.values()), seen
