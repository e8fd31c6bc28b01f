"""GPU parity of merge / unmerge of an adapter into the base weights and of the deLoRA compensation
op against oracle/lora_oracle.py.  Small-integer weights make the comparison bit-exact; random
weights are compared to one unit in the last place of the result (the accumulation order inside a
GEMM is not part of the reference's contract)."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import workloads as W
from valora_amd.merge import DeLoraPlan, merge_adapter, unmerge_adapter
from tests._util import assert_parity
from tests.test_merge_oracle_pins import int_pool

pytestmark = pytest.mark.gpu


def ulp_of(t):
    a = t.float().abs().clamp_min(2.0 ** -14)
    mant = 10 if t.dtype == torch.float16 else 7
    return torch.exp2(torch.floor(torch.log2(a)) - mant)


def run_merge(dev, Ws, pool, adapter, scaling, slots, sign, max_rank=None, ld=None):
    H_in, H_out = Ws[0].shape
    if ld is None:
        Wd = [w.clone().to(dev) for w in Ws]
    else:    # weights that are column slices of a wider matrix
        big = [torch.zeros(H_in, ld, dtype=Ws[0].dtype, device=dev) for _ in Ws]
        for b, w in zip(big, Ws):
            b[:, :H_out] = w.to(dev)
        Wd = [b[:, :H_out] for b in big]
    p = pool.to(dev)
    fn = merge_adapter if sign > 0 else unmerge_adapter
    fn(Wd, p.key_buffer, p.value_buffer, p.a_start, p.a_len, p.a_loc, adapter, scaling,
       max_rank or max(pool.ranks), slots=slots, n_slots=pool.n_slots)
    return [w.cpu() for w in Wd]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,ranks", [(64, [8, 16, 8]), (256, [32, 64, 8, 16]), (1000, [128, 8]), (4096, [16, 64])])
def test_merge_integer_weights_bit_exact(dev, dtype, H, ranks):
    pool = int_pool(H, ranks, dtype, seed=H)
    g = torch.Generator().manual_seed(H + 1)
    for adapter in range(len(ranks)):
        Ws = [torch.randint(-8, 9, (H, H), generator=g).to(dtype) for _ in range(4)]
        for sign in (1, -1):
            want = O.merge_adapter(Ws, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc,
                                   adapter, 2.0, sign=sign)
            got = run_merge(dev, Ws, pool, adapter, 2.0, (0, 1, 2, 3), sign)
            for k in range(4):
                assert torch.equal(got[k], want[k]), f"adapter {adapter} slot {k} sign {sign}"


@pytest.mark.parametrize("H_in,H_out,rank", [(3080, 3000, 128), (4104, 2064, 64), (136, 264, 128), (8, 4096, 64), (4096, 8, 128)])
def test_merge_several_slices_of_A_per_workgroup(dev, H_in, H_out, rank):
    """Shapes at the edges of the split over slices: several slices per workgroup with a ragged last one, a last
    workgroup with fewer slices than the others, matrices smaller than a tile in either direction."""
    g = torch.Generator().manual_seed(H_in + rank)
    pool = W.make_pool([rank], H_in, H_out, torch.bfloat16, g, True, heads=8)
    pool.key_buffer.copy_(torch.randint(-2, 3, pool.key_buffer.shape, generator=g))
    pool.value_buffer.copy_(torch.randint(-2, 3, pool.value_buffer.shape, generator=g))
    Ws = [torch.randint(-8, 9, (H_in, H_out), generator=g).to(torch.bfloat16) for _ in range(4)]
    want = O.merge_adapter(Ws, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, 0, 1.0, sign=1)
    got = run_merge(dev, Ws, pool, 0, 1.0, (0, 1, 2, 3), 1)
    for k in range(4):
        assert torch.equal(got[k], want[k]), f"slot {k}"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_merge_random_weights_and_views(dev, dtype):
    g = torch.Generator().manual_seed(8)
    H = 512
    pool = W.make_pool([16, 64, 32], H, H, dtype, g, True, std=0.05, scalings=[2.0, 0.5, 1.0], heads=8)
    Ws = [(torch.randn(H, H, generator=g) * 0.05).to(dtype) for _ in range(3)]
    for adapter, scaling in ((0, 2.0), (1, 0.3), (2, 1.7)):
        want = O.merge_adapter(Ws, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, adapter,
                               scaling, slots=(3, 0, 1))
        for ld in (None, H + 64):
            got = run_merge(dev, Ws, pool, adapter, scaling, (3, 0, 1), 1, ld=ld)
            for k in range(3):
                d = (got[k].float() - want[k].float()).abs()
                # one ulp of the rounded GEMM result (|ab| <= |W| + |W'|) may move the sum by as much
                big = torch.maximum(want[k].float().abs(), Ws[k].float().abs()).to(dtype)
                assert (d <= 2 * ulp_of(big)).all(), f"adapter {adapter} slot {k}: more than one ulp of ab"
                assert (d > 0).float().mean() < 0.02
        # merge then unmerge: back to within one rounding of the start, like the reference
        m = run_merge(dev, Ws, pool, adapter, scaling, (3, 0, 1), 1)
        back = run_merge(dev, m, pool, adapter, scaling, (3, 0, 1), -1)
        for k in range(3):
            big = torch.maximum(m[k].float().abs(), Ws[k].float().abs()).to(dtype)
            assert ((back[k].float() - Ws[k].float()).abs() <= 2 * ulp_of(big)).all()


def test_merge_rejects_bad_arguments(dev):
    g = torch.Generator().manual_seed(9)
    pool = W.make_pool([8], 64, 64, torch.float16, g, True, heads=8).to(dev)
    w = torch.zeros(64, 64, dtype=torch.float16, device=dev)
    args = (pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc)
    with pytest.raises(RuntimeError, match="adapter"):
        merge_adapter([w], *args, 5, 1.0, 8, slots=(0,))
    with pytest.raises(RuntimeError, match="slot"):
        merge_adapter([w], *args, 0, 1.0, 8, slots=(4,))
    with pytest.raises(RuntimeError, match="one shape"):
        merge_adapter([w, w[:32]], *args, 0, 1.0, 8, slots=(0, 1))
    with pytest.raises(RuntimeError, match="max_rank"):
        merge_adapter([w], *args, 0, 1.0, 12, slots=(0,))


@pytest.mark.parametrize("n", [2, 3, 5])
def test_delora_compensation(dev, n):
    """The merged adapter lives in W; every other request is compensated.  Compared with the oracle and,
    end to end, with base + LoRA of the token's own adapter."""
    small = {2: dict(hidden=512, n_tokens=96, n_adapters=24), 3: dict(hidden=256, mlp=704, len_div=8, n_decode=40),
             5: dict(hidden=256, mlp=704, len_div=8, n_decode=48, n_adapters=20)}[n]
    w = W.CONFIGS[n](**small)
    wd = w.to(dev)
    t = w.target("q"); p = t.pool; pd = wd.target("q").pool
    merged = int(torch.bincount(w.ids[w.ids >= 0]).argmax())
    R = max(p.ranks)
    plan = DeLoraPlan(wd.ids, merged, pd.a_start, pd.a_len, R, hidden=t.h_in)
    y = wd.y0["q"].clone()
    plan.apply(y, wd.x[t.h_in], pd.key_buffer, pd.value_buffer, pd.a_start, pd.a_len, pd.a_loc, t.slot, pd.a_scaling)
    want = O.delora_compensate(w.y0["q"], w.x[t.h_in], p.key_buffer, p.value_buffer, p.a_start, p.a_len, p.a_loc,
                               w.ids, merged, t.slot, p.a_scaling)
    assert_parity(y.cpu(), want, f"config{n} deLoRA compensation")
    same = (w.ids == merged)
    assert torch.equal(y.cpu()[same], w.y0["q"][same])

    # end to end: x @ W_merged + compensation == x @ W + LoRA_own(x)
    g = torch.Generator().manual_seed(n)
    H = t.h_in
    Wb = (torch.randn(H, H, generator=g) * 0.02).to(w.dtype)
    Wm = Wb.clone().to(dev)
    merge_adapter([Wm], pd.key_buffer, pd.value_buffer, pd.a_start, pd.a_len, pd.a_loc, merged,
                  float(p.a_scaling[merged]), R, slots=(t.slot,))
    x = wd.x[H]
    out = (x.float() @ Wm.float())
    comp = torch.zeros(w.T, H, dtype=w.dtype, device=dev)
    plan.apply(comp, x, pd.key_buffer, pd.value_buffer, pd.a_start, pd.a_len, pd.a_loc, t.slot, pd.a_scaling)
    out = (out + comp.float()).cpu()
    lora = O.lora_op(torch.zeros(w.T, H, dtype=w.dtype), w.x[H], p.key_buffer, p.value_buffer, p.a_start, p.a_len,
                     p.a_loc, w.ids, t.slot, p.a_scaling, round_v=False).float()
    ref = w.x[H].float() @ Wb.float() + lora
    has = w.ids >= 0
    err = (out - ref)[has].abs().max()
    assert err <= (6e-2 if w.dtype == torch.bfloat16 else 8e-3) * (1 + ref[has].abs().max()), err


@pytest.mark.parametrize("ranks,T,kw", [
    ([8], 1, {}), ([16, 8, 32], 33, {}), ([64, 8, 24], 300, dict(bm_shrink=32, ksplit=4, bm_expand=32)),
    ([128, 16, 64], 130, dict(bm_shrink=16, ksplit=2, bm_expand=16)), ([32, 64, 8], 517, dict(bm_shrink=64, ksplit=1, bm_expand=96)),
    ([64, 16], 700, dict(bm_shrink=128, ksplit=4, bm_expand=128)), ([16, 8, 64], 300, dict(bm_shrink=256, ksplit=2, bm_expand=48)),
    ([16, 40], 90, dict(bm_shrink=16, ksplit=4, bm_expand=16, shrink_recompute=True))])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_compensation_shapes(dev, ranks, T, kw, dtype):
    """The two products of a compensation call over every shrink tile height and way to finish the split-K sum: tiles
    of the merged adapter that cross the borders of the tokens' own tiles, ragged last tiles, a merged adapter of
    another rank, tokens without adapter, all tokens with the merged adapter, a merged adapter that does not exist."""
    g = torch.Generator().manual_seed(T + len(ranks))
    h_in, h_out = 520, 392
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, std=0.05, heads=1, scalings=[0.5 + 0.25 * i for i in range(len(ranks))])
    pd = pool.to(dev)
    idx = (pd.a_start, pd.a_len, pd.a_loc)
    x, y0 = torch.randn(T, h_in, generator=g).to(dtype), torch.randn(T, h_out, generator=g).to(dtype)
    mixed = torch.randint(-1, len(ranks), (T,), generator=g)
    for ids, merged in ((mixed, 0), (mixed, len(ranks) - 1), (torch.zeros(T, dtype=torch.long), 0), (mixed, -1)):
        plan = DeLoraPlan(ids.to(dev), merged, pd.a_start, pd.a_len, max(ranks), hidden=h_in, **kw)
        for slot in (0, 3):
            y = y0.to(dev)
            plan.apply(y, x.to(dev), pd.key_buffer, pd.value_buffer, *idx, slot, pd.a_scaling)
            if merged < 0:
                want = O.lora_op(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, ids, slot,
                                 pool.a_scaling)
            else:
                want = O.delora_compensate(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc,
                                           ids, merged, slot, pool.a_scaling)
            assert_parity(y.cpu(), want, f"ranks {ranks} T {T} merged {merged} slot {slot}")
            same = (ids == merged) | (ids < 0)
            assert torch.equal(y.cpu()[same], y0[same])


@pytest.mark.parametrize("T,kw", [
    (1, {}), (33, {}), (300, dict(bm_shrink=16, ksplit=1, bm_expand=16)), (300, dict(bm_shrink=32, ksplit=4, bm_expand=32)),
    (517, dict(bm_shrink=64, ksplit=2, bm_expand=96)), (700, dict(bm_shrink=128, ksplit=4, bm_expand=128)),
    (1300, dict(bm_shrink=256, ksplit=2, bm_expand=256)), (90, dict(bm_shrink=16, ksplit=4, bm_expand=16, shrink_recompute=True))])
def test_compensation_of_unusable_own_ranks(dev, T, kw):
    """A token whose own adapter has no usable rank (0, not a multiple of 8, above 128) has no product of its own, and the
    merged adapter comes off it all the same; its scale is not looked at.  With a merged adapter that has no usable rank
    such a token is left alone."""
    g = torch.Generator().manual_seed(T)
    h_in, h_out, dtype = 520, 392, torch.float16
    ranks = [32, 8, 16, 8, 64]
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, std=0.05, heads=1, scalings=[0.5 + 0.25 * i for i in range(len(ranks))])
    a_len, usable = pool.a_len.clone(), pool.a_len.clone()
    for a, rank in ((1, 0), (2, 12), (3, 136)):
        a_len[a], usable[a] = 4 * rank, 0
    scales = pool.a_scaling.clone()
    scales[1:4] = torch.tensor([float("nan"), float("inf"), 2.0])
    pd = pool.to(dev)
    idx = (pd.a_start, a_len.to(dev), pd.a_loc)
    x, y0 = torch.randn(T, h_in, generator=g).to(dtype), torch.randn(T, h_out, generator=g).to(dtype)
    ids = torch.randint(-1, len(ranks), (T,), generator=g)
    ids[0] = 1
    for merged in (0, 4, 1, 2):
        plan = DeLoraPlan(ids.to(dev), merged, idx[0], idx[1], 64, hidden=h_in, **kw)
        y = y0.to(dev)
        plan.apply(y, x.to(dev), pd.key_buffer, pd.value_buffer, *idx, 2, scales.to(dev))
        want = O.delora_compensate(y0, x, pool.key_buffer, pool.value_buffer, pool.a_start, usable, pool.a_loc, ids, merged, 2,
                                   scales)
        assert_parity(y.cpu(), want, f"T {T} merged {merged}")
        same = (ids == merged) | (ids < 0)
        if merged in (1, 2):
            same |= (ids >= 1) & (ids <= 3)
        assert torch.equal(y.cpu()[same], y0[same])


@pytest.mark.parametrize("seed", range(24))
def test_merge_random_shapes(dev, seed):
    """Non-square weights, widths that are multiples of 8 only, 1-5 pool slots, any subset of slots,
    weights that are column slices of a wider matrix (whose other columns must stay untouched)."""
    import random
    rnd = random.Random(seed)
    dtype = rnd.choice([torch.float16, torch.bfloat16])
    h_in, h_out = (rnd.choice([8, 24, 72, 136, 264, 520, 1000, 1032, 2056]) for _ in range(2))
    ranks = [rnd.choice([8, 16, 24, 32, 40, 64, 128]) for _ in range(rnd.choice([1, 2, 4]))]
    n_slots = rnd.choice([1, 2, 4, 5])
    slots = rnd.sample(range(n_slots), rnd.randint(1, min(4, n_slots)))
    adapter, scaling, sign = rnd.randrange(len(ranks)), rnd.choice([1.0, 2.0, 0.5, 1.7, 0.3]), rnd.choice([1, -1])
    pad = rnd.choice([0, 8, 64])
    what = f"seed {seed} {dtype} {h_in}x{h_out} ranks {ranks} slots {slots}/{n_slots} s {scaling} sign {sign} pad {pad}"
    print(what, flush=True)
    g = torch.Generator().manual_seed(seed)
    pool = W.make_pool(ranks, h_in, h_out, dtype, g, True, n_slots=n_slots, std=0.05, heads=1)
    Ws = [(torch.randn(h_in, h_out, generator=g) * 0.05).to(dtype) for _ in slots]
    want = O.merge_adapter(Ws, pool.key_buffer, pool.value_buffer, pool.a_start, pool.a_len, pool.a_loc, adapter,
                           scaling, slots=slots, n_slots=n_slots, sign=sign)
    big = [torch.zeros(h_in, h_out + pad, dtype=dtype, device=dev) for _ in Ws]
    for b, w in zip(big, Ws):
        b[:, :h_out] = w.to(dev)
    Wd = [b[:, :h_out] for b in big]
    p = pool.to(dev)
    fn = merge_adapter if sign > 0 else unmerge_adapter
    fn(Wd, p.key_buffer, p.value_buffer, p.a_start, p.a_len, p.a_loc, adapter, scaling, max(ranks), slots=slots,
       n_slots=n_slots)
    for k in range(len(slots)):
        d = (Wd[k].cpu().float() - want[k].float()).abs()
        lim = 2 * ulp_of(torch.maximum(want[k].float().abs(), Ws[k].float().abs()).to(dtype))
        assert (d <= lim).all(), what + f" target {k}: more than one ulp of ab"
        assert (d > 0).float().mean() < 0.03, what
        assert not big[k][:, h_out:].any(), what + " wrote outside the weight's columns"
