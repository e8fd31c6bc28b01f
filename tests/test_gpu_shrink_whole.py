"""Shrinks of one target over a few thousand tokens, all of K in one workgroup of eight waves: at the edges of the pieces and of K,
through every entry point that writes such a result and over plans of other tile heights, against the oracle at the
tolerance of the whole op; then on both sides of every bound of the rule that takes them."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import _lib, workloads as W
from valora_amd.plan import LoraPlan
from tests._util import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,h_in,ranks", [
    (4479, 520, (8, 16)),           # below the rule: the table's tiles
    (4480, 520, (8, 16)),
    (4480, 72, (16,)),              # one step and an eighth of K: most waves have none
    (4800, 8, (8, 8)),
    (5001, 1032, (32, 8, 24)),
    (4700, 5120, (16, 8)),
    (6080, 3080, (32, 16)),         # too few pieces with rank above 16 and more than 3072 wide: the table's tiles
    (6112, 3080, (32, 16)),
    (6000, 584, (64, 40, 8, 16, 128)),
    (4600, 1096, (32,) * 100),      # a tail per adapter
    (8191, 264, (16,)),             # the last of one round of 32-token pieces
    (12000, 264, (16, 8, 8)),       # past it and too narrow for 64-token ones: the table's tiles
    (16383, 136, (8,)),
    (16448, 136, (8,)),
])
def test_entry_points(dev, T, h_in, ranks):
    from valora_amd.atmm_ops import dispatch_bgmv as dispatch_sgmm, shrink_accumulate
    from valora_amd.kernels import dispatch_bgmv
    from valora_amd.lora_prefill import lora_get_qkvo_fwd_shrink
    g = torch.Generator().manual_seed(T + h_in)
    dtype = torch.bfloat16 if T % 2 else torch.float16
    A, R, slot = len(ranks), min(max(ranks), 64), 2
    pool = W.make_pool(list(ranks), h_in, h_in, dtype, g, True, std=0.05, heads=1)
    cut = torch.sort(torch.randint(0, T, (max(A, 3) * 2 - 1,), generator=g)).values.tolist()
    seq = torch.tensor([b - a for a, b in zip([0] + cut, cut + [T])], dtype=torch.int32)   # some of them empty
    req = torch.arange(len(seq)) % A
    start = (torch.cumsum(seq, 0) - seq).to(torch.int32)
    ids = torch.repeat_interleave(req, seq.long())
    x = torch.randn(T, h_in, generator=g).to(dtype)
    pd, xd = pool.to(dev), x.to(dev)
    idx = (pool.a_start, pool.a_len, pool.a_loc)
    idxd = (pd.a_start, pd.a_len, pd.a_loc)
    fresh = O.bgmv_shrink(torch.zeros(T, max(ranks)), x.float(), pool.key_buffer.float(), *idx, ids, slot)[:, :R]

    def start_of(ids_):   # columns past an adapter's rank and tokens without an adapter keep what is there
        had = torch.tensor(ranks)[ids_.clamp(min=0)].unsqueeze(1) > torch.arange(R)
        had &= (ids_ >= 0).unsqueeze(1)
        d0 = torch.randn(T, R, generator=g).to(dtype)
        return d0, torch.where(had, fresh.to(dtype), d0), had

    holes = torch.where(torch.rand(T, generator=g) < 0.1, -1, ids)
    holes = torch.where(torch.arange(T) == 0, ids, holes)
    for given in (ids, holes):
        d0, want, had = start_of(given)
        d = d0.to(dev)
        dispatch_bgmv(d, xd, pd.key_buffer, *idxd, given.to(dev), slot, pd.a_scaling)
        assert_parity(d.cpu(), want, f"bgmv {T} {h_in}")
        assert torch.equal(d.cpu()[~had], d0[~had])
    # a plan of the caller's: taller tiles go in pieces, lower ones stay
    d0, want, had = start_of(ids)
    for bm in (16, 32, 64, 128):
        plan = LoraPlan(ids.to(dev), pd.a_start, pd.a_len, R, hidden=h_in, bm_shrink=bm, bm_expand=32, one_launch=False)
        pk = _lib.make_pool(pd.key_buffer, *idxd, h_in)
        ws = torch.empty(_lib.lib().mlora_workspace_bytes(T, A, R), dtype=torch.uint8, device=dev)
        d = d0.to(dev)
        _lib.check(_lib.lib().mlora_dispatch_bgmv(_lib.current_stream(dev), _lib.ptr(d), _lib.ptr(xd), pk, None, slot, None, T,
                                                  h_in, R, _lib.dtype_code(dtype), _lib.ptr(ws), ws.numel(), plan.handle))
        assert_parity(d.cpu(), want, f"plan of {bm} {T} {h_in}")
        assert torch.equal(d.cpu()[~had], d0[~had])
    shrink_accumulate(True)
    try:
        d0 = torch.randn(T, R, generator=g).to(dtype)
        d = d0.to(dev)
        oc, rc, li, st = O.count_consecutive_requests(pool.a_len, ids)
        t = lambda l: torch.tensor(l + [1] * 4, dtype=torch.long, device=dev)
        tmp = torch.zeros(64 * max(8, len(oc)), dtype=torch.int8, device=dev)
        dispatch_sgmm(d, xd, pd.key_buffer, *idxd, ids.to(dev), slot, pd.a_scaling, t(oc), t(rc), t(li), t(st), tmp, len(oc),
                      64, 32, 32, 32, 32, 32)
        assert_parity(d.cpu(), (d0.float() + fresh).to(dtype), f"accumulate {T} {h_in}")
    finally:
        shrink_accumulate(False)
    o = torch.full((T, R), 2.5, dtype=dtype, device=dev)
    lora_get_qkvo_fwd_shrink(xd, pd.key_buffer.view(-1, h_in), o, pd.a_loc, pd.a_start, pd.a_len, start.to(dev), seq.to(dev),
                             req.to(dev), h_in, slot, R, int(seq.max()))
    assert_parity(o.cpu(), fresh.to(dtype), f"prefill shrink {T} {h_in}")


@pytest.mark.parametrize("T,h_in,ranks,tile", [
    (4480, 72, (16,), 32), (4479, 72, (16,), 0), (8192, 264, (16,), 32), (8193, 264, (16,), 0),     # 256 pieces
    (4600, 136, (32,) * 212, 32), (4600, 136, (32,) * 214, 0),                                      # 144 and 112 or 113 tails
    (5001, 2048, (32, 8), 32), (5001, 2056, (32, 8), 0), (5001, 2056, (32, 8) * 4, 32), (5001, 3064, (32, 8), 0), (5001, 3072, (32, 8), 32),
    (6368, 3080, (32, 16), 0), (6369, 3080, (32, 16), 32), (4600, 1032, (64, 16), 32),              # 199 and 200 pieces at least
    (8896, 3080, (16,), 0), (8897, 3080, (16, 8, 8), 64), (16384, 3072, (8,), 64), (16385, 3072, (8,), 0), (12000, 3064, (16,), 0),
])
@pytest.mark.parametrize("missing", [False, True])
def test_both_sides_of_the_rule(dev, T, h_in, ranks, tile, missing):
    """Which calls take the kernel, and their results with every pool row there and with rows outside the index or the pool."""
    from valora_amd._ext import binding
    from valora_amd.kernels import dispatch_bgmv
    A, R, slot = len(ranks), max(ranks), 1
    assert binding.one_call_tile(T, A, R, h_in) == tile
    g = torch.Generator().manual_seed(T + h_in)
    dtype = torch.bfloat16 if T % 2 else torch.float16
    pool = W.make_pool(list(ranks), h_in, h_in, dtype, g, True, std=0.05, heads=1, extra_rows=1)
    seen = pool.a_loc.clone()
    if missing:
        spare = pool.key_buffer.shape[0] - 1   # zeros for the oracle, out of the pool's bounds for the op
        pool.key_buffer[-1] = 0
        pool.a_loc[pool.a_loc == spare] = 0
        seen = pool.a_loc.clone()
        for a in range(0, A, 2):
            for i, bad in enumerate((-1, spare + 1, 1 << 40)):
                at = int(pool.a_start[a]) + ranks[a] * slot + 2 * i + 1
                seen[at], pool.a_loc[at] = spare, bad
    ids = torch.randint(-1, A, (T,), generator=g)
    x, d0 = torch.randn(T, h_in, generator=g).to(dtype), torch.randn(T, R, generator=g).to(dtype)
    want = O.bgmv_shrink(d0, x, pool.key_buffer, pool.a_start, pool.a_len, seen, ids, slot)
    pd, d = pool.to(dev), d0.to(dev)
    dispatch_bgmv(d, x.to(dev), pd.key_buffer, pd.a_start, pd.a_len, pd.a_loc, ids.to(dev), slot, pd.a_scaling)
    assert_parity(d.cpu(), want, f"{T} {h_in} {missing}")
    had = (torch.tensor(ranks)[ids.clamp(min=0)].unsqueeze(1) > torch.arange(R)) & (ids >= 0).unsqueeze(1)
    assert torch.equal(d.cpu()[~had], d0[~had])
