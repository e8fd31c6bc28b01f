"""The 128- and 256-token shrink tiles at the edges of their K steps (64 elements; whole steps are loaded without looking
at any lane, a last step that is not whole is masked) and of their tiles and waves (rows past the tile's end read another
row), against the oracle at the tolerance of the whole op."""
import pytest
import torch

from oracle import lora_oracle as O
from valora_amd import workloads as W
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
