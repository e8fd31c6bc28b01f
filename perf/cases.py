"""Performance cases: the work a serving process has this package do, through its public entry points.

A case is one forward pass's share of LoRA work over some layers (each layer with its own adapter weights and
activations, as in a model), or one change of the resident / merged adapters between forward passes.

* ``plan``       the planned op (``valora_amd.plan.LoraPlan`` / ``valora_amd.layer.LayerPlans``): the tiles of the batch
                 are cut once per pass -- in place for a decode batch that keeps its size, a new plan for a batch with
                 prefill requests -- then q+k+v in one call, o, and with ``mlp`` gate+up in one call and down, per layer
* ``bgmv``       the reference caller's eight ``valora._kernels.dispatch_bgmv`` calls per layer (per-token ids)
* ``sgmm``       the same eight calls through ``atmm_ops.dispatch_bgmv``, with the segment tensors of the batch
* ``requests``   the same eight calls through the ``lora_prefill`` pair (per-request operands)
* ``compensate`` one adapter merged into the base weights, every other request corrected (``valora_amd.merge.DeLoraPlan``)
* ``switch``     the merged adapter of every layer exchanged (``unmerge_adapter`` + ``merge_adapter``)
* ``residency``  adapters of the next requests loaded from pinned host memory, those no longer wanted dropped
                 (``valora_amd.infer_adapter.InferAdapter``)
"""
from __future__ import annotations

import numpy as np
import torch

from valora_amd import atmm_ops, kernels, lora_prefill, segments
from valora_amd.infer_adapter import InferAdapter, LoraAdapterWeights, MemoryAllocator
from valora_amd.layer import LayerPlans
from valora_amd.merge import DeLoraPlan, merge_adapter, unmerge_adapter
from valora_amd.plan import LoraPlan

DEVICE = "cuda"
HEADS = 32
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
WEIGHT_STD = 0.02          # adapter weights, as the package's own workloads draw them
IMAGE_SCALE = 4.0          # image tokens have larger activations than text
MAX_BYTES = 4.0e9          # no drawn case moves more than the largest listed ones


def _case(name, kind, dtype, **kw):
    c = {"name": name, "kind": kind, "dtype": dtype, "hidden": 4096, "mlp": 0, "layers": 32, "adapters": 64, "ranks": "16",
         "skew": 0.6, "decode": 0, "prefill": 0, "shortest": 0, "longest": 0, "image": 0}
    c.update(kw)
    return c


def listed():
    return [
        # a lone request decoding: nothing but latency, launches and host work
        _case("decode_1", "plan", "fp16", adapters=8, decode=1),
        # a small server's decode batch on a 13B shape: odd size, adapters of many ranks, all seven projections
        _case("decode_77_ranks", "plan", "bf16", hidden=5120, mlp=13824, layers=8, adapters=33, ranks="8,16,32,64", skew=0.8,
              decode=77),
        # the headline decode batch: 256 requests over 64 adapters of rank 16, attention projections of 32 layers
        _case("decode_256", "plan", "fp16", decode=256),
        # decode where the adapters' weights are the traffic: 128 resident adapters of rank 128
        _case("decode_512_rank128", "plan", "fp16", layers=4, adapters=128, ranks="128", skew=0.7, decode=512),
        # the headline decode batch through the reference caller's own calls
        _case("bgmv_256", "bgmv", "fp16", decode=256),
        # four prefill requests of 128 tokens with an adapter each, through the segment signature
        _case("sgmm_4x128", "sgmm", "fp16", adapters=4, skew=0.0, prefill=4, shortest=128, longest=128),
        # a long ragged prefill batch through the per-request signature
        _case("requests_prefill", "requests", "fp16", layers=4, adapters=24, ranks="16,32", skew=0.8, prefill=19, shortest=33,
              longest=783),
        # continuous batching: ragged prefill requests among decoding ones, mixed ranks, all seven projections
        _case("mixed_ranks", "plan", "bf16", mlp=11008, layers=2, adapters=32, ranks="8,16,32,64", skew=0.8, decode=192,
              prefill=8, shortest=32, longest=1024),
        # vision requests: 256 image tokens and some text each, an adapter of rank 64 per request
        _case("vision_prefill", "plan", "bf16", mlp=11008, layers=2, adapters=16, ranks="64", skew=0.0, prefill=16,
              shortest=16, longest=128, image=256),
        # most requests use the merged adapter, the others are compensated
        _case("compensate_mixed", "compensate", "fp16", layers=8, adapters=12, ranks="16,32,64", skew=1.2, decode=61, prefill=5,
              shortest=40, longest=300),
        # another adapter becomes the merged one
        _case("switch_rank64", "switch", "bf16", layers=8, adapters=2, ranks="64"),
        # four adapters come, four go, eight stay
        _case("residency_4_of_12", "residency", "fp16", adapters=4, ranks="16,32,64"),
    ]


def draw(rng):
    def between(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["plan", "plan", "plan", "plan", "bgmv", "bgmv", "sgmm", "requests", "compensate", "switch", "residency"])
    c = _case("", kind, rng.choice(["fp16", "bf16"]))
    del c["name"]
    hidden, mlp = rng.choice([(2048, 8192), (3072, 8192), (4096, 11008), (4096, 14336), (5120, 13824)])
    c["hidden"] = hidden
    c["ranks"] = rng.choice(["8", "16", "32", "64", "128", "8,16,32,64", "16,32,64", "16,64"])
    c["skew"] = round(rng.uniform(0.0, 1.2), 2)
    c["adapters"] = between(1, 128)
    if kind == "switch":
        c.update(adapters=2, layers=between(2, 8), skew=0.0)
        return _fit(c)
    if kind == "residency":
        c.update(adapters=between(1, 6), layers=between(8, 32), skew=0.0)
        return _fit(c)
    c["layers"] = between(4, 32)
    if kind in ("plan", "compensate") and rng.random() < 0.5:
        c["mlp"] = mlp if kind == "plan" else 0
    if kind in ("sgmm", "requests") or rng.random() < 0.4:
        c["prefill"] = between(1, 24)
        c["longest"] = between(24, 1024)
        c["shortest"] = between(8, c["longest"])
        c["image"] = rng.choice([0, 0, 0, 256])
    if not c["prefill"] or (kind in ("plan", "bgmv", "compensate") and rng.random() < 0.5):
        c["decode"] = between(1, 1024)
    if kind == "compensate":         # the merged adapter has part of the requests only
        c.update(adapters=max(3, c["adapters"] // 4), decode=between(32, 1024))
    return _fit(c)


def _fit(c):
    """Fewer layers, then fewer requests and adapters, until the case moves no more than MAX_BYTES and its state is
    small enough to be held several times."""
    while (c["layers"] > 2 and (work(c)["bytes"] > MAX_BYTES or _pool_bytes(c) > 12e9)):
        c["layers"] = max(2, c["layers"] * 3 // 4)
    while work(c)["bytes"] > MAX_BYTES and max(c["prefill"], c["adapters"], c["decode"]) > 2:
        for k in ("prefill", "adapters", "decode"):
            c[k] = max(min(c[k], 2), c[k] * 3 // 4)
    return c


# ---- the batch ---------------------------------------------------------------------------------------------------
def _ranks(c, n):
    """Ranks of n adapters: the case's, in turn."""
    r = [int(v) for v in c["ranks"].split(",")]
    return [r[i % len(r)] for i in range(n)]


def _batch(c, seed):
    """(adapter of each request, tokens of each request, activation scale of each token or None).  The lengths are
    the case's own, who asks for what is the seed's; prefill requests come first, as in the reference's batches."""
    shape = np.random.RandomState(c["prefill"] * 7919 + c["longest"])
    lens = (shape.randint(c["shortest"], c["longest"] + 1, c["prefill"]) if c["prefill"] else np.zeros(0, dtype=np.int64))
    lens = np.concatenate([lens + c["image"], np.ones(c["decode"], dtype=np.int64)]).astype(np.int64)
    n = c["adapters"]
    p = np.arange(1, n + 1, dtype=np.float64) ** -c["skew"]
    rng = np.random.RandomState(seed % (1 << 31))
    if c["skew"] == 0.0 and len(lens) <= n:
        bins = rng.permutation(n)[: len(lens)]          # an adapter per request
    else:
        bins = rng.choice(n, size=len(lens), p=p / p.sum())
    scale = None
    if c["image"]:
        scale = np.ones(int(lens.sum()), dtype=np.float32)
        for s, l in zip(np.cumsum(lens) - lens, lens):
            if l > 1:
                scale[s:s + c["image"]] = IMAGE_SCALE
    return bins.astype(np.int64), lens, scale


def _index(ranks, rng, dtype):
    """The pool index of adapters whose rows lie scattered over the pool, as they do after a while of serving."""
    lens = np.array([4 * r for r in ranks], dtype=np.int64)
    scaling = np.array([(0.5, 1.0, 2.0)[i % 3] for i in range(len(ranks))], dtype=np.float32)
    to = lambda a: torch.from_numpy(a).to(DEVICE)  # noqa: E731
    return {"a_start": to(np.cumsum(lens) - lens), "a_len": to(lens), "a_loc": to(rng.permutation(int(lens.sum())).astype(np.int64)),
            "a_scaling": to(scaling).to(dtype), "rows": int(lens.sum()), "max_rank": max(ranks)}


def _pool_bytes(c):
    rows = 4 * sum(_ranks(c, c["adapters"]))
    width = 2 * c["hidden"] + (2 * c["hidden"] + 2 * c["mlp"] if c["mlp"] else 0)
    return 2 * rows * width * c["layers"]


class _State:
    """What a program holds between passes.  Tensors of all layers are allocated as one and held as a view per layer, as
    the layers of a model hold theirs; ``y`` keeps the whole output tensors."""

    def per_layer(self, **tensors):
        for name, t in tensors.items():
            setattr(self, name, list(t.unbind(0)))


def prepare(case, seed):
    c, s = case, _State()
    s.case, s.kind, s.layers = c, c["kind"], c["layers"]
    dtype = DTYPES[c["dtype"]]
    h, mlp, L = c["hidden"], c["mlp"], c["layers"]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    rng = np.random.RandomState((seed + 1) % (1 << 31))

    def normal(*shape, std=1.0):
        return torch.empty(*shape, dtype=dtype, device=DEVICE).normal_(0.0, std, generator=g)

    if s.kind == "residency":
        return _prepare_residency(s, c, dtype, normal)

    ranks = _ranks(c, c["adapters"])
    s.index = _index(ranks, rng, dtype)
    rows = s.index["rows"]
    # pool rows of A and of B: [layer, row, heads, head_dim]
    s.per_layer(key=normal(L, rows, HEADS, h // HEADS, std=WEIGHT_STD), value=normal(L, rows, HEADS, h // HEADS, std=WEIGHT_STD))
    if s.kind == "switch":
        s.w = normal(L, 4, h, h, std=h ** -0.5)                     # q, k, v, o weights, the first adapter merged in
        s.layer_w = [list(w.unbind(0)) for w in s.w.unbind(0)]
        s.rank, s.scaling, s.merged = ranks, s.index["a_scaling"].tolist(), 0
        return s
    if mlp:
        s.per_layer(key_up=normal(L, rows, HEADS, h // HEADS, std=WEIGHT_STD),
                    value_up=normal(L, rows, HEADS, mlp // HEADS, std=WEIGHT_STD),
                    key_down=normal(L, rows, HEADS, mlp // HEADS, std=WEIGHT_STD),
                    value_down=normal(L, rows, HEADS, h // HEADS, std=WEIGHT_STD))

    bins, lens, scale = _batch(c, seed)
    T = int(lens.sum())
    s.T, s.lens, s.bins = T, lens, bins
    s.req_bins = torch.from_numpy(bins).to(DEVICE)
    s.b_seq_len = torch.from_numpy(lens.astype(np.int32)).to(DEVICE)
    s.b_start_loc = torch.from_numpy((np.cumsum(lens) - lens).astype(np.int32)).to(DEVICE)
    s.longest = int(lens.max())
    s.ids = torch.from_numpy(np.repeat(bins, lens)).to(DEVICE)
    rowscale = None if scale is None else torch.from_numpy(scale).to(DEVICE, dtype)[:, None]

    def acts(width):
        x = normal(L, T, width)
        return x if rowscale is None else x.mul_(rowscale)

    # what the base model hands over: the inputs of the projections and their outputs, which the op adds to
    s.per_layer(x=acts(h), attn=acts(h))
    s.y = {n: normal(L, T, h) for n in ("q", "k", "v", "o")}
    if mlp:
        s.per_layer(h2=acts(h), m=acts(mlp))
        s.y["gate"], s.y["up"], s.y["down"] = normal(L, T, mlp), normal(L, T, mlp), normal(L, T, h)
    s.per_layer(**s.y)

    i = s.index
    if s.kind == "plan" and not c["prefill"]:   # a decode batch keeps its plan and cuts it again in place
        s.plans = _plans(s)
    if s.kind == "sgmm":
        s.dirs = ["adapter%d" % b for b in bins]
        s.rank_counts = torch.full((segments.SGMM_BUFFER_LEN,), i["max_rank"], dtype=torch.long, device=DEVICE)
        s.tmp = torch.zeros(128 * 60, dtype=torch.int8, device=DEVICE)
    if s.kind == "compensate":
        s.merged = int(np.bincount(bins, weights=lens, minlength=c["adapters"]).argmax())
    return s


def _prepare_residency(s, c, dtype, normal):
    h, L = c["hidden"], c["layers"]
    cfg = {"num_hidden_layers": L, "hidden_size": h}

    def adapter(name, r):
        home = torch.empty(L, 2, 4 * r, h, dtype=dtype, pin_memory=True)
        home.copy_(normal(L, 2, 4 * r, h, std=WEIGHT_STD))
        return LoraAdapterWeights(name, r, 2.0 * r, cfg, home)

    n = c["adapters"]
    coming = _ranks(c, n)
    staying = [adapter("stays%d" % i, 16) for i in range(2 * n)]
    s.sets = [[adapter("set%d_%d" % (k, i), r) for i, r in enumerate(coming)] for k in (0, 1)]
    total = 4 * 16 * 2 * n + 2 * 4 * sum(coming)
    mem = MemoryAllocator(total, total, dtype, HEADS, h // HEADS, L, device=DEVICE)
    mem.key_buffer.zero_()
    mem.value_buffer.zero_()
    s.adapters = InferAdapter.init(mem)
    s.adapters.load_adapters(staying)
    s.adapters.load_adapters(s.sets[0])
    s.stays, s.now = [a.lora_dir for a in staying], 0
    return s


def _plans(s):
    """The plan(s) of the batch: one for hidden-wide inputs and, with the MLP targets, one for MLP-wide inputs."""
    i, c = s.index, s.case
    if c["mlp"]:
        return LayerPlans(s.ids, i["a_start"], i["a_len"], i["max_rank"], c["hidden"], c["mlp"])
    return LoraPlan(s.ids, i["a_start"], i["a_len"], i["max_rank"], hidden=c["hidden"])


# ---- one pass ----------------------------------------------------------------------------------------------------
def run(state):
    return _RUN[state.kind](state)


def _run_plan(s):
    i = s.index
    idx = (i["a_start"], i["a_len"], i["a_loc"])
    sc = i["a_scaling"]
    if s.case["prefill"]:
        plans = _plans(s)
    else:
        plans = s.plans
        for p in ((plans.h, plans.m) if s.case["mlp"] else (plans,)):
            p.rebuild(s.ids)
    ph, pm = (plans.h, plans.m) if s.case["mlp"] else (plans, None)
    for l in range(s.layers):
        kb, vb = s.key[l], s.value[l]
        ph.apply_multi([s.q[l], s.k[l], s.v[l]], s.x[l], kb, vb, *idx, [0, 1, 2], sc)
        ph.apply(s.o[l], s.attn[l], kb, vb, *idx, 3, sc)
        if pm is not None:
            ph.apply_multi([s.gate[l], s.up[l]], s.h2[l], s.key_up[l], s.value_up[l], *idx, [0, 1], sc)
            pm.apply(s.down[l], s.m[l], s.key_down[l], s.value_down[l], *idx, 0, sc)
    return s.y


def _eight_calls(s, shrink, expand):
    """The reference caller's order: three shrinks into delta[0..2], three expands, then o through delta[0]."""
    delta = [torch.zeros(s.T, s.index["max_rank"], dtype=DTYPES[s.case["dtype"]], device=DEVICE) for _ in range(3)]
    for l in range(s.layers):
        kb, vb = s.key[l], s.value[l]
        for t in range(3):
            shrink(delta[t], s.x[l], kb, t)
        for t, y in enumerate((s.q[l], s.k[l], s.v[l])):
            expand(y, delta[t], vb, t)
        shrink(delta[0], s.attn[l], kb, 3)
        expand(s.o[l], delta[0], vb, 3)
    return s.y


def _run_bgmv(s):
    i = s.index
    idx = (i["a_start"], i["a_len"], i["a_loc"])
    ids = segments.batch_req_bins(s.req_bins, s.b_seq_len)
    op, sc = kernels.dispatch_bgmv, i["a_scaling"]
    return _eight_calls(s, lambda d, x, w, t: op(d, x, w, *idx, ids, t, sc), lambda y, d, w, t: op(y, d, w, *idx, ids, t, sc))


def _run_sgmm(s):
    i = s.index
    idx = (i["a_start"], i["a_len"], i["a_loc"])
    counts, lora_ids, starts, problems = segments.set_sgmm_args(s.dirs, s.lens, True, None, device=DEVICE)
    ids = segments.batch_req_bins(s.req_bins, s.b_seq_len)
    op, sc = atmm_ops.dispatch_bgmv, i["a_scaling"]
    seg = (counts, s.rank_counts, lora_ids, starts, s.tmp, problems[0])
    return _eight_calls(s, lambda d, x, w, t: op(d, x, w, *idx, ids, t, sc, *seg, 64, 32, 32, 32, 32, 32),
                        lambda y, d, w, t: op(y, d, w, *idx, ids, t, sc, *seg, 64, 64, 32, 64, 64, 32))


def _run_requests(s):
    i, h = s.index, s.case["hidden"]
    req = (i["a_loc"], i["a_start"], i["a_len"], s.b_start_loc, s.b_seq_len, s.req_bins)
    r, n = i["max_rank"], s.longest
    return _eight_calls(
        s, lambda d, x, w, t: lora_prefill.lora_get_qkvo_fwd_shrink(x, w.view(-1, h), d, *req, h, t, r, n),
        lambda y, d, w, t: lora_prefill.lora_get_qkvo_fwd_expand(d, w.view(-1, h), y, i["a_scaling"], *req, h, t, r, n))


def _run_compensate(s):
    i = s.index
    idx = (i["a_start"], i["a_len"], i["a_loc"])
    plan = DeLoraPlan(s.ids, s.merged, i["a_start"], i["a_len"], i["max_rank"], s.case["hidden"])
    for l in range(s.layers):
        for slot, (y, x) in enumerate(((s.q, s.x), (s.k, s.x), (s.v, s.x), (s.o, s.attn))):
            plan.apply(y[l], x[l], s.key[l], s.value[l], *idx, slot, i["a_scaling"])
    return s.y


def _run_switch(s):
    i = s.index
    idx = (i["a_start"], i["a_len"], i["a_loc"])
    old, new = s.merged, 1 - s.merged
    for l in range(s.layers):
        w = s.layer_w[l]
        unmerge_adapter(w, s.key[l], s.value[l], *idx, old, s.scaling[old], i["max_rank"])
        merge_adapter(w, s.key[l], s.value[l], *idx, new, s.scaling[new], i["max_rank"])
    s.merged = new
    return s.w


def _run_residency(s):
    a = s.adapters
    s.now = 1 - s.now
    coming = s.sets[s.now]
    a.load_adapters(coming)
    a.offload_adapters(s.stays + [x.lora_dir for x in coming])
    m = a.mem_manager
    return [a.a_loc, a.a_start, a.a_len, a.a_scaling, m.mem_state, m.key_buffer, m.value_buffer]


_RUN = {"plan": _run_plan, "bgmv": _run_bgmv, "sgmm": _run_sgmm, "requests": _run_requests, "compensate": _run_compensate,
        "switch": _run_switch, "residency": _run_residency}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def work(case):
    c = case
    h, mlp, L = c["hidden"], c["mlp"], c["layers"]
    ranks = _ranks(c, c["adapters"])
    if c["kind"] == "residency":     # host memory read, pool rows written
        return {"bytes": 2.0 * 2 * 2 * L * 4 * sum(ranks) * h, "flops": 0}
    if c["kind"] == "switch":        # four weights read and written by either call, A and B of the adapter read
        r = _ranks(c, 2)
        return {"bytes": 2.0 * L * (2 * 2 * 4 * h * h + 4 * sum(r) * 2 * h), "flops": 2.0 * L * 4 * sum(r) * h * h}
    bins, lens, _ = _batch(c, 0)
    T = int(lens.sum())
    tok = np.bincount(bins, weights=lens, minlength=c["adapters"])     # tokens of each adapter
    r = np.array(ranks, dtype=np.float64)
    extra_rank, extra_flops = 0.0, 0.0
    if c["kind"] == "compensate":    # rows of the merged adapter are left alone; the others need the merged one's weights too
        m = int(tok.argmax())
        tok[m] = 0
        T = int(tok.sum())
        extra_rank, extra_flops = (r[m], r[m] * T) if T else (0.0, 0.0)
    touched = float(r[tok > 0].sum()) + extra_rank
    rank_tokens = float((r * tok).sum()) + extra_flops
    # per layer: x of q, k, v once, x of o; four outputs read and written; A and B of four slots
    elements = 2.0 * T * h + 8.0 * T * h + 4 * touched * 2 * h
    flops = 4 * 2 * rank_tokens * 2 * h
    if mlp:
        elements += T * (h + mlp) + 2.0 * T * (2 * mlp + h) + 3 * touched * (h + mlp)
        flops += 3 * 2 * rank_tokens * (h + mlp)
    return {"bytes": 2.0 * L * elements, "flops": L * flops}


def tolerance(case):
    """Outputs are rounded to the 16-bit type once, from sums of 32 bits taken in any order (the intermediate of rank
    width is rounded to the type as well): an odd value lands on the neighbour, a few units at most after two passes."""
    if case["kind"] == "residency":
        return "exact"
    return {"rel": 5e-4, "max": 4e-3} if case["dtype"] == "fp16" else {"rel": 4e-3, "max": 2e-2}
