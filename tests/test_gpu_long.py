"""The two-launch path of long segments (lora_long_stacked) at the edges of its tiles, against the oracle.

Segments around one, two and four 16-token tiles; K around one wave's step and
a turn of the four waves; N around an MFMA tile and a workgroup's chunk; ranks
around a pass (and two passes, above 64); a second module that some adapters
do not have; plans of 16- and 64-token groups, and one with enough tiles for
the two-tile shrink.  Then units of two and four tiles of several slots, for
launches large enough to have them; infinities and NaN; HIP graphs, streams.

Reference: the fallback of layers.py:112-134 (reference_forward).
"""

from __future__ import annotations

import pytest
import torch

from oracle.lora import reference_forward
from polylora_amd import sgmv
from tests._util import make_cache, oracle_slot_tensors, peft_layer, tol_for

pytestmark = pytest.mark.gpu

CASES = [
    # rows, row_len, K, (N of the two modules), ranks
    (3, 1, 8, (8, 16), [1, 2]),
    (9, 15, 64, (520, 8), [8, 16, 3]),
    (6, 17, 264, (504, 512), [16, 15]),
    (5, 65, 256, (1032, 24), [17, 32, 33]),
    (12, 33, 1000, (136, 264), [64, 5]),
    (4, 100, 520, (72, 640), [65, 128, 16]),
    (17, 16, 72, (48, 56), [40, 9, 1, 24]),
    (40, 256, 136, (264, 16), [16, 31, 64]),
    (3, 50, 128, (88, 16), [256, 129, 70]),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("group_tokens", [16, 64])
@pytest.mark.parametrize("rows,row_len,K,Ns,ranks", CASES)
def test_long_path_edges_match_the_oracle(gpu, dtype, group_tokens, rows, row_len, K, Ns, ranks):
    print("case:", dtype, group_tokens, rows, row_len, K, Ns, ranks, flush=True)
    if dtype == torch.float32 and max(ranks) > sgmv.LONG_MAX_RANK // 2:
        ranks = [min(r, sgmv.LONG_MAX_RANK // 2) for r in ranks]
    g = torch.Generator().manual_seed(rows * 1000 + K + Ns[0])
    # weights N(0, 0.02): |t| and the deltas stay near 1 or below, so that fp32 sums in two orders differ by at most
    # some sqrt(terms) * 2^-24 < 4e-6, inside the fp32 tolerance of 1e-5
    adapters = {}
    for i, r in enumerate(ranks):
        adapters[f"a{i}"] = {"m0": peft_layer(g, K, Ns[0], r, 2.0 * r)}
        if i % 2 == 0:
            adapters[f"a{i}"]["m1"] = peft_layer(g, K, Ns[1], max(1, r // 2), 1.0 * r)
    cache = make_cache(adapters, {"m0": (K, Ns[0]), "m1": (K, Ns[1])}, len(ranks), max(ranks), gpu, dtype)
    ids = list(adapters) + ["__base__"]
    row_slot = cache.ensure_resident([ids[i] for i in torch.randint(0, len(ids), (rows,), generator=g).tolist()])
    seq = torch.randint(0, row_len + 2, (rows,), generator=g, dtype=torch.int32)
    seq[0] = row_len
    plan = sgmv.SgmvPlan(row_slot, seq.to(gpu), row_len, cache.num_slots, distinct_slots=len(ranks),
                         group_tokens=group_tokens)
    x = torch.randn(rows, row_len, K, generator=g).to(dtype)
    bases = [torch.randn(rows, row_len, n, generator=g).to(dtype) for n in Ns]
    dx = x.to(gpu).view(-1, K)
    for epilogue in (0, 1):
        # the modules one by one, then stacked, with bit-equal outputs
        one = [b.to(gpu).view(-1, b.shape[-1]) for b in bases]
        both = [t.clone() for t in one]
        for name, y in zip(("m0", "m1"), one):
            sgmv.lora_long_stacked(dx, [y], cache, [name], plan, epilogue=epilogue)
        sgmv.lora_long_stacked(dx, both, cache, ["m0", "m1"], plan, epilogue=epilogue)
        assert all(torch.equal(a, b) for a, b in zip(one, both))
        for name, y, base in zip(("m0", "m1"), both, bases):
            got = y.cpu().view(base.shape)
            A, B, rk, sc = oracle_slot_tensors(cache, adapters, name, dtype)
            torch.testing.assert_close(got, reference_forward(x, base, seq, row_slot.cpu(), A, B, rk, sc), **tol_for(dtype))
            keep = torch.tensor([[int(rk[s]) == 0 or m >= int(n) for m in range(row_len)]
                                 for s, n in zip(row_slot.tolist(), seq)])
            assert torch.equal(got[keep], base[keep])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("ranks,Ns", [
    ([32, 5, 17, 0, 16], (2048,)),  # expand units of two tiles
    ([64, 33, 0, 8, 48], (2048,)),  # of four
    ([128, 65, 40, 0, 9, 100], (2048,)),  # four, intermediates of up to 8 rank steps in fp32, 4 in 16 bits
    ([256, 129, 70, 0, 40, 64], (2048,)),  # 8 rank steps in 16 bits; 64-rank shrink passes
    ([64, 40, 0, 16], (1024, 256, 256, 512))])  # 64-rank shrink passes of four modules
def test_units_of_several_slots_match_the_oracle(gpu, dtype, ranks, Ns):
    """Many short segments of interleaved adapters, some without the modules, in launches large enough for shrink
    units of two tiles and expand units of two or four: neighbouring tiles of a unit belong to different slots."""
    print("case:", dtype, ranks, Ns, flush=True)
    if dtype == torch.float32:
        ranks = [min(r, sgmv.LONG_MAX_RANK // 2) for r in ranks]
    rows, row_len, K, n_adapters = 220, 30, 72, 100
    g = torch.Generator().manual_seed(sum(ranks) + len(Ns))
    mods = [f"m{i}" for i in range(len(Ns))]
    adapters = {}
    for i in range(n_adapters):
        r = ranks[i % len(ranks)]
        adapters[f"a{i}"] = ({m: peft_layer(g, K, n, r, 2.0 * r) for m, n in zip(mods, Ns)} if r else
                             {"other": peft_layer(g, 8, 8, 2, 4.0)})
    shapes = dict({m: (K, n) for m, n in zip(mods, Ns)}, other=(8, 8))
    cache = make_cache(adapters, shapes, n_adapters, max(ranks), gpu, dtype)
    ids = list(adapters) + ["__base__"]
    # every adapter first, so that all hold slots, then at random
    pick = [ids[i] for i in range(n_adapters)] + [ids[i] for i in torch.randint(0, len(ids), (rows - n_adapters,), generator=g).tolist()]
    row_slot = cache.ensure_resident(pick)
    seq = torch.randint(0, row_len + 2, (rows,), generator=g, dtype=torch.int32)
    plan = sgmv.SgmvPlan(row_slot, seq.to(gpu), row_len, cache.num_slots, distinct_slots=n_adapters, group_tokens=16)
    # what the launch's choices look at: tiles, and workgroups of one-tile units
    es = torch.empty((), dtype=dtype).element_size()
    ldt, tiles = cache.rank8_cap, -(-plan.group_cap // 8) * 8
    chunk = (512 if ldt * es > 128 else 1024) // es
    assert tiles >= 512 and all(n * es % 128 == 0 for n in Ns)
    assert tiles * sum(-(-n // chunk) for n in Ns) >= 2048
    if len(Ns) == 4 or ldt == 256:
        assert tiles // 2 * len(Ns) * -(-ldt // 32) >= 1536  # 64-rank passes
    slots = plan.groups.cpu()[: int(plan.meta[3]), 0].view(-1, 8)  # [position on the XCD][XCD]
    for unit in (2, 4):
        several = sum(len(set(slots[i : i + unit, x].tolist())) > 1 for x in range(8) for i in range(0, slots.shape[0], unit))
        assert several > slots.shape[0] // unit * 8 // 4, unit
    x = torch.randn(rows, row_len, K, generator=g).to(dtype)
    bases = [torch.randn(rows, row_len, n, generator=g).to(dtype) for n in Ns]
    got = [b.to(gpu).view(-1, b.shape[-1]) for b in bases]
    sgmv.lora_long_stacked(x.to(gpu).view(-1, K), got, cache, mods, plan)
    for m, y, base in zip(mods, got, bases):
        A, B, rk, sc = oracle_slot_tensors(cache, adapters, m, dtype)
        y = y.cpu().view(base.shape)
        torch.testing.assert_close(y, reference_forward(x, base, seq, row_slot.cpu(), A, B, rk, sc), **tol_for(dtype))
        keep = torch.tensor([[int(rk[s]) == 0 or i >= int(n) for i in range(row_len)] for s, n in zip(row_slot.tolist(), seq)])
        assert torch.equal(y[keep], base[keep])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank,N", [(5, 264), (40, 2048), (100, 264)])
def test_infinities_and_nans_stay_in_their_tokens(gpu, dtype, rank, N):
    """An infinity or NaN in x or in one adapter's weights gives the oracle's values, in its own tokens alone: rows of
    a tile past its tokens, ranks past the slot's and K past the range are left out, not multiplied by zero."""
    print("case:", dtype, rank, N, flush=True)
    g = torch.Generator().manual_seed(rank)
    rows, row_len, K = 40, 27, 72
    adapters = {f"a{i}": {"m": peft_layer(g, K, N, max(1, rank - 2 * i), 2.0 * rank)} for i in range(3)}
    adapters["a2"]["m"][0][0, 5] = float("inf")  # A of one adapter
    cache = make_cache(adapters, {"m": (K, N)}, 3, rank, gpu, dtype)
    row_slot = cache.ensure_resident([["a0", "a1", "a2", "__base__"][i % 4] for i in range(rows)])
    seq = torch.randint(1, row_len + 1, (rows,), generator=g, dtype=torch.int32)
    plan = sgmv.SgmvPlan(row_slot, seq.to(gpu), row_len, cache.num_slots, distinct_slots=3, group_tokens=16)
    x = torch.randn(rows, row_len, K, generator=g).to(dtype)
    x[0, 0, 3], x[5, 0, K - 1], x[8, 0, 0] = float("inf"), float("nan"), float("-inf")
    x[4, int(seq[4]) - 1, K - 1] = float("inf")  # the last token of a row, last of its slot's tile or not
    x[9, :, :][int(seq[9]):] = float("nan")  # padding positions
    base = torch.randn(rows, row_len, N, generator=g).to(dtype)
    y = base.to(gpu).view(-1, N)
    sgmv.lora_long_stacked(x.to(gpu).view(-1, K), [y], cache, ["m"], plan)
    A, B, rk, sc = oracle_slot_tensors(cache, adapters, "m", dtype)
    want = reference_forward(x, base, seq, row_slot.cpu(), A, B, rk, sc)
    got = y.cpu().view(base.shape)
    assert bool(want.isnan().any()) and bool(want.isfinite().any())
    assert torch.equal(got.isfinite(), want.isfinite())
    ok = want.isfinite()
    torch.testing.assert_close(got[ok], want[ok], **tol_for(dtype))


def _long_case(gpu, seed, rank=24):
    g = torch.Generator().manual_seed(seed)
    K, shapes, tokens = 520, {"q": 1032, "k": 264}, 1300
    adapters = {f"a{i}": {m: peft_layer(g, K, n, r, 2.0 * r) for m, n in shapes.items()} for i, r in enumerate([rank, 7])}
    cache = make_cache(adapters, {m: (K, n) for m, n in shapes.items()}, 2, rank, gpu, torch.bfloat16)
    slots = cache.ensure_resident(["a0", "a1", "__base__", "a0"])
    plan = sgmv.SgmvPlan(slots, torch.tensor([325, 99, 200, 16], dtype=torch.int32, device=gpu), 325, cache.num_slots,
                         distinct_slots=2)
    x = torch.randn(tokens, K, generator=g).bfloat16().to(gpu)
    bases = [torch.randn(tokens, n, generator=g).bfloat16().to(gpu) for n in shapes.values()]
    return cache, list(shapes), plan, x, bases


@pytest.mark.parametrize("rank", [24, 100])
def test_long_path_in_a_graph(gpu, rank):
    """Captured with its workspace (an allocation inside the capture), between other captured work; every replay,
    with eager long calls between replays, equals the eager result."""
    cache, mods, plan, x, bases = _long_case(gpu, 90 + rank, rank)
    want = sgmv.lora_long_stacked(x, [b.clone() for b in bases], cache, mods, plan)
    ys = [torch.empty_like(b) for b in bases]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for y, b in zip(ys, bases):
            y.copy_(b)
        sgmv.lora_long_stacked(x, ys[:1], cache, mods[:1], plan)
        more = torch.ones(1 << 18, device=gpu)  # may take the first call's workspace
        sgmv.lora_long_stacked(x, ys[1:], cache, mods[1:], plan)
        more.add_(1.0)
    for i in range(4):
        for y in ys:
            y.fill_(float(i))
        eager = sgmv.lora_long_stacked(x, [b.clone() for b in bases], cache, mods, plan)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(ys, want)), i
        assert all(torch.equal(a, b) for a, b in zip(eager, want)), i
        assert bool((more == 2.0).all()), i


def test_long_calls_on_two_streams(gpu):
    """Calls that overlap on two streams have workspaces of their own: equal to the calls one after the other."""
    cases = [_long_case(gpu, seed, rank) for seed, rank in ((101, 24), (102, 64))]
    want = [sgmv.lora_long_stacked(x, [b.clone() for b in bases], cache, mods, plan) for cache, mods, plan, x, bases in cases]
    streams = [torch.cuda.Stream() for _ in cases]
    outs = [[[b.clone() for b in bases] for _ in range(20)] for *_, bases in cases]
    torch.cuda.synchronize()
    for i in range(20):
        for (cache, mods, plan, x, _), s, ys in zip(cases, streams, outs):
            with torch.cuda.stream(s):
                sgmv.lora_long_stacked(x, ys[i], cache, mods, plan)
    torch.cuda.synchronize()
    for ys, ref in zip(outs, want):
        for i, y in enumerate(ys):
            assert all(torch.equal(a, b) for a, b in zip(y, ref)), i


def test_a_stream_other_than_the_current_one_keeps_the_fused_kernel(gpu, monkeypatch):
    """The workspace is allocated on the current stream, so lora_fused(stream=other) stays off the long path."""
    cache, mods, plan, x, bases = _long_case(gpu, 103)
    calls = []
    launch = sgmv._long_launch
    monkeypatch.setattr(sgmv, "_long_launch", lambda *a: (calls.append(1), launch(*a))[1])
    monkeypatch.setattr(sgmv, "long_ok", lambda *a: True)
    here = sgmv.lora_fused(x, bases[0].clone(), cache, mods[0], plan)
    assert calls == [1]
    both = sgmv.lora_fused_stacked(x, [b.clone() for b in bases], cache, mods, plan, stream=torch.cuda.current_stream().cuda_stream)
    assert calls == [1, 1]
    there, there2 = bases[0].clone(), [b.clone() for b in bases]
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    sgmv.lora_fused(x, there, cache, mods[0], plan, stream=other.cuda_stream)
    sgmv.lora_fused_stacked(x, there2, cache, mods, plan, stream=other.cuda_stream)
    torch.cuda.synchronize()
    assert calls == [1, 1]
    assert torch.equal(here, there) and all(torch.equal(a, b) for a, b in zip(both, there2))


def test_the_dispatch_takes_the_long_path_where_its_rule_says(gpu, monkeypatch):
    """lora_apply and lora_fused_stacked go through it for large outputs and for high ranks, and only there."""
    calls = []
    launch = sgmv._long_launch
    monkeypatch.setattr(sgmv, "_long_launch", lambda x, ys, *a: (calls.append(len(ys)), launch(x, ys, *a))[1])
    g = torch.Generator().manual_seed(5)
    # (rank 96, 64 outputs: a call that the host paces keeps the split pair)
    for rank, rows, n, want in ((16, 20, 1024, []), (16, 20, 17000, [1, 1]), (96, 40, 64, [1]), (96, 20, 64, []),
                                (96, 20, 2048, [1]), (96, 8, 2048, []), (160, 20, 64, [1])):
        adapters = {"a": {"m": peft_layer(g, 64, n, rank, 2.0 * rank)}}
        cache = make_cache(adapters, {"m": (64, n)}, 1, rank, gpu, torch.bfloat16)
        row_slot = cache.ensure_resident(["a"] * rows)
        seq = torch.full((rows,), 128, dtype=torch.int32)
        plan = sgmv.SgmvPlan(row_slot, seq.to(gpu), 128, cache.num_slots, distinct_slots=1)
        x, base = (torch.randn(rows, 128, k, generator=g).bfloat16() for k in (64, n))
        A, B, rk, sc = oracle_slot_tensors(cache, adapters, "m", torch.bfloat16)
        ref = reference_forward(x, base, seq, row_slot.cpu(), A, B, rk, sc)
        calls.clear()
        ops = [lambda x, y: sgmv.lora_apply(x, y, cache, "m", plan)]
        if rank <= sgmv.FUSED_MAX_RANK:  # lora_fused_stacked refuses higher ranks
            ops.append(lambda x, y: sgmv.lora_fused_stacked(x, [y], cache, ["m"], plan))
        for op in ops:
            y = base.to(gpu).view(-1, n)
            op(x.to(gpu).view(-1, 64), y)
            torch.testing.assert_close(y.cpu().view(base.shape), ref, **tol_for(torch.bfloat16))
        assert calls == want, (rank, rows, n)


@pytest.mark.parametrize("K,rank", [(768, 8), (4096, 64), (4096, 128)])
def test_long_fp32_sums_in_short_chains(gpu, K, rank):
    """The delta's rms error against 64 bits stays below 0.42 * 2^-24 * sqrt(additions of one sum).

    An addition rounds by 2^-24 / sqrt(3) of its power of two, 0.42 * 2^-24 of the running sum on average, independently
    of the others.  The shrink adds 4 products, 4 words, K / 64 chunks and 4 waves (4 + 2 + K / 64 + 3), the expand
    `rank` products.  One running sum over each wave's K / 4 elements is past the bound (2.6e-7, 5.9e-7 and 6.0e-7).
    """
    print("case:", K, rank, flush=True)
    g = torch.Generator().manual_seed(K + rank)
    N, tokens = 512, 1024
    layer = peft_layer(g, K, N, rank, 2.0 * rank)
    cache = make_cache({"a": {"m": layer}}, {"m": (K, N)}, 1, rank, gpu, torch.float32)
    slots = cache.ensure_resident(["a"])
    x = torch.randn(tokens, K, generator=g)
    y = torch.zeros(tokens, N, device=gpu)
    seq = torch.tensor([tokens], dtype=torch.int32, device=gpu)
    plan = sgmv.SgmvPlan(slots, seq, tokens, cache.num_slots, distinct_slots=1)
    sgmv.lora_long_stacked(x.to(gpu), [y], cache, ["m"], plan)
    want = 2.0 * ((x.double() @ layer[0].double().T) @ layer[1].double().T)
    err = float((y.cpu().double() - want).norm() / want.norm())
    assert err < 0.42 * 2.0**-24 * (9 + K / 64 + rank) ** 0.5, err


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,row_len,K,N,ranks", [
    (4, 40, 8, 24, [1, 16]), (3, 70, 64, 520, [8, 15]), (5, 33, 136, 264, [17, 32, 3]), (2, 100, 520, 1032, [33, 64]),
    (3, 50, 2056, 72, [16, 64, 40]), (2, 90, 4104, 512, [32, 5]), (40, 256, 1000, 136, [64, 16, 31])])
def test_long_and_fused_paths_give_the_same_bits(gpu, dtype, rows, row_len, K, N, ranks):
    """In 16 bits the two paths make every sum of the same additions in the same order, so a Linear's output does not
    depend on which of them its call took: K around shares of one to several step pairs, ranks around a tile."""
    print("case:", dtype, rows, row_len, K, N, ranks, flush=True)
    g = torch.Generator().manual_seed(K + N)
    adapters = {f"a{i}": {"m": peft_layer(g, K, N, r, 2.0 * r)} for i, r in enumerate(ranks)}
    cache = make_cache(adapters, {"m": (K, N)}, len(ranks), max(ranks), gpu, dtype)
    ids = list(adapters) + ["__base__"]
    row_slot = cache.ensure_resident([ids[i] for i in torch.randint(0, len(ids), (rows,), generator=g).tolist()])
    seq = torch.randint(0, row_len + 1, (rows,), generator=g, dtype=torch.int32).to(gpu)
    x = torch.randn(rows * row_len, K, generator=g).to(dtype).to(gpu)
    base = torch.randn(rows * row_len, N, generator=g).to(dtype).to(gpu)
    for group_tokens in (16, 64):
        plan = sgmv.SgmvPlan(row_slot, seq, row_len, cache.num_slots, distinct_slots=len(ranks), group_tokens=group_tokens)
        fused = sgmv.lora_fused(x, base.clone(), cache, "m", plan, slices=1)
        (long,) = sgmv.lora_long_stacked(x, [base.clone()], cache, ["m"], plan)
        assert torch.equal(fused, long) and not torch.equal(fused, base)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rank", [16, 64])
def test_a_linear_alone_and_with_its_siblings_gives_the_same_bits(gpu, monkeypatch, dtype, rank):
    """A rule by which a Linear alone takes the fused kernel and with its siblings the long path (the first forward
    runs Linears alone, later ones the learned siblings together): equal outputs, and both kernels really ran."""
    ran = []
    calls = sgmv._native.calls()

    class Spy:
        def __getattr__(self, name):
            f = getattr(calls, name)
            return lambda *a: (ran.append(name), f(*a))[1]

    spy = Spy()
    monkeypatch.setattr(sgmv._native, "calls", lambda: spy)
    g = torch.Generator().manual_seed(rank)
    K, shapes, tokens = 1000, {"q": 1536, "k": 264, "v": 264}, 1200
    # a line between k or v alone and q alone or all together
    monkeypatch.setattr(sgmv, "long_ok", lambda plan, cache, fin, fout, modules=1: fout >= 1000)
    adapters = {f"a{i}": {m: peft_layer(g, K, n, r, 2.0 * r) for m, n in shapes.items()} for i, r in enumerate([rank, 5])}
    cache = make_cache(adapters, {m: (K, n) for m, n in shapes.items()}, 2, rank, gpu, dtype)
    slots = cache.ensure_resident(["a0", "a1", "a0"])
    plan = sgmv.SgmvPlan(slots, torch.tensor([400, 333, 17], dtype=torch.int32, device=gpu), 400, cache.num_slots,
                         distinct_slots=2)
    x = torch.randn(tokens, K, generator=g).to(dtype).to(gpu)
    bases = [torch.randn(tokens, n, generator=g).to(dtype).to(gpu) for n in shapes.values()]
    alone = [sgmv.lora_apply(x, b.clone(), cache, m, plan) for m, b in zip(shapes, bases)]
    assert ran == ["pl_lora_long_stacked", "pl_lora_fused", "pl_lora_fused"]
    ran.clear()
    together = sgmv.lora_fused_stacked(x, [b.clone() for b in bases], cache, list(shapes), plan)
    assert ran[0] == "pl_lora_long_stacked" and len(ran) == (2 if dtype == torch.float32 else 1)
    for m, a, b in zip(shapes, alone, together):
        assert torch.equal(a, b), m
