"""The wide-workgroup row kernel (lora_apply_rows) at the edges of its tiles, against the oracle.

K and N around a chunk, a wave load and a 16-wave column step; ranks around a
pass and past one; rows around a 16-position tile, some empty, some on the base
adapter; x and y with odd row strides from an odd element, so no access is
16-byte aligned.  Rank capacities above 256 take the plain row kernels.

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
    # rows, row_len, K, N, ranks
    (3, 1, 1, 1, [1, 2]),
    (5, 15, 7, 9, [3, 16]),
    (4, 16, 31, 63, [15, 16]),
    (4, 17, 33, 65, [17, 32]),
    (6, 33, 520, 513, [16, 33]),
    (2, 40, 1025, 1023, [4, 64]),
    (9, 1, 1031, 1025, [8, 16, 1]),
    (7, 3, 2050, 2049, [100, 5, 64]),
    (3, 20, 64, 48, [256, 255, 31]),
    (3, 5, 40, 24, [300, 7]),
    (600, 1, 65, 3000, [16, 8]),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,row_len,K,N,ranks", CASES)
@pytest.mark.parametrize("aligned", [True, False])
def test_row_kernel_edges_match_the_oracle(gpu, dtype, rows, row_len, K, N, ranks, aligned):
    print("case:", dtype, rows, row_len, K, N, ranks, aligned, flush=True)
    g = torch.Generator().manual_seed(rows * 1000 + K + N)
    # weights N(0, 0.02): |t| stays near 0.02 * sqrt(K) < 1 and the delta near 2 * 0.02 * |t| * sqrt(rank) < 1, so that
    # fp32 sums in two orders differ by at most some sqrt(terms) * 2^-24 < 4e-6, inside the fp32 tolerance of 1e-5
    # (with N(0, 0.1) both factors grow five times and two fp32 orders differ by up to 25 times as much)
    adapters = {f"a{i}": {"m": peft_layer(g, K, N, r, 2.0 * r)} for i, r in enumerate(ranks)}
    cache = make_cache(adapters, {"m": (K, N)}, len(ranks), max(ranks), gpu, dtype, tiled=False)
    ids = list(adapters) + ["__base__"]
    row_slot = cache.ensure_resident([ids[i] for i in torch.randint(0, len(ids), (rows,), generator=g).tolist()])
    seq = torch.randint(0, row_len + 2, (rows,), generator=g, dtype=torch.int32)
    seq[0] = row_len
    x = torch.randn(rows, row_len, K, generator=g).to(dtype)
    base = torch.randn(rows, row_len, N, generator=g).to(dtype)
    pad = 0 if aligned else 1

    def strided(t):
        flat = t.view(-1, t.shape[-1])
        big = torch.full((flat.shape[0] + 1, flat.shape[1] + 2 * pad), 7.0, dtype=dtype, device=gpu)
        out = big.view(-1)[pad:].as_strided(flat.shape, (big.shape[1], 1))
        out.copy_(flat)
        return out, big

    dx, _ = strided(x)
    dy, around = strided(base)
    sgmv.lora_apply_rows(dx, dy, cache, "m", row_slot, seq.to(gpu), row_len)
    A, B, rk, sc = oracle_slot_tensors(cache, adapters, "m", dtype)
    want = reference_forward(x, base, seq, row_slot.cpu(), A, B, rk, sc)
    torch.testing.assert_close(dy.cpu().view(rows, row_len, N), want, **tol_for(dtype))
    untouched = torch.tensor([[int(s) == 0 or m >= int(n) for m in range(row_len)] for s, n in zip(row_slot.tolist(), seq)])
    assert torch.equal(dy.cpu().view(rows, row_len, N)[untouched], base[untouched])
    if not aligned:  # nothing between or around the rows was written
        gaps = torch.ones(around.numel(), dtype=torch.bool)
        gaps[1:].as_strided(dy.shape, dy.stride()).fill_(False)
        assert torch.equal(around.view(-1).cpu()[gaps], torch.full((int(gaps.sum()),), 7.0, dtype=dtype))


@pytest.mark.parametrize("K,rank", [(192, 4), (768, 16), (2000, 16), (4096, 64)])
def test_row_kernel_fp32_sums_in_short_chains(gpu, K, rank):
    """The delta's rms error against 64 bits stays below 0.42 * 2^-24 * sqrt(additions of one sum).

    An addition rounds by 2^-24 / sqrt(3) of its power of two, 0.42 * 2^-24 of the running sum on average, independently
    of the others.  The shrink adds 4 products, 4 words, K / 256 chunks and 16 waves pairwise (4 + 2 + K / 256 + 4), the
    expand `rank` products.  One running sum over each wave's K / 16 elements and the waves in turn is past the
    bound (1.06e-7, 1.62e-7, 2.25e-7 and 3.25e-7 for these sizes).
    """
    print("case:", K, rank, flush=True)
    g = torch.Generator().manual_seed(K + rank)
    N, tokens = 512, 256
    layer = peft_layer(g, K, N, rank, 2.0 * rank)
    cache = make_cache({"a": {"m": layer}}, {"m": (K, N)}, 1, rank, gpu, torch.float32, tiled=False)
    slots = cache.ensure_resident(["a"])
    x = torch.randn(tokens, K, generator=g)
    y = torch.zeros(tokens, N, device=gpu)
    seq = torch.tensor([tokens], dtype=torch.int32, device=gpu)
    sgmv.lora_apply_rows(x.to(gpu), y, cache, "m", slots, seq, tokens)
    want = 2.0 * ((x.double() @ layer[0].double().T) @ layer[1].double().T)
    err = float((y.cpu().double() - want).norm() / want.norm())
    assert err < 0.42 * 2.0**-24 * (10 + K / 256 + rank) ** 0.5, err


def _overlapping(kind, T, K, N, dtype, g, device):
    """x [T, K] and y [T, N] in one buffer: y is x, beside it in packed rows, its last columns, or one row further."""
    ld = {"same": K, "beside": K + N, "tail": K + 7, "next row": K}[kind]
    buf = torch.randn(T + 1, ld, generator=g).to(dtype).to(device)
    x = buf[:T, :K]
    y = {"same": buf[:T, :N], "beside": buf[:T, K:], "tail": buf[:T, ld - N:], "next row": buf[1:, :N]}[kind]
    return x, y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["same", "beside", "tail", "next row"])
@pytest.mark.parametrize("rows,row_len,rank", [(3, 20, 16), (2, 7, 40)])
def test_row_kernel_reads_x_before_an_overlapping_y(gpu, dtype, kind, rows, row_len, rank):
    """y over x in one buffer gives what separate buffers give; wide outputs, so that a tile has several column ranges."""
    print("case:", dtype, kind, rows, row_len, rank, flush=True)
    g = torch.Generator().manual_seed(rank)
    K, N, T = 2050, 2050, rows * row_len
    cache = make_cache({"a": {"m": peft_layer(g, K, N, rank, 2.0 * rank)}}, {"m": (K, N)}, 1, rank, gpu, dtype, tiled=False)
    slots = cache.ensure_resident(["a"] * rows)
    seq = torch.full((rows,), row_len, dtype=torch.int32, device=gpu)
    x, y = _overlapping(kind, T, K, N, dtype, g, gpu)
    want = y.clone()
    sgmv.lora_apply_rows(x.clone(), want, cache, "m", slots, seq, row_len)
    sgmv.lora_apply_rows(x, y, cache, "m", slots, seq, row_len)
    if kind == "next row":  # the plain kernels, whose sums have another order
        torch.testing.assert_close(y, want, **tol_for(dtype))
    else:
        assert torch.equal(y, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,N,rank", [(71, 65, 5), (1031, 1025, 16), (72, 264, 40)])
def test_infinities_and_nans_stay_in_their_positions(gpu, dtype, K, N, rank):
    """An infinity or NaN in x or in one adapter's weights gives the oracle's values, in its own positions alone."""
    print("case:", dtype, K, N, rank, flush=True)
    g = torch.Generator().manual_seed(K)
    rows, row_len = 12, 21
    adapters = {f"a{i}": {"m": peft_layer(g, K, N, max(1, rank - 2 * i), 2.0 * rank)} for i in range(3)}
    adapters["a2"]["m"][0][0, 5] = float("inf")  # A of one adapter
    cache = make_cache(adapters, {"m": (K, N)}, 3, rank, gpu, dtype, tiled=False)
    row_slot = cache.ensure_resident([["a0", "a1", "a2", "__base__"][i % 4] for i in range(rows)])
    seq = torch.randint(1, row_len + 1, (rows,), generator=g, dtype=torch.int32)
    x = torch.randn(rows, row_len, K, generator=g).to(dtype)
    x[0, 0, 3], x[5, 0, K - 1], x[8, 0, 0] = float("inf"), float("nan"), float("-inf")
    x[4, int(seq[4]) - 1, K - 1] = float("inf")
    x[9, :, :][int(seq[9]):] = float("nan")  # padding positions
    base = torch.randn(rows, row_len, N, generator=g).to(dtype)
    y = base.to(gpu).view(-1, N)
    sgmv.lora_apply_rows(x.to(gpu).view(-1, K), y, cache, "m", row_slot, seq.to(gpu), row_len)
    A, B, rk, sc = oracle_slot_tensors(cache, adapters, "m", dtype)
    want = reference_forward(x, base, seq, row_slot.cpu(), A, B, rk, sc)
    got = y.cpu().view(base.shape)
    assert bool(want.isnan().any()) and torch.equal(got.isfinite(), want.isfinite())
    ok = want.isfinite()
    torch.testing.assert_close(got[ok], want[ok], **tol_for(dtype))


@pytest.mark.parametrize("dtype,rows,row_len,K,N,rank,plain", [
    (torch.bfloat16, 4096, 1, 768, 768, 1, True), (torch.bfloat16, 4096, 1, 16, 16, 16, True),
    (torch.bfloat16, 4096, 1, 768, 768, 64, False), (torch.bfloat16, 1024, 3, 100, 100, 2, True),
    (torch.bfloat16, 64, 17, 1024, 1003, 4, False), (torch.float32, 256, 1, 4096, 1003, 1, True),
    (torch.float32, 256, 1, 4096, 1003, 16, False), (torch.float32, 64, 1, 1000, 2000, 4, False)])
def test_many_rows_of_low_rank_take_the_plain_kernels(gpu, dtype, rows, row_len, K, N, rank, plain):
    """The row kernels' route, seen from the scratch (only the plain kernels write it), and the result on both."""
    print("case:", dtype, rows, row_len, K, N, rank, flush=True)
    g = torch.Generator().manual_seed(rows + K)
    adapters = {"a": {"m": peft_layer(g, K, N, rank, 2.0 * rank)}}
    cache = make_cache(adapters, {"m": (K, N)}, 1, rank, gpu, dtype, tiled=False)
    row_slot = cache.ensure_resident([["a", "__base__"][i % 3 == 2] for i in range(rows)])
    seq = torch.randint(1, row_len + 1, (rows,), generator=g, dtype=torch.int32)
    x = torch.randn(rows, row_len, K, generator=g).to(dtype)
    base = torch.randn(rows, row_len, N, generator=g).to(dtype)
    dx, y, lens = x.to(gpu).view(-1, K), base.to(gpu).view(-1, N), seq.to(gpu)
    tmp = torch.full((rows * row_len, rank), 12345.0, device=gpu)
    arena, table, n_mod, column, _ = sgmv._cache_args(cache, "m")
    rc = sgmv._native.calls().pl_lora_apply_rows(
        sgmv._native.dtype_code(dtype), dx.data_ptr(), K, K, y.data_ptr(), N, N, arena, table, cache.num_slots, n_mod,
        column, row_slot.data_ptr(), lens.data_ptr(), rows, row_len, tmp.data_ptr(), rank, 0, sgmv._stream(gpu))
    sgmv._native.check(rc, "pl_lora_apply_rows")
    assert bool((tmp != 12345.0).any()) == plain
    A, B, rk, sc = oracle_slot_tensors(cache, adapters, "m", dtype)
    want = reference_forward(x, base, seq, row_slot.cpu(), A, B, rk, sc)
    torch.testing.assert_close(y.cpu().view(base.shape), want, **tol_for(dtype))
