"""Kernels of steps of few rows alone, at the edges of the sizes they take."""
import types

import pytest
import torch

from kernel_refs import PlainOps
from plain import dolidra_plain as plain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from tokenizer_amd.kernels import get_ops
    return get_ops()


def rounded(t):
    return t.to(torch.bfloat16).to(torch.float64)


def sum_slack(x, w, *more):
    """How far x w^T + more, added in floats, may be off, output by output: a product joins up to 32 in its matrix instruction, the steps of
    32 of K that a wave has (four waves at least share K), two sums of each of sixteen waves and what else is added; each of these
    roundings is of a sum no larger than that of the magnitudes, by 2^-23 (nothing says that a matrix instruction does not cut off)."""
    k, mags = x.shape[1], x.double().abs() @ w.double().abs().t()
    for t in more:
        mags = mags + t.double().abs()
    return (32 + -(-k // 128) + 32 + len(more)) * 2.0 ** -23 * mags


def rand_bf16(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).cuda()


# Inner widths with a block of sixteen columns left over, a shared expert wider than four others (four parts), narrower than one
# (one part), with parts that whole turns of 64 leave no columns for (104 in four parts of 24 are two of 64) and a last part of eight
# (72 in two); one row and sixteen, one expert and all of them.
@pytest.mark.parametrize("width,inner,shared,experts,top,rows", [(64, 24, 104, 8, 2, 1), (1032, 40, 8, 3, 1, 16), (72, 1032, 1040, 4, 4, 5),
                                                                 (896, 64, 72, 8, 3, 16), (1536, 72, 200, 1, 1, 3)])
@pytest.mark.parametrize("weighted", [False, True])
def test_chosen_experts_beside_one_that_all_rows_use(ops, width, inner, shared, experts, top, rows, weighted):
    gen = torch.Generator().manual_seed(width + rows)
    rand = lambda *shape: torch.randn(*shape, generator=gen, dtype=torch.float64)
    sizes = [inner] * experts + [shared]
    first = [rounded(rand(2, n, width) / width ** 0.5 * 2) for n in sizes]
    second = [rounded(rand(width, n) / n ** 0.5) for n in sizes]
    x = rounded(rand(rows, width))
    chosen = torch.stack([torch.randperm(experts, generator=gen)[:top] for _ in range(rows)]).to(torch.int32)
    weights = (0.2 + torch.rand(rows, top, generator=gen)).float()
    share = (0.2 + torch.rand(rows, generator=gen)).float() if weighted else None
    for e in range(experts):                                  # an expert nobody chose is not read
        if not bool((chosen == e).any()):
            first[e], second[e] = torch.full_like(first[e], float("nan")), torch.full_like(second[e], float("nan"))
    on = lambda t: t.to(torch.bfloat16).cuda().contiguous()
    parts = ops.experts_few(on(x), chosen.cuda(), weights.cuda(), experts, on(torch.cat([m.reshape(-1, width) for m in first])), True,
                            inner, on(torch.cat(second, dim=1)), shared=shared, shared_weight=None if share is None else share.cuda())
    expert = lambda t, e: second[e] @ (plain.silu(first[e][0] @ x[t]) * (first[e][1] @ x[t]))
    want = torch.zeros(rows, width, dtype=torch.float64)
    for t in range(rows):
        want[t] = sum(float(weights[t, k]) * expert(t, int(chosen[t, k])) for k in range(top))
        want[t] += (1.0 if share is None else float(share[t])) * expert(t, experts)
    # Gate, up and their product are rounded to bfloat16 (2^-9 each), so a result is off by less than four such roundings of sums
    # whose terms are as large as the largest result.
    got = parts.resolve().double().cpu()
    # (As many parts of the shared expert as the others are long, four at most, of whole turns of 64: none is empty.)
    length = -(-(-(-shared // min(4, -(-shared // inner)))) // 64) * 64
    assert parts.partial.shape[0] == top + -(-shared // length)
    assert float((got - want).abs().max()) <= 2e-2 * float(want.abs().max())


@pytest.mark.parametrize("gated,shared,weigh_input", [(True, 48, False), (True, 0, True), (False, 0, False)])
def test_a_pick_that_weighs_nothing_adds_nothing(ops, gated, shared, weigh_input):
    """Expert 1 overflows on every row and is chosen with a weight of zero: the rows are those of expert 0 (and the shared one)."""
    width, inner, experts, rows, halves = 64, 32, 3, 4, 2 if gated else 1
    first, second = rand_bf16((halves * (experts * inner + shared), width), 51) / 8, rand_bf16((width, experts * inner + shared), 52)
    x = rand_bf16((rows, width), 53).abs()
    first[halves * inner:2 * halves * inner] = 3e38
    chosen = torch.tensor([[0, 1]] * rows, dtype=torch.int32, device="cuda")
    weights = torch.tensor([[0.75, 0.0]] * rows, device="cuda")
    run = lambda: ops.experts_few(x, chosen, weights, experts, first, gated, inner, second, weigh_input=weigh_input, shared=shared).resolve()
    got = run()
    first[halves * inner:2 * halves * inner] = 0.25
    assert bool(torch.isfinite(got).all()) and torch.equal(got, run())


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("width", [896, 1536])
def test_chosen_experts_are_the_same_in_every_call(ops, gated, width):
    """More workgroups than the device holds at once: a sum read before it is there would differ from call to call."""
    inner, experts, top, rows, halves = 3648, 8, 2, 4, 2 if gated else 1
    first, second = rand_bf16((halves * experts * inner, width), 61) / 32, rand_bf16((width, experts * inner), 62) / 64
    x, weights = rand_bf16((rows, width), 63), (0.2 + torch.rand(rows, top, generator=torch.Generator().manual_seed(64))).cuda()
    chosen = torch.tensor([[5, 4], [4, 3], [5, 2], [2, 1]], dtype=torch.int32, device="cuda")
    run = lambda: ops.experts_few(x, chosen, weights, experts, first, gated, inner, second).partial
    got = run()
    for _ in range(24):
        assert torch.equal(run(), got)
    # Rounded to bfloat16: the first product's results, and what the second is handed (2^-9 each).
    for t in range(rows):
        for k in range(top):
            e = int(chosen[t, k])
            each = (first[e * halves * inner:(e + 1) * halves * inner].double() @ x[t].double()).bfloat16().double()
            act = plain.silu(each[:inner]) * each[inner:] if gated else each.clamp(min=0) ** 2
            want = second[:, e * inner:(e + 1) * inner].double() @ (float(weights[t, k]) * act).bfloat16().double()
            assert float((got[k, t] - want).abs().max()) <= 2e-2 * float(want.abs().max())


@pytest.mark.parametrize("experts,shared,taken", [(65535, 0, True), (65534, 8, True), (65533, 264, False), (65535, 8, False)])
def test_as_many_experts_as_a_grid_has_places_for(ops, experts, shared, taken):
    """The last experts of a full grid; where the shared one's parts have no place left, the call is handed back, not refused."""
    width = inner = 8
    total = experts * inner + shared
    first = torch.randn((2 * total, width), device="cuda", dtype=torch.float32).to(torch.bfloat16)
    second = torch.randn((width, total), device="cuda", dtype=torch.float32).to(torch.bfloat16)
    x = rand_bf16((2, width), 55)
    chosen = torch.tensor([[0, experts - 1], [experts - 2, 31]], dtype=torch.int32, device="cuda")
    weights = torch.tensor([[0.75, 0.5], [1.25, 0.25]], device="cuda")
    parts = ops.experts_few(x, chosen, weights, experts, first, True, inner, second, shared=shared)
    assert (parts is not None) == taken
    if not taken:
        return
    expert = lambda t, at, n: second[:, at:at + n].double().cpu() @ (
        plain.silu(first[2 * at:2 * at + n].double().cpu() @ x[t].double().cpu()) * (first[2 * at + n:2 * at + 2 * n].double().cpu() @ x[t].double().cpu()))
    want = torch.stack([sum(float(weights[t, k]) * expert(t, int(chosen[t, k]) * inner, inner) for k in range(2))
                        + (expert(t, experts * inner, shared) if shared else 0) for t in range(2)])
    assert float((parts.resolve().double().cpu() - want).abs().max()) <= 2e-2 * float(want.abs().max())


@pytest.mark.parametrize("width", [8, 520, 2048, 2056, 4096])
@pytest.mark.parametrize("dim", [8, 16])
@pytest.mark.parametrize("rows", [1, 256])
def test_norm_with_the_token_input_of_few_rows(ops, width, dim, rows):
    gen = torch.Generator().manual_seed(width + dim)
    rand = lambda *shape: torch.randn(*shape, generator=gen, dtype=torch.float64)
    table, ids = rounded(rand(31, 3 * dim)), torch.randint(0, 31, (rows,), generator=gen)
    x, delta = rand(rows, width).float().double(), rounded(5 * rand(rows, width))
    w = {"gate": rounded(rand(dim, width) / width ** 0.5), "proj": rounded(rand(width, dim)), "norm": rand(width).float().double()}
    behind, nxt = rand(width).float().double(), rand(width).float().double()
    on = lambda t, kind=torch.bfloat16: t.to(kind).cuda().contiguous()
    for post, last in ((behind, nxt), (None, None)):
        first = x + (plain.weighted_norm(delta, post, 3e-5) if post is not None else delta)
        after = first + plain.token_side_input(first, ids, table, w, 1, dim, 1e-5)
        want = plain.weighted_norm(after, last, 1e-6) if last is not None else after
        vector = lambda t: None if t is None else on(t, torch.float32)
        for picked in (None, torch.tensor([rows - 1, 0], dtype=torch.int32, device="cuda")):
            stream = on(x, torch.float32)
            out = torch.empty((rows if picked is None else 2, width), dtype=torch.bfloat16, device="cuda")
            ops.norm_side_norm(stream, on(delta), vector(post), 3e-5, on(w["gate"]), on(w["proj"]), vector(w["norm"]), 1e-5, on(table),
                               on(ids, torch.int32), dim, dim, vector(last), 1e-6, out, picked)
            # The stream is a float sum throughout; a row of the result is rounded to bfloat16 once.
            stored = after if picked is None else x
            assert float((stream.double().cpu() - stored).abs().max()) <= 1e-4 * float(stored.abs().max())
            rows_want = want if picked is None else want[[rows - 1, 0]]
            assert float((out.double().cpu() - rows_want).abs().max()) <= 2 ** -8 * float(rows_want.abs().max()) + 1e-4


# K of one, two, three and four steps of 32 (rounds of three, and what is left of one) and of no whole step; columns of one strip, one
# past it, no multiple of four; an expert nobody chose, one with a single pair, one with several tiles.
@pytest.mark.parametrize("k", [32, 64, 96, 160, 136])
@pytest.mark.parametrize("n_out", [256, 257, 90, 520])
@pytest.mark.parametrize("bm", [64, 128])
def test_sorted_products_in_either_kernel(ops, k, n_out, bm, monkeypatch):
    gen = torch.Generator().manual_seed(k + n_out)
    experts, rows, ldw = 4, 150, k + 24
    rand = lambda *shape: rounded(torch.randn(*shape, generator=gen, dtype=torch.float64))
    chosen = torch.where(torch.arange(rows) < 149, torch.tensor(2), torch.tensor(0)).to(torch.int32)[:, None]
    chosen[:5] = 3
    x, w = rand(rows, k), rand(experts, n_out, k) / k ** 0.5
    w = rounded(w)
    joined = torch.full((experts * n_out, ldw), float("nan"), dtype=torch.bfloat16)        # columns behind K are not read
    joined[:, :k] = w.reshape(-1, k).to(torch.bfloat16)
    slot_of, row_of, tile_expert = ops.expert_slots(chosen.cuda(), experts, bm)
    on = lambda t: t.to(torch.bfloat16).cuda().contiguous()
    want = torch.stack([w[int(chosen[t, 0])] @ x[t] for t in range(rows)])
    slots = slot_of.cpu().long()
    by_slot = torch.zeros(row_of.numel(), k, dtype=torch.float64)
    by_slot[slots] = x
    for wide in (-1, 1):                                      # (the wide kernel where K goes in whole steps)
        monkeypatch.setattr(ops, "grouped_wide", wide)
        for dtype in (torch.float32, torch.bfloat16):
            for rows_of, source in ((row_of, x), (None, by_slot)):
                got = ops.grouped_linear(on(source), rows_of, tile_expert, bm, joined.cuda(), n_out * ldw, n_out, k, dtype)
                error = (got.double().cpu()[slots] - want).abs().max() / want.abs().max()
                assert float(error) <= (2e-6 * k ** 0.5 if dtype == torch.float32 else 2 ** -8)


# A list of more than 64 tiles, and sixteen tiles at a time with a few left over, over several strips of columns.
@pytest.mark.parametrize("bm,rows", [(64, 900), (128, 2700)])
def test_sorted_products_of_many_tiles_in_either_kernel(ops, bm, rows, monkeypatch):
    experts, top, k, n_out = 45, 2, 96, 520
    gen = torch.Generator().manual_seed(bm)
    chosen = torch.stack([torch.randperm(experts - 2, generator=gen)[:top] for _ in range(rows)]).to(torch.int32).cuda()
    x, w = rand_bf16((rows, k), 45), rand_bf16((experts * n_out, k), 46)
    slot_of, row_of, on_tiles = ops.expert_slots(chosen, experts, bm)
    used = int((on_tiles >= 0).sum())
    assert on_tiles.numel() > 64 and used > 16 and used % 16
    want = torch.empty((rows * top, n_out), dtype=torch.float64, device="cuda")
    for e in range(experts):
        at = (chosen.reshape(-1) == e).nonzero()[:, 0]
        want[at] = x[at // top].double() @ w[e * n_out:(e + 1) * n_out].double().t()
    for wide in (-1, 1):
        monkeypatch.setattr(ops, "grouped_wide", wide)
        got = ops.grouped_linear(x, row_of, on_tiles, bm, w, n_out * k, n_out, k, torch.float32)[slot_of.long()]
        assert float((got.double() - want).abs().max()) <= 2e-6 * k ** 0.5 * float(want.abs().max())


# The ring kernel's tiles: K of one step and of every number of steps past the first round of two, three or four buffers, with and
# without half a step behind them; columns of one tile, one past it, no multiple of four.
@pytest.mark.parametrize("bm,width", [(64, 64), (64, 128), (64, 256), (128, 128), (128, 256)])
@pytest.mark.parametrize("k", [64, 96, 128, 192, 224, 256, 320, 416, 448])
def test_sorted_products_of_every_ring(ops, bm, width, k, monkeypatch):
    experts, tiles, ldw = 2, 3, k + 24
    x = rand_bf16((tiles * bm, k + 8), k)
    x[:, k:] = float("nan")                                   # columns behind K are not read, on either side
    on_tiles = torch.tensor([1, -1, 0], dtype=torch.int32, device="cuda")
    row_of = torch.randperm(tiles * bm, generator=torch.Generator().manual_seed(k)).to(torch.int32).cuda()
    row_of[5] = -1
    for n_out in (width, width + 1, 90):
        joined = torch.full((experts * n_out, ldw), float("nan"), dtype=torch.bfloat16, device="cuda")
        joined[:, :k] = rand_bf16((experts * n_out, k), n_out)
        monkeypatch.setattr(ops, "grouped_wide", width)
        for dtype in (torch.float32, torch.bfloat16):
            got = ops.grouped_linear(x, row_of, on_tiles, bm, joined, n_out * ldw, n_out, k, dtype)
            for tile, expert in ((0, 1), (2, 0)):
                at = torch.arange(tile * bm, tile * bm + bm, device="cuda")
                at = at[row_of[at] >= 0]
                want = x[row_of[at].long(), :k].double() @ joined[expert * n_out:(expert + 1) * n_out, :k].double().t()
                # Float sums of K exact products: at most K / 2 roundings of 2^-24 of the largest partial sum, fewer in practice.
                error = float((got[at].double() - want).abs().max() / want.abs().max())
                assert error <= (2e-6 * k ** 0.5 if dtype == torch.float32 else 2 ** -8), (n_out, tile)


@pytest.mark.parametrize("bm", [64, 128])
def test_sorted_products_pass_over_tiles_without_slots_anywhere_in_the_list(ops, bm, monkeypatch):
    k, n_out, experts = 64, 256, 3
    of_tile = [2, -1, 0, -1, -1, 1, -1]
    x, w = rand_bf16((len(of_tile) * bm, k), 41), rand_bf16((experts * n_out, k), 42)
    on_tiles = torch.tensor(of_tile, dtype=torch.int32, device="cuda")
    for wide in (-1, 1):
        monkeypatch.setattr(ops, "grouped_wide", wide)
        got = ops.grouped_linear(x, None, on_tiles, bm, w, n_out * k, n_out, k, torch.float32)
        for tile, expert in enumerate(of_tile):
            if expert >= 0:
                at = slice(tile * bm, tile * bm + bm)
                want = x[at].double() @ w[expert * n_out:(expert + 1) * n_out].double().t()
                assert float((got[at].double() - want).abs().max()) <= 2e-6 * k ** 0.5 * float(want.abs().max())


def test_sorted_products_take_rows_far_apart(ops, monkeypatch):
    """More than 2^31 elements from the first row to the last that a single tile names."""
    k, n_out, bm, rows = 64, 256, 64, 2100
    x = torch.empty((rows, (1 << 20) + 8), dtype=torch.bfloat16, device="cuda")
    x[:, :k] = rand_bf16((rows, k), 43)
    w = rand_bf16((n_out, k), 44)
    row_of = (torch.arange(bm, dtype=torch.int32, device="cuda") * 33 + 5).contiguous()
    want = x[row_of.long(), :k].double() @ w.double().t()
    for wide in (-1, 1):
        monkeypatch.setattr(ops, "grouped_wide", wide)
        got = ops.grouped_linear(x, row_of, torch.zeros(1, dtype=torch.int32, device="cuda"), bm, w, n_out * k, n_out, k, torch.float32)
        assert float((got.double() - want).abs().max()) <= 2e-6 * k ** 0.5 * float(want.abs().max())


# Rows of one piece a lane, of two and an incomplete one, the longest; fewer experts than waves, one more, many; more rows than compute
# units (four waves a row).
@pytest.mark.parametrize("width,experts,top,rows", [(8, 3, 2, 1), (512, 8, 2, 5), (1032, 9, 4, 3), (4096, 17, 1, 2), (896, 8, 2, 300),
                                                    (2056, 64, 6, 7)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_routers_of_few_rows(ops, width, experts, top, rows, dtype):
    width = min(width, 2048) if dtype == torch.float32 else width         # (the longest rows the kernels take, in bytes)
    gen = torch.Generator().manual_seed(width + experts)
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(dtype)
    x, router = rand(rows, width), rand(experts, width)
    logits = x.double() @ router.double().t()
    chosen = torch.empty((rows, top), dtype=torch.int32, device="cuda")
    weights = torch.empty((rows, top), dtype=torch.float32, device="cuda")
    assert ops.route_rows(x.cuda(), router.cuda(), chosen, weights)
    best = torch.topk(logits, top, dim=-1)
    assert torch.equal(chosen.cpu().long(), best.indices)
    # (Logits of about sqrt(width) from float sums of `width` products.)
    torch.testing.assert_close(weights.double().cpu(), torch.softmax(best.values, -1), rtol=3e-6 * width, atol=1e-6)
    gate = torch.empty(rows, dtype=torch.float32, device="cuda")
    both = torch.cat([router, rand(1, width)])
    assert ops.route_rows_scores(x.cuda(), both.cuda(), None, experts, 0, 0, chosen, weights, softmax=True, group_max=False, gate=gate)
    assert torch.equal(chosen.cpu().long(), best.indices)
    picked = torch.softmax(logits, -1).gather(1, best.indices)
    torch.testing.assert_close(weights.double().cpu(), picked / (picked.sum(-1, keepdim=True) + 1e-20), rtol=3e-6 * width, atol=1e-6)
    torch.testing.assert_close(gate.double().cpu(), torch.sigmoid(x.double() @ both[-1].double()), rtol=3e-6 * width, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_router_over_nothing_takes_the_first_experts_alike(ops, dtype):
    x, router = torch.empty((1, 0), dtype=dtype, device="cuda"), torch.empty((11, 0), dtype=dtype, device="cuda")
    chosen, weights = torch.empty((1, 3), dtype=torch.int32, device="cuda"), torch.empty((1, 3), device="cuda")
    first = torch.arange(3, dtype=torch.int32, device="cuda")[None]
    for route in (lambda: ops.route_rows(x, router, chosen, weights),
                  lambda: ops.route_rows_scores(x, router, None, 11, 0, 0, chosen, weights, softmax=True),
                  lambda: ops.route_rows_sigmoid(x, router, torch.zeros(11, device="cuda"), 0, 0, chosen, weights)):
        chosen.fill_(-1)
        assert route() and torch.equal(chosen, first)
        torch.testing.assert_close(weights, torch.full_like(weights, 1 / 3), rtol=1e-6, atol=0)


@pytest.mark.parametrize("width", [4, 1028, 4096])
@pytest.mark.parametrize("count,normed", [(0, True), (0, False), (2, False), (3, False)])
def test_terms_onto_the_stream_without_terms_or_norm(ops, width, count, normed):
    rows = 5
    gen = torch.Generator().manual_seed(width + count)
    rand = lambda *shape: torch.randn(*shape, generator=gen, dtype=torch.float64)
    stream, weight = rand(rows, width).float(), rand(width).float()
    terms = [(rounded(rand(rows, width)), 0.5 + k, rand(width).float()) for k in range(count)]
    want = stream.double() + sum((f * s.double() * t for t, f, s in terms), torch.zeros(rows, width, dtype=torch.float64))
    wide = torch.full((rows, 2 * width), 7.0, dtype=torch.bfloat16, device="cuda")        # the result is a half of wider rows
    residual = stream.cuda()
    ops.add_terms_rmsnorm(residual, [(t.to(torch.bfloat16).cuda(), f, s.cuda()) for t, f, s in terms], weight.cuda() if normed else None,
                          1e-5, wide[:, :width], store_residual=True)
    torch.testing.assert_close(residual.double().cpu(), want, rtol=1e-6, atol=1e-6)
    result = plain.weighted_norm(want, weight.double(), 1e-5) if normed else want
    torch.testing.assert_close(wide[:, :width].double().cpu(), result, rtol=2 ** -8, atol=1e-6)
    assert bool((wide[:, width:] == 7.0).all())


# More tokens than compute units (256 threads a token) and the same tokens in calls of few (1,024), each against the reference: rows
# shorter than either workgroup, a row that 1,024 threads go through in turns with a rest, a whole-head and a partial rotation.
@pytest.mark.parametrize("n_q,n_k,n_v,d,dims", [(2, 1, 1, 24, 8), (14, 2, 2, 64, 64), (16, 16, 8, 128, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_norm_rotation_and_store_of_many_tokens_and_of_few(ops, n_q, n_k, n_v, d, dims, dtype):
    gen = torch.Generator().manual_seed(d + dims)
    count = torch.cuda.get_device_properties(0).multi_processor_count + 45
    rows = torch.randn(count, (n_q + n_k + n_v) * d, generator=gen).to(dtype).cuda()
    positions = torch.randint(0, 4096, (count,), generator=gen, dtype=torch.int32).cuda()
    slots = torch.randperm(count, generator=gen).to(torch.int32).cuda()
    rates, wq, wk = torch.rand(dims // 2, generator=gen).cuda(), torch.rand(n_q * d, generator=gen).cuda(), torch.rand(n_k * d, generator=gen).cuda()
    pages = lambda device: (torch.zeros(count // 16 + 1, n_k, 16, d, dtype=dtype, device=device),
                            torch.zeros(count // 16 + 1, n_v, d, 16, dtype=dtype, device=device))
    want = (rows.cpu(), *pages("cpu"))
    PlainOps(torch.float64).norm_rotate_store(want[0], None, positions.cpu(), rates.cpu(), dims, slots.cpu(), *want[1:], n_q, n_k, n_v,
                                              d, d, wq.cpu(), wk.cpu(), 1e-5)
    # Both results are rounded to bfloat16, where sums that differ by float32 rounding can end as neighbours (2^-7 of the value
    # apart at most); float32: sums of up to 2,048 squares.  Two terms of up to about 5 may cancel.
    bound = 2.0 ** -7 if dtype == torch.bfloat16 else 2e-5
    for step in (count, 40):
        got = (rows.clone(), *pages("cuda"))
        for at in range(0, count, step):
            part = slice(at, at + step)
            ops.norm_rotate_store(got[0][part], None, positions[part], rates, dims, slots[part], *got[1:], n_q, n_k, n_v, d, d,
                                  wq, wk, 1e-5)
        for mine, right in zip(got, want):
            torch.testing.assert_close(mine.cpu().float(), right.float(), rtol=bound, atol=1e-5)


# Weights read by whole cache lines (a K of whole lines, more than a trip of them) against the plain product: rows on either side of
# eight and up to sixteen, blocks of sixteen weight rows with only some of them there, K that leaves some waves a line less than
# others, that is one trip of a wave's whole share and that is several, four to sixteen waves, and a K that is no multiple of a line.
@pytest.mark.parametrize("rows", [1, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(24, 1088), (24, 1536), (4104, 1536), (20, 4160), (40, 5184), (16400, 640), (1540, 8256), (60, 3840), (40, 5192)])
def test_weights_by_whole_lines(ops, rows, n, k):
    x, w = rand_bf16((rows, k + 8), 7)[:, :k], (rand_bf16((2 * n, k), 8).float() * 0.05).to(torch.bfloat16)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(9)).cuda()
    exact = x.double() @ w.double().t()
    first, second = exact[:, :n], exact[:, n:]
    gated = first / (1 + torch.exp(-first)) * second

    def near(got, want):                       # float sums of K terms, and one rounding of the result to bfloat16 (2^-9)
        assert float((got.double() - want).abs().max()) <= 2 ** -8 * max(1.0, float(want.abs().max()))

    near(ops.linear(x, w[:n], bias), first + bias)
    parts = ops.linear(x, w[:n], bias, pending=True)
    near(parts if isinstance(parts, torch.Tensor) else parts.resolve(), first + bias)
    near(ops.linear_silu_gate(x, w), gated)
    near(ops.fused_norm_gated(x.contiguous(), None, 1e-6, w), gated)
    residual = torch.randn(rows, n, generator=torch.Generator().manual_seed(10)).cuda()
    want = residual.double() + first + bias
    ops.linear_add(x.contiguous(), w[:n], bias, residual)
    near(residual, want)


# Rows that a wave brings through its own part of LDS: one load and as many as eight rows take, nine rows beside them (straight from
# memory), a K of less than a wave's first line, with a last step of 32, with a tail of eight, and shares of 4, 8 and 10 steps; rows
# with a stride of their own and what lies beyond K in them no number.
@pytest.mark.parametrize("rows", [1, 2, 3, 5, 6, 8, 9])
@pytest.mark.parametrize("n,k", [(20, 8), (20, 40), (896, 480), (896, 896), (100, 1352), (1536, 1536), (900, 4064), (896, 4864), (52, 5000)])
def test_rows_staged_by_their_waves(ops, rows, n, k):
    x = torch.full((rows, k + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    x[:, :k] = rand_bf16((rows, k), 21)
    w = (rand_bf16((n, k), 22).float() * 0.05).to(torch.bfloat16)
    bias, residual = torch.randn(n, device="cuda"), torch.randn(rows, n, device="cuda")
    want = residual.double() + bias.double() + x[:, :k].double() @ w.double().t()
    slack = sum_slack(x[:, :k], w, bias, residual)
    ops.linear_add(x[:, :k], w, bias, residual)
    assert bool(((residual.double() - want).abs() <= slack).all())


# Choices counted in registers (up to 64 experts) and searched for (more): ties, logits and choice scores of minus infinity (with too few others to
# pick), an infinite logit and one that is no number, groups of one and of many, worth their largest score or their two largest, weights
# over their sum and as they are; the logits form, whose kernels search, is the reference.
@pytest.mark.parametrize("experts,groups,keep,top", [(8, 0, 0, 2), (8, 4, 2, 2), (8, 8, 3, 3), (1, 0, 0, 1), (64, 8, 2, 7), (60, 4, 1, 15), (64, 0, 0, 64), (72, 8, 2, 5)])
@pytest.mark.parametrize("softmax", [False, True])
@pytest.mark.parametrize("group_max", [False, True])
@pytest.mark.parametrize("renormalize", [False, True])
def test_choice_counted_is_choice_searched(ops, experts, groups, keep, top, softmax, group_max, renormalize):
    rows, width, inf = 5, 64, float("inf")
    x, router = torch.zeros((rows, width), dtype=torch.bfloat16), torch.zeros((experts, width), dtype=torch.bfloat16)
    x[:, :rows] = torch.eye(rows)
    router[:, 0] = rand_bf16((experts,), 41).cpu()
    router[:, 1] = torch.arange(experts) % 3                                    # ties
    router[:, 2] = torch.where(torch.arange(experts) < 1, 1.0, -3e38)           # all but one weigh nothing
    router[:, 3] = -torch.arange(experts) / 64
    router[:, 4] = torch.arange(experts) % 5 - 2
    noted = torch.randn(experts, generator=torch.Generator().manual_seed(42)).round(decimals=1)
    barred = torch.where(torch.arange(experts) % 4 == 1, noted, -inf)           # fewer than are picked are left
    # A row of one in column 0 alone against logits of minus infinity but for one, an infinite one among others, and one that is no number.
    single = torch.zeros((1, width), dtype=torch.bfloat16)
    single[0, 0] = 1
    columns = [torch.where(torch.arange(experts) == experts // 2, 1.0, -inf), router[:, 0].float(), router[:, 0].float()]
    columns[1][experts - 1], columns[2][experts // 2] = inf, float("nan")
    batches = [(x, router)]
    for column in columns:
        special = torch.zeros_like(router)
        special[:, 0] = column
        batches.append((single, special))
    for rows_in, matrix in batches:
        logits = (rows_in.float() @ matrix.float().t()) if len(rows_in) > 1 else matrix[:, 0].float()[None]      # (exact: one product a sum)
        shape = (len(rows_in), top)

        def chosen_by(route):
            chosen, weights = torch.full(shape, -1, dtype=torch.int32, device="cuda"), torch.full(shape, 7.0, device="cuda")
            assert route(chosen, weights) in (None, True)
            return chosen, weights

        def same(got, want):
            assert bool((want[0] >= 0).all()) and torch.equal(got[0], want[0])
            # (a weight is a quotient of terms of two roundings and sums of at most `experts` of them, in either order)
            assert torch.allclose(got[1], want[1], rtol=2 * (experts + 4) * 2.0 ** -24, atol=0, equal_nan=True)
        on = lambda t: None if t is None else t.contiguous().cuda()
        for correction in (None, noted, barred):
            more = dict(softmax=softmax, group_max=group_max, renormalize=renormalize)
            same(chosen_by(lambda c, w: ops.route_rows_scores(on(rows_in), on(matrix), on(correction), experts, groups, keep, c, w, **more)),
                 chosen_by(lambda c, w: ops.route_scores(on(logits), on(correction), experts, groups, keep, c, w, **more)))
        if not groups:
            same(chosen_by(lambda c, w: ops.route_rows(on(rows_in), on(matrix), c, w)), chosen_by(lambda c, w: ops.route_top(on(logits), c, w)))


# Rows in LDS beside the waves' sums at what a launch has of it unasked, 64 KB: just below, above, and at the most that is taken.
@pytest.mark.parametrize("rows,k", [(16, 1488), (16, 1520), (16, 1528), (12, 2040), (6, 4008), (6, 4096), (16, 3832)])
@pytest.mark.parametrize("normed", [False, True])
def test_fused_products_whose_rows_fill_local_memory(ops, rows, k, normed):
    gen = torch.Generator(device="cuda").manual_seed(k)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    x, w, weight = rand(rows, k), (rand(256, k) * k ** -0.5).bfloat16(), 1 + 0.3 * rand(k)
    if not normed:
        x, weight = x.bfloat16(), None
    unit = x.double() if weight is None else (x.double() / (x.double().square().mean(1, keepdim=True) + 1e-5).sqrt() * weight.double())
    # bfloat16 has eight bits: a rounding is 2^-8 of its value at most, and one that falls to the other side 2^-7.  A result is rounded once; the
    # normed rows before it, each |x| |w| of a sum by 2^-7; the K products are added in float (K units of 2^-24).
    rows_in = unit.bfloat16().double()
    product, mags = rows_in @ w.double().t(), rows_in.abs() @ w.double().t().abs()
    slack = (2.0 ** -7 * normed + k * 2.0 ** -24) * mags
    q = ops.fused_norm_qkv_rope(x, weight, 1e-5, w, None, torch.zeros(rows, dtype=torch.int32, device="cuda"), None, None, None, None, 2, 1, 64)
    assert bool(((q.double() - product[:, :128]).abs() <= 2.0 ** -8 * product[:, :128].abs() + slack[:, :128]).all())
    gated = ops.fused_norm_gated(x, weight, 1e-5, w)
    gate, up = product.chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    # (silu's slope is at most 1.1, silu(z) at most |z|; the exponential and the quotient are units of 2^-22.)
    slack = 1.1 * slack[:, :128] * (up.abs() + slack[:, 128:]) + gate.abs() * slack[:, 128:] + (2.0 ** -8 + 2.0 ** -20) * want.abs()
    assert bool(((gated.double() - want).abs() <= slack).all())


# Gated products of as many workgroups as pass their results by the chiplet's caches at most, and of more, in one block of rows and in two; silu and the
# capped activation.
@pytest.mark.parametrize("rows", [1, 8, 9])
@pytest.mark.parametrize("inner", [8192, 8200, 17000])
@pytest.mark.parametrize("capped", [False, True])
def test_gated_products_of_many_columns(ops, rows, inner, capped):
    x, w, k = rand_bf16((rows, 64), 33), rand_bf16((2 * inner, 64), 34), 64
    gate, up = (x.double() @ w.double().t()).chunk(2, 1)
    off_gate, off_up = (k * 2.0 ** -24 * x.double().abs() @ w.double().t().abs()).chunk(2, 1)      # K products added in float
    act = torch.tensor([1.7, 7.0, 1.0], device="cuda") if capped else None
    if capped:
        gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0) + 1
    alpha = 1.7 if capped else 1.0
    want = gate * torch.sigmoid(alpha * gate) * up
    # z sigmoid(alpha z) has a slope of at most 1.1; the exponential's argument is below 128 and rounded twice, the rest are units of 2^-22.
    slack = 1.1 * off_gate * (up.abs() + off_up) + gate.abs() * off_up + (2.0 ** -8 + 2.0 ** -15) * want.abs()
    assert bool(((ops.fused_norm_gated(x, None, 0.0, w, act).double() - want).abs() <= slack).all())


# Workgroups of four, seven, nine and sixteen weight rows with a last one that is not full; K below a step, with a tail, of one trip and
# of several, by steps and by lines; rows that are staged in one load and in as many as eight rows take, and that come straight from
# memory, at the last share of K that is staged and the first that is not; rows of a longer stride with no numbers beyond K; the gate with few
# and with many columns.
@pytest.mark.parametrize("rows", [1, 3, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(8, 8), (20, 40), (900, 904), (1544, 2112), (2060, 1536), (900, 4864), (1100, 6720), (4100, 904), (16400, 1536),
                                 (300, 768), (300, 776), (300, 1032), (300, 2056), (4100, 1032), (16400, 392), (16400, 1000), (16400, 1064)])
def test_products_of_few_rows_spread_over_the_device(ops, rows, n, k):
    x = torch.full((rows, k + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    x[:, :k] = rand_bf16((rows, k), 31)
    w = (rand_bf16((2 * n, k), 32).float() * 0.05).to(torch.bfloat16)
    bias = torch.randn(n, device="cuda")
    exact = x[:, :k].double() @ w.double().t()
    got = ops.linear(x[:, :k], w[:n], bias, out_dtype=torch.float32)
    assert bool(((got.double() - exact[:, :n] - bias.double()).abs() <= sum_slack(x[:, :k], w[:n], bias)).all())
    gate = exact[:, :n]
    want = gate / (1 + torch.exp(-gate)) * exact[:, n:]
    got = ops.linear_silu_gate(x[:, :k], w)
    assert float((got.double() - want).abs().max()) <= 2 ** -8 * max(1.0, float(want.abs().max()))     # (one rounding to bfloat16)


@pytest.mark.parametrize("rows", [1, 16])
@pytest.mark.parametrize("k", [2112, 3584])
def test_qkv_by_whole_lines(ops, rows, k):
    heads, kv, d, page = 3, 1, 32, 16
    x, w = rand_bf16((rows, k), 11), (rand_bf16(((heads + 2 * kv) * d, k), 12).float() * 0.05).to(torch.bfloat16)
    positions = torch.arange(rows, dtype=torch.int32, device="cuda")
    k_pages = torch.zeros(1, kv, page, d, dtype=torch.bfloat16, device="cuda")
    v_pages = torch.zeros(1, kv, d, page, dtype=torch.bfloat16, device="cuda")
    q = ops.fused_norm_qkv_rope(x, None, 1e-6, w, None, positions, None, positions, k_pages, v_pages, heads, kv, d)
    want = x.double() @ w.double().t()
    got = torch.cat([q, k_pages[0, 0, :rows], v_pages[0, 0, :, :rows].t()], dim=1)
    assert float((got.double() - want).abs().max()) <= 2 ** -8 * float(want.abs().max())


# The float32 products of few rows: a K of whole lines and not, that leaves a wave's last pair of units empty, whose parts are cut, weight
# rows that end inside a tile, one to sixteen rows on both sides of the choice between matrix and vector instructions, and more workgroups
# than compute units.
@pytest.mark.parametrize("rows", [1, 2, 4, 5, 16])
@pytest.mark.parametrize("n,k", [(24, 96), (20, 1056), (36, 4864), (4200, 2016), (40, 1004)])
def test_float32_weights_by_whole_lines(ops, rows, n, k):
    gen = torch.Generator().manual_seed(n + rows)
    x, w = torch.randn(rows, k + 4, generator=gen).cuda()[:, :k], torch.randn(2 * n, k, generator=gen).cuda() * 0.05
    bias = torch.randn(n, generator=gen).cuda()
    exact = x.double() @ w.double().t()
    first, second = exact[:, :n], exact[:, n:]

    def near(got, want):                       # sums of K products of numbers around 0.05: K 2^-24 of their absolute sum at most, far less in fact
        assert got.dtype == torch.float32 and float((got.double() - want).abs().max()) <= 1e-5 * max(1.0, float(want.abs().max()))

    near(ops.linear(x, w[:n], bias), first + bias)
    parts = ops.linear(x, w[:n], bias, pending=True)
    near(parts if isinstance(parts, torch.Tensor) else parts.resolve(), first + bias)
    near(ops.linear_silu_gate(x, w), first / (1 + torch.exp(-first)) * second)


@pytest.mark.parametrize("rows", [1, 5, 16])
@pytest.mark.parametrize("heads,kv,d,k", [(3, 1, 32, 96), (14, 2, 64, 896), (2, 2, 96, 1000)])
@pytest.mark.parametrize("rotate", [False, True])
def test_float32_qkv_with_rotation_and_store(ops, rows, heads, kv, d, k, rotate):
    gen = torch.Generator().manual_seed(d + rows)
    rand = lambda *shape: torch.randn(*shape, generator=gen).cuda()
    x, w, bias = rand(rows, k), rand((heads + 2 * kv) * d, k) * 0.05, rand((heads + 2 * kv) * d)
    positions = torch.randint(0, 40, (rows,), generator=gen, dtype=torch.int32).cuda()
    slots = torch.randperm(48, generator=gen)[:rows].to(torch.int32).cuda()
    slots[rows // 2] = -1                                     # this row's keys and values are not stored
    table = rand(40, d) if rotate else None
    pages = [(torch.full((3, kv, 16, d), 7.0, device="cuda"), torch.full((3, kv, d, 16), 7.0, device="cuda")) for _ in range(2)]
    q = ops.fused_norm_qkv_rope(x, None, 0.0, w, bias, positions, table, slots, *pages[0], heads, kv, d)
    qkv = (x.double() @ w.double().t() + bias).float()
    ops.rope_store(qkv, None, positions, table, slots, *pages[1], heads, kv, d)
    torch.testing.assert_close(q, qkv[:, :heads * d], rtol=1e-5, atol=2e-5)
    for got, want in zip(*pages):
        torch.testing.assert_close(got, want, rtol=1e-5, atol=2e-5)
    silent = ops.fused_norm_qkv_rope(x, None, 0.0, w, bias, positions, table, None, *pages[0], heads, kv, d)
    assert torch.equal(silent, q)


# The short convolution of steps of a token an entry: entries of none, one of two, one that starts and one that goes on, a row that only fills the
# batch up, two to four taps and (five: the kernels of long portions) more, three runs of channels past a workgroup's 256; as many rows as
# entries (one kernel for all of it) and one row more (the two kernels of long portions).
@pytest.mark.parametrize("lengths,starts", [([1, 0, 2, 0, 1, 1], [0, 0, 7, 5, 3, 0]), ([1, 0, 2, 1, 1], [0, 0, 7, 3, 0])])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("biased", [False, True])
def test_short_convolution_of_single_tokens(ops, lengths, starts, dtype, taps, biased):
    gen = torch.Generator().manual_seed(taps)
    widths, offsets, fill = (96, 200, 40), (4, 300, 104), 1
    channels, n, keep = sum(widths), sum(lengths) + fill, taps - 1
    rows = torch.randn(n, 512, generator=gen).to(dtype)
    weights, bias = torch.randn(channels, taps, generator=gen), torch.randn(channels, generator=gen) if biased else None
    state = torch.randn(8, 5 + keep * channels + 3, generator=gen)
    slots = torch.randperm(8, generator=gen)[:len(lengths)]
    entry = [e for e, count in enumerate(lengths) for _ in range(count)] + [-1] * fill
    cu = [0]
    for count in lengths:
        cu.append(cu[-1] + count)
    x = torch.cat([rows[:, o:o + w] for o, w in zip(offsets, widths)], dim=1).double()
    want, behind = torch.zeros(n, channels, dtype=torch.float64), state.double().clone()
    for e, s in enumerate(slots.tolist()):
        kept = state[s, 5:5 + keep * channels].double().reshape(keep, channels) * (starts[e] > 0)
        for t in range(cu[e], cu[e + 1]):
            window = torch.cat([kept, x[t:t + 1]])
            y = (weights.double() * window.t()).sum(1) + (bias.double() if biased else 0)
            want[t] = y / (1 + torch.exp(-y))
            kept = window[1:]
        if lengths[e]:
            behind[s, 5:5 + keep * channels] = kept.reshape(-1)
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    held, out = state.cuda(), torch.full((n, channels), 7.0, dtype=dtype, device="cuda")
    ops.short_conv_silu(rows.cuda(), offsets, widths, weights.cuda(), held, 5, ints(cu), ints(starts), ints(slots.tolist()), ints(entry), out,
                        **({"bias": bias.cuda()} if biased else {}))
    rounding = 2 ** -8 if dtype == torch.bfloat16 else 1e-6   # the result's rounding; float sums of five terms
    assert float((out.double().cpu() - want).abs().max()) <= rounding * max(1.0, float(want.abs().max()))
    torch.testing.assert_close(held.double().cpu(), behind, rtol=0, atol=0)


# Products head by head with a gate a head and a gate a result: rows on either side of eight and of sixteen (the kernels of more rows, and the gate's
# own), heads whose results end inside a workgroup's four, a K of several trips and of less than one.
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17])
@pytest.mark.parametrize("heads,n,k", [(3, 10, 40), (14, 64, 136), (2, 33, 1032)])
@pytest.mark.parametrize("each", [False, True])
def test_head_products_with_gates(ops, rows, heads, n, k, each):
    x, w = rand_bf16((rows, heads * k), 3), (rand_bf16((heads, n, k), 4).float() * 0.1).to(torch.bfloat16)
    units = n if each else 1
    gates = rand_bf16((rows, 5 + heads * units + 2), 5)
    out = torch.full((rows, heads * n), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.head_linear(x, 0, k, w, out, 0, n, gate=(gates, 5, units))
    product = torch.stack([x[:, h * k:(h + 1) * k].double() @ w[h].double().t() for h in range(heads)], dim=1)
    factor = 1 / (1 + torch.exp(-gates[:, 5:5 + heads * units].double().reshape(rows, heads, units)))
    want = (product * factor).reshape(rows, heads * n)
    assert float((out.double() - want).abs().max()) <= 2 ** -7 * max(1.0, float(want.abs().max()))     # two roundings to bfloat16


# Rows of pieces of eight, a thread a piece: a norm over the queries alone, over the keys alone and over neither, a bias, values narrower than keys, no rotation
# and one of whole heads, tokens that store nothing, a wave of threads and just over the most (the general kernel).
@pytest.mark.parametrize("n_q,n_k,n_v,d,dv,dims,norms,biased", [(4, 2, 1, 48, 16, 16, (True, False), True), (3, 1, 1, 32, 32, 0, (False, True), False),
                                                                (24, 4, 2, 128, 128, 64, (True, True), False), (6, 6, 6, 64, 24, 64, (False, False), True),
                                                                (62, 1, 1, 128, 128, 128, (True, True), True), (64, 33, 32, 64, 64, 32, (True, True), True)])
def test_norm_rotation_and_store_by_pieces(ops, n_q, n_k, n_v, d, dv, dims, norms, biased):
    gen = torch.Generator().manual_seed(d + n_q)
    rand = lambda *shape: torch.rand(*shape, generator=gen) + 0.2
    count, used = 7, (n_q + n_k) * d + n_v * dv
    rows = torch.randn(count, used + 8, generator=gen).to(torch.bfloat16)
    positions = torch.tensor([0, 1, 63, 64, 1000, 4095, 17], dtype=torch.int32)
    slots = torch.tensor([3, -1, 47, 16, 0, 31, 5], dtype=torch.int32)
    rates, wq, wk, bias = rand(dims // 2), rand(n_q * d) if norms[0] else None, rand(n_k * d) if norms[1] else None, rand(used + 8) if biased else None
    pages = lambda device: (torch.zeros(3, n_k, 16, d, dtype=torch.bfloat16, device=device),
                            torch.zeros(3, n_v, dv, 16, dtype=torch.bfloat16, device=device))
    on = lambda t: None if t is None else t.cuda()
    want, got = (rows.clone(), *pages("cpu")), (rows.cuda(), *pages("cuda"))
    PlainOps(torch.float64).norm_rotate_store(want[0], bias, positions, rates if dims else None, dims, slots, *want[1:], n_q, n_k, n_v, d, dv, wq, wk, 1e-5)
    ops.norm_rotate_store(got[0], on(bias), positions.cuda(), on(rates) if dims else None, dims, slots.cuda(), *got[1:], n_q, n_k, n_v, d, dv,
                          on(wq), on(wk), 1e-5)
    for mine, right in zip(got, want):                        # neighbours in bfloat16; angles of up to 4,095 in float32 (3e-4 of a radian)
        torch.testing.assert_close(mine.cpu().float(), right.float(), rtol=2.0 ** -7, atol=4e-3)


# Two latents and a turned tail, a thread keeping one, two, four or eight of a latent's elements: latents on either side of each of those and longer than the
# most that is kept, one of each far shorter than the other, a tail of none, of two, and of more pairs than threads, tokens that store nothing.
@pytest.mark.parametrize("q_rank,kv_rank,rot", [(256, 1, 2), (257, 96, 0), (96, 513, 64), (1024, 1025, 16), (2049, 8, 600), (40, 2305, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("neighbours,values", [(False, True), (True, False)])
def test_latents_kept_in_registers(ops, q_rank, kv_rank, rot, dtype, neighbours, values):
    gen = torch.Generator().manual_seed(q_rank + kv_rank)
    width, slots = kv_rank + rot, torch.tensor([3, -1, 47, 16, 0], dtype=torch.int32)
    rows = torch.randn(5, 3 + q_rank + kv_rank + rot, generator=gen).to(dtype)
    q_norm, kv_norm, rates = (torch.rand(n, generator=gen) + 0.2 for n in (q_rank, kv_rank, rot // 2))
    positions = torch.tensor([0, 1, 63, 100, 17], dtype=torch.int32)
    got_q = torch.full((5, q_rank), 7.0, dtype=dtype, device="cuda")
    k_pages = torch.zeros(3, 1, 16, width, dtype=dtype, device="cuda")
    v_pages = torch.zeros(3, 1, width, 16, dtype=dtype, device="cuda") if values else None
    ops.latent_store(rows.cuda(), 3, q_rank, q_norm.cuda(), 3 + q_rank, kv_rank, kv_norm.cuda(), rot, rates.cuda() if rot else None, 1e-5,
                     positions.cuda(), slots.cuda(), k_pages, v_pages, got_q, neighbours)
    unit = lambda x, w: x / (x.square().mean(1, keepdim=True) + 1e-5).sqrt() * w.double()
    x = rows.double()
    want_q, kept = unit(x[:, 3:3 + q_rank], q_norm), unit(x[:, 3 + q_rank:3 + q_rank + kv_rank], kv_norm)
    angles = (positions.float()[:, None] * rates[None, :]).double()       # the angle is a float product
    tail, half = x[:, 3 + q_rank + kv_rank:], rot // 2
    a, b = (tail[:, 0::2], tail[:, 1::2]) if neighbours else (tail[:, :half], tail[:, half:])
    lo, hi = a * angles.cos() - b * angles.sin(), b * angles.cos() + a * angles.sin()
    kept = torch.cat([kept, torch.stack([lo, hi], -1).flatten(1) if neighbours else torch.cat([lo, hi], 1)], 1)
    want_k = torch.zeros(3 * 16, width, dtype=torch.float64)
    for t, slot in enumerate(slots.tolist()):
        if slot >= 0:
            want_k[slot] = kept[t]
    # A rounding to the type; in 32 bits sums of 2,305 squares and a root's and a quotient's roundings, 16 units of 2^-23 on values below 8.
    tol = dict(rtol=2 ** -8, atol=1e-6) if dtype == torch.bfloat16 else dict(rtol=16 * 2 ** -23, atol=8 * 16 * 2 ** -23)
    torch.testing.assert_close(got_q.double().cpu(), want_q, **tol)
    torch.testing.assert_close(k_pages.double().cpu().reshape(48, width), want_k, **tol)
    if values:
        torch.testing.assert_close(v_pages.double().cpu()[:, 0].transpose(1, 2).reshape(48, width), want_k, **tol)


# Many rows, whose two latents share a workgroup where one is short, and the same rows a few at a time, which have one each: latents of one wave and of
# four, and longer, either of them the short one, tails of none and of more pairs than the keys' waves have threads, tokens that store nothing.
@pytest.mark.parametrize("q_rank,kv_rank,rot", [(64, 64, 0), (192, 64, 64), (100, 600, 32), (256, 129, 2), (1030, 40, 300), (2100, 128, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_latents_of_many_rows_have_the_bits_of_few(ops, q_rank, kv_rank, rot, dtype):
    gen = torch.Generator().manual_seed(q_rank + rot)
    n, width, few = 2 * ops.compute_units + 7, kv_rank + rot, 61
    rows, norms = torch.randn(n, q_rank + kv_rank + rot, generator=gen).to(dtype).cuda(), [torch.rand(r, generator=gen).cuda() for r in (q_rank, kv_rank)]
    rates, positions = torch.rand(rot // 2, generator=gen).cuda(), torch.randint(0, 4000, (n,), generator=gen, dtype=torch.int32).cuda()
    slots = torch.randperm(n, generator=gen).int()
    slots[::9] = -1
    slots, results = slots.cuda(), []
    for step in (n, few):
        q = torch.full((n, q_rank), 7.0, dtype=dtype, device="cuda")
        k_pages = torch.full((-(-n // 16), 1, 16, width), 7.0, dtype=dtype, device="cuda")
        v_pages = torch.full((-(-n // 16), 1, width, 16), 7.0, dtype=dtype, device="cuda")
        for i in range(0, n, step):
            at = slice(i, i + step)
            ops.latent_store(rows[at], 0, q_rank, norms[0], q_rank, kv_rank, norms[1], rot, rates if rot else None, 1e-5, positions[at], slots[at],
                             k_pages, v_pages, q[at])
        results.append((q, k_pages, v_pages))
    for many, one in zip(*results):
        assert many.isfinite().all() and torch.equal(many, one)


# A matrix memory stepped a token at a time against the recurrence in 64 bits.  Widths on either side of the rows a thread holds and of the columns of a workgroup;
# an entry that goes on, one that only fills the batch up, one that starts (in a state row full of NaN), state rows in another order.
@pytest.mark.parametrize("heads,d,dv", [(1, 16, 16), (3, 33, 40), (2, 128, 256), (3, 72, 17), (1, 200, 3), (1, 256, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_matrix_memory_of_single_tokens(ops, heads, d, dv, dtype):
    gen = torch.Generator().manual_seed(d + dv)
    slots, steps, cap = [2, 1, 0], 4, 15.0
    keys, values = 2 * heads * d, heads * d * dv
    state = torch.rand(3, values + heads * d + heads + 4, generator=gen)
    state[0, :values + heads * d + heads] = float("nan")
    held, ints = state.cuda(), lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    C, n, m = (state[[2, 0], a:b].double().reshape(2, heads, *shape) for a, b, shape in
               ((0, values, (d, dv)), (values, values + heads * d, (d,)), (values + heads * d, values + heads * d + heads, ())))
    C[1], n[1], m[1] = 0.0, 0.0, 0.0
    # An exponent's argument (below 48) is rounded three times and a product twice a step; sums of d and of sixteen rows.
    unit = (steps * (3 * 48 + 4) + d) * 2.0 ** -24
    for i in range(steps):
        x = torch.randn(2, keys + heads * dv + 5, generator=gen).to(dtype)
        gates = 3 * torch.randn(2, 2 * heads + 1, generator=gen)
        out = torch.full((2, heads * dv), 7.0, device="cuda")
        ops.mlstm_scan(x.cuda(), gates.cuda(), held, ints([0, 1, 1, 2]), ints([7 + i, 0, i]), ints(slots), out, heads, d, dv, cap)
        q, k = (x.double()[:, a:a + heads * d].reshape(2, heads, d) for a in (0, heads * d))
        v, q = x.double()[:, keys:keys + heads * dv].reshape(2, heads, dv), q / d ** 0.5
        g = cap * torch.tanh(gates.double() / cap)
        gi, gf = g[:, :heads], torch.nn.functional.logsigmoid(g[:, heads:2 * heads])
        after = torch.maximum(gf + m, gi)
        keep, take = (gf + m - after).exp(), (gi - after).exp()
        C = keep[..., None, None] * C + take[..., None, None] * k[..., :, None] * v[..., None, :]
        n, m = keep[..., None] * n + take[..., None] * k, after
        least = torch.maximum((n * q).sum(-1).abs(), (-m).exp()) + 1e-6
        want = (C * q[..., None]).sum(-2) / least[..., None]
        mags = [(a.abs().amax() * q.abs().sum(-1) / least)[..., None] for a in (C, n)]
        slack = unit * (mags[0] + want.abs() * mags[1] + want.abs())
        assert bool(((out.double().cpu().reshape(2, heads, dv) - want).abs() <= slack).all())
    got = held[[2, 0]].double().cpu()
    for a, want in ((0, C), (values, n), (values + heads * d, m)):
        part = got[:, a:a + want[0].numel()].reshape(want.shape)
        assert float((part - want).abs().max()) <= unit * max(1.0, float(want.abs().max()))
    assert torch.equal(held[1].cpu(), state[1])


# The streams' step with the token shift behind it, against 64 bits: one to four streams, columns of one wave and of sixteen, a last wave that is
# partly empty, few rows and (at up to 256 columns) more than twice the compute units; a write pending and none.  Of five rows one only fills the
# batch up (it takes no state and leaves none), one starts over a state row of NaN; entries and state rows lie in other orders.
@pytest.mark.parametrize("streams", [1, 2, 3, 4])
@pytest.mark.parametrize("width,rows", [(52, 5), (200, 700), (256, 5), (896, 10), (1000, 5), (1024, 15)])
@pytest.mark.parametrize("written,out_dtype", [(None, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                               (torch.float32, torch.float32)])
def test_streams_step_with_the_token_shift(ops, streams, width, rows, written, out_dtype):
    gen = torch.Generator().manual_seed(width + streams)
    rand = lambda *shape: torch.randn(*shape, generator=gen)
    x, read, gain, mu, eps = rand(rows, streams, width), rand(streams), torch.tensor([1.7]), torch.rand(width, generator=gen), 1e-5
    y, mix, coef, scale = rand(rows, width).to(written or torch.float32), rand(streams, streams), rand(streams), rand(width)
    entry = torch.randperm(rows, generator=gen).int()
    filler, fresh = torch.arange(rows) % 5 == 1, torch.arange(rows) % 5 == 2
    entry[filler] = -1
    slots = torch.randperm(rows + 3, generator=gen)[:rows].int()              # by entry
    positions = torch.where(fresh, 0, 3 + torch.arange(rows)).int()
    row_of = slots[entry.clamp(min=0).long()].long()                          # by row
    state = rand(rows + 3, width)
    state[row_of[fresh & ~filler]] = float("nan")
    kept = state.clone()
    ctx = types.SimpleNamespace(entry_of_token=entry.cuda(), state_slots=slots.cuda(), positions=positions.cuda())
    held, on_state = x.cuda(), state.cuda()
    write = types.SimpleNamespace(y=y.cuda(), mix=mix.cuda(), out=coef.cuda(), scale=scale.cuda()) if written else None
    got = torch.empty((rows, width), dtype=out_dtype, device="cuda")
    ops.streams_step(held, write, read.cuda(), gain.cuda(), eps, got, shift=(mu.cuda(), on_state, ctx))
    new, mags = x.double(), x.double().abs()
    if written:
        add = scale.double() * y.double()
        new = torch.einsum("tsw,sr->trw", new, mix.double()) + coef.double()[None, :, None] * add[:, None]
        mags = torch.einsum("tsw,sr->trw", mags, mix.double().abs()) + coef.double().abs()[None, :, None] * add.abs()[:, None]
    # A stream is a sum of at most five terms, the read one of four, each term rounded twice; the root mean square adds sums of sixty-four,
    # of sixteen waves, a quotient and a root to what the squares are off by.
    unit = 2.0 ** -24
    assert bool(((held.double().cpu() - new).abs() <= 12 * unit * mags).all())
    u, off = torch.einsum("tsw,s->tw", new, read.double()), 20 * unit * torch.einsum("tsw,s->tw", mags, read.double().abs())
    rms = (u.square().mean(1, keepdim=True) + eps).sqrt()
    h = u / rms * 1.7
    off = 1.7 * off / rms + h.abs() * (off.norm(dim=1, keepdim=True) / u.norm(dim=1, keepdim=True) + 40 * unit)
    live = ~filler
    before = torch.where(fresh[:, None], 0.0, kept[row_of].double())
    want = torch.where(live[:, None], h + (before - h) * mu.double(), h)
    slack = 2 * off + 4 * unit * (h.abs() + before.nan_to_num().abs()) + (2.0 ** -8 * want.abs() if out_dtype == torch.bfloat16 else 0.0)
    assert bool(((got.double().cpu() - want).abs() <= slack).all())
    after = on_state.cpu()
    assert bool(((after[row_of[live]].double() - h[live]).abs() <= off[live]).all())
    untouched = torch.ones(rows + 3, dtype=torch.bool)
    untouched[row_of[live]] = False
    assert torch.equal(after[untouched], kept[untouched])
