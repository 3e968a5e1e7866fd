"""In which order the products of few rows and the sums over a wave add up.  Reading the weights by whole cache lines, or a sum through
other instructions, must leave the sums as they were: a product's bits decide a router's near ties, and with them whole rows of logits."""
from ctypes import c_void_p

import pytest
import torch

pytestmark = pytest.mark.gpu
BIG = 2.0 ** 30       # (in float32 a one that meets it before its negative does is lost)


@pytest.fixture(scope="module")
def ops():
    from tokenizer_amd.kernels import get_ops
    return get_ops()


def rand(shape, seed, scale=1.0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=gen, device="cuda") * scale).bfloat16()


def pattern(k, *places):
    """Elements of K that add up to one if `places` (the big number, its negative, the one) meet in this order, else to zero."""
    row = torch.zeros(k, dtype=torch.bfloat16, device="cuda")
    for place, value in zip(places, (BIG, -BIG, 1.0)):
        row[place] = value
    return row


# Columns and K by the launcher's sixteen, eight and four sums a tile, its lines a trip (1, 2, 3, 4 and 6), one workgroup a compute unit,
# and columns that end inside a tile.
@pytest.mark.parametrize("rows", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n, k, gated", [(1000, 2240, False), (1000, 3584, False), (4200, 1344, False), (4200, 1984, False),
                                         (4096, 4160, False), (16400, 704, False), (1000, 2240, True), (4200, 1344, True),
                                         (4200, 1984, True), (4200, 2048, True), (16400, 704, True), (16400, 2048, True)])
def test_product_by_whole_lines_has_the_bits_of_half_lines(ops, rows, n, k, gated):
    x, w = rand((rows, k + 8), 1)[:, :k], rand((n * (2 if gated else 1), k), 2, 0.05)
    bias = rand((n,), 3).float()
    run = (lambda: ops.linear_silu_gate(x, w)) if gated else (lambda: ops.linear(x, w, bias, out_dtype=torch.float32))
    got = run()
    ops.lib.ta_skinny_lines(0)
    try:
        want = run()
    finally:
        ops.lib.ta_skinny_lines(1)
    assert got.isfinite().all() and torch.equal(got, want)


@pytest.mark.parametrize("rows", [1, 16])
@pytest.mark.parametrize("k", [896, 1536, 3584, 4864, 8960])
def test_fused_products_add_32_elements_of_k_at_a_time(ops, rows, k):
    x = torch.ones((rows, k), dtype=torch.bfloat16, device="cuda")
    w = pattern(k, 0, 8, 33).repeat(80, 1)
    residual = torch.zeros((rows, 80), device="cuda")
    ops.linear_add(x, w, None, residual)
    assert (residual == 1).all()
    gated = ops.fused_norm_gated(x, None, 0.0, w)
    want = torch.nn.functional.silu(torch.ones(1)).bfloat16().item()
    assert ((gated.float() - want).abs() <= 2 ** -8).all()


@pytest.mark.parametrize("rows", [1, 12])
@pytest.mark.parametrize("hidden, inner", [(512, 64), (1536, 1088)])
def test_experts_of_few_rows_add_32_elements_of_k_at_a_time(ops, rows, hidden, inner):
    x = torch.ones((rows, hidden), dtype=torch.bfloat16, device="cuda")
    first = pattern(hidden, 0, 8, 33).repeat(2 * inner, 1)                 # (two experts; relu squared of one is one)
    second = torch.cat([pattern(inner, 0, 8, 33)] * 2).repeat(hidden, 1)
    chosen = torch.zeros((rows, 1), dtype=torch.int32, device="cuda")
    chosen[1::2] = 1
    got = ops.experts_few(x, chosen, torch.ones((rows, 1), device="cuda"), 2, first, False, inner, second)
    assert (got.partial == 1).all()


@pytest.mark.parametrize("rows", [1, 8, 11])
def test_sum_over_a_wave_starts_with_lanes_32_apart(ops, rows):
    # A lane holds eight elements of K: lanes 0 and 32 meet first, lane 1's one afterwards.
    heads, n, k = 3, 20, 512
    x = torch.ones((rows, heads * k), dtype=torch.bfloat16, device="cuda")
    w = pattern(k, 0, 256, 8).repeat(heads, n, 1)
    out = torch.empty((rows, heads * n), dtype=torch.bfloat16, device="cuda")
    ops.head_linear(x, 0, k, w, out, 0, n)
    assert (out == 1).all()
    gate = torch.zeros((rows, heads * n), dtype=torch.bfloat16, device="cuda")
    ops.head_linear(x, 0, k, w, out, 0, n, gate=(gate, 0, n))
    assert (out == 0.5).all()


@pytest.mark.parametrize("hidden, inner, shared", [(512, 1040, 0), (1000, 1040, 64), (2056, 520, 0), (520, 512, 0), (512, 520, 40)])
def test_experts_of_one_row_and_of_many_have_the_same_bits(ops, hidden, inner, shared):
    # Few workgroups ask for four turns of K at once, many for one: shares of K that end inside a trip, K that is no whole line.
    experts, top = 8, 2
    x = rand((16, hidden), 4)
    first, second = rand((2 * (experts * inner + shared), hidden), 5, hidden ** -0.5), rand((hidden, experts * inner + shared), 6, inner ** -0.5)
    gen = torch.Generator().manual_seed(7)
    chosen = torch.stack([torch.randperm(experts, generator=gen)[:top] for _ in range(16)]).int().cuda()
    weights = torch.rand((16, top), generator=gen).cuda()
    run = lambda rows: ops.experts_few(x[:rows], chosen[:rows].contiguous(), weights[:rows].contiguous(), experts, first, True, inner,
                                       second, shared=shared).partial
    many, one = run(16), run(1)
    assert many.isfinite().all() and torch.equal(many[:, :1], one)


def test_merged_parts_join_their_neighbours_in_one_rounding(ops):
    # Part 0 has x, part 1 -x under the same weight w = exp(-0.3): joined in one rounding, x w - round(x w) is what the rounding left, at most
    # half a unit in the last place of a product below 4; joined after two roundings it is zero.  Part 2 has the largest maximum and the
    # whole denominator, so that the result is the sum itself.
    heads, splits = 3, 4
    for d, single in ((32, True), (64, True), (96, False), (128, False)):
        part_o = torch.zeros((16, heads, splits, d), device="cuda")
        part_o[:, :, 0] = torch.rand((16, heads, d), generator=torch.Generator(device="cuda").manual_seed(d), device="cuda") + 1
        part_o[:, :, 1] = -part_o[:, :, 0]
        part_ml = torch.zeros((16, heads, splits, 2), device="cuda")
        part_ml[:, :, :2, 0], part_ml[:, :, 3, 0], part_ml[:, :, 2, 1] = -0.3, -0.3, 1.0
        ints = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
        tiles, cu_q = ints(0, 0), ints(0, 16)
        out = torch.full((16, heads * d), 7.0, dtype=torch.bfloat16, device="cuda")
        assert ops.lib.ta_attention_merge_tiles(*(c_void_p(t.data_ptr()) for t in (part_o, part_ml, tiles)), 1, c_void_p(cu_q.data_ptr()),
                                                c_void_p(out.data_ptr()), heads, d, splits, ops._stream()) == 0
        assert bool((out.abs() <= 2.0 ** -23).all())
        assert float((out != 0).float().mean()) > 0.9 if single else not out.any()


@pytest.mark.parametrize("heads,d,dv", [(1, 16, 16), (3, 33, 40), (2, 128, 256), (1, 256, 17)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_matrix_memory_of_tokens_one_by_one_has_the_bits_of_a_walk(ops, heads, d, dv, dtype):
    # Tokens a step each and all of them in one portion; one request from its start and one that goes on.
    steps, cap, width = 6, 15.0, heads * (2 * d + dv)
    gen = torch.Generator(device="cuda").manual_seed(d + dv)
    x = torch.randn((2, steps, width), generator=gen, device="cuda").to(dtype)
    gates = 3 * torch.randn((2, steps, 2 * heads), generator=gen, device="cuda")
    start = torch.rand((2, heads * (d * dv + d + 1)), generator=gen, device="cuda")
    ints = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    walked, stepped = start.clone(), start.clone()
    want, got = (torch.empty((2, steps, heads * dv), device="cuda") for _ in range(2))
    ops.mlstm_scan(x.reshape(2 * steps, width), gates.reshape(2 * steps, -1), walked, ints(0, steps, 2 * steps), ints(0, 9), ints(1, 0),
                   want.view(2 * steps, -1), heads, d, dv, cap)
    for i in range(steps):
        out = torch.empty((2, heads * dv), device="cuda")
        ops.mlstm_scan(x[:, i].contiguous(), gates[:, i].contiguous(), stepped, ints(0, 1, 2), ints(i, 9 + i), ints(1, 0), out, heads, d, dv, cap)
        got[:, i] = out
    assert want.isfinite().all() and torch.equal(got, want) and torch.equal(stepped, walked)


# Rows in LDS at eight waves by lines (K 2,112, or float rows), at four waves and by half lines, and rows straight from memory (16 of 4,096).
@pytest.mark.parametrize("rows,k,waves,sine_first", [(1, 2112, 8, True), (16, 2112, 8, True), (1, 2112, 4, False), (3, 2120, 8, False),
                                                     (8, 896, 8, False), (2, 1536, 8, False), (16, 4096, 8, True), (16, 4096, 4, False),
                                                     (16, 4104, 8, False)])
def test_rotation_rounds_the_products_it_did(ops, rows, k, waves, sine_first):
    # Both elements of a pair are x (exact).  Sine s, cosine -s: the second result is what the rounding of one product left, its sign says
    # of which; sine and cosine s: the first is x s - round(x s).  x has 8 bits, s 24, so that what is left is a bfloat16.
    heads, kv, d = 2, 1, 64
    x = rand((rows, k), 5)
    w = torch.zeros(((heads + 2 * kv) * d, k), dtype=torch.bfloat16, device="cuda")
    w[:, 0] = 1
    s = torch.rand((1, d // 2), generator=torch.Generator(device="cuda").manual_seed(6), device="cuda") + 0.5
    product = x[:, :1].double() * s.double()
    left = (product - product.float().double()).float()       # x s - round(x s)
    assert float((left != 0).float().mean()) > 0.5
    positions = torch.zeros(rows, dtype=torch.int32, device="cuda")
    ops.fused_waves = waves
    try:
        run = lambda cosine: ops.fused_norm_qkv_rope(x, None, 0.0, w, None, positions, torch.cat([cosine, s], 1), None, None, None, heads, kv, d)
        opposed, alike = (run(c).float().view(rows, heads, 2, d // 2) for c in (-s, s))
    finally:
        ops.fused_waves = 0
    assert torch.equal(alike[:, :, 0], left[:, None].expand(-1, heads, -1))
    assert torch.equal(opposed[:, :, 1], (-left if sine_first else left)[:, None].expand(-1, heads, -1))


# Rows of one, two and four pieces a thread, the product in parts and as it is, results of both types.
@pytest.mark.parametrize("hidden,post_groups,groups", [(896, 2, 2), (1024, 1, 4), (1536, 2, 2), (4096, 8, 2)])
@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_grouped_norm_joins_the_stream_in_one_rounding(ops, hidden, post_groups, groups, parts, dtype):
    from tokenizer_amd.kernels import PendingSum
    gen = torch.Generator(device="cuda").manual_seed(hidden + parts)
    slabs = torch.randn((max(1, parts), 3, hidden), generator=gen, device="cuda")
    delta = PendingSum(ops, slabs, None, dtype) if parts else slabs[0].to(dtype)
    behind = 1 + 0.3 * torch.randn(hidden, generator=gen, device="cuda")

    def stream_after(before, weight, normed=True):
        kept, out = before.clone(), torch.empty((3, hidden), dtype=dtype, device="cuda")
        ops.norm_add_rmsnorm(kept, delta, weight, 1e-5, torch.ones_like(behind) if normed else None, 1e-5, out, post_groups=post_groups, groups=groups)
        return kept
    nothing = torch.zeros((3, hidden), device="cuda")
    factor = stream_after(nothing, torch.ones_like(behind))   # the product over its root mean square, rounded
    rounded = stream_after(nothing, behind)
    left = (factor.double() * behind.double() - rounded.double()).float()      # (exact: 48 bits without their first 24)
    assert float((left != 0).float().mean()) > 0.9
    assert torch.equal(stream_after(-rounded, behind), left) and torch.equal(stream_after(-rounded, behind, False), left)
