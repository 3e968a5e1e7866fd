"""Products of many rows in the ring kernel, tile by tile, against the same products in 64 bits."""
import ctypes

import pytest
import torch

from tokenizer_amd.kernels import KernelError, PendingSum, _ptr, get_ops

pytestmark = pytest.mark.gpu
TILES = [(64, 64), (64, 128), (64, 256), (128, 128), (128, 256), (256, 128), (256, 192), (256, 256)]


@pytest.fixture(scope="module")
def ops():
    return get_ops()


def rand(shape, seed, spread=1.0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=gen, device="cuda") * spread).to(torch.bfloat16)


def strided(rows, k, lda, seed):
    x = torch.full((rows, lda), float("nan"), dtype=torch.bfloat16, device="cuda")      # columns behind K are not read
    x[:, :k] = rand((rows, k), seed)
    return x[:, :k]


# Float sums of K exact products, of which each rounding takes 2^-24 of a partial sum: 2e-6 sqrt(K) of the largest result is some
# eight times what is seen; a result rounded to bfloat16 is within 2^-8 of its own size.
def close(got, want, k, rounded):
    bound = 2e-6 * k ** 0.5 * float(want.abs().max()) + (2.0 ** -8 * want.abs() if rounded else 0.0)
    return bool(((got.double() - want).abs() <= bound).all())


# Rows and columns of one tile, one past it and a remainder; K of one step, of every number of steps past the buffers, of half a step more.
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("k", [64, 96, 192, 320, 352, 448])
def test_plain_products_of_every_tile(ops, tile, k):
    bm, bn = TILES[tile]
    for m, n in ((bm, bn), (bm + 1, bn + 4), (65, 100)):
        x, w = strided(m, k, k + 40, k + m), rand((n, k), k + n, 0.1)
        bias = torch.randn(n, device="cuda")
        want = x.double() @ w.double().t() + bias.double()
        for dtype, code in ((torch.float32, 0), (torch.bfloat16, 1)):
            out = torch.full((m, n + 12), float("nan"), dtype=dtype, device="cuda")
            assert ops.lib.ta_gemm_ring(_ptr(x), _ptr(w), _ptr(bias), _ptr(out), None, m, n, k, k + 40, n + 12, 1, code, tile, ops._stream()) == 0
            assert close(out[:, :n], want, k, dtype == torch.bfloat16) and bool(out[:, n:].isnan().all())


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("k,parts", [(576, 3), (1056, 4), (2080, 7), (544, 5)])     # (the last: a part of half a step)
def test_products_in_parts_of_every_tile(ops, tile, k, parts):
    m, n = TILES[tile][0] + 3, TILES[tile][1] + 8
    x, w, bias = rand((m, k), 1), rand((n, k), 2, 0.1), torch.randn(n, device="cuda")
    want = x.double() @ w.double().t()
    partial = torch.full((parts, m, n), float("nan"), device="cuda")
    assert ops.lib.ta_gemm_ring(_ptr(x), _ptr(w), None, None, _ptr(partial), m, n, k, k, n, parts, 1, tile, ops._stream()) == 0
    assert close(partial.double().sum(0), want, k, False)
    out = torch.empty((m, n), device="cuda")
    assert ops.lib.ta_gemm_ring(_ptr(x), _ptr(w), _ptr(bias), _ptr(out), _ptr(partial), m, n, k, k, n, parts, 0, tile, ops._stream()) == 0
    assert close(out, want + bias.double(), k, False)


# Parts are worth their trip to the norm where a whole K would be a long walk of few tiles, and not where the tiles fill the chip.
def test_how_many_parts_a_product_is_cut_into(ops):
    parts = ops.lib.ta_gemm_ring_parts
    for m, n, k in ((700, 1536, 1536), (850, 1536, 1536), (600, 2048, 1536), (700, 2048, 2048), (700, 1024, 2816), (1024, 768, 3072)):
        assert parts(m, n, k, 1) == 1, (m, n, k)
    for m, n, k in ((64, 1536, 8960), (130, 1536, 1536), (300, 896, 4864), (512, 1536, 8960), (2048, 1536, 8960)):
        assert parts(m, n, k, 1) > 1, (m, n, k)


# Results of few tiles and long K go to the ring kernel, large results to the library; float results, which it does not give, never do.
def test_which_products_of_many_rows_are_whose(ops):
    def ring(m, n, k, dtype=torch.bfloat16, pending=False):
        return ops._to_ring(m, n, k, k, dtype, pending)
    for m, n, k in ((65, 512, 512), (512, 1536, 1536), (2048, 896, 896), (2048, 896, 4864), (400, 4096, 4096), (2048, 3584, 18944), (2048, 1536, 8960)):
        assert ring(m, n, k, pending=True), (m, n, k)
    for m, n, k in ((2048, 1536, 1536), (2048, 2560, 2560), (3000, 4096, 11008), (2600, 3584, 18944), (4096, 896, 896), (4096, 1152, 896)):
        assert not ring(m, n, k, pending=True), (m, n, k)
    for m, n, k in ((512, 1152, 896), (1024, 2048, 1536), (512, 1536, 8960), (2048, 1536, 8960)):
        assert ring(m, n, k), (m, n, k)
    for m, n, k in ((1536, 2048, 1536), (512, 4608, 3584), (300, 4096, 4096), (4096, 896, 896)):
        assert not ring(m, n, k), (m, n, k)
    assert ring(6000, 4096, 4096, torch.float32) and ring(4100, 32768, 1024, torch.float32)
    assert not ring(512, 1536, 80) and not ring(512, 1534, 1536)


def test_which_gated_products_are_whose(ops):
    for m, inner, k in ((33, 4864, 896), (64, 8960, 1536), (65, 4864, 896), (512, 4864, 896), (2048, 8960, 1536), (2048, 18944, 3584), (400, 18944, 3584)):
        assert ops._gated_to_ring(m, inner, k), (m, inner, k)
    for m, inner, k in ((32, 4864, 896), (64, 2432, 896), (64, 8192, 2048), (64, 18944, 3584), (224, 18944, 3584), (300, 11008, 4096), (800, 11008, 4096)):
        assert not ops._gated_to_ring(m, inner, k), (m, inner, k)


# (The two after the tiles: large tiles in front, small ones behind.  None, none, none and one strip of 128 columns is in front here, none and two
# for the wider; the next test has more.)
@pytest.mark.parametrize("tile", range(1, len(TILES) + 2))
@pytest.mark.parametrize("act", [None, "gelu_tanh", "relu", (1.702, 2.0, 1.0)])
def test_gated_products_of_every_tile(ops, tile, act):
    bm, bn = (TILES + [(128, 256), (256, 256)])[tile]
    numbers = act if isinstance(act, tuple) else (0.0, 0.0, 0.0)
    code = 4 if isinstance(act, tuple) else {None: 1, "gelu_tanh": 2, "relu": 3}[act]
    for m, inner, k in ((bm, bn // 2, 64), (bm + 1, bn // 2 + 4, 352), (70, 52, 224), (bm + 70, 300, 192)):
        x, w = strided(m, k, k + 8, m), rand((2 * inner, k), inner, 0.2)
        gate, up = (x.double() @ half.double().t() for half in (w[:inner], w[inner:]))
        if act is None:
            want = gate * torch.sigmoid(gate) * up
        elif act == "gelu_tanh":
            want = torch.nn.functional.gelu(gate, approximate="tanh") * up
        elif act == "relu":
            want = torch.relu(gate) * up
        else:
            g = gate.clamp(max=act[1])
            want = g * torch.sigmoid(act[0] * g) * (up.clamp(-act[1], act[1]) + act[2])
        out = torch.full((m, inner), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert ops.lib.ta_gemm_ring_gated(_ptr(x), _ptr(w), _ptr(out), m, inner, k, k + 8, code, *map(ctypes.c_float, numbers), tile,
                                          ops._stream()) == 0
        # The activation in float: 2^-20 of the product of its factors, beside the rounding of the result.
        slack = 2.0 ** -20 * float(gate.abs().max() * up.abs().max())
        assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 4e-5 * float(want.abs().max()) + slack).all())


# More tiles of rows than go in a group (sixteen), a number that is no multiple of it, over several strips of columns and parts of K: every tile
# of the result is somebody's.  Plain, in parts, gated; the gated product in large tiles and small ones behind with several strips of either.
@pytest.mark.parametrize("tile", range(len(TILES) + 2))
def test_products_of_more_tiles_of_rows_than_a_group_has(ops, tile):
    bm, bn = (TILES + [(128, 256), (256, 256)])[tile]
    m, n, k = 17 * bm + 3, 2 * bn + 100, 96
    x, w = strided(m, k, k + 8, tile), rand((n, k), 3, 0.1)
    if tile < len(TILES):
        out = torch.full((m, n), float("nan"), device="cuda")
        assert ops.lib.ta_gemm_ring(_ptr(x), _ptr(w), None, _ptr(out), None, m, n, k, k + 8, n, 1, 0, tile, ops._stream()) == 0
        assert close(out, x.double() @ w.double().t(), k, False)
        long, wide = rand((m, 288), 5), rand((n, 288), 6, 0.1)
        partial = torch.full((3, m, n), float("nan"), device="cuda")
        assert ops.lib.ta_gemm_ring(_ptr(long), _ptr(wide), None, None, _ptr(partial), m, n, 288, 288, n, 3, 1, tile, ops._stream()) == 0
        assert close(partial.double().sum(0), long.double() @ wide.double().t(), 288, False)
    if tile > 0:
        inner = 1500 if tile >= len(TILES) else n // 8 * 4
        w = rand((2 * inner, k), 4, 0.2)
        gate, up = (x.double() @ half.double().t() for half in (w[:inner], w[inner:]))
        out = torch.full((m, inner), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert ops.lib.ta_gemm_ring_gated(_ptr(x), _ptr(w), _ptr(out), m, inner, k, k + 8, 1, *map(ctypes.c_float, (0.0, 0.0, 0.0)), tile,
                                          ops._stream()) == 0
        want = gate * torch.sigmoid(gate) * up
        slack = 2.0 ** -20 * float(gate.abs().max() * up.abs().max())
        assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 4e-5 * float(want.abs().max()) + slack).all())


# The gated product where the launcher's own choice is whole rounds of large tiles with the columns behind them in small ones.
def test_gated_product_of_two_kinds_of_tiles_by_the_launchers_choice(ops):
    m, inner, k = 2048, 4864, 896
    x, w = rand((m, k), 1), rand((2 * inner, k), 2, 0.05)
    got = ops.linear_silu_gate(x, w)
    for rows in range(0, m, 512):
        gate, up = (x[rows:rows + 512].double() @ half.double().t() for half in (w[:inner], w[inner:]))
        want = gate * torch.sigmoid(gate) * up
        slack = 2.0 ** -20 * float(gate.abs().max() * up.abs().max())
        assert bool(((got[rows:rows + 512].double() - want).abs() <= 2.0 ** -8 * want.abs() + 4e-5 * float(want.abs().max()) + slack).all())


# Heads of one pair of blocks, of two and of three, more columns than a tile and fewer; tokens that are stored nowhere, pages in any order.
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("n_q,n_kv,d,page_size", [(3, 1, 64, 16), (5, 2, 32, 16), (2, 1, 96, 32), (4, 2, 128, 16)])
def test_projections_with_rotation_and_store_of_every_tile(ops, tile, n_q, n_kv, d, page_size):
    m, k, n = TILES[tile][0] + 5, 96 + 64 * (tile % 3), (n_q + 2 * n_kv) * d
    x, w, bias = strided(m, k, k + 8, tile), rand((n, k), d, 0.1), torch.randn(n, device="cuda")
    gen = torch.Generator().manual_seed(d)
    positions = torch.randint(0, 500, (m,), generator=gen).int().cuda()
    table = torch.randn((500, d), device="cuda")
    pages = (m + page_size - 1) // page_size + 1
    slots = torch.randperm(pages * page_size, generator=gen)[:m].int().cuda()
    slots[3] = -1
    for use_bias, turn, store in ((True, True, True), (False, True, True), (True, False, True), (True, True, False)):
        out = x.double() @ w.double().t() + (bias.double() if use_bias else 0.0)
        heads = out.view(m, n_q + 2 * n_kv, d).clone()
        if turn:
            cos, sin = (t[:, None] for t in table.double()[positions.long()].split(d // 2, 1))
            u, v = heads[:, :n_q + n_kv, :d // 2].clone(), heads[:, :n_q + n_kv, d // 2:].clone()
            heads[:, :n_q + n_kv] = torch.cat([u * cos - v * sin, v * cos + u * sin], -1)
        keys = torch.zeros((pages, n_kv, page_size, d), dtype=torch.float64, device="cuda")
        values = torch.zeros((pages, n_kv, d, page_size), dtype=torch.float64, device="cuda")
        if store:
            for t in torch.nonzero(slots >= 0)[:, 0].tolist():
                page, off = divmod(int(slots[t]), page_size)
                keys[page, :, off], values[page, :, :, off] = heads[t, n_q:n_q + n_kv], heads[t, n_q + n_kv:]
        q = torch.full((m, n_q * d), float("nan"), dtype=torch.bfloat16, device="cuda")
        k_pages, v_pages = keys.to(torch.bfloat16) * 0, values.to(torch.bfloat16) * 0
        at = lambda t, given=True: _ptr(t if given else None)
        assert ops.lib.ta_gemm_ring_qkv(_ptr(x), k + 8, _ptr(w), at(bias, use_bias), _ptr(q), _ptr(positions), at(table, turn), at(slots, store),
                                        _ptr(k_pages), _ptr(v_pages), m, k, n_q, n_kv, d, page_size, tile, ops._stream()) == 0
        # Float throughout, one rounding of the result: 2^-8 of itself, and of the float sums what a turn by these angles leaves.
        slack = 8 * 2e-6 * k ** 0.5 * float(out.abs().max())
        for got, want in ((q, heads[:, :n_q].reshape(m, -1)), (k_pages, keys), (v_pages, values)):
            assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + slack).all())


# The same of more tiles of rows than go in a group, over several strips of columns: against the product and the rotation one by one.
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_projections_of_more_tiles_of_rows_than_a_group_has(ops, tile):
    n_q, n_kv, d, page_size, k = 9, 1, 64, 16, 96
    m, n = 17 * TILES[tile][0] + 5, (n_q + 2 * n_kv) * d
    x, w, bias = rand((m, k), tile), rand((n, k), d, 0.1), torch.randn(n, device="cuda")
    positions, slots = torch.arange(m, dtype=torch.int32, device="cuda"), torch.randperm(m, device="cuda").int()
    table, pages = torch.randn((m, d), device="cuda"), -(-m // page_size)
    k_pages, v_pages = (torch.zeros(shape, dtype=torch.bfloat16, device="cuda") for shape in ((pages, n_kv, page_size, d), (pages, n_kv, d, page_size)))
    q = torch.full((m, n_q * d), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert ops.lib.ta_gemm_ring_qkv(_ptr(x), k, _ptr(w), _ptr(bias), _ptr(q), _ptr(positions), _ptr(table), _ptr(slots), _ptr(k_pages),
                                    _ptr(v_pages), m, k, n_q, n_kv, d, page_size, tile, ops._stream()) == 0
    heads = (x.double() @ w.double().t() + bias.double()).view(m, -1, d)
    cos, sin = (t[:, None] for t in table.double().split(d // 2, 1))
    u, v = heads[..., :d // 2], heads[..., d // 2:]
    turned = torch.cat([u * cos - v * sin, v * cos + u * sin], -1)
    page, off = slots.long() // page_size, slots.long() % page_size
    slack = 8 * 2e-6 * k ** 0.5 * float(heads.abs().max())
    for got, want in ((q, turned[:, :n_q].reshape(m, -1)), (k_pages[page, 0, off], turned[:, n_q]), (v_pages[page, 0, :, off], heads[:, n_q + 1])):
        assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + slack).all())


# Through the entry point: a width that the ring kernel does not take comes back from the two kernels before it, keys and values stored alike.
@pytest.mark.parametrize("width", [96, 104])
def test_projection_of_many_rows_whatever_the_width(ops, width):
    m, n_q, n_kv, d = 70, 2, 1, 32
    n = (n_q + 2 * n_kv) * d
    x, w, bias = rand((m, width), 1), rand((n, width), 2, 0.1), torch.randn(n, device="cuda")
    positions, slots = (torch.arange(m, dtype=torch.int32, device="cuda") for _ in range(2))
    table = torch.randn((m, d), device="cuda")
    k_pages, v_pages = (torch.zeros(shape, dtype=torch.bfloat16, device="cuda") for shape in ((5, n_kv, 16, d), (5, n_kv, d, 16)))
    got = ops.fused_norm_qkv_rope(x, None, 0.0, w, bias, positions, table, slots, k_pages, v_pages, n_q, n_kv, d)[:, :n_q * d]
    qkv = ops.linear(x, w, bias)
    keys, values = torch.zeros_like(k_pages), torch.zeros_like(v_pages)
    ops.rope_store(qkv, None, positions, table, slots, keys, values, n_q, n_kv, d)
    for a, b in ((got, qkv[:, :n_q * d]), (k_pages, keys), (v_pages, values)):
        assert float((a.float() - b.float()).abs().max()) <= 3 * 2.0 ** -8 * float(b.float().abs().max())


# What goes to the ring kernel comes back as the general kernels give it: rows and sizes on either side of its lines, an activation of
# each kind, infinities and NaN in a row, which stay in that row.
@pytest.mark.parametrize("m,n,k", [(65, 96, 64), (300, 128, 2080), (1025, 64, 256), (70, 4100, 512), (33, 96, 64), (257, 8, 96)])
def test_the_choice_of_kernel_does_not_change_the_product(ops, m, n, k, monkeypatch):
    x, w, bias = rand((m, k), m), rand((n, k), n, 0.1), torch.randn(n, device="cuda")
    x[1, 3], x[2, 5] = float("inf"), float("nan")
    for act in (None, "gelu_tanh", "relu", (1.702, 2.0, 1.0)):
        got = ops.linear_silu_gate(x, w, act=act)
        with monkeypatch.context() as only:
            only.setattr(ops, "use_ring", False)
            want = ops.linear_silu_gate(x, w, act=act)
        rest = torch.arange(m, device="cuda") > 2
        # (There the sums are rounded to bfloat16 before the activation: 2^-8 of either factor.)
        assert float((got[rest].double() - want[rest].double()).abs().max()) <= 4 * 2.0 ** -8 * float(want[rest].double().abs().max())
        assert torch.equal(got[1:3].isfinite(), want[1:3].isfinite())
    for pending in (False, True):
        for dtype in (torch.bfloat16, torch.float32):
            got = ops.linear(x, w, bias, out_dtype=dtype, pending=pending)
            got = got.resolve() if isinstance(got, PendingSum) else got
            with monkeypatch.context() as only:
                only.setattr(ops, "use_ring", False)
                want = ops.linear(x, w, bias, out_dtype=dtype)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
            fine = want.isfinite()
            limit = 2.0 ** -7 if dtype == torch.bfloat16 else 2e-6 * k ** 0.5
            assert float((got[fine].double() - want[fine].double()).abs().max()) <= limit * float(want[fine].double().abs().max())


# Decode attention of few rows at head size 128: whole where a step may have any context up to 512, in parts where a window's range is known to lie
# past 384 keys.
def test_ranges_of_keys_that_are_whole(ops, monkeypatch):
    seen, kernel = [], ops.lib.ta_decode_attention_bf16
    monkeypatch.setattr(ops.lib, "ta_decode_attention_bf16", lambda *args: (seen.append(args[20]), kernel(*args))[1])
    for d, window, context, whole in ((128, None, 500, True), (128, 300, 2000, True), (128, 400, 2000, False), (96, 400, 2000, True), (64, 400, 2000, True)):
        n_q, n_kv, pages = 4, 2, 128
        q = rand((2, (n_q + 2 * n_kv) * d), d)
        keys, values = rand((pages, n_kv, 16, d), 1), rand((pages, n_kv, d, 16), 2)
        table = torch.arange(128, dtype=torch.int32, device="cuda").expand(2, -1).contiguous()
        positions, out = torch.full((2,), context - 1, dtype=torch.int32, device="cuda"), torch.empty((2, n_q * d), dtype=torch.bfloat16, device="cuda")
        ops._decode_attention(q, out, keys, values, positions, None, table, n_q, n_kv, d, 16, window, d ** -0.5, context - 1, identity_entries=True)
        assert (seen[-1] == 1) == whole, (d, window)


# The capped gate's three numbers may come as any sequence, with few rows and with many.
@pytest.mark.parametrize("m", [9, 40, 300])
def test_numbers_of_the_capped_gate_as_a_list(ops, m):
    x, w = rand((m, 96), m), rand((64, 96), 2, 0.2)
    assert torch.equal(ops.linear_silu_gate(x, w, act=[1.702, 2.0, 1.0]), ops.linear_silu_gate(x, w, act=(1.702, 2.0, 1.0)))


def test_operands_that_are_refused(ops):
    x, w, out = rand((80, 96), 1), rand((64, 96), 2), torch.empty((80, 64), dtype=torch.bfloat16, device="cuda")
    call = lambda m, n, k, lda, ldc, parts=1, partial=None, xp=None: ops.lib.ta_gemm_ring(
        xp or _ptr(x), _ptr(w), None, _ptr(out), partial, m, n, k, lda, ldc, parts, 1, -1, ops._stream())
    assert call(80, 64, 32, 96, 64) == -2                     # less than a step of K
    assert call(80, 64, 80, 96, 64) == -2                     # no whole half step
    assert call(80, 62, 96, 96, 64) == -2                     # columns no multiple of four
    assert call(80, 64, 96, 92, 64) == -2                     # rows not sixteen bytes apart
    assert call(80, 64, 96, 96, 64, xp=ctypes.c_void_p(x.data_ptr() + 2)) == -2
    assert call(80, 64, 96, 96, 64, parts=2) == -1            # parts without a place
    assert call(80, 64, 96, 96, 64, parts=3, partial=_ptr(out)) == -1      # more parts than steps
    assert call(0, 64, 96, 96, 64) == 0


# The first product of a routed layer with its activation, in every tile: against 64 bits, an expert without a pair, one with several tiles,
# slots that only fill a tile up, columns past a tile and no multiple of four, widths with half a step.
@pytest.mark.parametrize("bm,width", [(64, 64), (64, 128), (64, 256), (128, 128), (128, 256)])
@pytest.mark.parametrize("act", ["silu", "weighed", "relu2"])
@pytest.mark.parametrize("inner,k", [(64, 64), (132, 96), (90, 224)])
def test_sorted_products_with_their_activation(ops, bm, width, act, inner, k, monkeypatch):
    experts, top, rows = 5, 2, 2 * bm + 9
    gen = torch.Generator().manual_seed(inner + k)
    first = torch.where(torch.arange(rows) < rows - 4, 2, 4)
    chosen = torch.stack([first, (first + 1 + torch.arange(rows) % 2) % 4], 1).to(torch.int32)
    chosen[3, 1] = -1                                         # a pair that is passed over
    wide = (1 if act == "relu2" else 2) * inner
    x, w = rand((rows, k + 8), k), rand((experts * wide, k + 16), inner, 0.2)
    x[:, k:], w[:, k:] = float("nan"), float("nan")             # columns behind K are not read
    weights = torch.rand((rows, top), generator=gen).cuda() + 0.5
    slot_of, row_of, tile_expert = ops.expert_slots(chosen.cuda(), experts, bm)
    monkeypatch.setattr(ops, "grouped_wide", width)
    out = ops.grouped_act(x, row_of, tile_expert, bm, w, wide * (k + 16), inner, k, act, slot_of, weights)
    slots = slot_of.cpu().view(rows, top)
    for e in range(experts):
        t, p = (chosen == e).nonzero(as_tuple=True)
        if not len(t):
            continue
        z = x[t.cuda(), :k].double() @ w[e * wide:(e + 1) * wide, :k].double().t()
        if act == "relu2":
            want, parts = torch.relu(z) ** 2, float(z.abs().max()) ** 2
        else:
            a = weights[t.cuda(), p.cuda()].double()[:, None] if act == "weighed" else 1.0
            gate, up = a * z[:, :inner], a * z[:, inner:]
            want, parts = gate * torch.sigmoid(gate) * up, float(gate.abs().max() * up.abs().max())
        got = out[slots[t, p].long().cuda()].double()
        # Float sums and activation (2^-19 of the product of its factors), one rounding of the result.
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -19 * parts + 4e-5 * float(want.abs().max())).all()), e


def test_sorted_products_with_activation_leave_other_operands_to_the_two_kernels(ops, monkeypatch):
    x, w = rand((64, 104), 1), rand((128, 104), 2)
    tile_expert, row_of = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.arange(64, dtype=torch.int32, device="cuda")
    assert ops.grouped_act(x, row_of, tile_expert, 64, w, 128 * 104, 64, 104, "silu") is None
    monkeypatch.setattr(ops, "grouped_wide", -1)
    assert ops.grouped_act(x, row_of, tile_expert, 64, w, 128 * 104, 64, 96, "silu") is None


# A product whose parts the grouped norms add themselves: rows of one piece a thread and of several, the last ones partly filled, a number of
# parts that is no multiple of the four asked for at a time, rows picked out, and rows that only the general kernel takes (40 in 4 groups of
# ten, 5,120).  float results: 2^-24 of the sums' size for each of the few dozen roundings; bfloat16 ones 2^-8 of their own size more.
@pytest.mark.parametrize("hidden,post_groups,groups", [(1536, 2, 2), (1024, 1, 4), (1028, 257, 1), (2048, 8, 1), (4096, 2, 1024), (896, 2, 2),
                                                       (40, 4, 4), (5120, 4, 2)])
@pytest.mark.parametrize("parts", [1, 2, 4, 5, 11])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_grouped_norms_add_the_parts_of_a_product(ops, hidden, post_groups, groups, parts, dtype):
    rows = 5
    gen = torch.Generator(device="cuda").manual_seed(hidden + parts)
    draw = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    stream, slabs = draw(rows, hidden), draw(parts, rows, hidden)
    behind, weight = 1 + 0.3 * draw(hidden), 1 + 0.3 * draw(hidden)

    def norm(v, w, count, eps):
        runs = v.reshape(len(v), count, -1)
        return (runs / (runs.square().mean(-1, keepdim=True) + eps).sqrt()).reshape(v.shape) * w.double()
    pending = lambda: PendingSum(ops, slabs, None, dtype)
    # (The general kernel takes the product as it comes without parts: added, and rounded to its own type.)
    general = hidden % (4 * post_groups) or hidden % (4 * groups) or hidden > 4096
    product = pending().resolve().double() if general else slabs.double().sum(0)
    x = stream.double() + norm(product, behind, post_groups, 1e-5)
    y = norm(x, weight, groups, 1e-3)
    near = lambda got, want: bool(((got.double() - want).abs() <= 2e-6 * want.abs().max()
                                   + (2.0 ** -8 * want.abs() if got.dtype == torch.bfloat16 else 0.0)).all())
    args = dict(post_groups=post_groups, groups=groups)
    kept, out = stream.clone(), torch.empty(rows, hidden, dtype=dtype, device="cuda")
    ops.norm_add_rmsnorm(kept, pending(), behind, 1e-5, weight, 1e-3, out, **args)
    assert near(kept, x) and near(out, y)
    again, same = stream.clone(), torch.empty_like(out)
    ops.norm_add_rmsnorm(again, pending(), behind, 1e-5, None, 0.0, same, **args)              # the sum itself
    assert torch.equal(again, kept) and near(same, x)
    pick = torch.tensor([4, 0], dtype=torch.int32, device="cuda")
    again, some = stream.clone(), torch.empty(2, hidden, dtype=dtype, device="cuda")
    ops.norm_add_rmsnorm(again, pending(), behind, 1e-5, weight, 1e-3, some, pick, store_residual=False, **args)
    assert torch.equal(again, stream) and torch.equal(some, out[[4, 0]])
    with pytest.raises(KernelError):                                                          # slabs of other rows
        ops.norm_add_rmsnorm(kept[:3].contiguous(), pending(), behind, 1e-5, weight, 1e-3, out[:3], **args)
