"""The 32-bit path's matrix-core kernels alone against plain references, at the edges of their tiles, units and parts."""
import math

import pytest
import torch

from tokenizer_amd.kernels import KernelError, PendingSum

from kernel_refs import PlainOps
from test_kernels_gpu import linear_tol, make_batch, make_paged_case, rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from tokenizer_amd.kernels import get_ops
    return get_ops()


@pytest.fixture(scope="module")
def ref():
    return PlainOps(torch.float64)


# Few rows: one and sixteen, K of one piece, of one unit and a piece, no multiple of four (the element form); vector multiply-adds
# of one, two, four and eight rows of long K, columns that are no multiple of a wave's four; many rows: around a
# tile's 64 and 128, K of a step and a piece, of no multiple of four, N of one column past a tile, K cut over workgroups.
@pytest.mark.parametrize("shape", [(1, 16, 4), (16, 17, 36), (3, 40, 33), (7, 896, 4864), (15, 1152, 896), (2, 50, 260),
                                   (1, 899, 896), (2, 2049, 4100), (4, 50, 4096), (3, 2052, 4104), (6, 38, 16384), (8, 21, 16388),
                                   (17, 64, 32), (64, 65, 36), (65, 63, 30), (129, 257, 100), (128, 128, 4864), (300, 896, 4864),
                                   (1280, 132, 896), (513, 1000, 64)])
def test_products(ops, ref, shape):
    m, n, k = shape
    x, w, bias = rand((m, k), torch.float32, 60), rand((n, k), torch.float32, 61, 0.1), rand((n,), torch.float32, 62)
    for b in (bias, None):
        want = ref.linear(x, w, b, out_dtype=torch.float64)
        torch.testing.assert_close(ops.linear(x, w, b).double(), want, **linear_tol(torch.float32, x, w))
        left = ops.linear(x, w, b, pending=True)               # parts for the next norm, or the product itself
        left = left.resolve() if isinstance(left, PendingSum) else left
        torch.testing.assert_close(left.double(), want, **linear_tol(torch.float32, x, w))
    assert torch.equal(ops.linear(x, w, bias), ops.linear(x, w, bias))
    wide = rand((m, k + 5), torch.float32, 63)                 # rows that do not lie on sixteen bytes
    torch.testing.assert_close(ops.linear(wide[:, 1:k + 1], w).double(), ref.linear(wide[:, 1:k + 1], w, out_dtype=torch.float64),
                               **linear_tol(torch.float32, wide, w))
    # What lies behind the rows and behind K must not reach a sum.
    framed = torch.full((m + 1, k + 4), float("inf"), device="cuda")
    framed[:m, :k] = x
    torch.testing.assert_close(ops.linear(framed[:m, :k], w).double(), ref.linear(x, w, out_dtype=torch.float64),
                               **linear_tol(torch.float32, x, w))


# Few rows staged by their waves (three and four in one load, five and eight in two, nine not at all) and workgroups of four, seven and sixteen
# weight rows with a last one that is not full; one unit, units for some of the waves, for two pairs of each, and many; the gate with
# rows in LDS and without; rows of a longer stride with no numbers between them.
@pytest.mark.parametrize("rows", [3, 4, 5, 8, 9])
@pytest.mark.parametrize("n,k", [(20, 32), (100, 608), (900, 896), (1540, 1536), (2500, 4896)])
def test_few_rows_spread_over_the_device(ops, ref, rows, n, k):
    x = torch.full((rows, k + 4), float("nan"), device="cuda")
    x[:, :k] = rand((rows, k), torch.float32, 71)
    x, w, bias = x[:, :k], rand((n, k), torch.float32, 72, 0.1), rand((n,), torch.float32, 73)
    want = ref.linear(x, w, bias, out_dtype=torch.float64)
    torch.testing.assert_close(ops.linear(x, w, bias).double(), want, **linear_tol(torch.float32, x, w))
    left = ops.linear(x, w, bias, pending=True)
    left = left.resolve() if isinstance(left, PendingSum) else left
    torch.testing.assert_close(left.double(), want, **linear_tol(torch.float32, x, w))
    got, gate = ops.linear_silu_gate(x, w), want - bias.double()
    exact = gate[:, :n // 2] / (1 + torch.exp(-gate[:, :n // 2])) * gate[:, n // 2:]
    # (each factor is off by a product's bound, the other one is at most the largest sum)
    bound = linear_tol(torch.float32, x, w)["atol"] * (2 + 2 * float(gate.abs().max()))
    assert float((got.double() - exact).abs().max()) <= bound


def test_a_product_of_infinities_keeps_them_to_their_row(ops):
    x, w = rand((4, 100), torch.float32, 64), rand((32, 100), torch.float32, 65)
    x[1, 0] = float("inf")
    got = ops.linear(x, w)
    assert torch.isfinite(got[[0, 2, 3]]).all() and not torch.isfinite(got[1]).any()


@pytest.mark.parametrize("rows", [1, 3, 16, 17, 70])
def test_a_product_over_nothing_is_its_bias(ops, rows):
    x, w, bias = rand((rows, 0), torch.float32, 71), rand((20, 0), torch.float32, 72), rand((20,), torch.float32, 73)
    for pending in (False, True):
        assert torch.equal(ops.linear(x, w, bias, pending=pending), bias.expand(rows, 20))
        assert torch.equal(ops.linear(x, w, pending=pending), torch.zeros(rows, 20, device="cuda"))


@pytest.mark.parametrize("shape", [(1, 8, 4), (4, 4864, 896), (16, 100, 260), (9, 33, 64), (5, 24, 30), (1, 4863, 896), (2, 33, 260),
                                   (4, 19, 4096), (7, 22, 16384)])
def test_gated_product_of_few_rows(ops, shape):
    m, inner, k = shape
    x, w = rand((m, k), torch.float32, 66), rand((2 * inner, k), torch.float32, 67, 0.1)
    got = ops.linear_silu_gate(x, w)
    both = x.double() @ w.double().t()
    want = torch.nn.functional.silu(both[:, :inner]) * both[:, inner:]
    # Each factor errs as a sum of K products does; the other is at most its largest value.
    bound = linear_tol(torch.float32, x, w)["atol"] * 2.2 * float(both.abs().max())
    torch.testing.assert_close(got.double(), want, rtol=2e-5, atol=bound)


@pytest.mark.parametrize("rows", [1, 16, 17])
def test_gated_product_over_nothing_is_zero(ops, rows):
    x, w = rand((rows, 0), torch.float32, 74), rand((24, 0), torch.float32, 75)
    assert torch.equal(ops.linear_silu_gate(x, w), torch.zeros(rows, 12, device="cuda"))


@pytest.mark.parametrize("rows", [4, 20])
def test_gated_product_refuses_a_result_on_the_host(ops, rows):
    x, w = rand((rows, 64), torch.float32, 76), rand((24, 64), torch.float32, 77)
    with pytest.raises(KernelError):
        ops.linear_silu_gate(x, w, out=torch.empty(rows, 12))


FORMS = [dict(), dict(window=37), dict(chunk=50), dict(slopes=True, sinks=True), dict(softcap=3.0, sinks=True),
         dict(window=29, keep_first=21), dict(value_heads=1), dict(value_dim=40)]


@pytest.mark.parametrize("geometry", [(6, 2, 64, 16), (20, 1, 16, 16), (4, 2, 100, 48), (2, 2, 256, 32), (4, 2, 32, 16),
                                      (6, 2, 96, 32), (4, 4, 192, 16), (5, 1, 96, 16), (17, 1, 128, 16)])
@pytest.mark.parametrize("form", FORMS, ids=str)
def test_attention(ops, ref, geometry, form, monkeypatch):
    """Portions that start and end inside pages, tiles and blocks of keys, single tokens whose keys are cut over workgroups (also
    into more parts than there are blocks), against the reference and, form by form, the generic kernel."""
    n_q, n_kv, d, page_size = geometry
    form = dict(form)
    lengths, q_lens = [1, 300, 64, 17, 200, 33], [1, 5, 64, 1, 100, 2]
    dv, n_v = form.get("value_dim", d), form.get("value_heads", n_kv)
    qkv, k_pages, v_pages, positions, entry_of_token, table = make_paged_case(
        torch.float32, n_q, n_kv, d, page_size, lengths=lengths, q_lens=q_lens, seed=31)
    if dv != d or n_v != n_kv:
        written = torch.isfinite(v_pages[:, :1, :1]).expand(-1, n_v, dv, -1)
        v_pages = torch.where(written, rand((v_pages.shape[0], n_v, dv, page_size), torch.float32, 68), float("nan"))
    for name, seed in (("slopes", 69), ("sinks", 70)):
        if form.get(name):
            form[name] = rand((n_q,), torch.float32, seed, 0.1 if name == "slopes" else 2.0)
    window = form.pop("window", None)
    scale = 1.0 / math.sqrt(d)

    def run(which, batch=None):
        on = (lambda v: v.cpu() if isinstance(v, torch.Tensor) else v) if which is ref else (lambda v: v)
        out = on(torch.full((qkv.shape[0], n_q * dv), float("nan"), device="cuda"))
        which.paged_attention(*map(on, (qkv, out, k_pages, v_pages, positions, entry_of_token, table)), n_q, n_kv, d, window, scale,
                              max_position=max(lengths) - 1, **({"batch": batch} if batch else {}),
                              **{name: on(value) for name, value in form.items()})
        return out.cuda()

    want = run(ref)
    # (Scores of about 1 from sums of d products, weighted sums of at most 300 values of about 1.)
    close = dict(rtol=2e-5, atol=4e-6)
    batch = make_batch(lengths, q_lens)
    tiled, ran = ops._attention_f32, []
    monkeypatch.setattr(ops, "_attention_f32", lambda *args: ran.append(tiled(*args)) or ran[-1])
    torch.testing.assert_close(run(ops, batch), want, **close)
    torch.testing.assert_close(run(ops), want, **close)
    assert ran == [True, True]                                # (not the generic kernel in its place)
    monkeypatch.setattr(ops, "min_split_keys_f32", 16)
    torch.testing.assert_close(run(ops), want, **close)
    monkeypatch.setattr(ops, "target_workgroups", 1)
    torch.testing.assert_close(run(ops), want, **close)
    monkeypatch.setattr(ops, "use_fast_attention", False)
    torch.testing.assert_close(run(ops), want, **close)


@pytest.mark.parametrize("geometry", [(6, 2, 64, 16), (20, 1, 16, 16), (2, 2, 256, 32)])
@pytest.mark.parametrize("form", [dict(), dict(window=29), dict(chunk=50), dict(window=29, keep_first=21)], ids=str)
def test_attention_keeps_an_infinite_value_to_the_queries_that_see_its_key(ops, ref, geometry, form):
    """Values that are infinite or no number at keys that some queries of a tile see and others do not (later tokens of the
    tile, keys that have just left the window or lie in front of the run), and at ones just outside a single token's reach."""
    n_q, n_kv, d, page_size = geometry
    lengths, q_lens = [300, 64, 90], [100, 1, 21]
    qkv, k_pages, v_pages, positions, entry_of_token, table = make_paged_case(
        torch.float32, n_q, n_kv, d, page_size, lengths=lengths, q_lens=q_lens, seed=32)
    infinity, nothing = float("inf"), float("nan")
    for entry, key, coordinate, value in ((0, 205, 3, infinity), (0, 250, 4, nothing), (0, 268, 5, -infinity), (0, 180, 6, infinity),
                                          (0, 5, 7, infinity), (1, 25, 2, nothing), (1, 33, 1, infinity), (1, 49, 5, -infinity),
                                          (2, 40, 9, infinity), (2, 89, 10, nothing)):
        v_pages[int(table[entry, key // page_size]), n_kv - 1, coordinate, key % page_size] = value

    def run(which, batch=None):
        on = (lambda t: t.cpu()) if which is ref else (lambda t: t)
        out = on(torch.full((qkv.shape[0], n_q * d), 7.0, device="cuda"))
        which.paged_attention(*map(on, (qkv, out, k_pages, v_pages, positions, entry_of_token, table)), n_q, n_kv, d,
                              form.get("window"), 1.0 / math.sqrt(d), max_position=max(lengths) - 1,
                              **({"batch": batch} if batch else {}), **{name: v for name, v in form.items() if name != "window"})
        return out.cuda()

    want = run(ref)
    clean = torch.isfinite(want)
    assert 0 < int((~clean).sum()) < want.numel() // 2
    for got in (run(ops, make_batch(lengths, q_lens)), run(ops)):
        assert torch.equal(torch.isfinite(got), clean)
        torch.testing.assert_close(got, want, rtol=2e-5, atol=4e-6, equal_nan=True)


@pytest.mark.parametrize("head_dim,page_size,tied", [(64, 16, True), (260, 16, False), (30, 16, False), (64, 24, False)])
def test_attention_of_other_forms_stays_with_the_generic_kernel(ops, ref, head_dim, page_size, tied, monkeypatch):
    n_q, n_kv, lengths, q_lens = 4, 2, [40, 1, 70], [9, 1, 1]
    qkv, k_pages, v_pages, positions, entry_of_token, table = make_paged_case(
        torch.float32, n_q, n_kv, head_dim, page_size, lengths=lengths, q_lens=q_lens, seed=34)
    tiled, ran = ops._attention_f32, []
    monkeypatch.setattr(ops, "_attention_f32", lambda *args: ran.append(tiled(*args)) or ran[-1])

    def run(which):
        on = (lambda t: t.cpu()) if which is ref else (lambda t: t)
        out = on(torch.full((qkv.shape[0], n_q * head_dim), float("nan"), device="cuda"))
        which.paged_attention(on(qkv), out, on(k_pages), None if tied else on(v_pages), on(positions), on(entry_of_token), on(table),
                              n_q, n_kv, head_dim, None, 1.0 / math.sqrt(head_dim), max_position=max(lengths) - 1,
                              **({"tied_values": True} if tied else {}))
        return out.cuda()

    torch.testing.assert_close(run(ops), run(ref), rtol=2e-5, atol=4e-6)
    assert ran == [False]


def test_attention_passes_over_a_description_of_other_tokens(ops, ref):
    n_q, n_kv, d, page_size, lengths, q_lens = 6, 2, 64, 16, [1, 300, 64], [1, 100, 2]
    qkv, k_pages, v_pages, positions, entry_of_token, table = make_paged_case(
        torch.float32, n_q, n_kv, d, page_size, lengths=lengths, q_lens=q_lens, seed=33)

    def run(which, batch=None):
        on = (lambda t: t.cpu()) if which is ref else (lambda t: t)
        out = on(torch.full((qkv.shape[0], n_q * d), float("nan"), device="cuda"))
        which.paged_attention(*map(on, (qkv, out, k_pages, v_pages, positions, entry_of_token, table)), n_q, n_kv, d, None,
                              1.0 / math.sqrt(d), max_position=max(lengths) - 1, **({"batch": batch} if batch else {}))
        return out.cuda()

    want = run(ref)
    for batch in (make_batch(lengths, [1, 101, 2]), make_batch(lengths + [30], [1, 98, 2, 2])):    # other tokens, other entries
        torch.testing.assert_close(run(ops, batch), want, rtol=2e-5, atol=4e-6)


# The merge of a single token's parts: 8, 16, 24, 48, 64 and (another walk) 80 of them, head sizes of a part of 64 coordinates, of a few and of four
# times 64; rows whose contexts end in an early part; an infinite value among the last part's, which its coordinate alone has.
@pytest.mark.parametrize("keys", [500, 900, 1500, 3000, 4000, 5000])
@pytest.mark.parametrize("d", [32, 64, 100, 128, 192, 256])
def test_merge_of_many_parts(ops, keys, d):
    rows, heads, kv, page = 3, 4, 2, 16
    gen = torch.Generator(device="cuda").manual_seed(keys + d)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    pages = -(-keys // page)
    k, v = rand(rows * pages, kv, page, d), rand(rows * pages, kv, d, page)
    last = [keys - 1, keys // 2, 70]
    v[last[0] // page, 1, 5, last[0] % page] = float("inf")
    q = rand(rows, (heads + 2 * kv) * d)
    ints = lambda t: torch.tensor(t, dtype=torch.int32, device="cuda")
    out = torch.empty((rows, heads * d), device="cuda")
    ops.paged_attention(q, out, k, v, ints(last), ints([0, 1, 2]), ints(range(rows * pages)).view(rows, pages), heads, kv, d, None, d ** -0.5,
                        max_position=keys - 1)
    for r in range(rows):
        n, mine = last[r] + 1, slice(r * pages, (r + 1) * pages)
        keys_of = k[mine].transpose(1, 2).reshape(-1, kv, d)[:n].double().repeat_interleave(heads // kv, 1)
        values = v[mine].permute(0, 3, 1, 2).reshape(-1, kv, d)[:n].double().repeat_interleave(heads // kv, 1)
        query = q[r, :heads * d].view(heads, d).double() * d ** -0.5
        weights = torch.softmax((keys_of * query).sum(-1), 0)[..., None]
        want = (weights * values).sum(0)
        # A weight is off by what its score is (d products, each sum rounded) and a few roundings more; sums of a wave's keys, of four waves and of the parts.
        slack = (2 * (d + 8) * (keys_of * query).abs().sum(-1).max() + n / 4 + 100) * 2.0 ** -24 * (weights * values.abs()).sum(0)
        got = out[r].view(heads, d).double()
        assert bool((((got - want).abs() <= slack) | (got == want)).all())
    assert int(torch.isinf(out).sum()) == heads // kv and not torch.isnan(out).any()
