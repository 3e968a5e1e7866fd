"""Norm kernels that add a product's parts themselves, and the token input's kernel with several rows a workgroup, against float64.

Bounds: a bfloat16 result is within half a unit of its last place (2^-9 of itself) of the float32 one, which 2^-8 of the largest
covers; the float32 stream is a sum of at most parts + 3 terms, each within 2^-24 of the largest partial sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _pending(ops, slabs):
    from tokenizer_amd.kernels import PendingSum
    return PendingSum(ops, slabs.cuda(), None, torch.bfloat16)


def test_rounded_sums_are_the_whole_product():
    """A sum of parts that is to be rounded gives bit for bit what the product added up first gives."""
    from tokenizer_amd.kernels import PendingSum, get_ops
    ops, gen, n, hidden, dim = get_ops(), torch.Generator().manual_seed(3), 600, 1536, 16
    residual, slabs = torch.randn(n, hidden, generator=gen).cuda(), torch.randn(5, n, hidden, generator=gen).cuda()
    other, w = torch.randn(n, hidden, generator=gen).to(torch.bfloat16).cuda(), torch.rand(hidden, generator=gen).cuda() + 0.5
    small = [torch.randn(*shape, generator=gen).to(torch.bfloat16).cuda() for shape in ((dim, hidden), (hidden, dim), (9, dim))]
    ids = torch.randint(0, 9, (n,), generator=gen, dtype=torch.int32).cuda()
    got = []
    for whole in (False, True):
        parts = PendingSum(ops, slabs, None, torch.bfloat16)
        parts.rounded = True
        delta, outs = parts.resolve() if whole else parts, []
        for run in (lambda x, out: ops.add_terms_rmsnorm(x, [(other, 1.0, None), (delta, 1.0, None)], w, 1e-5, out),
                    lambda x, out: ops.norm_add_rmsnorm(x, delta, w, 1e-5, w, 1e-5, out),
                    lambda x, out: ops.norm_side_norm(x, delta, w, 1e-5, small[0], small[1], w, 1e-5, small[2], ids, 0, dim, w, 1e-5, out)):
            stream, out = residual.clone(), torch.empty_like(other)
            run(stream, out)
            outs += [stream, out]
        got.append(outs)
    for a, b in zip(*got):
        assert torch.equal(a, b)


def _near(got, want, bound):
    assert torch.isfinite(got).all()
    assert float((got.double().cpu() - want).abs().max()) <= bound * float(want.abs().max())


@pytest.mark.parametrize("hidden", [4, 64, 1024, 1028, 3584, 4096])
@pytest.mark.parametrize("parts", [1, 4, 5, 9])
@pytest.mark.parametrize("scaled,second,normed", [(True, True, True), (False, False, True), (True, False, False)])
def test_two_terms_and_one_in_parts(hidden, parts, scaled, second, normed):
    from tokenizer_amd.kernels import get_ops
    ops, gen, n = get_ops(), torch.Generator().manual_seed(hidden + parts), 7
    residual, slabs = torch.randn(n, hidden, generator=gen), torch.randn(parts, n, hidden, generator=gen)
    rows = [torch.randn(n, hidden, generator=gen).to(torch.bfloat16) for _ in range(2)]
    scales = [1 + 0.4 * torch.randn(hidden, generator=gen) if scaled else None for _ in range(3)]
    w1, w2 = (1 + 0.4 * torch.randn(hidden, generator=gen) for _ in range(2))
    on = lambda s: None if s is None else s.cuda()
    want = residual.double()
    for term, factor, scale in zip(rows + [slabs.double().sum(0)], (0.7, 0.4, 1.0), scales):
        want = want + factor * term.double() * (1.0 if scale is None else scale.double())
    terms = [(rows[0].cuda(), 0.7, on(scales[0])), (rows[1].cuda(), 0.4, on(scales[1])), (_pending(ops, slabs), 1.0, on(scales[2]))]
    assert ops._add_slabs(residual.cuda(), terms, None, 0.0, torch.empty(n, hidden, dtype=torch.bfloat16, device="cuda"), None, False,
                          None, 0.0, None) is not None                       # (this kernel, not the parts added first)
    for picked in (None, [6, 2]):
        stream = residual.cuda()
        pick = None if picked is None else torch.tensor(picked, dtype=torch.int32, device="cuda")
        count, x = (n, want) if picked is None else (2, want[picked])
        wide = torch.full((count, hidden + 8), 3.0, dtype=torch.bfloat16, device="cuda")      # rows that lie apart
        other = torch.empty(count, hidden, dtype=torch.bfloat16, device="cuda") if second else None
        more = dict(weight2=w2.cuda(), eps2=1e-3, out2=other) if second else {}
        ops.add_terms_rmsnorm(stream, terms, w1.cuda() if normed else None, 1e-5, wide[:, :hidden], pick, store_residual=pick is None, **more)
        _near(wide[:, :hidden], _unit(x, 1e-5) * w1.double() if normed else x, 2.0 ** -8)
        assert bool((wide[:, hidden:] == 3.0).all())
        if second:
            _near(other, _unit(x, 1e-3) * w2.double(), 2.0 ** -8)
        _near(stream, want if pick is None else residual.double(), (parts + 3) * 2.0 ** -24 * 4)


@pytest.mark.parametrize("hidden", [4, 300, 1024, 1540, 4096])
@pytest.mark.parametrize("parts", [1, 2, 5, 8])
@pytest.mark.parametrize("post,weighted", [(True, True), (True, False), (False, True)])
def test_norm_behind_a_product_in_parts(hidden, parts, post, weighted):
    from tokenizer_amd.kernels import get_ops
    ops, gen, n = get_ops(), torch.Generator().manual_seed(hidden * parts), 5
    residual, slabs = torch.randn(n, hidden, generator=gen), torch.randn(parts, n, hidden, generator=gen)
    w1, w2 = (1 + 0.4 * torch.randn(hidden, generator=gen) for _ in range(2))
    delta = slabs.double().sum(0)
    want = residual.double() + (_unit(delta, 1e-4) * w1.double() if post else delta)
    for picked, dtype in ((None, torch.bfloat16), ([4, 1], torch.bfloat16), (None, torch.float32)):
        stream = residual.cuda()
        pick = None if picked is None else torch.tensor(picked, dtype=torch.int32, device="cuda")
        x = want if picked is None else want[picked]
        out = torch.empty(x.shape, dtype=dtype, device="cuda")
        ops.norm_add_rmsnorm(stream, _pending(ops, slabs), w1.cuda() if post else None, 1e-4, w2.cuda() if weighted else None, 1e-5, out,
                             pick, store_residual=pick is None)
        # (Sums of squares over a row add `hidden` rounded terms: far below 2^-18 of them for these lengths.)
        _near(out, _unit(x, 1e-5) * w2.double() if weighted else x, 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -18)
        _near(stream, want if pick is None else residual.double(), 2.0 ** -18)


@pytest.mark.parametrize("hidden,dim", [(8, 8), (896, 16), (2048, 8), (2056, 16), (4096, 16), (1536, 24)])
@pytest.mark.parametrize("per_unit", [0, 1, 2, 3, 4, 9])
@pytest.mark.parametrize("parts", [0, 1, 3, 6])
def test_token_input_of_many_rows(hidden, dim, per_unit, parts):
    """One row, and one more than so many for every compute unit (the kernel takes 1, 2, 4 or 8 a workgroup)."""
    from tokenizer_amd.kernels import get_ops
    ops, gen = get_ops(), torch.Generator().manual_seed(hidden + dim + per_unit)
    n = per_unit * ops.compute_units + 1
    bf = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16)
    residual, slabs = torch.randn(n, hidden, generator=gen), torch.randn(max(parts, 1), n, hidden, generator=gen)
    gate, proj, table = bf(dim, hidden) * hidden ** -0.5, bf(hidden, dim), bf(50, 3 * dim)
    gate = gate.to(torch.bfloat16)
    w = [1 + 0.3 * torch.randn(hidden, generator=gen) for _ in range(3)]
    ids = torch.randint(0, 50, (n,), generator=gen, dtype=torch.int32)
    delta = slabs.double().sum(0) if parts else slabs[0].to(torch.bfloat16).double()
    x = residual.double() + _unit(delta, 1e-5) * w[0].double()
    g = torch.nn.functional.gelu(x @ gate.double().T, approximate="tanh") * table.double()[ids.long(), dim:2 * dim]
    want = x + _unit(g @ proj.double().T, 1e-6) * w[1].double()
    for picked in (None, list(range(n - 1, -1, -2))):
        stream = residual.cuda()
        pick = None if picked is None else torch.tensor(picked, dtype=torch.int32, device="cuda")
        y = want if picked is None else want[picked]
        out = torch.empty(y.shape, dtype=torch.bfloat16, device="cuda")
        done = ops.norm_side_norm(stream, _pending(ops, slabs) if parts else slabs[0].to(torch.bfloat16).cuda(), w[0].cuda(), 1e-5,
                                  gate.cuda(), proj.cuda(), w[1].cuda(), 1e-6, table.cuda(), ids.cuda(), dim, dim, w[2].cuda(), 1e-5, out, pick)
        assert done is out
        # (Parts that this kernel does not take, dim 24, are added into bfloat16 first.)
        _near(out, _unit(y, 1e-5) * w[2].double(), 2.0 ** -8 if dim <= 16 or not parts else 2.0 ** -6)
        if dim <= 16 or not parts:
            _near(stream, want if pick is None else residual.double(), 2.0 ** -16)
