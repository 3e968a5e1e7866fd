"""Kernels of steps of few rows alone, at the edges of the sizes they take."""
import pytest
import torch

from plain import dolidra_plain as plain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from tokenizer_amd.kernels import get_ops
    return get_ops()


def rounded(t):
    return t.to(torch.bfloat16).to(torch.float64)


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
