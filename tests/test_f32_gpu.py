"""The 32-bit path's matrix-core kernels alone against plain references, at the edges of their tiles, units and parts."""
import pytest
import torch

from tokenizer_amd.kernels import PendingSum

from kernel_refs import PlainOps
from test_kernels_gpu import linear_tol, rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from tokenizer_amd.kernels import get_ops
    return get_ops()


@pytest.fixture(scope="module")
def ref():
    return PlainOps(torch.float64)


# Few rows: one and sixteen, K of one piece, of one unit and a piece, no multiple of four (the element form); many rows: around a
# tile's 64 and 128, K of a step and a piece, of no multiple of four, N of one column past a tile, K cut over workgroups.
@pytest.mark.parametrize("shape", [(1, 16, 4), (16, 17, 36), (3, 40, 33), (7, 896, 4864), (15, 1152, 896), (2, 50, 260),
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


def test_a_product_of_infinities_keeps_them_to_their_row(ops):
    x, w = rand((4, 100), torch.float32, 64), rand((32, 100), torch.float32, 65)
    x[1, 0] = float("inf")
    got = ops.linear(x, w)
    assert torch.isfinite(got[[0, 2, 3]]).all() and not torch.isfinite(got[1]).any()


@pytest.mark.parametrize("shape", [(1, 8, 4), (4, 4864, 896), (16, 100, 260), (9, 33, 64), (5, 24, 30)])
def test_gated_product_of_few_rows(ops, shape):
    m, inner, k = shape
    x, w = rand((m, k), torch.float32, 66), rand((2 * inner, k), torch.float32, 67, 0.1)
    got = ops.linear_silu_gate(x, w)
    both = x.double() @ w.double().t()
    want = torch.nn.functional.silu(both[:, :inner]) * both[:, inner:]
    # Each factor errs as a sum of K products does; the other is at most its largest value.
    bound = linear_tol(torch.float32, x, w)["atol"] * 2.2 * float(both.abs().max())
    torch.testing.assert_close(got.double(), want, rtol=2e-5, atol=bound)

