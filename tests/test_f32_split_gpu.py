"""32-bit products of many rows, whose operands are split into three bfloat16 numbers, against 64 bits and against the float instructions."""
import pytest
import torch

from tokenizer_amd.kernels import PendingSum, get_ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    return get_ops()


def rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def both_ways(ops, x, w, bias=None, pending=False):
    """The product from aligned rows (split) and, the same numbers in rows no sixteen bytes apart, from the float instructions."""
    whole = lambda y: y.resolve() if isinstance(y, PendingSum) else y
    apart = torch.zeros((x.shape[0], x.shape[1] + 1), device="cuda")
    apart[:, :x.shape[1]] = x
    return whole(ops.linear(x, w, bias, pending=pending)), whole(ops.linear(apart[:, :x.shape[1]], w, bias))


# One row past the few-rows kernel, tile edges of 64 and 128 and past them; K shorter than a step, no whole step, of every number of steps
# on their way; columns that leave the last tile almost empty, and no multiple of four; parts of K.
@pytest.mark.parametrize("m", [17, 64, 65, 129, 300])
@pytest.mark.parametrize("n,k", [(64, 4), (65, 36), (130, 96), (96, 132), (1152, 896), (66, 160), (256, 4864)])
def test_split_products_are_no_further_from_64_bits(ops, m, n, k):
    x, w, bias = rand((m, k), m + k) * torch.exp(2 * rand((m, 1), k)), rand((n, k), n) * 0.1, rand((n,), 3)
    want = x.double() @ w.double().t() + bias.double()
    for pending in (False, True):
        split, plain = both_ways(ops, x, w, bias, pending)
        error = lambda y: float((y.double() - want).norm() / want.norm())
        # Float sums either way; a tenth for short K, whose few roundings differ by chance.
        assert error(split) <= max(1.1 * error(plain), 1.5e-7), (error(split), error(plain))


# Infinities, no numbers, numbers past the largest bfloat16 and small ones, in either operand: the same places are no finite numbers, and
# the rest is as far from 64 bits as ever.
@pytest.mark.parametrize("odd", [float("inf"), float("-inf"), float("nan"), 3.4e38, 1e-36])
@pytest.mark.parametrize("m,k", [(70, 200), (260, 1024)])
def test_split_products_of_numbers_that_cannot_be_split(ops, odd, m, k):
    n = 140
    x, w = rand((m, k), 1), rand((n, k), 2) * 0.1
    x[3, 5] = odd
    w[17, 9], w[17, 5], w[18, 5] = odd, 0.0, 1.0
    split, plain = both_ways(ops, x, w)
    assert torch.equal(split.isnan(), plain.isnan()) and torch.equal(split.isinf(), plain.isinf())
    assert torch.equal(split[split.isinf()], plain[plain.isinf()])
    fine = plain.isfinite()
    want = x.double() @ w.double().t()
    size = (x.double().abs() @ w.double().abs().t())[fine]
    assert bool(((split.double() - want)[fine].abs() <= 2.0 ** -22 * size).all())


# Whole rows of small numbers, of either operand, down to those that are no normal floats any more: against 64 bits relative to the row's
# own sums, whose terms the other operand lifts back to ordinary sizes.  Float sums of K products: 2^-22 of the sum of their sizes is
# some sixteen times a rounding; operands of which a bit was lost would miss it from 1e-35 on.
@pytest.mark.parametrize("size", [1e-30, 1e-34, 1e-36, 1e-38, 1e-41])
@pytest.mark.parametrize("m,n,k", [(70, 96, 200), (260, 140, 1024)])
def test_split_products_of_small_numbers(ops, size, m, n, k):
    x, w = rand((m, k), m), rand((n, k), n)
    x[::2] *= size
    w[1::2] *= size
    x[::3] *= 1e16
    w[::3] *= 1e16
    split, _ = both_ways(ops, x, w)
    want, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # (Below the smallest normal float there are only multiples of 2^-149: up to eight parts of K, each within half of one.)
    assert bool(((split.double() - want).abs() <= 2.0 ** -22 * terms + 2.0 ** -146).all())


def test_split_products_repeat_bit_for_bit(ops):
    x, w = rand((300, 896), 5), rand((1152, 896), 6)
    first = ops.linear(x, w)
    for _ in range(5):
        assert torch.equal(ops.linear(x, w), first)


@pytest.mark.parametrize("m,n,k", [(70, 96, 200), (260, 1152, 896)])
def test_split_products_of_a_row_do_not_hang_on_other_rows(ops, m, n, k):
    x, w = rand((m, k), 7), rand((n, k), 8)
    alone = ops.linear(x, w)
    x[m - 1], x[20, 3] = float("nan"), float("inf")
    beside = ops.linear(x, w)
    rest = [t for t in range(m) if t not in (20, m - 1)]
    assert torch.equal(beside[rest], alone[rest]) and not beside[m - 1].isfinite().any() and not beside[20].isfinite().any()
