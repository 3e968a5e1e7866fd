"""The delta rule of long portions, which walk in blocks of eight tokens, against the rule token by token in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def token_by_token(fresh, z, rate, beta, state, portions, heads, groups, d, dv, eps):
    """(out [T, heads dv], the states behind) for portions of (first row, rows, starts from zeros)."""
    out, states = torch.zeros(fresh.shape[0], heads, dv, dtype=torch.float64), []
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + eps)
    for e, (lo, n, fresh_start) in enumerate(portions):
        S = torch.zeros(heads, d, dv, dtype=torch.float64) if fresh_start else state[e].clone()
        for t in range(lo, lo + n):
            q = unit(fresh[t, :groups * d].reshape(groups, d)).repeat_interleave(heads // groups, 0) / d ** 0.5
            k = unit(fresh[t, groups * d:2 * groups * d].reshape(groups, d)).repeat_interleave(heads // groups, 0)
            v = fresh[t, 2 * groups * d:].reshape(heads, dv)
            g = torch.exp(rate[:, None] * torch.nn.functional.softplus(z[t].reshape(heads, d)))
            S = g[:, :, None] * S
            u = torch.sigmoid(beta[t])[:, None] * (v - (S * k[:, :, None]).sum(1))
            S = S + k[:, :, None] * u[:, None, :]
            out[t] = (S * q[:, :, None]).sum(1)
        states.append(S)
    return out.reshape(fresh.shape[0], heads * dv), states


# Portions of whole blocks, of one token more or less, of less than a block, of none; from zeros and from a state; rows behind the last
# portion that only fill the batch up; key channels that fill a lane's rows and not, one to sixteen of them; decays from nearly one to
# ones whose products are no numbers a float can hold.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,groups,d,dv", [(2, 1, 16, 16), (3, 3, 20, 24), (4, 2, 64, 40), (2, 2, 128, 16), (2, 1, 200, 8)])
@pytest.mark.parametrize("strong", [False, True])
def test_blocks_of_eight_tokens(dtype, heads, groups, d, dv, strong):
    from tokenizer_amd.kernels import get_ops
    ops, gen = get_ops(), torch.Generator().manual_seed(d + heads)
    rand = lambda *shape: torch.randn(*shape, generator=gen, dtype=torch.float64)
    lengths, from_zero, eps = [37, 0, 16, 3, 33, 1, 20], [True, True, False, False, True, True, False], 1e-6
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    T = cu[-1] + 5
    fresh = rand(T, 2 * groups * d + heads * dv).to(dtype)
    rows = rand(T, heads + 3).to(dtype)
    z = (rand(T, heads * d) * (20.0 if strong else 1.5)).float()
    rate = -(torch.rand(heads, generator=gen, dtype=torch.float64) * (30.0 if strong else 0.2) + 0.01).float()
    state = rand(len(lengths) + 2, heads * d * dv + 7).float() * 0.3
    slots = torch.randperm(len(lengths) + 2, generator=gen)[:len(lengths)]
    want, behind = token_by_token(fresh.double(), z.double(), rate.double(), rows[:, 2:2 + heads].double(),
                                  [state[s, :heads * d * dv].double().reshape(heads, d, dv) for s in slots.tolist()],
                                  list(zip(cu, lengths, from_zero)), heads, groups, d, dv, eps)
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    results = []
    for rows_from in (0, 1 << 30):                            # in blocks; token by token
        held, out = state.cuda(), torch.zeros(T, heads * dv, device="cuda")
        kept, ops.DELTA_BLOCK_ROWS = ops.DELTA_BLOCK_ROWS, (rows_from, rows_from)
        try:
            ops.delta_scan(fresh.cuda(), z.cuda(), rate.cuda(), rows.cuda(), 2, held, ints(cu), ints([0 if f else 9 for f in from_zero]),
                           ints(slots.tolist()), out, heads, groups, d, dv, eps)
        finally:
            ops.DELTA_BLOCK_ROWS = kept
        results.append((out.cpu().double(), held.cpu().double()))
    for out, held in results:                                 # float sums of up to 200 terms over 37 dependent steps
        assert float((out[:cu[-1]] - want[:cu[-1]]).abs().max()) <= 2e-5 * float(want.abs().max())
        for e, s in enumerate(slots.tolist()):
            if lengths[e]:
                got = held[s, :heads * d * dv].reshape(heads, d, dv)
                assert float((got - behind[e]).abs().max()) <= 2e-5 * max(1.0, float(behind[e].abs().max()))
            else:
                assert torch.equal(held[s], state[s].double())
            assert torch.equal(held[s, heads * d * dv:], state[s, heads * d * dv:].double())
    # (Numbers that are not finite reach the tokens behind their own and no others, as they do token by token.)
    bad = fresh.clone()
    bad[cu[4] + 13, 2 * groups * d] = float("nan")
    bad[cu[4] + 14, 2 * groups * d + 1] = float("inf")
    held, out = state.cuda(), torch.zeros(T, heads * dv, device="cuda")
    ops.DELTA_BLOCK_ROWS = (0, 0)
    try:
        ops.delta_scan(bad.cuda(), z.cuda(), rate.cuda(), rows.cuda(), 2, held, ints(cu), ints([0 if f else 9 for f in from_zero]),
                       ints(slots.tolist()), out, heads, groups, d, dv, eps)
    finally:
        ops.DELTA_BLOCK_ROWS = kept
    hit = (out.cpu().double() - want).isfinite()
    assert hit[:cu[4] + 13].all() and hit[cu[5]:cu[-1]].all() and not hit[cu[4] + 13:cu[5], 0].any() and hit[cu[4]:cu[5], 2:].all()
    assert hit[cu[4] + 13, 1] and not hit[cu[4] + 14:cu[5], 1].any()
    error = lambda out: float((out[:cu[-1]] - want[:cu[-1]]).norm())
    assert error(results[0][0]) <= 2 * error(results[1][0])    # no less exact than the walk token by token (a factor for chance)


def random_step(lengths, heads, groups, d, seed):
    """A step's operands on the device, bfloat16, and a run of them that gives (out, state)."""
    from tokenizer_amd.kernels import get_ops
    ops, gen = get_ops(), torch.Generator().manual_seed(seed)
    rand = lambda *shape: torch.randn(*shape, generator=gen)
    T, cu = sum(lengths), [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    fresh, rows = rand(T, (2 * groups + heads) * d).bfloat16().cuda(), rand(T, heads).bfloat16().cuda()
    z, rate, state = rand(T, heads * d).cuda(), -torch.rand(heads, generator=gen).cuda(), rand(len(lengths), heads * d * d).cuda() * 0.3
    first, slots = ints([9 * (i % 2) for i in range(len(lengths))]), ints(list(range(len(lengths))))

    def run(blocks=None, prepared=None, **more):
        held, out = state.clone(), torch.zeros(T, heads * d, device="cuda")
        kept = ops.DELTA_BLOCK_ROWS, ops.DELTA_PREPARED
        ops.DELTA_BLOCK_ROWS = kept[0] if blocks is None else (0, 0) if blocks else (1 << 30, 1 << 30)
        ops.DELTA_PREPARED = kept[1] if prepared is None else prepared
        try:
            ops.delta_scan(fresh, z, rate, rows, 0, held, ints(cu), first, slots, out, heads, groups, d, d, 1e-6, **more)
        finally:
            ops.DELTA_BLOCK_ROWS, ops.DELTA_PREPARED = kept
        return out, held
    return run


def test_a_long_portion_beside_single_tokens_walks_in_blocks():
    from tokenizer_amd.parts.delta import portion_rows
    lengths = [300] + [1] * 15
    run = random_step(lengths, 4, 2, 64, 1)
    same = lambda a, b: all(torch.equal(x, y) for x, y in zip(a, b))
    scan, blocks = run(blocks=False), run(blocks=True)
    assert not same(scan, blocks)
    assert same(run(portion_rows=portion_rows(sum(lengths), len(lengths), 15)), blocks)
    assert same(run(), scan)                                  # (who calls without: the average over all entries)


# Slices of one block a portion, of three (which end inside and at the end of a portion), and portions of less than one.
@pytest.mark.parametrize("d", [16, 64, 200])
@pytest.mark.parametrize("each", [1, 3])
def test_blocks_slice_by_slice_are_the_same(d, each):
    lengths = [53, 0, 24, 1, 8, 17]
    run = random_step(lengths, 2, 1, d, d)
    size = next(s for s in (16, 64, 256) if d <= s)
    want, got = run(blocks=True), run(blocks=True, prepared=each * len(lengths) * 2 * (25 * size + 128))
    assert all(torch.equal(x, y) for x, y in zip(got, want))
