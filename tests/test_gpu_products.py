"""The products' kernels at the edges of their dispatch rules: every kernel that serves a shape gives
what float64 gives, and where the order of the sums is fixed, the same bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# N and K: one part and several, a last part that is short, K no multiple of a stage of 32 (528), of a
# block of 16 (1000: the kernel of any length), more parts than the norm kernel adds is out of reach here
@pytest.mark.parametrize("N,K", [(70, 528), (896, 4864), (130, 1000), (64, 48), (1000, 896)])
def test_float32_rows_have_the_same_bits_in_every_kernel(N, K):
    """Up to 16 rows, 17 to 32, tiles of 64, tiles of 32, planes of partial sums: a row alone and among
    others, and the planes added in order."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(300, K, device=DEV, generator=gen)
    w = torch.randn(N, K, device=DEV, generator=gen)
    b = torch.randn(N, device=DEV, generator=gen)
    want = x.double() @ w.double().t()
    whole = ops.linear(x, w, b)
    # a sum of 16 rounds at 4 units at most and the sums of 16 are added one by one: sqrt(16) + sqrt(K / 16) roundings
    # of values of about sqrt(K), in 2^-24; ten times their spread over all elements
    bound = 10 * (4 + math.sqrt(K / 16)) * math.sqrt(K) * 2.0 ** -24
    assert float((whole.double() - want - b.double()).abs().max()) < bound
    plain = ops.linear(x, w)
    for rows in (1, 15, 16, 17, 32, 33, 64, 65, 256, 257):
        part = x[:rows].contiguous()
        assert torch.equal(ops.linear(part, w, b), whole[:rows]), rows
        got = ops.linear(part, w, partial_ok=True)
        if isinstance(got, ops.PartialSums):
            got = got.sum()
        assert torch.equal(got, plain[:rows]), rows


def test_float32_infinities_stay_in_their_rows_and_columns():
    """What lies past K is not multiplied: an infinite weight or input reaches its own outputs only."""
    from clockwork_amd import ops

    x, w = torch.ones(40, 528, device=DEV), torch.ones(70, 528, device=DEV)
    x[39, 527] = float("inf")
    w[69, 0] = float("inf")
    for rows in (slice(0, 40), slice(30, 40)):
        got = ops.linear(x[rows].contiguous(), w)
        assert bool(torch.isinf(got[-1]).all()) and bool(torch.isinf(got[:, 69]).all())
        assert bool((got[:-1, :69] == 528).all())
